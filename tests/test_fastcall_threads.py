"""Calls through aetherkv._fastcall that must let other Python threads run while they wait.

The module is built here over a stand-in for the library whose functions wait (at most two seconds)
until another Python thread lets them go on, which it can only do without the interpreter lock.
"""
from __future__ import annotations

import ctypes
import importlib.util
import re
import subprocess
import sysconfig
import threading
import time

import pytest

from conftest import PKG_DIR, ROOT

SRC = PKG_DIR / "aetherkv" / "_fastcall.c"
RELEASING = ("aekv_tq_encode", "aekv_tq_decode", "aekv_hca_compress", "aekv_csa_indexer_topk",
             "aekv_csa_prefill_indexer_topk_quant", "aekv_quant_prefill_attention", "aekv_prefill_counts")


@pytest.fixture(scope="module")
def module(tmp_path_factory):
    text = SRC.read_text()
    args = {name: int(n) for n, name in re.findall(r'want_args\(nargs, (\d+), "(aekv_\w+)"\)', text)}
    stub = ["#include <time.h>", "volatile int stub_entered, stub_go;", "static int stub_wait(void) {",
            "  stub_entered = 1;", "  for (int i = 0; i < 2000 && !stub_go; ++i) {",
            "    struct timespec t = {0, 1000000};", "    nanosleep(&t, 0);", "  }", "  return stub_go ? 0 : 1;", "}"]
    stub += [f"int {name}(void) {{ return stub_wait(); }}" for name in args]
    d = tmp_path_factory.mktemp("fastcall")
    (d / "stub.c").write_text("\n".join(stub) + "\n")
    out = d / ("_fastcall" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-Wl,-Bsymbolic", f"-I{sysconfig.get_paths()['include']}",
                    f"-I{ROOT / 'include'}", str(SRC), str(d / "stub.c"), "-o", str(out)], check=True)
    spec = importlib.util.spec_from_file_location("_fastcall", out)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod, ctypes.CDLL(str(out)), args


@pytest.mark.parametrize("name", RELEASING)
def test_other_threads_run_during_the_call(module, name):
    mod, lib, args = module
    entered, go = (ctypes.c_int.in_dll(lib, n) for n in ("stub_entered", "stub_go"))
    entered.value = go.value = 0
    rc = []
    t = threading.Thread(target=lambda: rc.append(getattr(mod, name)(*[0] * args[name])))
    t.start()
    for _ in range(4000):
        if entered.value:
            break
        time.sleep(0.001)
    go.value = 1
    t.join()
    assert rc == [0]
