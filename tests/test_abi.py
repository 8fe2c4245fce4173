"""CPU (-m "not gpu"): the C-ABI library builds, loads without a GPU, exports every symbol include/*.h declares, and its
compute entry points fail loudly (no CPU fallback) when no MI355X is visible."""
import ctypes as C
import os

import pytest

from pipeinfer_amd import lib as L


def test_library_loads_and_exports_every_declared_symbol():
    lib = L.load()
    names = L.declared_symbols()
    assert len(names) >= 25
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_no_gpu_means_loud_failure():
    lib = L.load()
    if lib.pi_device_count() > 0:
        pytest.skip("a GPU is visible")
    assert lib.pi_device_init(0) != 0
    assert b"no HIP device" in lib.pi_last_error()


def test_product_never_touches_the_oracle():
    """the oracle is test infrastructure: nothing under pipeinfer_amd/ may reference it"""
    root = os.path.dirname(os.path.abspath(L.__file__))
    for dp, _, files in os.walk(root):
        if "build" in dp.split(os.sep):
            continue
        for f in files:
            if f.endswith((".py", ".cpp", ".hip", ".h", "Makefile")):
                text = open(os.path.join(dp, f), errors="ignore").read()
                assert "liboracle" not in text and "oracle/" not in text and "oracle_lib" not in text, os.path.join(dp, f)


@pytest.mark.parametrize("call,why", [
    (lambda lib, p: lib.pi_op_topk_merge(p, 1, 9, p, p, p, None), b"k=9 > 8"),
    (lambda lib, p: lib.pi_op_topk_merge(p, 1, -1, p, p, p, None), b"k=-1 < 0"),
    (lambda lib, p: lib.pi_op_topk_merge(None, 1, 8, p, p, p, None), b"scratch is NULL"),
    (lambda lib, p: lib.pi_op_topk_parts(p, 100, 1, 9, p, None), b"k=9 > 8"),
    (lambda lib, p: lib.pi_op_topk(p, 100, 1, -1, p, p, p, p, None), b"k=-1 < 0"),
    (lambda lib, p: lib.pi_op_topk_out(None, 0, 1, p, p, p, p, p, 4, None), b"scratch is NULL"),
    (lambda lib, p: lib.pi_op_topk_out(p, 0, 1, p, None, p, p, p, 4, None), b"are NULL"),
    (lambda lib, p: lib.pi_op_topk_out(p, 0, 0, None, None, None, p, None, 4, None), b"are NULL"),
    (lambda lib, p: lib.pi_op_topk_out(p, -1, 1, p, p, p, p, p, 4, None), b"rows [-1, + 1)"),
])
def test_both_halves_of_the_top_k_refuse_what_the_whole_refuses(call, why):
    """more bests than a row's share of the scratch holds, no scratch, no place for the results: an error ahead of any launch (the addresses are never used)"""
    lib = L.load()
    assert call(lib, 4096) != 0 and why in lib.pi_last_error()
