"""CPU checks of the C-ABI boundary: the library loads and exports every
function include/tncontract_amd.h declares (no compute calls: no GPU here)."""
import ctypes
import os
import re

import pytest

from tests.conftest import ROOT

HEADER = os.path.join(ROOT, "include", "tncontract_amd.h")
LIB = os.path.join(ROOT, "tncontract_amd", "libtncontract_amd.so")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"\b(tn_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_header_declares_entry_points():
    names = declared_functions()
    for n in ["tn_contract", "tn_qr", "tn_svd", "tn_permute", "tn_sumsq", "tn_last_error"]:
        assert n in names


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_library_exports_every_declared_symbol():
    import torch  # noqa: F401  (bind to torch's HIP runtime first)
    lib = ctypes.CDLL(LIB)
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_error_path_without_gpu_calls():
    import torch  # noqa: F401
    from tncontract_amd import _lib as L
    lib = L.lib()
    assert lib.tn_version() >= 1
    # invalid modes are rejected on the host before any device work
    m = L.tn_modes()
    m.nmodes = 99
    rc = lib.tn_permute(None, ctypes.byref(m), None, 0, None)
    assert rc == L.TN_ERR_INVALID
    assert b"modes" in lib.tn_last_error()
    with pytest.raises(ValueError):
        L.check(rc)


def test_merged_modes_reproduce_view_offsets():
    """The fused mode group of a strided view enumerates, in row-major
    order, exactly the element offsets of the view (host logic of the
    permute launches; no GPU call)."""
    import itertools
    import numpy as np
    from tncontract_amd._lib import _merged_modes
    rng = np.random.default_rng(0)
    for trial in range(200):
        nd = int(rng.integers(1, 11))
        shape = [int(x) for x in rng.integers(1, 4, nd)]
        base = np.arange(int(np.prod(shape))).reshape(shape)
        perm = list(rng.permutation(nd))
        view = base.transpose(perm)
        if trial % 3 == 0 and view.ndim and view.shape[0] > 1:
            view = view[1:]
        strides = [s // base.itemsize for s in view.strides]
        dims, st = _merged_modes(view.shape, strides)
        assert all(d > 1 for d in dims)
        off0 = view.reshape(-1)[0] if view.size else 0
        offs = [off0 + sum(i * s for i, s in zip(idx, st))
                for idx in itertools.product(*[range(d) for d in dims])]
        assert offs == list(view.reshape(-1))


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_contract_axes_rejects_bad_groups_on_the_host():
    import torch  # noqa: F401
    from tncontract_amd import _lib as L
    lib = L.lib()
    ok = [1, 1, 1] + [2, 1, 1] * 3
    for bad in ([9, 1, 1] + [2, 1, 1] * 11, [1, -1, 1] + [2, 1, 1] * 3,
                [1, 1, 1, -2, 1, 1] + [2, 1, 1] * 2, ok):  # ok: null operands
        axes = (ctypes.c_int64 * len(bad))(*bad)
        rc = lib.tn_contract_axes(None, None, None, axes, L.TN_F64, 0, 1.0, 0.0, None, 0, None)
        assert rc == L.TN_ERR_INVALID and lib.tn_last_error()


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_contract_workspace_only_for_products_that_split():
    import torch  # noqa: F401
    from tncontract_amd import _lib as L
    need = L.lib().tn_contract_workspace
    # FP64 products of few 32 x 32 tiles take one launch without partial sums
    for m, n, k in [(512, 512, 512), (256, 256, 128), (1024, 1024, 128), (64, 64, 512)]:
        assert need(m, n, k, L.TN_F64) == 0
    # the first sizes past them, long products of few outputs, and FP32 (whose
    # split-bf16 products split) keep theirs
    for m, n, k, dtype in [(512, 512, 513, L.TN_F64), (1024, 544, 512, L.TN_F64),
                           (8, 8, 70000, L.TN_F64), (512, 512, 512, L.TN_F32)]:
        assert need(m, n, k, dtype) > 0
