"""Host checks of the split-operand fp32 entry points (no GPU)."""
import ctypes

import pytest

from sparseattnfunctions_amd import _lib


@pytest.mark.parametrize("D", [64, 128])
def test_workspace_is_checked(D):
    lib = _lib.load()
    n = ctypes.c_int64(0)
    assert lib.sa_block_sparse_fwd_f32_terms_workspace(2, 3, 321, D, ctypes.byref(n)) == _lib.SA_OK
    assert n.value == 2 * 3 * 6 * (768 * D + 16)  # 12 D bytes per key of a 64-key block, and its flags
    assert lib.sa_block_sparse_fwd_f32_terms_workspace(2, 3, 321, 96, ctypes.byref(n)) == _lib.SA_ERR_UNSUPPORTED
    assert lib.sa_block_sparse_fwd_f32_terms_workspace(0, 3, 321, D, ctypes.byref(n)) == _lib.SA_ERR_INVALID
    assert lib.sa_block_sparse_fwd_f32_terms_workspace(2, 3, 321, D, None) == _lib.SA_ERR_INVALID
    lib.sa_block_sparse_fwd_f32_terms_workspace(2, 3, 321, D, ctypes.byref(n))
    p, st = 1 << 20, _lib.i64(D, D, D)

    def call(ws, nbytes, q=p, d=D, Lk=321):
        return lib.sa_block_sparse_fwd_f32_terms(q, st, p, st, p, st, p, st, 2, 3, 64, Lk, d, p, p, 6, 0.125, None, 0,
                                                 ws, nbytes, None)

    assert call(None, n.value) == _lib.SA_ERR_INVALID
    assert call(p + 16, n.value) == _lib.SA_ERR_INVALID
    assert call(p, n.value - 1) == _lib.SA_ERR_INVALID
    assert call(p, n.value, q=None) == _lib.SA_ERR_INVALID
    assert call(p, n.value, q=p + 4) == _lib.SA_ERR_UNSUPPORTED
    assert call(p, n.value, d=96) == _lib.SA_ERR_UNSUPPORTED
    assert call(p, 1 << 62, Lk=1 << 24) == _lib.SA_ERR_UNSUPPORTED  # past the 32-bit offsets of one head


def test_pooling_workspace_holds_the_split_operands():
    lib = _lib.load()
    n, base = ctypes.c_int64(0), ctypes.c_int64(0)
    assert lib.sa_attn_pooling_workspace(2, 4, 900, 32, ctypes.byref(base)) == _lib.SA_OK
    assert lib.sa_attn_pooling_workspace_f32(2, 4, 2, 900, 64, 32, ctypes.byref(n)) == _lib.SA_OK
    assert base.value % 256 == 0 and n.value == base.value + 2 * 2 * 15 * (768 * 64 + 16)
    assert lib.sa_attn_pooling_workspace_f32(2, 4, 3, 900, 64, 32, ctypes.byref(n)) == _lib.SA_ERR_INVALID
    assert lib.sa_attn_pooling_workspace_f32(2, 4, 2, 900, 96, 32, ctypes.byref(n)) == _lib.SA_ERR_UNSUPPORTED
    assert lib.sa_attn_pooling_workspace_f32(2, 4, 2, 900, 64, 48, ctypes.byref(n)) == _lib.SA_ERR_INVALID
