"""Host checks of the judges' entry points (no GPU)."""
import ctypes

from sparseattnfunctions_amd import _lib


def test_arguments_are_checked():
    lib = _lib.load()
    p, st = 1 << 20, _lib.i64(64, 64, 64)
    assert lib.sa_topk_mass(None, p, 2, 5, 32, 100, 128, 0.125, 20, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p + 2, p, 2, 5, 32, 100, 128, 0.125, 20, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p, p, 2, 33, 32, 100, 128, 0.125, 20, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p, p, 2, 5, 32, 100, 96, 0.125, 20, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p, p, 2, 5, 32, 100, 128, 0.125, 0, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p, p, 2, 5, 32, 100, 128, 0.125, 101, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_topk_mass(p, p, 2, 5, 32, 16385, 16416, 0.125, 20, p, None) == _lib.SA_ERR_UNSUPPORTED
    assert lib.sa_gather_key_operands(p, st, 1, 2, 50, 64, p, 33, p, None) == _lib.SA_ERR_INVALID
    assert lib.sa_gather_key_operands(p, st, 1, 2, 50, 128, p, 32, p, None) == _lib.SA_ERR_UNSUPPORTED
    assert lib.sa_gather_key_operands(p, _lib.i64(64, 64, 4), 1, 2, 50, 64, p, 32, p, None) == _lib.SA_ERR_UNSUPPORTED
    n = ctypes.c_int64(0)
    assert lib.sa_pattern_sim_gram_workspace(3, 11, 17, ctypes.byref(n)) == _lib.SA_OK
    assert n.value == 3 * 3 * 11 * 24 * 32 * 4  # heads x chunks x frames x products x (8 positions x 4)
    assert lib.sa_pattern_sim_gram_workspace(3, 13, 17, ctypes.byref(n)) == _lib.SA_ERR_INVALID

    def gram(ws, nbytes):
        return lib.sa_pattern_sim_gram_ws(p, p, 3, 11, 17, 4, 192, 192, 0.125, 0.0, p, ws, nbytes, None)

    assert gram(None, n.value) == _lib.SA_ERR_INVALID
    assert gram(p + 4, n.value) == _lib.SA_ERR_INVALID
    assert gram(p, n.value - 1) == _lib.SA_ERR_INVALID
