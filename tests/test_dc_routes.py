"""Which calls the divide and conquer route accepts (host side, no GPU)."""
import ctypes

import pytest

import eigeng_batched as eg

PHASES = [0x1000, 0x2000, 0x4000, 0x3000]
INVALID = 1


def refused(L, n, tb, solver):
    """The call returns hipErrorInvalidValue (nothing is launched then)."""
    f = eg.lib().eigen_GPU_batch_FP_x if tb == 4 else eg.lib().eigen_GPU_batch_DP_x
    buf = ctypes.create_string_buffer(4096)
    return f(L, n, n, n, ctypes.addressof(buf), ctypes.addressof(buf), ctypes.addressof(buf), None, solver, None) == INVALID


@pytest.mark.parametrize("ph", PHASES)
@pytest.mark.parametrize("L,n,tb", [(100, 48, 4), (100, 48, 8), (1000, 8, 8), (1000, 12, 4), (100, 20, 4), (100, 64, 8),
                                    (100, 100, 4), (100, 100, 8), (500, 200, 8), (100, 300, 4), (64, 512, 8)])
def test_phases_without_a_path_stay_refused_for_small_batches(L, n, tb, ph):
    """A single phase of a batch that has no QL path in separate kernels, and no path
    bit, was always invalid; so is a phase of the fused kernel with 0x8000000 beside it."""
    eg.tune_reset()
    assert refused(L, n, tb, eg.IMTQL2 | ph)
    assert refused(L, n, tb, eg.IMTQL2 | eg.FLAG_FUSED | ph)
    assert refused(L, n, tb, eg.IMTQL2 | eg.FLAG_FUSED | eg.FLAG_DC | ph)
