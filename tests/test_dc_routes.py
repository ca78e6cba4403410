"""Which calls the divide and conquer route accepts (host side, no GPU)."""
import ctypes

import pytest
import torch

import eigeng_batched as eg

# host memory stands for device memory: only where nothing can be launched
pytestmark = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="passes host pointers")
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


@pytest.mark.parametrize("L,n,tb,path", [(10000, 100, 4, 0), (16384, 65, 4, 0), (16384, 128, 4, 0),
                                         (5000, 100, 4, 1 << eg.CHUNK_SHIFT), (16384, 48, 4, 0), (8192, 128, 8, 0)])
def test_phases_are_taken_up_to_the_documented_batch(L, n, tb, path):
    """FP32 n <= 128 up to 16384 matrices (a chunk bit halves that), FP64 beyond 64 up to
    8192; one matrix more is refused."""
    eg.tune_reset()
    top = L if L in (16384, 8192) else (16384 if not path else 8192)
    for ph in PHASES:
        assert not refused(L, n, tb, eg.IMTQL2 | path | ph)
        assert refused(top + 1, n, tb, eg.IMTQL2 | path | ph)


@pytest.mark.parametrize("tb", [4, 8])
def test_launch_params_are_those_of_the_path_without_divide_and_conquer(tb):
    """The same numbers with and without it (bit 28 means nothing to IMTQL2 but keeps a
    call off that path)."""
    eg.tune_reset()
    for L in (1, 100, 257, 600, 1024, 2048, 8192, 16384):
        for n in (5, 8, 20, 32, 48, 64, 65, 100, 128, 129, 192, 200, 256, 257, 300, 512):
            p = eg.launch_params(L, n, tb)
            assert p["rc"] == 0
            assert p == eg.launch_params(L, n, tb, eg.IMTQL2 | (1 << 28)) == eg.launch_params(L, n, tb, eg.FLAG_DC)
