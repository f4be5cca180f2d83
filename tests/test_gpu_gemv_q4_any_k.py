"""Q4_K Q8-inline GEMV for long rows of any K on few rows: K split over the waves
of a workgroup, with the bits of the one-row-per-step kernel."""
import pytest
import torch

from rocmforge_amd import synth

from . import gpu_util as G

pytestmark = pytest.mark.gpu

# The same rows as part of a matrix that fills the other kernel's row slots (two
# rows for each of four waves a CU): a row's bits depend on neither N nor the grid.
# K: three slices, the last with one super-block, 11 of 16, 16 less one; five; the
# largest (eight, the last half full).  N: one row, an odd few, more than one a CU.
@pytest.mark.parametrize("k", [8448, 11008, 12032, 18944, 30720])
@pytest.mark.parametrize("n", [1, 37, 300, 1537])
def test_bits_of_the_row_step_kernel(rf, dev, n, k):
    full = 8 * torch.cuda.get_device_properties(0).multi_processor_count
    assert n <= 7 * full // 8
    w = synth.weights("q4_k", full, k, seed=k)
    x = synth.activations(k, seed=n)
    res = synth.activations(full, seed=k + 1)
    dw, dx, dr = G.to_dev(w), G.to_dev(x), G.to_dev(res)
    ref, got = G.empty(full, torch.float32), G.empty(n + 1, torch.float32)
    for residual in (False, True):
        got.fill_(-7.0)
        if residual:
            f = rf.gemv_q4_k_f32_q8_inline_residual_launch
            G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(dr), G.ptr(ref), k, full)
            G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(dr), G.ptr(got), k, n)
        else:
            f = rf.gemv_q4_k_f32_q8_inline_launch
            G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(ref), k, full)
            G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(got), k, n)
        assert torch.equal(got[:n], ref[:n])
        assert got[n].item() == -7.0
    # in place: output may alias the residual
    inout = dr[:n].clone()
    G.call(rf.gemv_q4_k_f32_q8_inline_residual_launch, G.ptr(dw), G.ptr(dx), G.ptr(inout), G.ptr(inout), k, n)
    assert torch.equal(inout, got[:n])


# the fullest the kernel takes (256 CUs: 2048 rows a step of the other kernel), by
# steps and slices of K, against the same rows of a matrix that fills the steps
@pytest.mark.parametrize("n,k", [(1536, 8448), (3072, 11008), (1536, 13824), (3584, 18944), (5120, 13824)])
def test_at_the_lines(rf, dev, n, k):
    step = 8 * torch.cuda.get_device_properties(0).multi_processor_count
    full = -(-n // step) * step
    part = synth.weights("q4_k", 512, k, seed=k).reshape(512, -1)
    w, x = part.repeat(-(-full // 512), axis=0)[:full].reshape(-1), synth.activations(k, seed=n)
    dw, dx = G.to_dev(w), G.to_dev(x)
    ref, got = G.empty(full, torch.float32), G.empty(n, torch.float32)
    f = rf.gemv_q4_k_f32_q8_inline_launch
    G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(ref), k, full)
    G.call(f, G.ptr(dw), G.ptr(dx), G.ptr(got), k, n)
    assert torch.equal(got, ref[:n])
