"""The sixteen-wave 64-row Q4_K tiles at the edges of their range."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from rocmforge_amd import synth

from . import gpu_util as G

pytestmark = pytest.mark.gpu


# one super-block (every prefetched stage clamped), two, three, five; one column
# tile and several; unsplit and split over K (4096 x 2048); two and four row tiles
@pytest.mark.parametrize("m,n,k", [(64, 64, 256), (64, 192, 512), (64, 64, 768), (128, 128, 1280), (256, 64, 256),
                                   (64, 64, 2048)])
def test_every_weight_bit_for_bit(rf, dev, m, n, k):
    # rows of A are unit vectors, so outputs are single dequantised weights
    w = synth.weights("q4_k", n, k, seed=n + k)
    deq = O.dequant_f16("q4_k", w, n, k).astype(np.float32)
    dw, d = G.to_dev(w), G.empty(m * n, torch.float32)
    for k0 in range(0, k, m):
        rows = min(m, k - k0)
        a = np.zeros((m, k), np.float16)
        a[np.arange(rows), k0 + np.arange(rows)] = 1.0
        G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(G.to_dev(a.view(np.int16))), G.ptr(dw), G.ptr(d), m, n, k)
        np.testing.assert_array_equal(G.host(d).reshape(m, n)[:rows], deq[:, k0:k0 + rows].T)


@pytest.mark.parametrize("m,n,k", [(64, 8448, 3072), (64, 1024, 4096), (192, 640, 1792), (64, 64, 256)])
def test_store_accumulate_and_swiglu(rf, dev, m, n, k):
    a = synth.activations(k, seed=m + n, m=m)
    w = synth.weights("q4_k", n, k, seed=k)
    rng = np.random.default_rng(k)
    r, g = rng.standard_normal((m, n)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    da, dw, dg = G.to_dev(a.astype(np.float16).view(np.int16)), G.to_dev(w), G.to_dev(g)
    d, acc = G.empty(m * n, torch.float32), G.to_dev(r)
    up, want = G.empty(m * n, torch.int16), G.empty(m * n, torch.int16)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(d), m, n, k)
    G.call(rf.rf_gemm_q4_k_f16_accumulate_launch, G.ptr(da), G.ptr(dw), G.ptr(acc), m, n, k)
    G.call(rf.rf_gemm_q4_k_f16_swiglu_up_launch, G.ptr(da), G.ptr(dw), G.ptr(dg), G.ptr(up), m, n, k)
    G.call(rf.rf_silu_mul_f16_on_stream, G.ptr(dg), G.ptr(d), G.ptr(want), m * n)
    got = G.host(d).reshape(m, n)
    np.testing.assert_array_equal(G.host(acc), r + got)
    np.testing.assert_array_equal(G.host(up), G.host(want))
    ref = O.gemm("q4_k", a, w, m, n, k)
    tol = 2e-3 * np.abs(ref) + 2e-5 * O.gemm_abs("q4_k", a, w, m, n, k)     # the GEMM bar
    assert (np.abs(got - ref) <= tol).all()


# Short ranges of a K split stay on eight waves with four K slices, as the segment
# launcher's tiles take them: its products of the ranges, added in order, have the
# same bits (these few tiles are split into one to three super-blocks; 128 tiles, with
# 256 CUs, in two of five)
@pytest.mark.parametrize("m,n,k,split", [(64, 64, 512, 2), (64, 192, 768, 3), (128, 64, 1024, 4), (64, 128, 4096, 8),
                                         (64, 64, 6144, 8), (2048, 256, 2560, 2)])
def test_short_k_ranges_on_eight_waves(rf, dev, m, n, k, split):
    if m > 1024 and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("split for 256 CUs")
    a = synth.activations(k, seed=m + n, m=m).astype(np.float16)
    w = synth.weights("q4_k", n, k, seed=k).reshape(n, k // 256, -1)
    z = None
    want, part = None, G.empty(m * n, torch.float32)
    for s in range(split):
        ks = slice(s * k // split, (s + 1) * k // split)
        da = G.to_dev(np.ascontiguousarray(a[:, ks]).view(np.int16))
        dw = G.to_dev(np.ascontiguousarray(w[:, ks.start // 256:ks.stop // 256]))
        G.call(rf.rf_gemm_qk_f16_segments_launch, G.ptr(da), G.ptr(dw), z, z, 12, 12, 12, G.ptr(part), z, z, m, n, 0,
               0, k // split)
        got = G.host(part).reshape(m, n)
        want = got if want is None else want + got
    d = G.empty(m * n, torch.float32)
    da, dw = G.to_dev(a.view(np.int16)), G.to_dev(w.reshape(-1))
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(d), m, n, k)
    np.testing.assert_array_equal(G.host(d).reshape(m, n), want)


# and from four super-blocks a workgroup on sixteen, with eight K slices: 64 rows of a
# product have the bits of one too few tiles wide to be split otherwise
@pytest.mark.parametrize("k", [8192, 8448])
def test_longer_k_ranges_keep_their_bits(rf, dev, k):
    a = synth.activations(k, seed=k, m=64).astype(np.float16)
    w = synth.weights("q4_k", 128, k, seed=k + 1)
    da, dw = G.to_dev(a.view(np.int16)), G.to_dev(w)
    wide, narrow = G.empty(64 * 128, torch.float32), G.empty(64 * 64, torch.float32)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(wide), 64, 128, k)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(narrow), 64, 64, k)
    got, ref = G.host(wide).reshape(64, 128), O.gemm("q4_k", a.astype(np.float32), w, 64, 128, k)
    np.testing.assert_array_equal(got[:, :64], G.host(narrow).reshape(64, 64))
    tol = 2e-3 * np.abs(ref) + 2e-5 * O.gemm_abs("q4_k", a.astype(np.float32), w, 64, 128, k)
    assert (np.abs(got - ref) <= tol).all()
