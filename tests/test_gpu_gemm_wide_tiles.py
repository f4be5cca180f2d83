"""The 256 x 128 Q4_K tiles from half the CUs on, storing and accumulating."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from rocmforge_amd import synth

from . import gpu_util as G

pytestmark = pytest.mark.gpu


# 256 CUs: 128 tiles (256 x 64 tiles still), 129 and 130 (one row tile and two,
# the second of 64 rows), 192, 257 (a second round); one, two and three super-blocks
@pytest.mark.parametrize("m,n,k", [(256, 16384, 256), (256, 16512, 256), (320, 8320, 512), (512, 12288, 768),
                                   (256, 32896, 256)])
def test_store_and_accumulate(rf, dev, m, n, k):
    a = synth.activations(k, seed=m + n, m=m)
    w = synth.weights("q4_k", n, k, seed=k)
    r = np.random.default_rng(k).standard_normal((m, n)).astype(np.float32)
    da, dw = G.to_dev(a.astype(np.float16).view(np.int16)), G.to_dev(w)
    d, acc = G.empty(m * n, torch.float32), G.to_dev(r)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(d), m, n, k)
    G.call(rf.rf_gemm_q4_k_f16_accumulate_launch, G.ptr(da), G.ptr(dw), G.ptr(acc), m, n, k)
    got = G.host(d).reshape(m, n)
    # both take the same tiles: the old contents plus the product, rounded once
    np.testing.assert_array_equal(G.host(acc), r + got)
    ref = O.gemm("q4_k", a, w, m, n, k)
    tol = 2e-3 * np.abs(ref) + 2e-5 * O.gemm_abs("q4_k", a, w, m, n, k)     # the GEMM bar
    assert (np.abs(got - ref) <= tol).all()


# up to 128 rows a 256-row tile would be half empty or more: whatever the width, the
# tiles of the row count, whose bits a product too narrow for the wide ones shows
# (16448 columns: 257 column tiles of 64, no whole number of 128)
@pytest.mark.parametrize("m,k", [(64, 768), (64, 1536), (128, 512), (128, 1536)])
@pytest.mark.parametrize("n", [16512, 18944, 27648])
def test_few_rows_keep_their_own_tiles(rf, dev, m, n, k):
    a = synth.activations(k, seed=m + n, m=m)
    w = synth.weights("q4_k", n, k, seed=k)
    da, dw = G.to_dev(a.astype(np.float16).view(np.int16)), G.to_dev(w)
    acc = np.random.default_rng(k).standard_normal((m, n)).astype(np.float32)
    wide, narrow, d_acc = G.empty(m * n, torch.float32), G.empty(m * 16448, torch.float32), G.to_dev(acc)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(wide), m, n, k)
    G.call(rf.rf_gemm_q4_k_f16_launch, G.ptr(da), G.ptr(dw), G.ptr(narrow), m, 16448, k)
    G.call(rf.rf_gemm_q4_k_f16_accumulate_launch, G.ptr(da), G.ptr(dw), G.ptr(d_acc), m, n, k)
    got = G.host(wide).reshape(m, n)
    np.testing.assert_array_equal(got[:, :16448], G.host(narrow).reshape(m, 16448))
    np.testing.assert_array_equal(G.host(d_acc).reshape(m, n), acc + got)
