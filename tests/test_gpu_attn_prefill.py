"""The prefill attention's routes (two, four or eight 32-query units a workgroup,
with and without a key split) at the edges of their ranges, against float64."""
import math

import pytest
import torch

from . import gpu_util as G

pytestmark = pytest.mark.gpu

D = 128
U16 = 2.0 ** -11     # half an ulp of fp16, relative


def reference(q, k, v, causal, scale):
    """(out, sum of p |v|) in float64, [seq][heads][D]."""
    seq, nq, group = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    out, mag = (torch.empty(seq, nq, D, dtype=torch.float64, device=q.device) for _ in range(2))
    mask = torch.ones(seq, seq, dtype=torch.bool, device=q.device).triu(1)
    for h in range(nq):
        s = (q[:, h].double() @ k[:, h // group].double().T) * scale
        if causal:
            s = s.masked_fill(mask, -math.inf)
        p, vh = s.softmax(-1), v[:, h // group].double()
        out[:, h], mag[:, h] = p @ vh, p @ vh.abs()
    return out, mag


def inputs(seq, nq, nkv, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 1000 * seq + nq)
    return [torch.randn(seq, n, D, device="cuda", generator=g).half() for n in (nq, nkv, nkv)]


def run(rf, q, k, v, causal, scale):
    out = torch.empty(q.shape, device="cuda")
    G.call(rf.wmma_attention_prefill_gqa_causal_launch, G.ptr(q), G.ptr(k), G.ptr(v), G.ptr(out), q.shape[0],
           q.shape[1], k.shape[1], causal, scale)
    torch.cuda.synchronize()
    return out.double()


# one tile; remainders of units (heads x blocks) per workgroup; each route's
# ends on 256 CUs: units <= 512, < 4096, beyond; GQA groups 1, 3, 5, 7, 8
@pytest.mark.parametrize("seq,nq,nkv,causal", [(64, 1, 1, 1), (64, 8, 1, 1), (128, 3, 1, 0), (192, 10, 2, 1),
                                               (448, 7, 1, 1), (512, 32, 8, 1), (576, 32, 8, 1), (1088, 15, 5, 1),
                                               (640, 28, 4, 0), (2048, 64, 8, 1), (2112, 63, 9, 1),
                                               (4096, 32, 8, 0)])
def test_routes_against_float64(rf, dev, seq, nq, nkv, causal):
    q, k, v = inputs(seq, nq, nkv)
    scale = 1.0 / math.sqrt(D)
    got = run(rf, q, k, v, causal, scale)
    ref, mag = reference(q, k, v, causal, scale)
    # each weight is rounded to fp16 once; fp32 sums and exp stay well below that
    bound = 1.25 * U16 * mag + 1e-5
    print(f"seq {seq} heads {nq}/{nkv}: largest error {((got - ref).abs() / bound).max().item():.2f} of the bound")
    assert bool(((got - ref).abs() <= bound).all())


@pytest.mark.parametrize("scale", [-0.07, 0.0, 1.0, 3.0])
def test_other_scales(rf, dev, scale):
    q, k, v = inputs(320, 4, 2, seed=5)
    got = run(rf, q, k, v, 1, scale)
    ref, mag = reference(q, k, v, 1, scale)
    # scores reach ~50 scale 1.44: an fp32 rounding of one moves its weight by up to that times 2^-23
    bound = 1.25 * U16 * mag + 1e-4
    assert bool(((got - ref).abs() <= bound).all())


@pytest.mark.parametrize("seq,nq,nkv", [(256, 4, 2), (1088, 32, 8), (4096, 32, 8)])
def test_masked_keys_of_any_value_stay_out(rf, dev, seq, nq, nkv):
    # keys behind a row's own position are masked whatever they hold
    q, k, v = inputs(seq, nq, nkv, seed=7)
    want = run(rf, q, k, v, 1, 0.09)
    k2 = k.clone()
    k2[seq - 20:seq - 10] = math.inf
    k2[seq - 10:] = math.nan
    got = run(rf, q, k2, v, 1, 0.09)
    assert bool((got[:seq - 20] == want[:seq - 20]).all())


def test_maximum_rising_tile_by_tile(rf, dev):
    # every tile's scores lie above the last one's, so O is rescaled on each
    seq, scale = 512, 1.0 / math.sqrt(D)
    q, k, v = inputs(seq, 2, 1, seed=9)
    q = torch.ones_like(q)
    ramp = torch.arange(seq, device="cuda") / 64 * 4.0 / math.sqrt(D)
    k = (ramp.view(seq, 1, 1) + 0.02 * k.float()).half()
    got = run(rf, q, k, v, 1, scale)
    ref, mag = reference(q, k, v, 1, scale)
    assert bool(((got - ref).abs() <= 1.25 * U16 * mag + 1e-5).all())


@pytest.mark.parametrize("seq,nq,nkv", [(64, 2, 1), (2048, 64, 8), (4096, 32, 8)])
def test_a_nan_scale_gives_nan(rf, dev, seq, nq, nkv):
    q, k, v = inputs(seq, nq, nkv, seed=11)
    assert bool(run(rf, q, k, v, 1, math.nan).isnan().all())


@pytest.mark.parametrize("seq,nq,nkv", [(64, 2, 1), (512, 4, 2), (2048, 64, 8), (4096, 32, 8)])
@pytest.mark.parametrize("size", [16.0, 300.0, 8000.0, 60000.0])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_large_scores(rf, dev, seq, nq, nkv, size, sign):
    # scores of up to +-128 size^2 scale (4e10), a multiple of each key's own size
    q, k, v = inputs(seq, nq, nkv, seed=13)
    q = torch.full_like(q, sign * size)
    k = (size * (1 - 0.1 * k[:, :, :1].float().abs())).expand(k.shape).half()
    scale = 1.0 / math.sqrt(D)
    got = run(rf, q, k, v, 1, scale)
    ref, mag = reference(q, k, v, 1, scale)
    # where a row's best score leads by more than the fp32 roundings of a score (the
    # dot of 128 terms, the scale: 2^-15 of it) and by a weight of e^-40, the row is
    # that key's V with a weight of exactly one
    s = (q[:, 0].double() @ k[:, 0].double().T) * scale
    top = s.masked_fill(torch.ones(seq, seq, dtype=torch.bool, device="cuda").triu(1), -math.inf).topk(2, 1).values
    clear = top[:, 0] - top[:, 1] > 40 + 2.0 ** -15 * top[:, 0].abs()
    assert bool(got.isfinite().all()) and int(clear.sum()) > 0
    group = nq // nkv
    bound = 1e-3 * U16 * mag[:, :group] + 1e-6
    assert bool(((got - ref)[:, :group].abs() <= bound)[clear].all())


# both sides of the lines between the routes (256 CUs): causal 768 and 2816 units of 32
# queries, without a mask 512, 1024, 2048 and 3072
@pytest.mark.parametrize("seq,nq,nkv,causal", [(768, 32, 8, 1), (832, 32, 8, 1), (1024, 88, 8, 1), (960, 90, 9, 1),
                                               (512, 32, 8, 0), (576, 32, 8, 0), (1024, 32, 8, 0), (1088, 32, 8, 0),
                                               (2048, 32, 8, 0), (2112, 32, 8, 0), (3136, 32, 8, 0)])
def test_both_sides_of_the_lines(rf, dev, seq, nq, nkv, causal):
    q, k, v = inputs(seq, nq, nkv, seed=17)
    scale = 1.0 / math.sqrt(D)
    got = run(rf, q, k, v, causal, scale)
    ref, mag = reference(q, k, v, causal, scale)
    assert bool(((got - ref).abs() <= 1.25 * U16 * mag + 1e-5).all())      # as above
