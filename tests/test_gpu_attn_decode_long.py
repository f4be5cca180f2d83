"""The decode attention's long-sequence form (head_dim 128, past 6144 positions
at 64 splits), at its line and at the ends of chunks, against float64."""
import ctypes
import math

import pytest
import torch

from . import gpu_util as G

pytestmark = pytest.mark.gpu

D = 128


def setup(seq, nh, nkv, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    # exactly seq rows: nothing past the sequence may be read
    return rnd(nh, D), rnd(seq, nkv, D).half(), rnd(seq, nkv, D).half()


def reference(q, k, v):
    group = q.shape[0] // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for h in range(q.shape[0]):
        s = (k[:, h // group].double() @ q[h].double()) / math.sqrt(D)
        out[h] = s.softmax(0) @ v[:, h // group].double()
    return out


def workspace(rf, nh):
    n = int(rf.rf_flash_attn_decode_workspace_bytes(nh, D))
    return torch.full((n // 4 + 1,), math.nan, device="cuda"), n


# the last short length and the first long one; a last chunk of one row, of 31,
# a whole one; groups of 1 (one wave, 16 loads each) to 8; splits of unequal
# chunk counts (S 64, 32)
@pytest.mark.parametrize("seq,nh,nkv", [(6144, 8, 2), (6145, 8, 2), (6177, 2, 2), (6176, 16, 2), (7167, 6, 2),
                                        (8192, 10, 2), (8193, 12, 2), (6500, 14, 2), (9001, 4, 2), (4300, 32, 16),
                                        (20011, 8, 1)])
def test_against_float64(rf, dev, seq, nh, nkv):
    q, k, v = setup(seq, nh, nkv, seq + nh)
    out = G.empty(nh * D, torch.float32)
    st = torch.tensor([seq - 1, seq], dtype=torch.int32, device="cuda")
    ws, n = workspace(rf, nh)
    G.call(rf.rf_flash_attn_decode_state_ws, G.ptr(out), G.ptr(q), G.ptr(k), G.ptr(v),
           ctypes.c_void_p(st.data_ptr() + 4), nh, nkv, D, 1.0 / math.sqrt(D), G.ptr(ws), n)
    ref = reference(q, k, v)
    err = (out.view(nh, D).double() - ref).abs().max().item()
    print(f"seq {seq}: {err / ref.abs().max().item():.2e}")
    assert err <= 1e-5 * ref.abs().max().item()      # the bar of the layer operations


@pytest.mark.parametrize("seq,nh,nkv", [(6145, 8, 2), (6208, 8, 2), (6175, 14, 2), (8224, 8, 1), (600, 8, 2), (640, 16, 2)])
def test_folded_step_gives_the_same(rf, dev, seq, nh, nkv):
    # per-head norm, RoPE and KV write folded in: as the step alone, then the attention
    q, k, v = setup(seq, nh, nkv, seq)
    rk, rv, qn, kn = (torch.randn(s, device="cuda") for s in (nkv * D, nkv * D, D, D))
    k[-1], v[-1] = math.nan, math.nan                # written by the launch, never read before
    k2, v2 = k.clone(), v.clone()
    st = torch.tensor([seq - 1, seq], dtype=torch.int32, device="cuda")
    a, b, q2 = G.empty(nh * D, torch.float32), G.empty(nh * D, torch.float32), q.clone()
    ws, n = workspace(rf, nh)
    scale = 1.0 / math.sqrt(D)
    G.call(rf.rf_attn_decode_qk_norm_rope_state, G.ptr(a), G.ptr(q), G.ptr(rk), G.ptr(rv), G.ptr(qn), G.ptr(kn),
           G.ptr(k), G.ptr(v), G.ptr(st), nh, nkv, D, 1e-6, 1e6, 1, None, None, None, scale, G.ptr(ws), n)
    G.call(rf.rf_qk_norm_rope_kv_write_state, G.ptr(q2), G.ptr(rk), G.ptr(rv), G.ptr(qn), G.ptr(kn), G.ptr(k2),
           G.ptr(v2), G.ptr(st), nh, nkv, D, 1e-6, 1e6, 1, None, None, None)
    G.call(rf.rf_flash_attn_decode_state_ws, G.ptr(b), G.ptr(q2), G.ptr(k2), G.ptr(v2),
           ctypes.c_void_p(st.data_ptr() + 4), nh, nkv, D, scale, G.ptr(ws), n)
    assert torch.equal(k.view(torch.int16), k2.view(torch.int16))
    assert torch.equal(v.view(torch.int16), v2.view(torch.int16))
    assert torch.equal(a, b) and bool(a.isfinite().all())


@pytest.mark.parametrize("shift", [1, 2, 4, 8])      # halves: 2-, 4-, 8- and 16-byte addresses
@pytest.mark.parametrize("seq,nh,nkv", [(6200, 8, 2), (7168, 16, 2), (600, 8, 2)])
def test_caches_off_a_16_byte_address(rf, dev, seq, nh, nkv, shift):
    # any address the cache's type allows, at every length
    q, k, v = setup(seq, nh, nkv, seq + shift)
    kb, vb = (torch.full((k.numel() + 8,), math.nan, dtype=torch.float16, device="cuda") for _ in range(2))
    ks, vs = (b[shift:shift + k.numel()] for b in (kb, vb))
    ks.copy_(k.view(-1))
    vs.copy_(v.view(-1))
    out, st = G.empty(nh * D, torch.float32), torch.tensor([seq - 1, seq], dtype=torch.int32, device="cuda")
    ws, n = workspace(rf, nh)
    scale = 1.0 / math.sqrt(D)
    G.call(rf.rf_flash_attn_decode_state_ws, G.ptr(out), G.ptr(q), G.ptr(ks), G.ptr(vs),
           ctypes.c_void_p(st.data_ptr() + 4), nh, nkv, D, scale, G.ptr(ws), n)
    ref = reference(q, k, v)
    assert (out.view(nh, D).double() - ref).abs().max().item() <= 1e-5 * ref.abs().max().item()
    # the folded step writes the last row: raw q, k and v in, no norm
    rk, rv, out2, q2 = torch.randn(nkv * D, device="cuda"), torch.randn(nkv * D, device="cuda"), out.clone(), q.clone()
    G.call(rf.rf_attn_decode_qk_norm_rope_state, G.ptr(out2), G.ptr(q), G.ptr(rk), G.ptr(rv), None, None, G.ptr(ks),
           G.ptr(vs), G.ptr(st), nh, nkv, D, 1e-6, 1e6, 1, None, None, None, scale, G.ptr(ws), n)
    G.call(rf.rf_qk_norm_rope_kv_write_state, G.ptr(q2), G.ptr(rk), G.ptr(rv), None, None, G.ptr(k), G.ptr(v),
           G.ptr(st), nh, nkv, D, 1e-6, 1e6, 1, None, None, None)
    assert torch.equal(ks, k.view(-1)) and torch.equal(vs, v.view(-1))
    assert bool(kb[:shift].isnan().all()) and bool(kb[shift + k.numel():].isnan().all())
    ref = reference(q2, k, v)
    assert (out2.view(nh, D).double() - ref).abs().max().item() <= 1e-5 * ref.abs().max().item()


@pytest.mark.parametrize("group,seq", [(1, 4096), (2, 1024), (2, 4096), (2, 16384)])
def test_a_grid_just_above_two_workgroups_a_cu(rf, dev, group, seq):
    # the split count is rounded up, so with most KV head counts the grid is a few more
    # than two workgroups a CU: they run beside the others, not in a round of their own
    # (which took 1.4 to 1.6 times as long), so the time follows the work
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    times = []
    for nkv in (cus // 2, cus // 2 + 1):             # 2 and 2 + 4 / CUs workgroups a CU
        nh = nkv * group
        q = torch.randn(nh, D, device="cuda")
        k, v = (torch.randn(seq, nkv, D, device="cuda", dtype=torch.float16) for _ in range(2))
        out, st = G.empty(nh * D, torch.float32), torch.tensor([seq - 1, seq], dtype=torch.int32, device="cuda")
        ws, n = workspace(rf, nh)
        best = math.inf
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                rc = rf.rf_flash_attn_decode_state_ws(
                    G.ptr(out), G.ptr(q), G.ptr(k), G.ptr(v), ctypes.c_void_p(st.data_ptr() + 4), nh, nkv, D,
                    1.0 / math.sqrt(D), G.ptr(ws), n, G.stream())
                assert rc == 0
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    print(f"group {group}, {seq} positions: {times[0] * 100:.1f} us, {times[1] * 100:.1f} us")
    assert times[1] < 1.2 * times[0]
