"""GPU parity of the paged causal window kernel (voom_paged_gqa_prefill, through
PagedKVCache.attend_prefill) against fp64 masked softmax attention over the same
bf16 K/V, at the edges of its tiles and splits.

Bar: relative L2 error of the whole output <= 4e-3.  The output is rounded to
bf16 (at most 2^-9 per value, 2^-9 / sqrt(3) = 1.1e-3 in the 2-norm) and so is
every softmax weight before the fp32 sums (the same 1.1e-3, less where many
weights average out); 4e-3 is twice the sum of the two worst cases' halves.
"""
import pytest
import torch

from voom_amd import ops
from voom_amd.kv_paged import PagedKVCache

pytestmark = pytest.mark.gpu

REL = 4e-3


def build(B, NQ, NKV, D, PT, S, L, seed=1, qstd=2.0):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * std).to(torch.bfloat16)

    k, v, q = rnd(B, NKV, S, D), rnd(B, NKV, S, D), rnd(B, NQ, L, D, std=qstd)
    kv = PagedKVCache(1, 1 << 40, page_positions=PT)
    # uneven appends, so that pages land at interleaved slots
    at = 0
    for n in (S // 3, S - S // 3):
        if n:
            kv.append(0, k[:, :, at:at + n], v[:, :, at:at + n])
        at += n
    return kv, q, k, v


def reference(q, k, v, scale):
    B, NQ, L, D = q.shape
    NKV, S = k.shape[1], k.shape[2]
    G = NQ // NKV
    hidden = torch.arange(S, device=q.device)[None, :] > \
        torch.arange(S - L, S, device=q.device)[:, None]
    out = torch.empty((B, NQ, L, D), dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(NQ):
            s = q[b, h].double() @ k[b, h // G].double().t().contiguous() * scale
            w = torch.softmax(s.masked_fill(hidden, -float("inf")), -1)
            out[b, h] = w @ v[b, h // G].double()
    return out


def check(out, ref):
    torch.cuda.synchronize()
    out = out.double()
    assert torch.isfinite(out).all()
    rel = ((out - ref).norm() / ref.norm()).item()
    assert rel <= REL, rel
    # no single row far off (a wrong row hides in the norm of a large output)
    row = ((out - ref).norm(dim=-1) / ref.norm(dim=-1).clamp(min=1e-3)).max().item()
    assert row <= 5 * REL, row


@pytest.mark.parametrize("B,NQ,NKV,D,PT,S,L", [
    (1, 9, 3, 64, 64, 2, 2),          # the smallest window
    (1, 4, 4, 64, 32, 65, 64),        # one head per group; one key past a tile; 32-token pages
    (2, 9, 3, 64, 64, 130, 129),      # rows that straddle wavefronts, batch
    (1, 28, 4, 128, 64, 63, 63),      # a group that does not divide 32; under one tile
    (1, 16, 1, 128, 32, 300, 37),     # the largest group
    (1, 32, 8, 128, 256, 1025, 5),    # a verify window: split over keys
    (1, 8, 1, 128, 64, 9000, 2),      # many splits, more than 64 pages
    (3, 32, 8, 128, 64, 700, 350),
    (1, 64, 8, 128, 64, 2500, 1100),  # full-width workgroups
    (1, 9, 3, 64, 4096, 5000, 200),   # the largest page
])
def test_window_against_fp64(B, NQ, NKV, D, PT, S, L):
    print(f"[prefill] B={B} NQ={NQ} NKV={NKV} D={D} PT={PT} S={S} L={L}", flush=True)
    kv, q, k, v = build(B, NQ, NKV, D, PT, S, L)
    check(kv.attend_prefill(0, q), reference(q, k, v, D ** -0.5))


@pytest.mark.parametrize("scale", [-0.1, 0.0, 1.5])
def test_scales(scale):
    print(f"[prefill] scale={scale}", flush=True)
    kv, q, k, v = build(1, 8, 2, 128, 64, 500, 90, seed=2)
    check(kv.attend_prefill(0, q, scale=scale), reference(q, k, v, scale))


@pytest.mark.parametrize("L,first,count", [(3, 64, 2900), (3, 2048, 700), (40, 512, 1600),
                                           (700, 0, 200)])
def test_keys_pushed_to_minus_infinity(L, first, count):
    """Whole tiles of visible keys that score -inf weigh nothing, at the start of the
    window and of a key split (3 queries: every fourth tile begins one) too."""
    print(f"[prefill] -inf keys {first} + {count}, window {L}", flush=True)
    S, D = 3000, 128
    kv, q, k, v = build(1, 8, 2, D, 64, S, L)
    k[:, :, first:first + count] = 0
    k[:, :, first:first + count, 5] = torch.finfo(torch.bfloat16).min
    q[..., 5] = 4.0  # 4 times the lowest value is past fp32's range
    kv = PagedKVCache(1, 1 << 40, page_positions=64)
    kv.append(0, k, v)
    k64 = k.double()
    k64[:, :, first:first + count, 5] = -float("inf")
    check(kv.attend_prefill(0, q, scale=0.1), reference(q, k64, v, 0.1))


def test_a_scale_of_zero_keeps_nan():
    """0 times an infinite or NaN query (or key) is NaN, as in the decode kernel;
    other rows average the values they see."""
    print("[prefill] scale 0, NaN in q and k", flush=True)
    kv, q, k, v = build(1, 8, 2, 64, 64, 300, 40)
    want = reference(q, k, v, 0.0)
    q[0, 3, 7, 5], q[0, 6, 39, 63] = float("nan"), float("inf")
    out = kv.attend_prefill(0, q, scale=0.0)
    torch.cuda.synchronize()
    hit = torch.zeros(out.shape[:3], dtype=torch.bool, device="cuda")
    hit[0, 3, 7] = hit[0, 6, 39] = True
    assert torch.isnan(out[hit]).all()
    check(out.masked_fill(hit[..., None], 0.0), want.masked_fill(hit[..., None], 0.0))


def test_rising_scores_move_the_reference_maximum():
    """Keys whose scores grow along the sequence: every tile's maximum is far
    above the last one's."""
    print("[prefill] rising scores", flush=True)
    kv, q, k, v = build(1, 8, 2, 128, 64, 600, 70, seed=3)
    ramp = (1 + torch.arange(600, device="cuda") / 20).view(1, 1, 600, 1)
    k2 = (k.abs() * ramp).to(torch.bfloat16)
    q2 = q.abs()
    kv2 = PagedKVCache(1, 1 << 40, page_positions=64)
    kv2.append(0, k2, v)
    check(kv2.attend_prefill(0, q2), reference(q2, k2, v, 128 ** -0.5))


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_values_behind_the_mask_do_not_leak(bad):
    """NaN and infinities in tokens that a query does not see, and in pool rows
    past the sequence, leave its output alone; queries that see them do not
    stay finite."""
    print(f"[prefill] {bad} behind the mask", flush=True)
    S, L, at = 200, 150, 100
    kv, q, k, v = build(1, 8, 2, 128, 64, S, L, seed=4)
    ref = kv.attend_prefill(0, q).clone()
    k2, v2 = k.clone(), v.clone()
    k2[:, :, at] = bad
    v2[:, :, at] = bad
    kv2 = PagedKVCache(1, 1 << 40, page_positions=64, initial_slots=8)
    kv2._init_geometry(k2)
    pool = kv2._pool(0)
    pool.k.fill_(bad)
    pool.v.fill_(bad)
    kv2.append(0, k2, v2)
    out = kv2.attend_prefill(0, q)
    torch.cuda.synchronize()
    first = at - (S - L)  # the first query that sees the token
    assert torch.equal(out[:, :, :first], ref[:, :, :first])
    assert not torch.isfinite(out[:, :, first:]).any(dim=-1).any()


def test_strides_offsets_and_part_of_the_batch():
    """Queries in another memory order, at an odd offset, and for the first
    sequences only give what the plain call gives."""
    print("[prefill] query layouts", flush=True)
    kv, q, _, _ = build(3, 8, 2, 64, 64, 210, 33, seed=5)
    ref = kv.attend_prefill(0, q)
    swapped = q.transpose(1, 2).contiguous().transpose(1, 2)
    odd = torch.empty(q.numel() + 1, dtype=q.dtype, device="cuda")[1:].view(q.shape).copy_(q)
    assert odd.data_ptr() % 16
    for other in (swapped, odd):
        assert torch.equal(kv.attend_prefill(0, other), ref)
    assert torch.equal(kv.attend_prefill(0, q[:2]), ref[:2])
    assert kv.attend_prefill(0, q[:, :, :0]).shape == (3, 8, 0, 64)


def test_one_token_is_the_decode_call_bitwise():
    print("[prefill] one token", flush=True)
    kv, q, _, _ = build(2, 32, 8, 128, 64, 1500, 1, seed=6)
    assert torch.equal(kv.attend_prefill(0, q), kv.attend(0, q))


def test_refusals():
    kv, q, _, _ = build(1, 8, 2, 64, 64, 100, 8, seed=7)
    for bad in (q.float(), q[..., :32], q.expand(2, 8, 8, 64)):
        with pytest.raises(ValueError):
            kv.attend_prefill(0, bad)
    wide = torch.zeros((1, 2 * 17, 8, 64), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError):
        kv.attend_prefill(0, wide)
    small, q2, _, _ = build(1, 8, 2, 64, 16, 100, 8, seed=8)
    with pytest.raises(ValueError):
        small.attend_prefill(0, q2)
    with pytest.raises(ValueError):
        ops.paged_gqa_prefill(q, kv._pool(0).k, kv._pool(0).v, kv._tables[0], 4)
