"""GPU parity of position-free attention with many (query, head) columns -- the
staged window kernels -- against fp64 attention over keys rotated as the entry
point rotates them, and against the same call made one query at a time.

Bars, relative L2 over the output: fp16 8e-4 (its own rounding is at most 2^-12 /
sqrt(3) = 1.4e-4 per value and the rotated keys carry one fp16 rounding that can
fall the other way than fp64's, 2^-11 of a key now and then; P is as good as in
32 bits), bf16 4e-3 (output and softmax weights rounded to bf16, 1.1e-3 each).
"""
import pytest
import torch

from voom_amd import ops

pytestmark = pytest.mark.gpu

REL = {torch.float16: 8e-4, torch.bfloat16: 4e-3}


def inputs(B, NQ, NKV, TQ, D, BLOCK, TK, dtype, seed, order="window", table_dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    blocks = -(-TK // BLOCK)
    P = max(1, blocks + 3)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)  # noqa: E731
    q = (2 * torch.randn((B, NQ, TQ, D), generator=g, device="cuda")).to(dtype)
    table = torch.randint(0, P, (blocks,), generator=g, device="cuda", dtype=torch.int32)
    kpos = torch.arange(TK, dtype=torch.int32, device="cuda")
    qpos = torch.arange(TK - TQ, TK, dtype=torch.int32, device="cuda").clamp(min=0)
    if order == "scattered":  # selected tokens anywhere, keys in any order
        qpos = torch.randint(0, TK, (TQ,), generator=g, device="cuda", dtype=torch.int32)
        kpos = kpos[torch.randperm(TK, generator=g, device="cuda")]
    elif order == "all":
        qpos = torch.full((TQ,), TK + 7, dtype=torch.int32, device="cuda")
    elif order == "none":
        kpos = kpos + 9
        qpos = torch.full((TQ,), 3, dtype=torch.int32, device="cuda")
    cos, sin = ops.rope_cache(TK + 16, D, 1e4, device="cuda")
    return (q, rnd(P, NKV, BLOCK, D), rnd(P, NKV, BLOCK, D), table, kpos, qpos,
            cos.to(table_dtype), sin.to(table_dtype))


def reference(q, kp, vp, table, kpos, qpos, cos, sin, scale):
    B, NQ, TQ, D = q.shape
    _, NKV, BLOCK, _ = kp.shape
    TK, half = kpos.numel(), D // 2
    k = kp[table.long()].permute(1, 0, 2, 3).reshape(NKV, -1, D)[:, :TK].double()
    v = vp[table.long()].permute(1, 0, 2, 3).reshape(NKV, -1, D)[:, :TK].double()
    c, s = cos[kpos.long()].double(), sin[kpos.long()].double()
    a, b = k[..., :half], k[..., half:]
    k = torch.cat([a * c - b * s, b * c + a * s], -1).to(q.dtype).double()
    hidden = kpos[None, :] > qpos[:, None]
    G = NQ // NKV
    out = torch.empty((B, NQ, TQ, D), dtype=torch.float64, device=q.device)
    for h in range(NQ):
        for b in range(B):
            x = (q[b, h].double() @ k[h // G].t().contiguous() * scale).masked_fill(
                hidden, -float("inf"))
            w = torch.softmax(x, -1).nan_to_num(0.0)  # no visible key: zeros
            out[b, h] = w @ v[h // G]
    return out


def check(got, ref, dtype):
    torch.cuda.synchronize()
    assert got.dtype == dtype and torch.isfinite(got).all()
    rel = ((got.double() - ref).norm() / ref.norm().clamp(min=1e-30)).item()
    assert rel <= REL[dtype], rel
    row = ((got.double() - ref).norm(dim=-1) / ref.norm(dim=-1).clamp(min=1e-2)).max().item()
    assert row <= 6 * REL[dtype], row


def staged_from(B, NQ, NKV, D, TK):
    """The fewest queries that take the staged route (kStageRules in
    position_free.hip)."""
    hw = next(h for h in (8, 4, 2, 1) if NKV % h == 0)
    least, extra = {(64, 1): (48, 140), (64, 2): (110, 300), (64, 4): (72, 70), (64, 8): (65, 60),
                    (128, 1): (48, 110), (128, 2): (65, 110), (128, 4): (56, 110),
                    (128, 8): (56, 17)}[D, hw]
    elems = TK * NKV * D
    least += min(elems >> 19, 16) if (D, hw) == (128, 8) else 0
    cols = least + -(-(extra << 19) // elems)
    return -(-cols // (B * (NQ // NKV)))


def test_staged_from_is_the_rule():
    """The workspace tells the routes apart: partials of many splits against the
    staged pages."""
    for B, NQ, NKV, D, TK in ((1, 28, 4, 128, 3000), (1, 32, 8, 128, 700), (1, 8, 8, 128, 9000),
                              (2, 9, 3, 64, 5000),
                              (1, 4, 2, 64, 8000), (1, 16, 2, 128, 900), (1, 8, 8, 64, 2000),
                              (1, 12, 12, 64, 1500), (1, 7, 1, 128, 20000)):
        TQ = staged_from(B, NQ, NKV, D, TK)
        need = [ops.position_free_workspace_bytes(B, NQ, n, NKV, D, TK, num_splits=1)
                for n in (TQ - 1, TQ)]
        staged = 4 * -(-TK // 64) * 64 * NKV * D
        assert need[0] < staged <= need[1], (need, staged)
        assert ops._may_stage_pages(B * (NQ // NKV) * TQ, TK * NKV * D)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,NQ,NKV,D,BLOCK,TK,order", [
    (1, 28, 4, 128, 1, 10, "scattered"),   # one partial block, very many rows
    (1, 32, 8, 128, 1, 63, "scattered"),   # one key short of a tile
    (1, 9, 3, 64, 16, 65, "window"),       # one key over; D = 64
    (2, 16, 1, 128, 4, 700, "window"),     # batch rows share the staged keys
    (1, 28, 4, 128, 1, 2100, "window"),    # key splits, a group that does not divide 32
    (1, 9, 3, 64, 1, 4500, "scattered"),   # more than 64 tiles, any order
    (1, 32, 8, 128, 16, 1000, "scattered"),
    (1, 8, 8, 64, 1, 300, "all"),          # no diagonal
    (1, 28, 4, 128, 8, 200, "none"),       # nothing visible: zeros
])
def test_windows_against_fp64(dtype, B, NQ, NKV, D, BLOCK, TK, order):
    """At the fewest columns that are staged, and one query below (the
    page-walking kernel)."""
    most = staged_from(B, NQ, NKV, D, TK)
    for TQ in (most, most - 1):
        print(f"[pf-window] {dtype} B={B} NQ={NQ} NKV={NKV} TQ={TQ} D={D} BLOCK={BLOCK} TK={TK} "
              f"{order}", flush=True)
        args = inputs(B, NQ, NKV, TQ, D, BLOCK, TK, dtype, seed=TK, order=order)
        out = ops.position_free_paged_attention(*args, scale=D ** -0.5)
        if order == "none":
            torch.cuda.synchronize()
            assert torch.all(out == 0)
        else:
            check(out, reference(*args, D ** -0.5), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_windows_equal_one_query_at_a_time(dtype):
    """The staged route against the page-walking one, over block sizes, table
    types, split counts and scales."""
    TQ = staged_from(1, 28, 4, 128, 500)
    for BLOCK, tdt, splits, scale in [(1, torch.float32, 0, 0.1), (4, dtype, 1, -0.09),
                                      (64, torch.float32, 7, 0.0), (1, dtype, 200, 0.2)]:
        print(f"[pf-window] routes {dtype} BLOCK={BLOCK} tables={tdt} splits={splits} scale={scale}",
              flush=True)
        q, kp, vp, table, kpos, qpos, cos, sin = inputs(1, 28, 4, TQ, 128, BLOCK, 500, dtype, seed=5,
                                                        order="scattered", table_dtype=tdt)
        out = ops.position_free_paged_attention(q, kp, vp, table, kpos, qpos, cos, sin, scale=scale,
                                                num_splits=splits)
        each = torch.cat([ops.position_free_paged_attention(
            q[:, :, i:i + 1].contiguous(), kp, vp, table, kpos, qpos[i:i + 1], cos, sin, scale=scale)
            for i in range(TQ)], 2)
        torch.cuda.synchronize()
        rel = ((out.double() - each.double()).norm() / each.double().norm()).item()
        assert rel <= 2 * REL[dtype], (BLOCK, splits, scale, rel)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_nan_keys_stay_nan(dtype):
    """Visible keys of NaN that fill whole splits (which then have no maximum) give
    NaN in either route, and only for the heads that read them."""
    print(f"[pf-window] NaN in K, {dtype}", flush=True)
    for TQ, splits in ((3, 0), (3, 1), (3, 5), (staged_from(1, 8, 2, 64, 800), 0)):
        args = list(inputs(1, 8, 2, TQ, 64, 1, 800, dtype, seed=3))
        args[3] = torch.arange(800, dtype=torch.int32, device="cuda")
        args[1][:300, 1] = float("nan")
        out = ops.position_free_paged_attention(*args, scale=0.1, num_splits=splits)
        torch.cuda.synchronize()
        assert torch.isnan(out[0, 4:]).all() and torch.isfinite(out[0, :4]).all(), (TQ, splits)


def test_weak_keys_keep_their_weight_in_fp16():
    """Weights far below fp16's normal range (2^-14 of the largest) still count:
    one key ahead of 4,000 others whose weights are 2^-16 of its own and whose
    values all point one way."""
    print("[pf-window] weak keys", flush=True)
    TK, D = 4000, 128
    for TQ in (1, staged_from(1, 2, 1, D, TK)):
        q = torch.zeros((1, 2, TQ, D), dtype=torch.float16, device="cuda")
        q[..., D // 2 - 1] = 1.0  # the slowest pair: hardly rotated
        kp = torch.zeros((TK, 1, 1, D), dtype=torch.float16, device="cuda")
        kp[0, 0, 0, D // 2 - 1] = 11.09  # 16 ln 2
        vp = torch.ones((TK, 1, 1, D), dtype=torch.float16, device="cuda")
        vp[0] = 0
        table = torch.arange(TK, dtype=torch.int32, device="cuda")
        qpos = torch.full((TQ,), TK, dtype=torch.int32, device="cuda")
        cos, sin = ops.rope_cache(TK + 1, D, 1e4, device="cuda")
        args = (q, kp, vp, table, table, qpos, cos, sin)
        out = ops.position_free_paged_attention(*args, scale=1.0)
        check(out, reference(*args, 1.0), torch.float16)


def slow_pair(dtype, TK, TQ, scores, values):
    """One kv head of 128 dims with two query heads.  The queries hold 1 in the
    slowest rotary pair, so that a key with s in its first dim scores s (its
    rotation is small); ``scores`` and ``values`` [TK, 128] fill K and V."""
    D = 128
    q = torch.zeros((1, 2, TQ, D), dtype=dtype, device="cuda")
    q[..., D // 2 - 1] = 1.0
    q[..., D - 1] = 2.0 ** -14  # the partner dim, so that infinities there keep their sign
    kp = torch.zeros((TK, 1, 1, D), dtype=dtype, device="cuda")
    kp[:, 0, 0, D // 2 - 1] = torch.as_tensor(scores, device="cuda").to(dtype)
    vp = values.to(dtype).reshape(TK, 1, 1, D)
    table = torch.arange(TK, dtype=torch.int32, device="cuda")
    qpos = torch.full((TQ,), TK + 1, dtype=torch.int32, device="cuda")
    cos, sin = ops.rope_cache(TK + 2, D, 1e4, device="cuda")
    return q, kp, vp, table, table + 1, qpos, cos, sin


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("first,count,splits", [(0, 200, 1), (0, 64, 0), (1000, 700, 3)])
def test_keys_pushed_to_minus_infinity(dtype, first, count, splits):
    """Whole tiles of visible keys that score -inf, at the start of a split too,
    weigh nothing."""
    print(f"[pf-window] -inf keys {dtype} {first} + {count}, splits={splits}", flush=True)
    TK = 2000
    g = torch.Generator(device="cuda").manual_seed(4)
    scores = torch.randn(TK, generator=g, device="cuda")
    scores[first:first + count] = -float("inf")
    args = slow_pair(dtype, TK, staged_from(1, 2, 1, 128, TK), scores,
                     torch.randn((TK, 128), generator=g, device="cuda"))
    out = ops.position_free_paged_attention(*args, scale=1.0, num_splits=splits)
    check(out, reference(*args, 1.0), dtype)


@pytest.mark.parametrize("wide", [False, True])
def test_infinite_values_in_fp16(wide):
    """An infinite V under a positive weight of any size gives that infinity
    (weights with an exact fp16 value, and far below fp16's range, among them),
    infinities of both signs and NaN give NaN, and the other dims keep their
    values."""
    TK, inf = 4000, float("inf")
    TQ = staged_from(1, 2, 1, 128, TK) if wide else 1
    print(f"[pf-window] infinite values, {TQ} queries", flush=True)
    g = torch.Generator(device="cuda").manual_seed(6)
    scores = torch.zeros(TK)  # equal scores: every weight is exactly 1
    scores[40] = -60.0        # e^-60
    values = torch.randn((TK, 128), generator=g, device="cuda")
    plain = values.clone()
    for key, dim, v in ((7, 3, inf), (100, 4, -inf), (3999, 5, inf), (40, 6, inf), (900, 7, -inf),
                        (901, 7, -inf), (5, 8, inf), (3000, 8, -inf), (64, 9, float("nan"))):
        values[key, dim] = v
    args = slow_pair(torch.float16, TK, TQ, scores, values)
    out = ops.position_free_paged_attention(*args, scale=1.0)
    ref = reference(*slow_pair(torch.float16, TK, TQ, scores, plain), 1.0)
    torch.cuda.synchronize()
    for dim, v in ((3, inf), (4, -inf), (5, inf), (6, inf), (7, -inf)):
        assert torch.all(out[..., dim] == v), dim
    assert torch.isnan(out[..., 8:10]).all()
    rest = [d for d in range(128) if not 3 <= d <= 9]
    check(out[..., rest], ref[..., rest], torch.float16)


@pytest.mark.parametrize("NQ,NKV,D,TK", [(28, 4, 128, 700), (16, 8, 64, 1500), (6, 2, 128, 900),
                                         (8, 8, 128, 333)])
def test_infinite_values_of_one_head(NQ, NKV, D, TK):
    """Infinities in single kv heads: every query that sees the key, nothing else;
    in the staged route also not the queries before it, a tile away or less."""
    G = NQ // NKV
    most = staged_from(1, NQ, NKV, D, TK)
    for TQ in (1, min(most, TK - 10)):
        print(f"[pf-window] infinite values NQ={NQ} NKV={NKV} D={D} TQ={TQ}", flush=True)
        args = list(inputs(1, NQ, NKV, TQ, D, 1, TK, torch.float16, seed=TK))
        args[3] = torch.arange(TK, dtype=torch.int32, device="cuda")
        want = reference(*args, D ** -0.5)
        late = TK - 3  # seen by the last three queries
        args[2][5, NKV - 1, 0, D - 1] = float("inf")
        args[2][late, 0, 0, 17] = -float("inf")
        out = ops.position_free_paged_attention(*args, scale=D ** -0.5)
        torch.cuda.synchronize()
        assert torch.all(out[:, -G:, :, D - 1] == float("inf"))
        sees = args[5] >= late
        assert torch.all(out[:, :G, sees, 17] == -float("inf"))
        if TQ > 1 and TQ == most:
            assert torch.isfinite(out[:, :G, ~sees, 17]).all()
        hit = torch.zeros_like(out, dtype=torch.bool)
        hit[:, -G:, :, D - 1] = True
        hit[:, :G, :, 17] = True
        check(out.masked_fill(hit, 0.0), want.masked_fill(hit, 0.0), torch.float16)


@pytest.mark.parametrize("wide", [False, True])
def test_weights_of_fp16_pages_to_32_bits(wide):
    """Two keys of a block with values +-2^15 whose weights differ by d = 2^-15 ..
    2^-13 (all others weigh nothing) leave 2^15 tanh(d / 2): what the weights' own
    rounding adds is not hidden by the output's.  Bound, for the weight just below 1: the exponential 2^-24 (an ulp),
    hi and lo halves 2^-24, the sums behind them as much again, times 2^14; fp16
    output 2^-12 of the value; scores of this size are exact to 2^-37."""
    TK = 4000
    TQ = staged_from(1, 2, 1, 128, TK) if wide else 40
    print(f"[pf-window] 32-bit weights, {TQ} queries", flush=True)
    scores = torch.full((TK,), -200.0)
    values = torch.zeros((TK, 128), device="cuda")
    values[10], values[12] = 2.0 ** 15, -2.0 ** 15
    steps = torch.linspace(1.0, 2.0, TQ, device="cuda").to(torch.float16)
    for e in (-15, -14):
        scores[10], scores[12] = 2.0 ** e, 0.0
        q, *args = slow_pair(torch.float16, TK, TQ, scores, values)
        q[..., 63] = steps
        q[..., 127] = 0.0
        out = ops.position_free_paged_attention(q, *args, scale=1.0)
        ref = reference(q, *args, 1.0)
        torch.cuda.synchronize()
        off = (out.double() - ref).abs()
        bound = 2.0 ** 14 * 3 * 2.0 ** -24 + ref.abs() * 2.0 ** -12
        assert bool((off <= bound).all()), (e, (off / bound).max().item())


def test_staged_pages_are_not_kept():
    """The staged copy of the pages is this call's own: the shared scratch does not
    grow, and past a gigabyte the pages are walked instead."""
    print("[pf-window] scratch", flush=True)
    for dtype in (torch.bfloat16, torch.float16):
        args = inputs(1, 28, 4, 250, 128, 1, 8000, dtype, seed=1)
        before = {k: t.numel() for k, t in ops._WORKSPACES.items()}
        ops.position_free_paged_attention(*args, scale=0.1)
        torch.cuda.synchronize()
        assert {k: t.numel() for k, t in ops._WORKSPACES.items()} == before
    need = [ops.position_free_workspace_bytes(1, 32, 250, 8, 128, n) for n in (200_000, 1_000_000)]
    assert need[0] > 4 * 200_000 * 8 * 128  # staged
    assert need[1] < 1 << 30, need


def test_windows_on_a_side_stream():
    """A window enqueued on another stream while the current one goes on allocating
    and computing: workspace and output keep their memory until it has run."""
    print("[pf-window] side stream", flush=True)
    args = inputs(1, 28, 4, 250, 128, 1, 8000, torch.float16, seed=2)
    want = ops.position_free_paged_attention(*args, scale=0.1)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(5):
        got = ops.position_free_paged_attention(*args, scale=0.1, stream=side)
        junk = [torch.full((1 << 22,), 7.0, device="cuda") for _ in range(8)]
        del junk
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_captured_windows_replay():
    """A captured window keeps its workspace: replays between eager calls of larger
    windows equal the eager result."""
    print("[pf-window] graph replay", flush=True)
    args = inputs(1, 28, 4, 100, 128, 1, 3000, torch.float16, seed=4)
    other = inputs(1, 28, 4, 250, 128, 1, 8000, torch.bfloat16, seed=5)
    want = ops.position_free_paged_attention(*args, scale=0.1)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            out = ops.position_free_paged_attention(*args, scale=0.1)
    torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        out.zero_()
        ops.position_free_paged_attention(*other, scale=0.1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
