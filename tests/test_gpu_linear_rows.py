"""GPU numerics of the many-row projections: products against float64, the
residual add bit for bit and the norm within an ulp of add_rms_norm's, SwiGLU and
the qkv form bit for bit against the plain form followed by silu_mul, or by
rope_split and append_kv."""
import pytest
import torch

from voom_amd import decoder, ops
from voom_amd.decoder import DecoderConfig, PagedDecoder, random_weights

pytestmark = pytest.mark.gpu


def bits(t: torch.Tensor) -> torch.Tensor:
    return t.view(torch.int16)


def randn(g, *shape, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(torch.bfloat16)


# rows around the 32-row tile; k at the ends of the LDS sizes (256 values) and of
# the weight buffers (12 or 6 k-steps of 32, two of them); n with a part of a
# 16-column tile, of the tiles of a workgroup, and of the 8 groups of the XCD map
@pytest.mark.parametrize("rows,k,n", [(2, 32, 8), (31, 384, 72), (32, 512, 64), (33, 544, 584),
                                      (65, 768, 136), (64, 800, 16), (5, 1536, 960), (40, 1056, 40),
                                      (34, 1408, 24), (3, 1792, 24), (97, 2048, 24)])
def test_linear_rows(rows, k, n):
    print(f"[linear-rows] {rows}x{k} -> {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + k + n)
    x, d, ln = randn(g, rows, k), randn(g, rows, k), randn(g, k)
    w = randn(g, 2 * n, k, std=k ** -0.5)
    y = ops.linear_rows(x, w)
    ref = x.double() @ w.double().T
    # fp32 sums of k exact products, then one rounding to bf16 (half an ulp: 2^-9)
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().T) * k * 2.0 ** -24
    assert bool(((y.double() - ref).abs() <= bound).all())
    for delta in (d, None):
        want = x.clone()
        h = ops.add_rms_norm(want, ln, 1e-5, delta=delta)
        out = torch.full_like(x, float("nan"))
        before = x.clone()
        act = ops.norm_swiglu_rows(x, w, ln, 1e-5, delta=delta, x_out=out)
        assert torch.equal(bits(x), bits(before)) and torch.equal(bits(out), bits(want))
        # a normed value may round to the neighbour of add_rms_norm's (2^-8 of it, the
        # statistics' order): first order through the two products and silu
        both = (h.double() @ w.double().T)
        e = (h.double().abs() @ w.double().abs().T) * (2.0 ** -8 + k * 2.0 ** -24)
        e = e + both.abs() * 2.0 ** -8
        gate, up, eg, eu = both[:, :n], both[:, n:], e[:, :n], e[:, n:]
        silu = gate * torch.sigmoid(gate)  # |silu'| <= 1.1
        bound = 1.1 * eg * (up.abs() + eu) + silu.abs() * eu + (silu * up).abs() * 2.0 ** -7
        assert bool(((act.double() - silu * up).abs() <= bound).all())


def test_norm_of_the_rows_within_an_ulp_and_swiglu_bitwise():
    """Unit weights pass the normed rows through the products exactly."""
    K, rows = 576, 45
    g = torch.Generator(device="cuda").manual_seed(5)
    x, d, ln = randn(g, rows, K), randn(g, rows, K), randn(g, K)
    eye = torch.eye(K, device="cuda").to(torch.bfloat16)
    h = ops.add_rms_norm(x.clone(), ln, 1e-5, delta=d)
    act = ops.norm_swiglu_rows(x, torch.cat([eye, eye]), ln, 1e-5, delta=d)
    ref = ops.silu_mul(torch.cat([h, h], -1))
    off = act != ref
    assert off.float().mean() < 1e-3
    assert bool(((act - ref).float().abs() <= 2.0 ** -5 * ref.float().abs()).all())
    # exact statistics (equal powers of two): nothing left to the order of sums
    x = torch.where(torch.rand((rows, K), generator=g, device="cuda") < 0.5, -2.0, 2.0)
    x = x.to(torch.bfloat16)
    w = randn(g, 2 * 72, K, std=K ** -0.5)
    h = ops.add_rms_norm(x.clone(), ln, 1e-5)
    act = ops.norm_swiglu_rows(x, w, ln, 1e-5)
    assert torch.equal(bits(act), bits(ops.silu_mul(ops.linear_rows(h, w))))


@pytest.mark.parametrize("B,L,nq,nkv,hd,pt,start", [(1, 2, 9, 3, 64, 64, 0), (1, 70, 9, 3, 64, 64, 61),
                                                    (2, 33, 4, 2, 32, 16, 15),
                                                    (3, 1, 4, 1, 128, 32, 31)])
def test_qkv_rope_append_rows(B, L, nq, nkv, hd, pt, start):
    print(f"[linear-rows] qkv B={B} L={L} hd={hd} pt={pt}", flush=True)
    K = 576
    g = torch.Generator(device="cuda").manual_seed(B * L + hd)
    # +-2 in every row: statistics that no order of sums changes
    x = torch.where(torch.rand((B, L, K), generator=g, device="cuda") < 0.5, -1.0, 1.0)
    x = x.to(torch.bfloat16)
    d, ln = x.clone(), randn(g, K)
    w = randn(g, (nq + 2 * nkv) * hd, K, std=K ** -0.5)
    ang = torch.rand((L, hd), generator=g, device="cuda") * 6
    cos, sin = ang.cos(), ang.sin()
    pages = -(-(start + L) // pt)
    slots = B * pages + 2
    table = torch.randperm(slots, generator=torch.Generator().manual_seed(1))[:B * pages]
    table = table.to(torch.int32).reshape(B, pages).cuda()
    pos = torch.full((B,), start, dtype=torch.int32, device="cuda")
    k1 = randn(g, slots, nkv, pt, hd)
    vshape = ops_v_shape(slots, nkv, hd, pt)
    v1 = randn(g, *vshape)
    k2, v2 = k1.clone(), v1.clone()
    xo = torch.empty_like(x)
    q = ops.qkv_rope_append_rows(x, w, cos, sin, k1, v1, table, start, nq, nkv, hd, ln_weight=ln,
                                 eps=1e-5, delta=d, x_out=xo)
    x2 = x.clone()
    h = ops.add_rms_norm(x2, ln, 1e-5, delta=d)
    q2, kn, vn = ops.rope_split(ops.linear_rows(h, w), cos, sin, nq, nkv, hd)
    ops.append_kv(kn, vn, k2, v2, table, pos)
    for a, b in ((q, q2), (k1, k2), (v1, v2), (xo, x2)):
        assert torch.equal(bits(a), bits(b))


def ops_v_shape(slots, nkv, hd, pt):
    vb = min(pt, 32)
    return slots, nkv, pt // vb, hd, vb


def test_refusals():
    x = torch.zeros((4, 64), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((16, 64), dtype=torch.bfloat16, device="cuda")
    for bad_x, bad_w in ((x[:, :48].contiguous(), w[:, :48].contiguous()),   # k % 32
                         (x, w[:12]),                                      # n % 8
                         (x.float(), w), (x, w[:, :32]),
                         (torch.zeros((4, 2080), dtype=torch.bfloat16, device="cuda"),
                          torch.zeros((16, 2080), dtype=torch.bfloat16, device="cuda"))):
        with pytest.raises(ValueError):
            ops.linear_rows(bad_x, bad_w)
    ln = torch.ones(64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError):
        ops.norm_swiglu_rows(x, w, ln, 1e-5, x_out=x)
    with pytest.raises(ValueError):
        ops.norm_swiglu_rows(x, w, ln[:32].contiguous(), 1e-5)
    flat = torch.zeros(4 * 64 + 1, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError):
        ops.linear_rows(flat[1:].view(4, 64), w)


@pytest.mark.parametrize("B,L", [(1, 6), (2, 37), (3, 1)])
def test_decoder_rows_route_against_the_separate_launches(B, L, monkeypatch):
    """Logits of a prompt through the fused row projections, through the separate
    launches (forced, and where the work is past FUSED_MAX_WORK), and through both
    (a layer with a misaligned weight), over the same weights, each counted to have
    run.  The routes round at the same points; their fp32 sums run in another order,
    so that now and then a bf16 value falls to its neighbour (2^-8 of it) and the
    layers behind carry that on.  Bar: as if every value of the twelve rounded results
    on the way (five a layer, the final norm, the logits) had: sqrt(12) * 2^-8 /
    sqrt(3) = 7.8e-3."""
    print(f"[linear-rows] decoder B={B} L={L}", flush=True)
    cfg = DecoderConfig(num_hidden_layers=2)
    dec = PagedDecoder(cfg, random_weights(cfg, seed=2))
    ids = torch.randint(0, cfg.vocab_size, (B, 2 * L), generator=torch.Generator().manual_seed(3))
    ran = []
    for name in ("_block_rows", "_block"):
        def counted(self, *a, _run=getattr(PagedDecoder, name), _name=name, **kw):
            ran.append(_name)
            return _run(self, *a, **kw)
        monkeypatch.setattr(PagedDecoder, name, counted)

    def logits(want):
        kv = dec.new_cache(page_positions=32)
        out = []
        for part, last in ((ids[:, :L], False), (ids[:, L:], False), (ids[:, :L], True)):
            ran.clear()
            out.append(dec.forward(part.cuda(), kv, last_only=last))
            assert ran == want, ran
        assert kv.offset == 3 * L
        return out

    fused = logits(["_block_rows"] * 2)
    with monkeypatch.context() as m:
        m.setattr(PagedDecoder, "_rows_fused", lambda self, x: False)
        ref = logits(["_block"] * 2)
    with monkeypatch.context() as m:
        m.setattr(decoder, "FUSED_MAX_WORK", B * L * 2_000_000)  # a layer has 3.5 million weights
        past = logits(["_block"] * 2)
    down = dec.layers[1]["down"]
    dec.layers[1]["down"] = torch.empty(down.numel() + 1, dtype=down.dtype,
                                        device="cuda")[1:].view(down.shape).copy_(down)
    mixed = logits(["_block_rows", "_block"])
    for got in (fused, mixed):
        for a, b in zip(got, ref):
            rel = ((a - b).norm() / b.norm()).item()
            print(f"[linear-rows] routes differ by {rel:.2e}", flush=True)
            assert a.shape == b.shape and rel < 7.8e-3, rel
    for a, b in zip(past, ref):
        assert torch.equal(a, b)
