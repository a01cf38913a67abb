"""GPU parity of the GroupQueryAttention prompt tiles against 64-bit attention, at the edges
of the tile (128 query rows, key blocks of 64 shared by two groups of waves) and of its
dispatch (key splits, rotary in the tile or staged, tensors that are not aligned).

Bound: rotated queries and keys are rounded to the type on both sides (a rounding that falls
the other way moves a score by one unit of one product, a few 2^-p of it), the probabilities
are rounded once (head 96: not), and so is the output: u * (4 P|V| + |out|) with u the
type's unit roundoff, P the exact probabilities."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch
from test_gpu_ops import _run_paged, assert_f16_close, dev, host

pytestmark = pytest.mark.gpu
U = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}
DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def rope(x, cos, sin, pos0, interleaved, dt):
    """x [B, S, heads, hd] float64, rotated and rounded to dt."""
    half = cos.shape[1]
    c = cos[pos0:pos0 + x.shape[1]].double()[None, :, None]
    s = sin[pos0:pos0 + x.shape[1]].double()[None, :, None]
    y = x.clone()
    a, b = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if interleaved else \
        (slice(0, half), slice(half, 2 * half))
    y[..., a] = x[..., a] * c - x[..., b] * s
    y[..., b] = x[..., b] * c + x[..., a] * s
    return y.to(dt).double()


def check(ortmi, dt, B, S, past, H, KV, hd, half=None, interleaved=False, shared=True, shift=0,
          scale=0.0, packed=False):
    tdt = DT[dt]
    g = torch.Generator().manual_seed(S * 131 + past + H + hd)
    half = hd // 2 if half is None else half

    def rnd(*shape):
        return torch.randn(shape, generator=g).to(tdt)

    def put(t):  # on the GPU, `shift` elements off an aligned address
        buf = torch.zeros(t.numel() + shift, dtype=tdt, device="cuda")
        buf[shift:] = t.flatten().cuda()
        return buf[shift:].view(t.shape)

    q, k, v = rnd(B, S, H * hd), rnd(B, S, KV * hd), rnd(B, S, KV * hd)
    cap = past + S + (5 if shared else 0)
    pk, pv = rnd(B, KV, cap if shared else past, hd), rnd(B, KV, cap if shared else past, hd)
    ang = torch.rand((past + S, max(half, 1)), generator=g) * 6
    cos, sin = ang.cos().to(tdt), ang.sin().to(tdt)
    kw = dict(num_heads=H, kv_num_heads=KV, scale=scale, rotary_interleaved=int(interleaved),
              do_rotary=int(half > 0))
    dpk, dpv = put(pk), put(pv)
    if shared:
        kw.update(present_key=dpk, present_value=dpv)
    qkv = (put(torch.cat([q, k, v], -1)), None, None) if packed else (put(q), put(k), put(v))
    out, ok, ov = ortmi.group_query_attention(*qkv, dpk, dpv, None, past + S,
                                              cos.cuda() if half else None,
                                              sin.cuda() if half else None, **kw)
    qd, kd = q.double().reshape(B, S, H, hd), k.double().reshape(B, S, KV, hd)
    if half:
        qd, kd = (rope(x, cos, sin, past, interleaved, tdt) for x in (qd, kd))
    keys = torch.cat([pk[:, :, :past].double(), kd.transpose(1, 2)], 2)
    vals = torch.cat([pv[:, :, :past].double(), v.double().reshape(B, S, KV, hd).transpose(1, 2)], 2)
    rep = torch.arange(H) // (H // KV)
    sc = qd.transpose(1, 2) @ keys[:, rep].transpose(-1, -2) * (scale or 1 / math.sqrt(hd))
    hide = torch.arange(past + S)[None] > past + torch.arange(S)[:, None]
    p = torch.softmax(sc.masked_fill(hide, -math.inf), -1)
    want = (p @ vals[:, rep]).transpose(1, 2)
    mag = (p @ vals[:, rep].abs()).transpose(1, 2)
    got = out.double().cpu().reshape(B, S, H, hd)
    if dt == "f32":
        bound = 2.0 ** -24 * ((past + S + 8 * hd) * mag + want.abs())
    else:
        bound = U[dt] * (4 * mag + want.abs())
    excess = ((got - want).abs() - bound).max().item()
    assert excess <= 1e-6, f"max excess {excess:.3e}"
    n = past + S
    err = (ok.double().cpu()[:, :, :n] - keys).abs().max().item()
    assert err <= (2.0 ** -20 if dt == "f32" else 2 * U[dt]) * keys.abs().max().item()
    assert torch.equal(ov.double().cpu()[:, :, :n], vals)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("hd", [64, 96, 128])
@pytest.mark.parametrize("B,S,past,H,KV", [
    (1, 2, 0, 4, 4),       # one block, the second key group without work
    (2, 33, 31, 14, 2),    # 18 tokens of 7 heads to a tile, a block cut at 64
    (1, 65, 0, 8, 8),      # one head per tile row group, one key past a block
    (1, 128, 64, 4, 1),
    (3, 129, 62, 16, 4),   # a tile with one token; odd number of blocks
    (1, 5, 1500, 32, 8),   # few rows, many keys: splits, merged
    (1, 20, 2000, 24, 8),  # the last split shorter
    (2, 1, 300, 6, 3),     # (fp32: one token on the tiles too)
])
def test_gqa_tile(ortmi, dt, hd, B, S, past, H, KV):
    check(ortmi, dt, B, S, past, H, KV, hd)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 96, 128])
@pytest.mark.parametrize("B,S,past,H,KV", [
    (2, 64, 0, 8, 2),     # one block of keys, full; two tiles
    (1, 31, 33, 12, 2),   # cached keys in it
    (9, 17, 0, 16, 16),   # a workgroup per head, ragged rows and keys
])
def test_gqa_tile_one_block(ortmi, dt, hd, B, S, past, H, KV):
    """All keys in one block: tiles of one key group."""
    check(ortmi, dt, B, S, past, H, KV, hd)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("opt", [
    dict(interleaved=True), dict(half=0), dict(half=16), dict(half=24, interleaved=True),
    dict(shared=False), dict(shift=1), dict(shift=3, interleaved=True), dict(scale=-0.2),
    dict(packed=True)])
@pytest.mark.parametrize("hd", [64, 96, 128])
def test_gqa_tile_options(ortmi, dt, hd, opt):
    check(ortmi, dt, 2, 37, 70, 8, 2, hd, **opt)


@pytest.mark.parametrize("opt", [dict(interleaved=True), dict(half=16), dict(shared=False),
                                 dict(shift=1), dict(scale=-0.2), dict(packed=True)])
@pytest.mark.parametrize("hd", [64, 96, 128])
def test_gqa_f32_tile_options(ortmi, hd, opt):
    """fp32: the sign branch, and the fallback for rows that are not 16-byte aligned."""
    check(ortmi, "f32", 2, 130, 150, 8, 2, hd, **opt)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,S,past,H,KV,opt", [
    (1, 300, 0, 4, 4, dict(shift=1)),               # several blocks and tiles, the last ragged
    (1, 5, 1500, 32, 8, dict(shift=7)),             # key splits
    (2, 1, 70, 18, 2, dict(shift=4)),               # one token the decode kernel does not take
    (2, 70, 33, 8, 2, dict(shift=5, shared=False)), # past rows copied from unaligned tensors
])
def test_gqa_tile_unaligned(ortmi, dt, hd, B, S, past, H, KV, opt):
    """Tensors that start at any element: the tiles' rows pass through registers."""
    check(ortmi, dt, B, S, past, H, KV, hd, **opt)


def test_gqa_tile_smallest_workspace(ortmi):
    """The smallest workspace of a prompt has room for two key splits instead of four; less
    is an error, and nothing is launched."""
    S, H, KV, hd, past = 40, 32, 8, 128, 1500
    lib = ortmi.load_kernels()
    g = torch.Generator().manual_seed(9)
    q, k, v, pk, pv = (torch.randn(n, generator=g).half().cuda() for n in (
        (1, S, H * hd), (1, S, KV * hd), (1, S, KV * hd), (1, KV, past + S, hd),
        (1, KV, past + S, hd)))
    full = lib.ortmi_group_query_attention_workspace_size(1, S, H, hd, past + S)
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    least = up(S * H * hd * 4) + up(S * H * 2 * (hd + 2) * 4) + up(S * H * 4)
    assert least < full
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    outs = []
    for size, status in ((full, 0), (least, 0), (least - 1, 3)):
        out = torch.zeros_like(q)
        rc = lib.ortmi_group_query_attention(
            *(x.data_ptr() for x in (q, k, v, pk, pv)), past + S, past + S, None, None, 0, 0,
            *(x.data_ptr() for x in (out, pk, pv)), 1, S, H, KV, hd, 0.0, 0, 10, ws.data_ptr(), size,
            torch.cuda.current_stream().cuda_stream)
        assert rc == status
        outs.append(out.double().cpu())
    assert_f16_close(outs[1].numpy(), outs[0].numpy(), what="two key splits")
    assert outs[0].abs().max() > 0 and outs[2].abs().max() == 0


def test_gqa_f32_tile_infinite_value_stays_in_its_rows(ortmi):
    """An infinite value of a key reaches the rows that see the key and no other."""
    S, H, hd = 45, 2, 64
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn((1, S, H * hd), generator=g) for _ in range(3))
    v[0, 20, 3] = math.inf
    z = torch.zeros((1, H, 0, hd), device="cuda")
    out, _, _ = ortmi.group_query_attention(q.cuda(), k.cuda(), v.cuda(), z, z, None, S, None, None,
                                            num_heads=H, kv_num_heads=H)
    out = out.cpu()[0]
    assert torch.isfinite(out[:20]).all() and (out[20:, 3] == math.inf).all()
    out[20:, 3] = 0
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("hd", [64, 96, 128])
@pytest.mark.parametrize("B,S,past,H,KV", [
    (1, 1, 16, 32, 8), (1, 17, 0, 14, 2), (2, 33, 16, 8, 8),    # few keys
    (32, 1, 90, 16, 16),                                        # one row to a tile
    (1, 60, 40, 32, 8), (1, 100, 0, 24, 8), (4, 9, 100, 32, 8),  # to both sides of the line
    (1, 257, 0, 8, 2),
])
def test_gqa_f32_few_keys(ortmi, hd, B, S, past, H, KV):
    """fp32 calls on both sides of the rule that chooses tiles or a workgroup per row."""
    check(ortmi, "f32", B, S, past, H, KV, hd)


@pytest.mark.parametrize("hd,at", [(64, 130), (96, 201), (128, 255)])
def test_gqa_f32_tile_infinite_value(ortmi, hd, at):
    """As above, with keys enough for the tiles."""
    S, H = 257, 8
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn((1, S, H * hd), generator=g) for _ in range(3))
    v[0, at, 3] = math.inf
    z = torch.zeros((1, H, 0, hd), device="cuda")
    out, _, _ = ortmi.group_query_attention(q.cuda(), k.cuda(), v.cuda(), z, z, None, S, None, None,
                                            num_heads=H, kv_num_heads=H)
    out = out.cpu()[0]
    assert torch.isfinite(out[:at]).all() and (out[at:, 3] == math.inf).all()
    out[at:, 3] = 0
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("S,past,H,KV,at", [
    (45, 0, 2, 2, 20),     # one block
    (128, 0, 4, 4, 120),   # hidden to whole waves of the tile
    (100, 70, 6, 2, 3),    # 42 tokens to a tile, a block that holds cached keys too
    (40, 1500, 2, 1, 39),  # key splits
])
def test_gqa_tile_head96_value_stays_in_its_rows(ortmi, dt, value, S, past, H, KV, at):
    """A value of a new token that is not finite reaches the rows of head 96 that see the
    token, in its dim, and no other; the finite outputs are those of finite values."""
    hd, tdt = 96, DT[dt]
    g = torch.Generator().manual_seed(S + past)

    def rnd(*shape):
        return torch.randn(shape, generator=g).to(tdt).cuda()

    q, k, v = rnd(1, S, H * hd), rnd(1, S, KV * hd), rnd(1, S, KV * hd)
    pk, pv = rnd(1, KV, past, hd), rnd(1, KV, past, hd)
    kw = dict(num_heads=H, kv_num_heads=KV)
    want, _, _ = ortmi.group_query_attention(q, k, v, pk, pv, None, past + S, None, None, **kw)
    v[0, at, 3] = value  # of KV head 0
    out, _, _ = ortmi.group_query_attention(q, k, v, pk, pv, None, past + S, None, None, **kw)
    out, want = (x.cpu()[0].reshape(S, H, hd) for x in (out, want))
    hit = torch.zeros((S, H, hd), dtype=torch.bool)
    hit[at:, :H // KV, 3] = True
    bad = out[hit].double()
    assert (torch.isnan(bad) if math.isnan(value) else bad == value).all()
    # The block's sums run in another order: fp32 accumulation, and one rounding.
    torch.testing.assert_close(out[~hit].double(), want[~hit].double(), rtol=2 * U[dt],
                               atol=2.0 ** -16)


def test_gqa_tile_head96_keeps_probabilities(ortmi):
    """Head 96 rounds no probability: with large values that cancel, the error stays at that
    of fp32 arithmetic and one rounding of the output."""
    B, S, H, hd = 1, 64, 2, 96
    g = torch.Generator().manual_seed(3)
    q, k = (torch.randn((B, S, H * hd), generator=g).half() * 0.1 for _ in range(2))
    v = (torch.randn((B, S, H * hd), generator=g).sign() * 1000).half()
    z = torch.zeros((B, H, 0, hd), dtype=torch.float16, device="cuda")
    out, _, _ = ortmi.group_query_attention(q.cuda(), k.cuda(), v.cuda(), z, z, None, S, None, None,
                                            num_heads=H, kv_num_heads=H)
    qd, kd, vd = (x.double().reshape(S, H, hd).transpose(0, 1) for x in (q, k, v))
    sc = (qd @ kd.transpose(-1, -2)) / math.sqrt(hd)
    sc = sc.masked_fill(torch.ones(S, S).triu(1).bool(), -math.inf)
    want = (torch.softmax(sc, -1) @ vd).transpose(0, 1).reshape(S, H * hd)
    err = (out.double().cpu()[0] - want).abs()
    assert (err <= 2.0 ** -11 * want.abs() + 1000 * 2.0 ** -19).all(), err.max().item()


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("nats", [9.0, 12.0])
def test_gqa_tile_head96_keeps_small_probabilities(ortmi, dt, nats):
    """Probabilities of e^-9 and e^-12 beside one near 1 (whose value is 0) keep their bits:
    large values that cancel leave the fp32 errors of the exponential, its argument (up to 16:
    2^-21 of P each) and the sums, and the output's rounding."""
    S, H, hd, tdt = 64, 2, 96, DT[dt]
    g = torch.Generator().manual_seed(11)
    q, k = (torch.randn((1, S, H, hd), generator=g) * 0.1 for _ in range(2))
    q[..., 0] = math.sqrt(nats * math.sqrt(hd))
    k[..., 0] = 0
    k[:, 0, :, 0] = q[0, 0, 0, 0]
    v = torch.full((1, S, H, hd), 30000.0)
    v[:, 1::2] *= -1
    v[:, 0] = 0
    q, k, v = (x.to(tdt).reshape(1, S, H * hd) for x in (q, k, v))
    z = torch.zeros((1, H, 0, hd), dtype=tdt, device="cuda")
    out, _, _ = ortmi.group_query_attention(q.cuda(), k.cuda(), v.cuda(), z, z, None, S, None, None,
                                            num_heads=H, kv_num_heads=H)
    qd, kd, vd = (x.double().reshape(S, H, hd).transpose(0, 1) for x in (q, k, v))
    sc = (qd @ kd.transpose(-1, -2)) / math.sqrt(hd)
    p = torch.softmax(sc.masked_fill(torch.ones(S, S).triu(1).bool(), -math.inf), -1)
    want, mag = ((p @ x).transpose(0, 1).reshape(S, H * hd) for x in (vd, vd.abs()))
    excess = (out.double().cpu()[0] - want).abs() - U[dt] * want.abs() - 2.0 ** -20 * mag
    assert excess.max().item() <= 0, excess.max().item()


@pytest.mark.parametrize("H,KV", [(6, 2), (14, 2)])
@pytest.mark.parametrize("d,new_max,interleaved", [(64, 1, 0), (128, 3, 1)])
def test_paged_group_sizes(ortmi, oracle, H, KV, d, new_max, interleaved):
    """Single tokens of 3 query heads per KV head (the decode kernel) and of 7 (the tiles),
    beside chunks on the tiles; long pasts split the keys."""
    _run_paged(ortmi, oracle, H, KV, d, nb=100 * 3, blk=16, batch=3, seed=H + d, new_max=new_max,
               rope=True, interleaved=interleaved)


@pytest.mark.parametrize("batch,maxb", [(4, 40), (26, 70)])
def test_paged_groups_of_three_beside_chunks(ortmi, oracle, batch, maxb):
    """Single tokens of 3 query heads per KV head beside chunks: on the tiles where those all
    run at once, on the decode kernel where they do not (26 sequences, 3 splits)."""
    _run_paged(ortmi, oracle, 24, 8, 64, nb=maxb * batch, blk=16, batch=batch, seed=batch,
               new_max=2, rope=True)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("hd,H,KV", [(64, 8, 8), (96, 6, 2), (128, 8, 1)])
@pytest.mark.parametrize("shared", [True, False])
def test_gqa_one_token_negative_scale(ortmi, dt, hd, H, KV, shared):
    """Scores of some +-100: the maximum that the exponents are taken from is that of the
    scaled scores, not of the raw products."""
    check(ortmi, dt, 2, 1, 300, H, KV, hd, half=0, scale=-4.0, shared=shared)


@pytest.mark.parametrize("H,KV", [(2, 2), (4, 2), (6, 2), (8, 2), (8, 1), (7, 1)])
def test_paged_one_token_negative_scale(ortmi, oracle, H, KV):
    """The same over a paged cache, for each group size of the decode kernel and one of the
    tiles; two sequences split their keys."""
    rng = np.random.default_rng(H)
    d, blk, batch, maxb = 64, 16, 3, 80
    past = np.array([37, 700, 1279], np.int32)
    cum = np.arange(batch + 1, dtype=np.int32)

    def rnd(*shape):
        return rng.standard_normal(shape).astype(np.float16)

    q, k, v = rnd(batch, H * d), rnd(batch, KV * d), rnd(batch, KV * d)
    kc, vc = rnd(maxb * batch, blk, KV, d), rnd(maxb * batch, blk, KV, d)
    bt = rng.permutation(maxb * batch).astype(np.int32).reshape(batch, maxb)
    out = ortmi.paged_attention(dev(q), dev(k), dev(v), dev(kc), dev(vc), dev(cum), dev(past),
                                dev(bt), num_heads=H, kv_num_heads=KV, scale=-4.0)
    want, _, _ = oracle.paged_attention(q, k, v, kc, vc, cum, past, bt, H, KV, scale=-4.0,
                                        round16=True)
    assert_f16_close(host(out), want, what="paged one token, scale -4")
