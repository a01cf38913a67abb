"""The work a user of the execution provider has it do, as timed cases.

Kinds of case ("kind" of the case dict):

  linear   one MatMulNBits call through the kernel C ABI (ortmi_matmul_nbits), as the
           execution provider and any other runtime on the library calls it: device
           buffers in place, the output buffer kept.
  gqa      one GroupQueryAttention call through the C ABI with a kept workspace
           (one-token decode or a prompt chunk, shared or growing KV cache).
  paged    one PagedAttention call over a paged cache through the C ABI.
  block    an attention block (QKV MatMulNBits, GroupQueryAttention, output
           MatMulNBits) through the Python op interface.
  decoder  one run of a whole int4 decoder graph through the plugin-EP boundary: a
           prompt (prefill) or one more token behind `context` cached ones (decode).

Sizes are those of this repository's benchmark (bench.py), its decoder layouts and
its tests. Inputs are made on the GPU from the seed alone.
"""

from __future__ import annotations

import ctypes
import importlib
import math

import numpy as np
import torch

PKG = "onnxruntime-mlx_amd"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
CODES = {"f16": 10, "bf16": 16, "f32": 1}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}

# Decoder layouts (hidden, query heads, KV heads, head size, SwiGLU width).
LAYOUTS = {
    "d1536": (1536, 12, 2, 128, 8960),
    "d896": (896, 14, 2, 64, 4864),
    "d2048": (2048, 32, 8, 64, 8192),
    "d3072": (3072, 24, 8, 128, 8192),
}


def _pkg(name=""):
    return importlib.import_module(PKG + name)


# ------------------------------------------------------------------------ cases --

def listed():
    return [
        # A 7B-class decoder's output projection for one token: the smallest call,
        # bound by launch and latency as much as by its 9 MB of weights.
        dict(name="linear_decode_o", kind="linear", dtype="f16", M=1, K=4096, N=4096, bits=4,
             block=32, zp=False),
        # The benchmark's headline GEMV: one token, fp32 activations.
        dict(name="linear_decode_mlp_f32", kind="linear", dtype="f32", M=1, K=4096, N=11008,
             bits=4, block=32, zp=True),
        # Eight requests decoded together (or eight drafted tokens verified at once)
        # through a 7B-class gate projection.
        dict(name="linear_batch8", kind="linear", dtype="f16", M=8, K=4096, N=14336, bits=4,
             block=32, zp=False),
        # The benchmark's prefill GEMM: a 512-token prompt.
        dict(name="linear_prefill_512", kind="linear", dtype="f16", M=512, K=4096, N=4096,
             bits=4, block=32, zp=True),
        # A long, ragged prompt through gate and up of a bf16 model, block 128.
        dict(name="linear_prefill_bf16", kind="linear", dtype="bf16", M=1999, K=1536, N=17920,
             bits=4, block=128, zp=False),
        # The 8-bit lm_head that int4 exports keep, one token.
        dict(name="linear_head_8bit", kind="linear", dtype="f16", M=1, K=3072, N=32064, bits=8,
             block=32, zp=False),
        # One decode step of eight sequences at a 4096-token context, cache in place.
        dict(name="gqa_decode_4k", kind="gqa", dtype="f16", B=8, S=1, past=4096, H=32, KV=8,
             hd=128, shared=True),
        # A 2048-token prompt's attention.
        dict(name="gqa_prefill_2k", kind="gqa", dtype="f16", B=1, S=2048, past=0, H=32, KV=8,
             hd=128, shared=True),
        # Continuous batching: four prefill chunks beside 28 decoding sequences.
        dict(name="paged_mixed", kind="paged", dtype="f16", nseq=32, prefill=4, chunk=256,
             lo=256, hi=8192, H=32, KV=8, hd=128, blk=16),
        # The attention block of an fp32-activation export over a 512-token prompt.
        dict(name="block_f32_prompt", kind="block", dtype="f32", S=512, hidden=896, H=14, KV=2,
             hd=64),
        # The benchmark decoder end to end: one greedy step, and a 512-token prompt.
        dict(name="decoder_step", kind="decoder", layout="d1536", layers=28, vocab=151936, S=1,
             context=576),
        dict(name="decoder_prompt", kind="decoder", layout="d1536", layers=28, vocab=151936,
             S=512, context=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "gqa", "paged", "block", "decoder"], [50, 24, 10, 10, 6])[0]
    if kind == "linear":
        dtype = rng.choices(["f16", "bf16", "f32"], [5, 3, 3])[0]
        bits = 8 if rng.random() < 0.2 else 4
        block = rng.choice([32, 32, 32, 64, 128])
        # One token, a small batch of sequences, or a prompt.
        M = rng.choices([1, _log_int(rng, 2, 32), _log_int(rng, 33, 2048)], [4, 3, 4])[0]
        K = _log_int(rng, 512, 14336)
        K -= K % (8 if rng.random() < 0.15 else block)
        N = _log_int(rng, 512, 17920)
        if M <= 32 and rng.random() < 0.15:
            N = rng.choice([32064, 128256, 151936])
            K = min(K, 4096)
        cap = 2.5e11 if dtype != "f32" and bits == 4 else 4e10
        M = max(1, min(M, int(cap / (2.0 * K * N))))
        return dict(kind=kind, dtype=dtype, M=M, K=K, N=N, bits=bits, block=block,
                    zp=rng.random() < 0.5)
    H, KV = rng.choice([(14, 2), (12, 2), (32, 8), (24, 8), (32, 32), (16, 4)])
    if kind == "gqa":
        dtype = rng.choices(["f16", "bf16", "f32"], [5, 4, 1])[0]
        hd = rng.choice([64, 96, 128, 128])
        S = 1 if rng.random() < 0.55 else _log_int(rng, 2, 2048)
        B = _log_int(rng, 1, 16) if S == 1 else _log_int(rng, 1, 4)
        past = _log_int(rng, 16, 8192) if S == 1 or rng.random() < 0.4 else 0
        if dtype == "f32":  # an fp32 export's sequences are short
            B, S, past = min(B, 2), min(S, 512), min(past, 2048)
        while B * KV * (past + S) * hd > 2 ** 27 or B * H * S * (past + S / 2) * hd > 2 ** 34:
            past, S, B = past // 2, max(1, S // 2), max(1, B // 2)
        return dict(kind=kind, dtype=dtype, B=B, S=S, past=past, H=H, KV=KV, hd=hd,
                    shared=past == 0 or rng.random() < 0.7)
    if kind == "paged":
        return dict(kind=kind, dtype=rng.choice(["f16", "bf16"]), nseq=_log_int(rng, 4, 40),
                    prefill=rng.randint(0, 4), chunk=_log_int(rng, 16, 256), lo=256,
                    hi=_log_int(rng, 512, 8192), H=H, KV=KV, hd=rng.choice([64, 128]),
                    blk=rng.choice([16, 32]))
    if kind == "block":
        hidden, H, KV, hd, _ = LAYOUTS[rng.choice(["d896", "d1536", "d2048"])]
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "f16"]),
                    S=_log_int(rng, 2, 640), hidden=hidden, H=H, KV=KV, hd=hd)
    prompt = rng.random() < 0.5
    return dict(kind=kind, layout=rng.choice(list(LAYOUTS)), layers=rng.randint(2, 6),
                vocab=32064, S=_log_int(rng, 2, 512) if prompt else 1,
                context=0 if prompt else _log_int(rng, 16, 2048))


# ----------------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, dtype, sd=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * sd).to(dtype)


def _quant(g, N, K, bits, block, zp, dtype):
    """Packed weights, scales and zero points of an [N, K] MatMulNBits."""
    nb = -(-K // block)
    B = torch.randint(0, 256, (N, nb, block * bits // 8), generator=g, device="cuda",
                      dtype=torch.uint8)
    s = torch.randn(N * nb, generator=g, device="cuda").abs() * 0.02 + 1e-4
    if bits == 8:
        s = s / 16
    z = None
    if zp:
        cols = (nb + 1) // 2 if bits == 4 else nb
        z = torch.randint(0, 256, (N * cols,), generator=g, device="cuda", dtype=torch.uint8)
    return B, s.to(dtype), z


def _rotary(max_pos, hd, dtype, base=10000.0):
    half = hd // 2
    inv = 1.0 / base ** (torch.arange(half, dtype=torch.float64) / half)
    ang = torch.arange(max_pos, dtype=torch.float64)[:, None] * inv[None, :]
    return ang.cos().to(dtype).cuda(), ang.sin().to(dtype).cuda()


def _linear_inputs(c, seed):
    g = _gen(seed)
    dt = DTYPES[c["dtype"]]
    A = _normal(g, (c["M"], c["K"]), dt)
    return (A,) + _quant(g, c["N"], c["K"], c["bits"], c["block"], c["zp"], dt)


def _gqa_inputs(c, seed):
    g = _gen(seed)
    dt, B, S, H, KV, hd = DTYPES[c["dtype"]], c["B"], c["S"], c["H"], c["KV"], c["hd"]
    cap = c["past"] + S if c["shared"] else c["past"]
    d = dict(q=_normal(g, (B, S, H * hd), dt), k=_normal(g, (B, S, KV * hd), dt),
             v=_normal(g, (B, S, KV * hd), dt), pk=_normal(g, (B, KV, cap, hd), dt),
             pv=_normal(g, (B, KV, cap, hd), dt))
    d["cos"], d["sin"] = _rotary(c["past"] + S, hd, dt)
    return d


def _paged_inputs(c, seed):
    """Contexts U[lo, hi]; the first `prefill` sequences bring `chunk` new tokens, the
    others one; a random block table over exactly the blocks in use."""
    g = _gen(seed)
    rng = np.random.default_rng(c["nseq"] * 7919 + c["hi"])  # the shape: the same for all seeds
    dt, KV, hd, blk = DTYPES[c["dtype"]], c["KV"], c["hd"], c["blk"]
    ctx = rng.integers(c["lo"], c["hi"] + 1, size=c["nseq"])
    new = np.array([c["chunk"]] * min(c["prefill"], c["nseq"]) +
                   [1] * max(0, c["nseq"] - c["prefill"]))
    nblocks = (ctx + blk - 1) // blk
    total, maxb = int(nblocks.sum()), int(nblocks.max())
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    bt = torch.zeros((c["nseq"], maxb), dtype=torch.int32, device="cuda")
    o = 0
    for b, n in enumerate(nblocks.tolist()):
        bt[b, :n] = perm[o:o + n]
        o += n
    T = int(new.sum())
    d = dict(q=_normal(g, (T, c["H"] * hd), dt), k=_normal(g, (T, KV * hd), dt),
             v=_normal(g, (T, KV * hd), dt), kc=_normal(g, (total, blk, KV, hd), dt),
             vc=_normal(g, (total, blk, KV, hd), dt), bt=bt, ctx=ctx, new=new)
    d["cum"] = torch.from_numpy(np.concatenate([[0], np.cumsum(new)]).astype(np.int32)).cuda()
    d["past"] = torch.from_numpy((ctx - new).astype(np.int32)).cuda()
    d["cos"], d["sin"] = _rotary(maxb * blk, hd, dt)
    return d


def _block_inputs(c, seed):
    g = _gen(seed)
    dt, H, KV, hd, D = DTYPES[c["dtype"]], c["H"], c["KV"], c["hd"], c["hidden"]
    nq = (H + 2 * KV) * hd
    d = dict(x=_normal(g, (1, c["S"], D), dt), qkv=_quant(g, nq, D, 4, 32, True, dt),
             o=_quant(g, D, H * hd, 4, 32, True, dt), nq=nq)
    d["pk"] = torch.zeros((1, KV, c["S"], hd), dtype=dt, device="cuda")
    d["pv"] = torch.zeros_like(d["pk"])
    d["cos"], d["sin"] = _rotary(c["S"], hd, dt)
    return d


def _decoder_config(c):
    D, H, KV, hd, inter = LAYOUTS[c["layout"]]
    return _pkg(".decoder").DecoderConfig(layers=c["layers"], hidden=D, heads=H, kv_heads=KV,
                                          head_dim=hd, inter=inter, vocab=c["vocab"])


def _decoder_inputs(c, seed):
    """Weights with the distributions of the repository's benchmark decoder (codes
    8 + Binomial(4, 1/2) - 2, scales |N(0, 0.02)|), ids, and the cached rows."""
    g = _gen(seed)
    D, H, KV, hd, inter = LAYOUTS[c["layout"]]
    table = torch.tensor([(6 + bin(b & 15).count("1")) | ((6 + bin(b >> 4).count("1")) << 4)
                          for b in range(256)], dtype=torch.uint8, device="cuda")
    w = {"embed": _normal(g, (c["vocab"], D), torch.float16)}

    def linear(key, N, K):
        raw = torch.randint(0, 256, (N, K // 32, 16), generator=g, device="cuda",
                            dtype=torch.uint8)
        w[key + ".B"] = table[raw.int()]
        w[key + ".s"] = (torch.randn(N * (K // 32), generator=g, device="cuda").abs() *
                         0.02).half()

    for i in range(c["layers"]):
        for name, N, K in (("q", H * hd, D), ("k", KV * hd, D), ("v", KV * hd, D),
                           ("o", D, H * hd), ("gate", inter, D), ("up", inter, D),
                           ("down", D, inter)):
            linear(f"l{i}.{name}", N, K)
        w[f"l{i}.ln1"] = _normal(g, (D,), torch.float16, 0.05) + 1
        w[f"l{i}.ln2"] = _normal(g, (D,), torch.float16, 0.05) + 1
    w["final_ln"] = _normal(g, (D,), torch.float16, 0.05) + 1
    linear("lm_head", c["vocab"], D)
    w["cos"], w["sin"] = _rotary(4096, hd, torch.float16, 1e6)
    cap = c["context"] + c["S"]
    kv = [[torch.cat([_normal(g, (1, KV, c["context"], hd), torch.float16, 0.8),
                      torch.zeros((1, KV, c["S"], hd), dtype=torch.float16, device="cuda")], 2)
           for _ in range(2)] for _ in range(c["layers"])]
    ids = torch.randint(0, c["vocab"], (1, c["S"]), generator=g, device="cuda")
    return w, kv, ids, cap


# ------------------------------------------------------------- prepare and run --

def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _state(fn, args, out, keep):
    return dict(fn=fn, args=args, out=out, keep=keep, check=_pkg().check)


def prepare(case, seed):
    kind = case["kind"]
    lib = _pkg().load_kernels()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "linear":
        c = case
        A, B, s, z = t = _linear_inputs(c, seed)
        Y = torch.empty((c["M"], c["N"]), dtype=A.dtype, device="cuda")
        args = (_ptr(A), _ptr(B), _ptr(s), _ptr(z), _ptr(Y), c["M"], c["N"], c["K"], c["bits"],
                c["block"], CODES[c["dtype"]], stream)
        return _state(lib.ortmi_matmul_nbits, args, Y, t)
    if kind == "gqa":
        c = case
        d = _gqa_inputs(c, seed)
        B, S, H, KV, hd, past = c["B"], c["S"], c["H"], c["KV"], c["hd"], c["past"]
        code, total, cap = CODES[c["dtype"]], past + S, d["pk"].shape[2]
        out = torch.empty((B, S, H * hd), dtype=d["q"].dtype, device="cuda")
        if c["shared"]:
            prk, prv = d["pk"], d["pv"]
        else:
            prk = torch.empty((B, KV, total, hd), dtype=d["q"].dtype, device="cuda")
            prv = torch.empty_like(prk)
        head = (_ptr(d["q"]), _ptr(d["k"]), _ptr(d["v"]), _ptr(d["pk"]), _ptr(d["pv"]), cap,
                total, _ptr(d["cos"]), _ptr(d["sin"]), hd // 2, d["cos"].shape[0])
        tail = (_ptr(out), _ptr(prk), _ptr(prv), B, S, H, KV, hd, 0.0, 0, code)
        if c["dtype"] == "f32":
            n = lib.ortmi_group_query_attention_ex_workspace_size(B, S, H, hd)
            fn, mid = lib.ortmi_group_query_attention_ex, (None, None, 1e-6, None, 0, 0, 0, 0)
        else:
            n = lib.ortmi_group_query_attention_workspace_size(B, S, H, hd, total)
            fn, mid = lib.ortmi_group_query_attention, ()
        ws = torch.empty(max(1, n), dtype=torch.uint8, device="cuda")
        return _state(fn, head + mid + tail + (_ptr(ws), n, stream),
                      dict(out=out, present_key=prk, present_value=prv), (d, ws))
    if kind == "paged":
        c = case
        d = _paged_inputs(c, seed)
        H, KV, hd, T = c["H"], c["KV"], c["hd"], d["q"].shape[0]
        nblk, maxb, batch = d["kc"].shape[0], d["bt"].shape[1], c["nseq"]
        ctx = maxb * c["blk"]
        out = torch.empty((T, H * hd), dtype=d["q"].dtype, device="cuda")
        n = lib.ortmi_paged_attention_workspace_size(T, batch, H, KV, hd, hd, ctx)
        ws = torch.empty(max(1, n), dtype=torch.uint8, device="cuda")
        args = (_ptr(d["q"]), _ptr(d["k"]), _ptr(d["v"]), _ptr(d["kc"]), _ptr(d["vc"]), nblk,
                c["blk"], _ptr(d["cum"]), _ptr(d["past"]), _ptr(d["bt"]), batch, maxb, T, ctx,
                _ptr(d["cos"]), _ptr(d["sin"]), hd // 2, d["cos"].shape[0], 0, 0, None, None,
                None, None, 1e-6, _ptr(out), H, KV, hd, hd, 0.0, CODES[c["dtype"]], _ptr(ws), n,
                stream)
        return _state(lib.ortmi_paged_attention, args,
                      dict(out=out, key_cache=d["kc"], value_cache=d["vc"]), (d, ws))
    if kind == "block":
        return dict(block=_block_inputs(case, seed), case=case, ops=_pkg(".ops"))
    w, kv, ids, cap = _decoder_inputs(case, seed)
    w = {k: v.cpu().numpy() for k, v in w.items()}
    runner = _pkg(".decoder").DecoderRunner(_decoder_config(case), w, cap, case["S"],
                                            argmax_node=True, host_feeds=True)
    for (k, v), (rk, rv) in zip(kv, runner.kv):
        rk.copy_(k)
        rv.copy_(v)
    runner.ids_host.copy_(ids)
    return dict(runner=runner, case=case)


def run(state):
    if "fn" in state:
        state["check"](state["fn"](*state["args"]))
        return state["out"]
    if "block" in state:
        c, d, ops = state["case"], state["block"], state["ops"]
        qkv = ops.matmul_nbits(d["x"], *d["qkv"], K=c["hidden"], N=d["nq"])
        attn, k, v = ops.group_query_attention(
            qkv, None, None, d["pk"], d["pv"], None, c["S"], d["cos"], d["sin"],
            num_heads=c["H"], kv_num_heads=c["KV"], do_rotary=1, present_key=d["pk"],
            present_value=d["pv"])
        y = ops.matmul_nbits(attn, *d["o"], K=c["H"] * c["hd"], N=c["hidden"])
        return dict(y=y, present_key=k, present_value=v)
    c, runner = state["case"], state["runner"]
    runner.length = c["context"]
    runner.run(runner.ids_host, c["S"])
    return dict(logits=runner.logits, kv=[list(p) for p in runner.kv])


# --------------------------------------------------------------- work and bounds --

def _linear_bytes(M, N, K, bits, block, zp, size):
    nb = -(-K // block)
    z = (N * ((nb + 1) // 2) if bits == 4 else N * nb) if zp else 0
    return M * K * size + N * nb * block * bits // 8 + N * nb * size + z + M * N * size


def _causal_pairs(S, past):
    return S * past + S * (S + 1) // 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        return dict(bytes=_linear_bytes(c["M"], c["N"], c["K"], c["bits"], c["block"], c["zp"],
                                        SIZE[c["dtype"]]), flops=2 * c["M"] * c["N"] * c["K"])
    if kind == "gqa":
        B, S, H, KV, hd, past = (c[k] for k in ("B", "S", "H", "KV", "hd", "past"))
        sz = SIZE[c["dtype"]]
        rows = B * KV * hd * sz * 2
        written = S if c["shared"] else past + S
        return dict(bytes=rows * (past + S + written) + 2 * B * S * H * hd * sz,
                    flops=4 * B * H * hd * _causal_pairs(S, past))
    if kind == "paged":
        rng = np.random.default_rng(c["nseq"] * 7919 + c["hi"])
        ctx = rng.integers(c["lo"], c["hi"] + 1, size=c["nseq"]).tolist()
        new = [c["chunk"] if i < c["prefill"] else 1 for i in range(c["nseq"])]
        row = c["KV"] * c["hd"] * SIZE[c["dtype"]] * 2
        T = sum(new)
        return dict(bytes=row * (sum(ctx) + T) + 2 * T * c["H"] * c["hd"] * SIZE[c["dtype"]],
                    flops=4 * c["H"] * c["hd"] *
                    sum(_causal_pairs(n, x - n) for x, n in zip(ctx, new)))
    if kind == "block":
        S, D, H, KV, hd, sz = c["S"], c["hidden"], c["H"], c["KV"], c["hd"], SIZE[c["dtype"]]
        nq = (H + 2 * KV) * hd
        return dict(bytes=_linear_bytes(S, nq, D, 4, 32, True, sz) - S * nq * sz +
                    _linear_bytes(S, D, H * hd, 4, 32, True, sz) - S * H * hd * sz +
                    2 * S * KV * hd * sz,
                    flops=2 * S * D * (nq + H * hd) + 4 * H * hd * _causal_pairs(S, 0))
    D, H, KV, hd, inter = LAYOUTS[c["layout"]]
    S, past, L = c["S"], c["context"], c["layers"]
    params = L * (D * (2 * H + 2 * KV) * hd + 3 * D * inter) + c["vocab"] * D
    return dict(bytes=params * 9 // 16 + L * KV * hd * 4 * (past + 2 * S) +
                S * D * 2 + S * c["vocab"] * 2,
                flops=2 * S * params + 4 * L * H * hd * _causal_pairs(S, past))


def tolerance(case):
    """About four times the distance from 64-bit arithmetic measured on MI355X: single
    layers 2.1e-4 to 3.6e-4 in fp16, 2.2e-3 in bf16, 1.4e-7 in fp32 (where another order
    of the sums gives up to 1e-5 at long K). A block chains three of them through a
    softmax (y: 5.4e-6 in fp32, 2e-2 in bf16); the 28-layer decoder adds up 2e-3 to 4e-3."""
    if case["kind"] == "decoder":
        return {"rel": 0.015, "max": 0.3}
    if case["kind"] == "block":
        return {"f16": {"rel": 1e-2, "max": 0.3}, "bf16": {"rel": 0.03, "max": 1.0},
                "f32": {"rel": 2e-5, "max": 1e-3}}[case["dtype"]]
    return {"f16": {"rel": 1.5e-3, "max": 0.05}, "bf16": {"rel": 1e-2, "max": 0.2},
            "f32": {"rel": 1e-5, "max": 1e-3}}[case["dtype"]]


# ------------------------------------------------------------- 64-bit arithmetic --

def _dequant(q, N, K, bits, block):
    """[N, K] float64 weights of a MatMulNBits triple."""
    B, s, z = q
    nb = -(-K // block)
    if bits == 4:
        codes = torch.stack([B & 15, B >> 4], -1).reshape(N, nb, block).double()
    else:
        codes = B.reshape(N, nb, block).double()
    if z is None:
        zero = torch.full((N, nb), float(1 << (bits - 1)), dtype=torch.float64, device="cuda")
    elif bits == 4:
        z = z.reshape(N, -1)
        zero = torch.stack([z & 15, z >> 4], -1).reshape(N, -1)[:, :nb].double()
    else:
        zero = z.reshape(N, nb).double()
    w = (codes - zero[:, :, None]) * s.reshape(N, nb, 1).double()
    return w.reshape(N, nb * block)[:, :K]


def _linear64(x, q, N, K, bits=4, block=32):
    """x [.., K] float64 times the dequantised weights, some rows of N at a time."""
    step = max(1, (1 << 26) // K)
    nb = -(-K // block)
    parts = []
    for n0 in range(0, N, step):
        n1 = min(N, n0 + step)
        B, s, z = q
        part = (B[n0:n1], s.reshape(N, nb)[n0:n1],
                None if z is None else z.reshape(N, -1)[n0:n1])
        parts.append(x @ _dequant(part, n1 - n0, K, bits, block).t())
    return torch.cat(parts, -1)


def _rope64(x, cos, sin, pos0):
    """Half-split rotation of x [B, S, heads, hd] at positions pos0, pos0 + 1, ..."""
    half = cos.shape[1]
    c = cos[pos0:pos0 + x.shape[1]].double()[None, :, None]
    s = sin[pos0:pos0 + x.shape[1]].double()[None, :, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend64(q, keys, values, past):
    """q [S, H, hd], keys/values [KV, n, hd], causal behind `past` rows: [S, H, hd]."""
    S, H, hd = q.shape
    KV, n, _ = keys.shape
    out = torch.empty_like(q)
    step = max(1, (1 << 25) // max(1, n))
    for h in range(H):
        k, v = keys[h * KV // H], values[h * KV // H]
        for s0 in range(0, S, step):
            s1 = min(S, s0 + step)
            sc = (q[s0:s1, h] @ k.t()) / math.sqrt(hd)
            hide = torch.arange(n, device="cuda")[None, :] > \
                past + torch.arange(s0, s1, device="cuda")[:, None]
            out[s0:s1, h] = torch.softmax(sc.masked_fill(hide, -math.inf), -1) @ v
    return out


def _gqa64(q, k, v, pk, pv, cos, sin, past, H, KV, hd, shared):
    """(output [B, S, H * hd], present key, present value), all float64."""
    B, S = q.shape[:2]
    q = _rope64(q.double().reshape(B, S, H, hd), cos, sin, past)
    k = _rope64(k.double().reshape(B, S, KV, hd), cos, sin, past).transpose(1, 2)
    v = v.double().reshape(B, S, KV, hd).transpose(1, 2)
    keys = torch.cat([pk[:, :, :past].double(), k], 2)
    vals = torch.cat([pv[:, :, :past].double(), v], 2)
    out = torch.stack([_attend64(q[b], keys[b], vals[b], past) for b in range(B)])
    if shared and pk.shape[2] > past + S:
        keys = torch.cat([keys, pk[:, :, past + S:].double()], 2)
        vals = torch.cat([vals, pv[:, :, past + S:].double()], 2)
    return out.reshape(B, S, H * hd), keys, vals


def _norm64(x, gamma, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma.double()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        A, *q = _linear_inputs(c, seed)
        return _linear64(A.double(), q, c["N"], c["K"], c["bits"], c["block"])
    if kind == "gqa":
        d = _gqa_inputs(c, seed)
        out, k, v = _gqa64(d["q"], d["k"], d["v"], d["pk"], d["pv"], d["cos"], d["sin"],
                           c["past"], c["H"], c["KV"], c["hd"], c["shared"])
        return dict(out=out, present_key=k, present_value=v)
    if kind == "paged":
        d = _paged_inputs(c, seed)
        H, KV, hd, blk = c["H"], c["KV"], c["hd"], c["blk"]
        kc = d["kc"].double().reshape(-1, KV, hd)
        vc = d["vc"].double().reshape(-1, KV, hd)
        outs, t = [], 0
        for b in range(c["nseq"]):
            n, ctx = int(d["new"][b]), int(d["ctx"][b])
            pos = torch.arange(ctx, device="cuda")
            rows = d["bt"][b].long()[pos // blk] * blk + pos % blk
            q = _rope64(d["q"][t:t + n].double().reshape(1, n, H, hd), d["cos"], d["sin"],
                        ctx - n)[0]
            kc[rows[ctx - n:]] = _rope64(d["k"][t:t + n].double().reshape(1, n, KV, hd),
                                         d["cos"], d["sin"], ctx - n)[0]
            vc[rows[ctx - n:]] = d["v"][t:t + n].double().reshape(n, KV, hd)
            outs.append(_attend64(q, kc[rows].transpose(0, 1), vc[rows].transpose(0, 1),
                                  ctx - n).reshape(n, H * hd))
            t += n
        return dict(out=torch.cat(outs), key_cache=kc.reshape(d["kc"].shape),
                    value_cache=vc.reshape(d["vc"].shape))
    if kind == "block":
        d, H, KV, hd = _block_inputs(c, seed), c["H"], c["KV"], c["hd"]
        qkv = _linear64(d["x"].double(), d["qkv"], d["nq"], c["hidden"])
        q, k, v = qkv.split([H * hd, KV * hd, KV * hd], -1)
        a, k, v = _gqa64(q, k, v, d["pk"], d["pv"], d["cos"], d["sin"], 0, H, KV, hd, True)
        return dict(y=_linear64(a, d["o"], c["hidden"], H * hd), present_key=k, present_value=v)
    w, kv, ids, _ = _decoder_inputs(c, seed)
    D, H, KV, hd, inter = LAYOUTS[c["layout"]]
    eps, past = _decoder_config(c).eps, c["context"]

    def lin(x, key, N, K):
        return _linear64(x, (w[key + ".B"], w[key + ".s"], None), N, K)

    h = w["embed"][ids].double()
    present = []
    for i in range(c["layers"]):
        x = _norm64(h, w[f"l{i}.ln1"], eps)
        a, k, v = _gqa64(lin(x, f"l{i}.q", H * hd, D), lin(x, f"l{i}.k", KV * hd, D),
                         lin(x, f"l{i}.v", KV * hd, D), kv[i][0], kv[i][1], w["cos"], w["sin"],
                         past, H, KV, hd, True)
        present.append([k, v])
        h = h + lin(a, f"l{i}.o", D, H * hd)
        x = _norm64(h, w[f"l{i}.ln2"], eps)
        gate = lin(x, f"l{i}.gate", inter, D)
        h = h + lin(gate * torch.sigmoid(gate) * lin(x, f"l{i}.up", inter, D), f"l{i}.down", D,
                    inter)
    return dict(logits=lin(_norm64(h, w["final_ln"], eps), "lm_head", c["vocab"], D), kv=present)
