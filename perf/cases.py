"""The calls whose speed this framework is judged by, through its public entry points.

Seven families cover what a program does with it: projections of a few rows
(decode) and of many (prefill) on dense and on affine-quantized weights, the
(M, K) x (K, N) product sweep, products whose rows are not 16-byte aligned,
attention over a KV cache for one token, for a chunk of tokens and for a whole
prompt, and a decoder run under batch_invariant_mode. Sizes are those of the
package's decoder, of its benchmark and of its tests.

listed() holds fixed cases, draw() makes more of the same ranges; prepare()
makes a case's inputs on the GPU, run() is one pass, work() what a pass cannot
do without, exact() the result in 64 bits and tolerance() how far another
correct implementation at the same precision may be from it.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

# The package of the tree that is the working folder.
sys.path.insert(0, os.path.abspath("mlx-batch-invariant_amd"))

import mlx_batch_invariant as bi  # noqa: E402
from mlx_batch_invariant import decoder  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}

# (K, N) of the product sweep (the benchmark's step runs all five), of the
# decoder's projections, and of the reference's published rows.
SWEEP = ((512, 512), (4096, 4096), (4096, 11008), (11008, 4096), (4096, 32000))
PROJECTIONS = SWEEP[1:] + ((4096, 1024), (2048, 2048), (2048, 12288), (6144, 2048), (512, 512))
HEADS = ((32, 8), (32, 8), (16, 8), (8, 8))
MAX_KV = 64 * 8192  # batch x keys of the largest decode case


def listed():
    return [
        # One generated token of three sequences through a 4096-wide
        # projection with bias: the shortest calls, one after the other.
        dict(name="linear_decode", kind="linear", M=3, K=4096, N=4096, dtype="bf16", bias=True),
        # The benchmark's step: the five products of the sweep at 256 rows.
        dict(name="sweep_256", kind="sweep", M=256, dtype="bf16"),
        # The same sweep for a small batch: weights are streamed once.
        dict(name="sweep_8", kind="sweep", M=8, dtype="f16"),
        # fp32 product with alpha, beta and a bias row.
        dict(name="addmm_f32", kind="addmm", M=100, K=4096, N=4096, dtype="f32"),
        # Rows that are not a multiple of 16 bytes, every size odd.
        dict(name="ragged", kind="ragged", M=301, K=1001, N=3001, layout="kn", dtype="bf16"),
        # One token through a 4-bit projection of the decoder's MLP.
        dict(name="qlinear_decode", kind="qlinear", M=1, K=4096, N=11008, bits=4, group=64,
             dtype="bf16"),
        # A 1024-token prompt through the same 4-bit projection.
        dict(name="qlinear_prefill", kind="qlinear", M=1024, K=4096, N=11008, bits=4, group=64,
             dtype="bf16"),
        # One user's next token over a long cache: one sequence, 32/8 heads.
        dict(name="decode_b1", kind="sdpa", B=1, H=32, Hkv=8, qL=1, N=8192, D=128, mask="none",
             dtype="bf16"),
        # A full serving batch over the same cache length.
        dict(name="decode_b64", kind="sdpa", B=64, H=32, Hkv=8, qL=1, N=8192, D=128, mask="none",
             dtype="bf16"),
        # Chunked prefill: 16 rows over a cache of 4200 keys of which a boolean
        # mask shows each row those written before it.
        dict(name="chunk_16", kind="sdpa", B=1, H=32, Hkv=8, qL=16, N=4200, D=128, mask="bool",
             dtype="bf16"),
        # A 2048-token prompt, causal.
        dict(name="prefill_2048", kind="sdpa", B=1, H=32, Hkv=8, qL=2048, N=2048, D=128,
             mask="causal", dtype="bf16"),
        # Two layers and the vocabulary head of the 4096-wide decoder on eight
        # 512-token prompts, under batch_invariant_mode: logits.
        dict(name="decoder", kind="decoder", B=8, L=512, layers=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "prefill", "sweep", "addmm", "ragged", "qlinear", "qprefill",
                       "decode", "chunk", "prompt", "decoder"))
    dtype16 = rng.choice(("bf16", "bf16", "f16"))
    if kind in ("linear", "prefill"):
        K, N = rng.choice(PROJECTIONS)
        M = _log_int(rng, 1, 64) if kind == "linear" else _log_int(rng, 65, 2048)
        return dict(kind="linear", M=M, K=K, N=N, dtype=dtype16, bias=rng.random() < 0.3)
    if kind == "sweep":
        return dict(kind="sweep", M=_log_int(rng, 1, 256),
                    dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
    if kind == "addmm":
        K, N = rng.choice(((512, 512), (4096, 4096), (4096, 11008), (2048, 2048)))
        return dict(kind="addmm", M=_log_int(rng, 1, 512), K=K, N=N,
                    dtype=rng.choice(("f32", "f32", "bf16")))
    if kind == "ragged":
        return dict(kind="ragged", M=_log_int(rng, 1, 1024), K=_log_int(rng, 200, 5000) | 1,
                    N=_log_int(rng, 100, 5000) | rng.choice((0, 1)),
                    layout=rng.choice(("kn", "nk")), dtype=rng.choice(("bf16", "f16", "f32")))
    if kind in ("qlinear", "qprefill"):
        K, N = rng.choice(PROJECTIONS)
        M = _log_int(rng, 1, 16) if kind == "qlinear" else _log_int(rng, 17, 1024)
        return dict(kind="qlinear", M=M, K=K, N=N, bits=rng.choice((4, 4, 8, 2)),
                    group=rng.choice((64, 64, 32, 128)), dtype=dtype16)
    if kind == "decoder":
        return dict(kind="decoder", B=_log_int(rng, 1, 8), L=_log_int(rng, 1, 512), layers=2)
    H, Hkv = rng.choice(HEADS)
    D = rng.choice((128, 128, 128, 64, 256))
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    if kind == "decode":
        B = _log_int(rng, 1, 64)
        N = _log_int(rng, 128, 8192)
        if D == 256 or dtype == "f32":  # keep the cache within the largest listed one's bytes
            N = max(128, min(N, MAX_KV // (4 * B)))
        return dict(kind="sdpa", B=B, H=H, Hkv=Hkv, qL=1, N=N, D=D,
                    mask=rng.choice(("none", "none", "bool", "additive")), dtype=dtype)
    if kind == "chunk":
        B, qL = _log_int(rng, 1, 8), _log_int(rng, 2, 32)
        return dict(kind="sdpa", B=B, H=H, Hkv=Hkv, qL=qL, N=_log_int(rng, 512, 8192), D=D,
                    mask=rng.choice(("causal", "bool", "additive")), dtype=dtype)
    L = _log_int(rng, 64, 2048)
    return dict(kind="sdpa", B=_log_int(rng, 1, max(1, 2048 // L)), H=H, Hkv=Hkv, qL=L, N=L, D=D,
                mask=rng.choice(("causal", "causal", "causal", "bool")), dtype=dtype)


# ------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rn(g, shape, dtype, std=1.0):
    t = torch.empty(shape, device="cuda", dtype=torch.float32).normal_(0.0, std, generator=g)
    return t.to(dtype)


def _weight(g, K, N, layout, dtype):
    return _rn(g, (N, K) if layout == "nk" else (K, N), dtype, K ** -0.5)


def _mask(c, g, dtype):
    """What a serving loop builds beside its cache: row s of the chunk sees the
    keys up to its own; a batch's sequences end at different cache positions,
    and the slots past them are not written yet."""
    B, qL, N = c["B"], c["qL"], c["N"]
    if c["mask"] in ("none", "causal"):
        return None if c["mask"] == "none" else "causal"
    spare = torch.randint(0, max(1, (N - qL) // 16) + 1, (B, 1, 1, 1), generator=g, device="cuda")
    rows = torch.arange(qL, device="cuda").view(1, 1, qL, 1)
    keep = torch.arange(N, device="cuda").view(1, 1, 1, N) <= rows + (N - qL) - spare
    if c["mask"] == "bool":
        return keep
    bias = _rn(g, (B, 1, qL, N), torch.float32, 0.5)
    return bias.masked_fill(~keep, float("-inf")).to(dtype)


def _decoder_weights(c, cfg, seed):
    g = _gen(seed)

    def uniform(n, k):
        t = torch.empty((n, k), device="cuda", dtype=torch.bfloat16)
        return t.uniform_(-k ** -0.5, k ** -0.5, generator=g)

    w = {"embed.weight": _rn(g, (cfg.vocab, cfg.hidden), torch.bfloat16),
         "norm.weight": 1 + _rn(g, (cfg.hidden,), torch.bfloat16, 0.1),
         "head.weight": uniform(cfg.vocab, cfg.hidden)}
    kv = cfg.kv_heads * cfg.head_dim
    qd = cfg.heads * cfg.head_dim
    for i in range(c["layers"]):
        p = "blocks.%d." % i
        w[p + "q.weight"] = uniform(qd, cfg.hidden)
        w[p + "k.weight"] = uniform(kv, cfg.hidden)
        w[p + "v.weight"] = uniform(kv, cfg.hidden)
        w[p + "o.weight"] = uniform(cfg.hidden, qd)
        w[p + "gate.weight"] = uniform(cfg.inter, cfg.hidden)
        w[p + "up.weight"] = uniform(cfg.inter, cfg.hidden)
        w[p + "down.weight"] = uniform(cfg.hidden, cfg.inter)
        w[p + "n1.weight"] = 1 + _rn(g, (cfg.hidden,), torch.bfloat16, 0.1)
        w[p + "n2.weight"] = 1 + _rn(g, (cfg.hidden,), torch.bfloat16, 0.1)
    ids = torch.randint(0, cfg.vocab, (c["B"], c["L"]), generator=g, device="cuda")
    return w, ids


def _config(c):
    return decoder.DecoderConfig(layers=c["layers"])


def prepare(c, seed):
    kind = c["kind"]
    if kind == "decoder":
        cfg = _config(c)
        w, ids = _decoder_weights(c, cfg, seed)
        model = decoder.Decoder(cfg, torch.device("meta"), torch.bfloat16)
        model.load_state_dict(w, assign=True)
        return dict(c=c, model=model.eval().requires_grad_(False), ids=ids)
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    if kind == "sdpa":
        q = _rn(g, (c["B"], c["H"], c["qL"], c["D"]), dt)
        k = _rn(g, (c["B"], c["Hkv"], c["N"], c["D"]), dt)
        v = _rn(g, (c["B"], c["Hkv"], c["N"], c["D"]), dt)
        return dict(c=c, q=q, k=k, v=v, mask=_mask(c, g, dt))
    if kind == "sweep":
        return dict(c=c, x={K: _rn(g, (c["M"], K), dt) for K in sorted({k for k, _ in SWEEP})},
                    w=[_weight(g, K, N, "kn", dt) for K, N in SWEEP])
    M, K, N = c["M"], c["K"], c["N"]
    x = _rn(g, (M, K), dt)
    if kind == "qlinear":
        words = torch.randint(-2 ** 31, 2 ** 31, (N, K * c["bits"] // 32), generator=g,
                              device="cuda").to(torch.int32)
        # A Gaussian weight's affine groups: about +-2.5 deviations over the codes.
        top = 2 ** c["bits"] - 1
        lo = -(2.5 + _rn(g, (N, K // c["group"]), torch.float32, 0.2)) * K ** -0.5
        return dict(c=c, x=x, w=words, s=(-2 * lo / top).to(dt), z=lo.to(dt))
    st = dict(c=c, x=x, w=_weight(g, K, N, c.get("layout", "nk" if kind == "linear" else "kn"), dt))
    if kind == "addmm" or c.get("bias"):
        st["b"] = _rn(g, (N,), dt)
    return st


# --------------------------------------------------------------------- pass


def run(st):
    c = st["c"]
    kind = c["kind"]
    if kind == "linear":
        return bi.linear(st["x"], st["w"], st.get("b"))
    if kind == "sweep":
        return [bi.matmul(st["x"][K], w) for (K, _), w in zip(SWEEP, st["w"])]
    if kind == "addmm":
        return bi.addmm(st["b"], st["x"], st["w"], 0.5, 2.0)
    if kind == "ragged":
        return (bi.linear if c["layout"] == "nk" else bi.matmul)(st["x"], st["w"])
    if kind == "qlinear":
        return bi.quantized_linear(st["x"], st["w"], st["s"], st["z"], c["group"], c["bits"])
    if kind == "sdpa":
        return bi.scaled_dot_product_attention(st["q"], st["k"], st["v"], mask=st["mask"])
    with torch.no_grad(), bi.batch_invariant_mode():
        return st["model"](st["ids"])


# ------------------------------------------------------------ what it needs


def _product(M, K, N, esz):
    return dict(bytes=(M * K + K * N + M * N) * esz, flops=2 * M * K * N)


def work(c):
    kind = c["kind"]
    if kind == "decoder":
        cfg = _config(c)
        h, kv, rows = cfg.hidden, cfg.kv_heads * cfg.head_dim, c["B"] * c["L"]
        qd = cfg.heads * cfg.head_dim
        layer = h * qd * 2 + h * kv * 2 + 3 * h * cfg.inter
        pairs = c["B"] * c["L"] * (c["L"] + 1) // 2
        return dict(bytes=2 * (c["layers"] * layer + cfg.vocab * h + rows * h + c["B"] * cfg.vocab),
                    flops=c["layers"] * (2 * rows * layer + 4 * pairs * qd)
                    + 2 * c["B"] * h * cfg.vocab)
    esz = BYTES[c["dtype"]]
    if kind == "sweep":
        parts = [_product(c["M"], K, N, esz) for K, N in SWEEP]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "sdpa":
        B, H, qL, N, D = c["B"], c["H"], c["qL"], c["N"], c["D"]
        by = (2 * B * c["Hkv"] * N * D + 2 * B * H * qL * D) * esz
        if c["mask"] in ("bool", "additive"):
            by += B * qL * N * (1 if c["mask"] == "bool" else esz)
        pairs = B * H * (qL * N - (qL * (qL - 1) // 2 if c["mask"] != "none" else 0))
        return dict(bytes=by, flops=4 * pairs * D)
    M, K, N = c["M"], c["K"], c["N"]
    if kind == "qlinear":
        return dict(bytes=(M * K + M * N) * 2 + N * K * c["bits"] // 8 + 2 * N * (K // c["group"]) * 2,
                    flops=2 * M * K * N)
    return _product(M, K, N, esz)


def tolerance(c):
    """Relative 2-norm, about four times the distance to the 64-bit result:
    1.7e-3 for one rounding to bf16, 2.1e-4 to f16, up to 1.4e-6 for fp32 sums
    of 11008 products; attention, which also rounds its probabilities, 2.4e-3,
    2.9e-4 and 3.5e-7. A change of rounding in the decoder's first layer
    travels through all that follow: 4.3e-3."""
    if c["kind"] == "decoder":
        return {"rel": 2e-2}
    if c["kind"] == "sdpa":
        return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 2e-6}[c["dtype"]]}
    return {"rel": {"bf16": 7e-3, "f16": 9e-4, "f32": 6e-6}[c["dtype"]]}


# ------------------------------------------------------------------- 64 bits


def _unpack(words, bits, K):
    w = words.to(torch.int64) & 0xFFFFFFFF
    sh = torch.arange(32 // bits, device=w.device, dtype=torch.int64) * bits
    return ((w.unsqueeze(-1) >> sh) & ((1 << bits) - 1)).reshape(w.shape[0], K)


def _attention(q, k, v, mask, scale=None, causal=False):
    """(H, L, D) x (Hkv, N, D): one sequence in 64 bits."""
    H, L, D = q.shape
    Hkv, N, _ = k.shape
    out = torch.empty(H, L, v.shape[-1], dtype=torch.float64, device=q.device)
    for h in range(H):
        kv = h // (H // Hkv)
        s = (q[h].double() @ k[kv].double().t().contiguous()) / math.sqrt(D)
        if causal:
            i = torch.arange(N, device=q.device)
            s = s.masked_fill(i > torch.arange(L, device=q.device)[:, None] + (N - L), -math.inf)
        if mask is not None:
            m = mask[0 if mask.shape[0] == 1 else h]
            s = s.masked_fill(~m, -math.inf) if m.dtype == torch.bool else s + m.double()
        out[h] = torch.softmax(s, -1).nan_to_num(0.0) @ v[kv].double()
    return out


def _exact_decoder(c, seed):
    cfg = _config(c)
    w, ids = _decoder_weights(c, cfg, seed)

    def lin(x, name):
        return x @ w[name + ".weight"].double().t().contiguous()

    def norm(x, name):
        return F.rms_norm(x, (cfg.hidden,), w[name + ".weight"].double(), cfg.eps)

    B, L, hd = c["B"], c["L"], cfg.head_dim
    x = w["embed.weight"][ids].double().reshape(B * L, cfg.hidden)
    for i in range(c["layers"]):
        p = "blocks.%d." % i
        y = norm(x, p + "n1")
        q, k, v = (lin(y, p + n).view(B, L, -1, hd).transpose(1, 2) for n in "qkv")
        a = torch.stack([_attention(q[b], k[b], v[b], None, causal=True) for b in range(B)])
        x = x + lin(a.transpose(1, 2).reshape(B * L, cfg.heads * hd), p + "o")
        y = norm(x, p + "n2")
        x = x + lin(F.silu(lin(y, p + "gate")) * lin(y, p + "up"), p + "down")
    return lin(norm(x.view(B, L, -1)[:, -1], "norm"), "head")


def exact(c, seed):
    kind = c["kind"]
    if kind == "decoder":
        return _exact_decoder(c, seed)
    st = prepare(c, seed)
    if kind == "sdpa":
        m = st["mask"]
        array = None if m is None or isinstance(m, str) else m
        return torch.stack([_attention(st["q"][b], st["k"][b], st["v"][b],
                                       None if array is None else array[b], causal=m == "causal")
                            for b in range(c["B"])])
    if kind == "sweep":
        return [st["x"][K].double() @ w.double() for (K, _), w in zip(SWEEP, st["w"])]
    x = st["x"].double()
    if kind == "qlinear":
        grp = c["group"]
        w = (st["s"].double().repeat_interleave(grp, 1) * _unpack(st["w"], c["bits"], c["K"])
             + st["z"].double().repeat_interleave(grp, 1))
        return x @ w.t().contiguous()
    w = st["w"].double()
    nk = kind == "linear" or c.get("layout") == "nk"
    y = x @ (w.t().contiguous() if nk else w)
    if kind == "addmm":
        return 0.5 * y + 2.0 * st["b"].double()
    return y if "b" not in st else y + st["b"].double()
