"""The work that a user of this framework has it do, as cases that can be timed and checked.

Three paths, each through its public Python entry points:

* ZipGEMM over compressed weights (`zipgemm`): one decode step's (or one prefill chunk's) projections
  through some layers, from the re-tiled layout and from the canonical streams;
* decode attention over compressed KV caches (`flash_attn_with_kvcache_zipserv`);
* the GPU codec: weights and KV caches compressed, weights decompressed for a dense consumer.

Weights are N(0, 0.02) with 0.1% of the entries scaled by 30 and KV caches N(0, 1) times a log-normal
scale per channel, the distributions that the benchmark uses.  A case that reads weights or caches holds
enough layers, where that is possible, that a pass finds them in HBM and not in the 256 MB cache in front
of it, as a whole model's pass does.
"""
import math

import torch

import zipserv_asplos26_amd as zs
from zipserv_asplos26_amd import attention as za

# the five projections of one decoder layer (qkv, o, gate, up, down), rows x columns
LAYER_8B = "6144x4096,4096x4096,14336x4096,14336x4096,4096x14336"
LAYER_70B = "10240x8192,8192x8192,28672x8192,28672x8192,8192x28672"

HEAD_DIM = 128
# compressed bytes per element of the two distributions (2 bytes over the ratios 1.4275 and 1.35)
WEIGHT_BYTES = 2 / 1.4275
KV_BYTES = 2 / 1.35


def listed():
    return [
        # One user's decode step at the smallest projection: launch- and latency-bound calls.
        dict(name="gemm_o_8b_n1", kind="gemm", fmt="retiled", shapes="4096x4096", layers=8, n=1, split_k=1),
        # One user's decode step through a layer of the large model: weight bytes from HBM.
        dict(name="gemm_layer_70b_n1", kind="gemm", fmt="retiled", shapes=LAYER_70B, layers=1, n=1, split_k=1),
        # A decode step of a small batch, split along K as the small model's shapes want it.
        dict(name="gemm_layer_8b_n16", kind="gemm", fmt="retiled", shapes=LAYER_8B, layers=2, n=16, split_k=4),
        # A decode step of a large batch of a ragged size.
        dict(name="gemm_layer_8b_n100", kind="gemm", fmt="retiled", shapes=LAYER_8B, layers=2, n=100, split_k=2),
        # A prefill chunk of a ragged length through an MLP's up and down projections: compute-bound.
        dict(name="gemm_mlp_8b_n500", kind="gemm", fmt="retiled", shapes="14336x4096,4096x14336", layers=1, n=500,
             split_k=1),
        # A decode step over the interchange format's own streams.
        dict(name="gemm_canonical_8b_n8", kind="gemm", fmt="canonical", shapes=LAYER_8B, layers=2, n=8, split_k=1),
        # One user with a long context, in a few layers.
        dict(name="attn_b1_t16k", kind="attn", fmt="retiled", layout="by_kv_head", batch=1, tokens=16384,
             ragged=False, heads=32, kv_heads=8, layers=4),
        # A batch of equally long contexts: cache bytes from HBM.
        dict(name="attn_b16_t8k", kind="attn", fmt="retiled", layout="by_kv_head", batch=16, tokens=8190,
             ragged=False, heads=64, kv_heads=8, layers=1),
        # A serving batch with contexts of all lengths, in the layout that a server appends to.
        dict(name="attn_token_major_b32", kind="attn", fmt="retiled", layout="token_major", batch=32, tokens=4000,
             ragged=True, heads=64, kv_heads=8, layers=1),
        # The KV caches of a prefilled batch of a ragged length are compressed.
        dict(name="kv_compress_b8_t4001", kind="kv_compress", fmt="retiled", layout="by_kv_head", batch=8,
             tokens=4001, kv_heads=8),
        # A layer's weights are compressed when a model is loaded.
        dict(name="weights_compress_8b", kind="weights_compress", fmt="retiled", shapes=LAYER_8B, layers=1),
        # Weights are decompressed for a consumer that wants them dense.
        dict(name="weights_decompress_70b", kind="decompress", fmt="retiled", shapes="10240x8192,8192x8192", layers=1),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _shapes(rng, count, most):
    """`count` matrices of multiples of 64, of at most `most` elements together."""
    out = []
    for _ in range(count):
        m = 64 * _spread(rng, 8, 448)
        k = 64 * _spread(rng, 8, 448)
        while m * k > most // count:
            if m > k:
                m = max(64, m // 2 // 64 * 64)
            else:
                k = max(64, k // 2 // 64 * 64)
        out.append("%dx%d" % (m, k))
    return ",".join(out)


def _sizes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")] * case["layers"]


def _cold_layers(shapes, most):
    """Layers that hold about 130 M elements (180 MB compressed), at most `most` outputs."""
    one = sum(m * k for m, k in _sizes(dict(shapes=shapes, layers=1)))
    return max(1, min(most // (shapes.count(",") + 1), 130_000_000 // one))


def draw(rng):
    kind = rng.choice(["narrow", "narrow", "wide", "wide", "prefill", "canonical", "attn", "attn", "kv_compress",
                       "weights_compress", "decompress"])
    if kind in ("narrow", "wide", "prefill", "canonical"):
        n = {"narrow": lambda: _spread(rng, 1, 16), "wide": lambda: _spread(rng, 17, 256),
             "prefill": lambda: _spread(rng, 257, 512), "canonical": lambda: _spread(rng, 1, 128)}[kind]()
        shapes = _shapes(rng, rng.randint(1, 3), 100_000_000 if kind in ("narrow", "wide") else 50_000_000)
        layers = _cold_layers(shapes, 24) if kind in ("narrow", "wide") else 1
        split_k = rng.choice([1, 1, 2, 4])
        if n <= 16 and kind == "narrow" and rng.random() < 0.1:
            split_k = 0  # the stream-K schedule
        return dict(kind="gemm", fmt="canonical" if kind == "canonical" else "retiled", shapes=shapes, layers=layers,
                    n=n, split_k=split_k)
    if kind == "attn":
        batch = _spread(rng, 1, 48)
        tokens = _spread(rng, 100, min(32768, 100_000 // batch))
        return dict(kind="attn", fmt=rng.choice(["retiled", "retiled", "retiled", "canonical"]),
                    layout=rng.choice(["by_kv_head", "token_major"]), batch=batch, tokens=tokens,
                    ragged=rng.random() < 0.5, heads=rng.choice([32, 64]), kv_heads=8,
                    layers=max(1, min(4, 40_000 // (batch * tokens))))
    if kind == "kv_compress":
        batch = _spread(rng, 1, 32)
        return dict(kind="kv_compress", fmt=rng.choice(["retiled", "retiled", "canonical"]),
                    layout=rng.choice(["by_kv_head", "by_kv_head", "token_major"]), batch=batch,
                    tokens=_spread(rng, 64, 32768 // batch), kv_heads=8)
    shapes = _shapes(rng, rng.randint(1, 4), 150_000_000)
    return dict(kind=kind, fmt=rng.choice(["retiled", "retiled", "canonical"]), shapes=shapes, layers=1)


# --------------------------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weight(m, k, g):
    w = torch.randn(m, k, device="cuda", generator=g).mul_(0.02)
    w[torch.rand(m, k, device="cuda", generator=g) < 0.001] *= 30
    return w.to(torch.bfloat16)


def _weights(case, g):
    """The case's matrices, one at a time."""
    for m, k in _sizes(case):
        yield _weight(m, k, g)


def _activations(case, seed):
    g = _generator(seed + 7_000_003)
    return {k: torch.randn(case["n"], k, device="cuda", generator=g).to(torch.bfloat16)
            for k in sorted({k for _, k in _sizes(case)})}


def _kv(case, g):
    """One K or V cache (batch, tokens, kv_heads, 128)."""
    scale = torch.randn(case["kv_heads"], HEAD_DIM, device="cuda", generator=g).exp_()
    x = torch.randn(case["batch"], case["tokens"], case["kv_heads"], HEAD_DIM, device="cuda", generator=g)
    return x.mul_(scale).to(torch.bfloat16)


def _redrawn(x, fixed, block, g):
    """`x` (..., rows, and `fixed` dimensions after) with its blocks of `block` rows in another order and other
    signs and mantissas.  Its exponents are the same ones in all, so the streams that it is compressed into
    keep their lengths."""
    rows = x.shape[-fixed - 1] // block
    order = torch.randperm(rows, device="cuda", generator=g)
    rows *= block
    at = (torch.arange(rows, device="cuda").view(-1, block)[order]).view(-1)
    bits = x.view(torch.int16).clone()
    dim = x.dim() - fixed - 1
    bits.narrow(dim, 0, rows).copy_(x.view(torch.int16).index_select(dim, at))
    other = torch.randint(-(1 << 15), 1 << 15, bits.shape, device="cuda", generator=g, dtype=torch.int16)
    return (bits.bitwise_and_(0x7F80).bitwise_or_(other.bitwise_and_(-(1 << 15) + 0x7F))).view(torch.bfloat16)


def _lengths(case):
    """Valid tokens of each sequence: all, or spread evenly up to all."""
    b, t = case["batch"], case["tokens"]
    if not case["ragged"]:
        return [t] * b
    lens = [max(1, t * (i + 1) // b) for i in range(b)]
    return lens[::2] + lens[1::2][::-1]


def _query(case, seed):
    g = _generator(seed + 7_000_003)
    return [torch.randn(case["batch"], 1, case["heads"], HEAD_DIM, device="cuda", generator=g).to(torch.bfloat16)
            for _ in range(case["layers"])]


def prepare(case, seed):
    g, kind = _generator(seed), case["kind"]
    state = dict(case=case)
    if kind == "gemm":
        compress = zs.compress_retiled if case["fmt"] == "retiled" else zs.compress
        state["x"] = _activations(case, seed)
        state["weights"] = [compress(w, window="weights") for w in _weights(case, g)]
    elif kind == "attn":
        state["q"] = _query(case, seed)
        state["kv"] = [tuple(za.compress_kv(_kv(case, g), case["layout"], retiled=case["fmt"] == "retiled")
                             for _ in range(2)) for _ in range(case["layers"])]
        state["lens"] = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda") if case["ragged"] else None
    elif kind == "kv_compress":
        base = _generator(1)
        state["kv"] = [_redrawn(_kv(case, base), 2, 64, g) for _ in range(2)]
    elif kind == "weights_compress":
        state["weights"] = [_redrawn(w, 1, 64, g) for w in _weights(case, _generator(1))]
    else:
        compress = zs.compress_retiled if case["fmt"] == "retiled" else zs.compress
        state["weights"] = [compress(w, window="weights") for w in _weights(case, g)]
    return state


# --------------------------------------------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------------------------------------------
def _streams(c):
    """Everything a compressed matrix holds, its streams at their own lengths."""
    if isinstance(c, zs.ZipservRetiled):
        return dict(fixed=c.fixed, exps=c.exps, eoff=c.eoff, start_exp=c.start_exp, outliers=c.num_outliers)
    return dict(sign_mantissa=c.sign_mantissa[: c.total_high_freq],
                full=c.compressed_full[: c.total_full].view(torch.int16), bitmap1=c.bitmap1, bitmap2=c.bitmap2,
                bitmap3=c.bitmap3, median=c.tile_offsets_median, tiles=c.tile_offsets_global,
                start_exp=c.start_exp, max_hf=c.max_high_freq_count, max_full=c.max_full_count)


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "gemm":
        return [zs.zipgemm(c, state["x"][c.cols], split_k=case["split_k"]) for c in state["weights"]]
    if kind == "attn":
        return [za.flash_attn_with_kvcache_zipserv(q, k, v, case["kv_heads"], case["tokens"], state["lens"],
                                                   return_softmax_lse=True)
                for q, (k, v) in zip(state["q"], state["kv"])]
    if kind == "kv_compress":
        return [_streams(za.compress_kv(x, case["layout"], retiled=case["fmt"] == "retiled")) for x in state["kv"]]
    if kind == "weights_compress":
        if case["fmt"] == "retiled":
            return [_streams(c) for c in zs.compress_retiled_many(state["weights"], window="weights")]
        return [_streams(zs.compress(w, window="weights")) for w in state["weights"]]
    decompress = zs.decompress_retiled if case["fmt"] == "retiled" else zs.decompress
    return [decompress(c) for c in state["weights"]]


# --------------------------------------------------------------------------------------------------------------
# What a pass has to move and compute, and how exact it is
# --------------------------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "gemm":
        n, sizes = case["n"], _sizes(case)
        return {"bytes": sum(WEIGHT_BYTES * m * k + 2 * n * (m + k) for m, k in sizes),
                "flops": sum(2 * n * m * k for m, k in sizes)}
    if kind == "attn":
        tokens, heads = sum(_lengths(case)), case["heads"]
        read = 2 * tokens * case["kv_heads"] * HEAD_DIM * KV_BYTES
        ends = 4 * case["batch"] * heads * HEAD_DIM + 4 * case["batch"] * heads
        return {"bytes": case["layers"] * (read + ends), "flops": case["layers"] * 4 * tokens * heads * HEAD_DIM}
    if kind == "kv_compress":
        n = 2 * case["batch"] * case["tokens"] * case["kv_heads"] * HEAD_DIM
        return {"bytes": n * (2 + KV_BYTES), "flops": 0}
    return {"bytes": sum(m * k for m, k in _sizes(case)) * (2 + WEIGHT_BYTES), "flops": 0}


def tolerance(case):
    # The codec's outputs are whole numbers, bytes and the very bf16 values that went in.  The others are bf16
    # results of fp32 sums: against `exact` a product shows 1.7e-3 (2.4e-3 with its bf16 split-K partial sums)
    # and attention, whose weights are rounded to bf16 before the second product, 1.7e-3.
    if case["kind"] == "gemm":
        return {"rel": 8e-3, "max": 0.04}
    if case["kind"] == "attn":
        return {"rel": 8e-3, "max": 0.05}
    return "exact"


def _exact_attention(q, k, v, lens):
    """softmax(q k / sqrt(d)) v and its log-sum-exp in float64; q (B, 1, H, D), k and v (B, T, Hkv, D)."""
    b, _, h, d = q.shape
    hk = k.shape[2]
    out = torch.zeros(b, 1, h, d, dtype=torch.float64, device=q.device)
    lse = torch.zeros(b, h, dtype=torch.float64, device=q.device)
    for i, n in enumerate(lens):
        kd = k[i, :n].double().permute(1, 2, 0).contiguous()
        vd = v[i, :n].double().permute(1, 0, 2).contiguous()
        s = torch.matmul(q[i, 0].double().view(hk, h // hk, d), kd) / math.sqrt(d)
        lse[i] = torch.logsumexp(s, -1).view(h)
        out[i, 0] = torch.matmul(torch.softmax(s, -1), vd).view(h, d)
    return out, lse


def exact(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "gemm":
        x = {k: v.double() for k, v in _activations(case, seed).items()}
        return [torch.matmul(x[w.shape[1]], w.double().t()) for w in _weights(case, g)]
    if kind == "attn":
        lens = _lengths(case)
        return [_exact_attention(q, _kv(case, g), _kv(case, g), lens) for q in _query(case, seed)]
    if kind == "decompress":
        return [w.double() for w in _weights(case, g)]
    return None  # whole numbers and bytes
