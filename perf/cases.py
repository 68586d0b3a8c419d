"""The work that users of this library have it do, as cases that can be timed and checked.

Every case goes through the C ABI of libquantlib_amd.so, called as a program calls it
(device addresses, sizes, a stream), on tensors that the program has in hand.  The
families, and what each stands for:

  sample        the tail and head of a decode step: greedy argmax over the logits of the
                active sequences, then the embedding rows of the sampled tokens
  layer_ops     the memory-bound operations of one decoder layer in their order: residual
                add + RMSNorm, RoPE with the KV-cache append, add + RMSNorm, SwiGLU
  softmax       row softmax of masked attention scores
  attn_prefill  causal attention of one fresh prompt over its own K/V rows
  attn_chunked  attention of a batch of prompt chunks over the paged KV cache
  attn_decode   one query row per sequence over the KV cache (paged, or contiguous with a
                key-split workspace for a single sequence)
  fp8_codec     quantizing a weight matrix to FP8 and dequantizing it
  fp8_gemm      activations times an FP8 weight matrix, decode rows up to prefill rows
  engine        a model step: embedding, decoder layers on fp16 or FP8 weights, logits

Sizes are those of the repository's benchmark and tests (hidden 4096, 32/8 heads of 128,
FFN 14336; hidden 2048, 32/4 heads of 64, FFN 5632) and generic ones around them.
"""
import ctypes
import math
import pathlib
import random
import sys

import torch

sys.path.insert(0, str(pathlib.Path.cwd() / "quant-lib_amd"))
import quantlib_amd as ql  # noqa: E402

DEV = "cuda"
PAGE = ql.PAGE_SIZE
EPS = 1e-5
FMAX = (448.0, 57344.0)  # E4M3, E5M2
F8 = (torch.float8_e4m3fn, torch.float8_e5m2)


# ---- the cases ------------------------------------------------------------------------------
def listed():
    return [
        # 8 active sequences, a 32000-word vocabulary: the smallest call, bound by launches
        dict(name="sample_8", family="sample", seqs=8, vocab=32000, hidden=2048),
        # the benchmark's layer chain: 8192 prompt tokens of the 4096-wide layer
        dict(name="layer_ops_8192", family="layer_ops", dtype="f16", tokens=8192, heads=32, kv_heads=8,
             head_dim=128, ffn=14336, pairing=1, fused=0),
        # a causal score matrix in fp32, the reference's headline softmax size
        dict(name="softmax_f32_4096", family="softmax", dtype="f32", rows=4096, cols=4096, causal=1),
        # a long prompt: the largest attention
        dict(name="attn_prefill_8192", family="attn_prefill", tokens=8192, heads=32, kv_heads=8,
             head_dim=128, fused=0),
        # four prompts that arrive in chunks of up to 300 rows over up to 3000 keys
        dict(name="attn_chunked_4x300", family="attn_chunked", seqs=4, rows=300, ctx=3000, heads=32,
             kv_heads=8, head_dim=128, ragged=3),
        # a batch of decoding sequences, contexts of 2048 to 4096 keys
        dict(name="attn_decode_48x4096", family="attn_decode", seqs=48, ctx=4096, heads=32, kv_heads=8,
             head_dim=128, layout="paged", ragged=5),
        # one FFN matrix of the 4096-wide layer to FP8 and back (loading a model)
        dict(name="fp8_codec_14336x4096", family="fp8_codec", rows=14336, cols=4096, format=0, granularity=2,
             group=128, mode=0),
        # 24 decode rows through the FFN down projection
        dict(name="fp8_gemm_24", family="fp8_gemm", m=24, n=4096, k=14336, format=0, granularity=2, group=128,
             mode=2),
        # a 333-token prompt through the FFN up projection
        dict(name="fp8_gemm_333", family="fp8_gemm", m=333, n=14336, k=4096, format=0, granularity=2,
             group=128, mode=0),
        # one decode step of 32 sequences, fp16 weights
        dict(name="engine_decode_f16_32", family="engine", phase="decode", weights="f16", seqs=32, ctx=1500,
             rows=1, layers=2, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000, ragged=7),
        # one decode step of one sequence, FP8 weights
        dict(name="engine_decode_fp8_1", family="engine", phase="decode", weights="fp8", seqs=1, ctx=2000,
             rows=1, layers=2, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000, ragged=1,
             granularity=2, group=128, mode=2),
        # a fresh prompt of 1531 tokens, fp16 weights
        dict(name="engine_prefill_f16_1531", family="engine", phase="prefill", weights="f16", seqs=1, ctx=1531,
             rows=1531, layers=2, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000, ragged=0),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def _heads(rng):
    return rng.choice([(32, 8, 128), (32, 4, 64), (24, 8, 128), (16, 16, 64), (16, 2, 128), (28, 4, 128),
                       (12, 12, 64), (20, 4, 128)])


def draw(rng):
    family = rng.choice(["sample", "layer_ops", "layer_ops", "softmax", "attn_prefill", "attn_chunked",
                         "attn_decode", "fp8_codec", "fp8_gemm", "fp8_gemm", "fp8_gemm", "engine", "engine",
                         "engine"])
    heads, kv_heads, head_dim = _heads(rng)
    h = dict(heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    if family == "sample":
        return dict(family=family, seqs=_log(rng, 1, 128), vocab=_log(rng, 8000, 160000), hidden=heads * head_dim)
    if family == "layer_ops":
        dtype = rng.choice(["f16", "f16", "f16", "f32"])
        return dict(family=family, dtype=dtype, tokens=_log(rng, 1, 8192 if dtype == "f16" else 4096), **h,
                    ffn=_log(rng, 2 * heads * head_dim, 14336, 8), pairing=rng.choice([0, 1, 1]),
                    fused=rng.choice([0, 1]))
    if family == "softmax":
        rows = _log(rng, 64, 8192)
        return dict(family=family, dtype=rng.choice(["f16", "f32"]), rows=rows,
                    cols=min(_log(rng, 64, 16384), 2 ** 25 // rows), causal=rng.choice([0, 1]))
    if family == "attn_prefill":
        return dict(family=family, tokens=_log(rng, 32, 8192), **h, fused=rng.choice([0, 1]))
    if family == "attn_chunked":
        seqs = _log(rng, 1, 8)
        rows = _log(rng, 16, 2048 // seqs)
        return dict(family=family, seqs=seqs, rows=rows, ctx=rows + _log(rng, 16, 8192 - rows), **h,
                    ragged=rng.randrange(1000))
    if family == "attn_decode":
        seqs = _log(rng, 1, 96)
        layout = rng.choice(["paged", "contiguous"]) if seqs == 1 else "paged"
        return dict(family=family, seqs=seqs, ctx=_log(rng, 64, min(16384, 262144 // seqs)), **h, layout=layout,
                    ragged=rng.randrange(1000))
    fp8 = dict(granularity=rng.choice([1, 2, 2]), group=rng.choice([64, 128, 128]), mode=rng.choice([0, 1, 2]))
    if family == "fp8_codec":
        odd = rng.random() < 0.3
        return dict(family=family, rows=_log(rng, 256, 14336), cols=_log(rng, 512, 4096, 1 if odd else 64),
                    format=rng.choice([0, 0, 1]), granularity=rng.choice([0, 1, 2, 2]), group=fp8["group"],
                    mode=min(1, fp8["mode"]))
    if family == "fp8_gemm":
        odd = rng.random() < 0.15
        m = _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 65, 4096)
        return dict(family=family, m=m, n=_log(rng, 512, 14336, 1 if odd else 16), k=_log(rng, 512, 14336, 128),
                    format=rng.choice([0, 0, 1]), **fp8)
    # a step of some 1500 rows at most
    phase = rng.choice(["decode", "decode", "prefill", "mixed"])
    weights = rng.choice(["f16", "fp8"])
    seqs = 1 if rng.random() < 0.3 else _log(rng, 2, 64) if phase == "decode" else rng.randint(2, 6)
    rows = 1 if phase == "decode" else _log(rng, 32, 1500 // seqs)
    ctx = _log(rng, 64, 4096) if phase == "decode" else rows
    return dict(family=family, phase=phase, weights=weights, seqs=seqs, ctx=ctx, rows=rows, layers=2, **h,
                ffn=_log(rng, 2 * heads * head_dim, 14336, 128), vocab=_log(rng, 8000, 64000, 8),
                ragged=rng.randrange(1000), **(fp8 if weights == "fp8" else {}))


# ---- what a program has in hand ---------------------------------------------------------------
class Inputs:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float16, clip=None):
        x = torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32)
        if clip:
            x.clamp_(-clip, clip)
        return x.mul_(scale).to(dtype)

    def uniform(self, lo, hi, *shape, dtype=torch.float16):
        return (torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo).to(dtype)

    def permutation(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)


def _dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _lengths(case):
    """(query rows, keys) of each sequence, from the case alone."""
    r = random.Random(case["ragged"])
    got = []
    for i in range(case["seqs"]):
        first = i == 0   # one sequence has the case's own sizes, the others up to half less
        ctx = case["ctx"] if first else r.randint((case["ctx"] + 1) // 2, case["ctx"])
        rows = min(ctx, case.get("rows", 1) if first else r.randint((case.get("rows", 1) + 1) // 2, case.get("rows", 1)))
        if case["family"] == "engine":
            if case["phase"] == "prefill":
                ctx = rows
            elif case["phase"] == "mixed" and i % 2:
                rows = 1   # every other sequence of a mixed step decodes
        got.append((rows, ctx))
    return got


class Pages:
    """A paged KV cache with the sequences' blocks in a permuted order, and its device tables."""

    def __init__(self, inputs, lengths, layers, kv_heads, head_dim, zero=False):
        need = [-(-ctx // PAGE) for _, ctx in lengths]
        n = self.blocks = sum(need) + 3
        shape = (n, layers, PAGE, kv_heads, head_dim)
        if zero:
            self.k, self.v = (torch.zeros(shape, dtype=torch.float16, device=DEV) for _ in range(2))
        else:
            self.k, self.v = inputs.normal(*shape), inputs.normal(*shape)
        order = inputs.permutation(n).tolist()
        step = layers * PAGE * kv_heads * head_dim * 2
        at = torch.arange(n, dtype=torch.int64, device=DEV) * step
        self.k_table, self.v_table = at + self.k.data_ptr(), at + self.v.data_ptr()
        self.max_blocks = max(need)
        self.rows_of, tables = [], []
        for blocks in need:
            mine = [order.pop() for _ in range(blocks)]
            self.rows_of.append(mine)
            tables.append(mine + [-1] * (self.max_blocks - blocks))
        self.tables = _int32(tables)
        self.slots = [[self.rows_of[s][p // PAGE] * PAGE + p % PAGE for p in range(ctx - rows, ctx)]
                      for s, (rows, ctx) in enumerate(lengths)]

    def rows(self, pool, layer, s, count):
        """The first `count` cached rows of sequence s, [count, kv_heads, head_dim]."""
        got = pool[torch.tensor(self.rows_of[s], device=DEV), layer]
        return got.reshape(-1, *got.shape[2:])[:count]


def _scales_of(w, fmt, granularity, group, mode):
    """Scales of a weight matrix: fmax over the largest magnitude of each group.  The
    reference codec's maximum takes the elements at offsets below 32 of every 128."""
    n = w.numel()
    size = {0: n, 1: w.shape[1], 2: group}[granularity]
    pad = -n % size
    flat = torch.nn.functional.pad(w.reshape(-1).abs().float(), (0, pad)).reshape(-1, size)
    if mode != 1:
        flat = flat[:, (torch.arange(size, device=w.device) % 128) < 32]
    m = flat.amax(dim=1).double()
    return torch.where(m < 1e-8, torch.ones_like(m), FMAX[fmt] / m).float(), size


def _per_element(scales, size, shape):
    n = shape[0] * shape[1]
    return scales.repeat_interleave(size)[:n].reshape(shape) if scales.numel() > 1 else scales.expand(shape)


def _quantize(w, fmt, granularity, group, mode):
    """FP8 codes and scales of a weight matrix in plain torch: round to nearest (OCP), or the
    reference's truncating encoder without subnormals."""
    scales, size = _scales_of(w, fmt, granularity, group, mode)
    v = (w.float() * _per_element(scales, size, w.shape)).clamp_(-FMAX[fmt], FMAX[fmt])
    if mode == 1:
        return v.to(F8[fmt]).view(torch.uint8), scales
    bits, mant, bias = v.view(torch.int32), (3, 2)[fmt], (7, 15)[fmt]
    e = ((bits >> 23) & 0xFF) - 127 + bias
    code = (e << mant) | ((bits >> (23 - mant)) & ((1 << mant) - 1))
    code = torch.where(e <= 0, torch.zeros_like(code), code) | ((bits >> 24) & 0x80)
    return code.to(torch.uint8), scales


def _decoded(codes, scales, fmt, granularity, group):
    """The weights that codes and scales stand for, in 64 bits."""
    size = {0: codes.numel(), 1: codes.shape[1], 2: group}[granularity]
    return codes.view(F8[fmt]).double() / _per_element(scales.double(), size, codes.shape)


def _bytes(entry, *args):
    got = ctypes.c_size_t(0)
    ql.call(entry, *args, ctypes.byref(got))
    return got.value


def _workspace(nbytes):
    return torch.empty(max(nbytes, 256), dtype=torch.uint8, device=DEV)


class Engine:
    """A decoder-layer engine that is destroyed with its owner."""

    def __init__(self, dims, rows, seqs, ctx, fp8=None):
        h = ctypes.c_void_p()
        if fp8:
            ql.call("ql_engine_create_fp8", ctypes.byref(dims), rows, seqs, ctx, *fp8, ctypes.byref(h))
        else:
            ql.call("ql_engine_create", ctypes.byref(dims), rows, seqs, ctx, ctypes.byref(h))
        self.h = h.value

    def __del__(self):
        if getattr(self, "h", None):
            torch.cuda.synchronize()
            ql.call("ql_engine_destroy", self.h)


def prepare(case, seed):
    return {"case": case, **_PREPARE[case["family"]](case, Inputs(seed))}


def run(state):
    return _RUN[state["case"]["family"]](state, state["case"], torch.cuda.current_stream().cuda_stream)


def exact(case, seed):
    return _EXACT[case["family"]](case, prepare(case, seed))


# ---- sample -----------------------------------------------------------------------------------
def _prepare_sample(c, r):
    return dict(logits=r.normal(c["seqs"], c["vocab"], scale=3.0), table=r.normal(c["vocab"], c["hidden"]),
                tokens=torch.empty(c["seqs"], dtype=torch.int32, device=DEV),
                x=torch.empty(c["seqs"], c["hidden"], dtype=torch.float16, device=DEV))


def _run_sample(s, c, stream):
    ql.call("ql_argmax_f16", s["logits"].data_ptr(), c["seqs"], c["vocab"], c["vocab"], s["tokens"].data_ptr(), stream)
    ql.call("ql_embed_f16", s["table"].data_ptr(), s["tokens"].data_ptr(), c["seqs"], c["vocab"], c["hidden"],
            s["x"].data_ptr(), stream)
    return {"tokens": s["tokens"], "x": s["x"]}


def _exact_sample(c, s):
    first = (s["logits"] == s["logits"].amax(dim=1, keepdim=True)).int().argmax(dim=1)
    return {"tokens": None, "x": s["table"][first].double()}


# ---- layer_ops ----------------------------------------------------------------------------------
LAYERS, LAYER = 4, 2   # layers of the cache, and the one that is written
THETA = 500000.0


def _prepare_layer_ops(c, r):
    t, hd, dt = c["tokens"], c["head_dim"], _dtype(c)
    width, kv = c["heads"] * hd, c["kv_heads"] * hd
    s = dict(x=r.normal(t, width, dtype=dt), d1=r.normal(t, width, dtype=dt), d2=r.normal(t, width, dtype=dt),
             w1=r.uniform(0.5, 1.5, width, dtype=dt), w2=r.uniform(0.5, 1.5, width, dtype=dt),
             y1=torch.empty(t, width, dtype=dt, device=DEV), y2=torch.empty(t, width, dtype=dt, device=DEV),
             gate=r.normal(t, c["ffn"], dtype=dt, clip=8), up=r.normal(t, c["ffn"], dtype=dt, clip=8),
             mid=torch.empty(t, c["ffn"], dtype=dt, device=DEV))
    if c["fused"]:   # views of one projection's rows
        qkv = r.normal(t, width + 2 * kv, dtype=dt)
        s.update(q=qkv[:, :width], k=qkv[:, width:width + kv], v=qkv[:, width + kv:])
    else:
        s.update(q=r.normal(t, width, dtype=dt), k=r.normal(t, kv, dtype=dt), v=r.normal(t, kv, dtype=dt))
    if c["dtype"] == "f16":   # the paged cache
        s["pages"] = p = Pages(r, [(t, t)], LAYERS, c["kv_heads"], hd, zero=True)
        s["slots"] = _int32(p.slots[0])
    else:                     # the contiguous cache
        s["k_cache"], s["v_cache"] = (torch.zeros(LAYERS, t, c["kv_heads"], hd, device=DEV) for _ in range(2))
    return s


def _run_layer_ops(s, c, stream):
    t, h, hk, hd, dt = c["tokens"], c["heads"], c["kv_heads"], c["head_dim"], c["dtype"]
    width = h * hd
    strides = (s["q"].stride(0), s["k"].stride(0), s["v"].stride(0))
    ql.call("ql_add_rmsnorm_" + dt, s["x"].data_ptr(), s["d1"].data_ptr(), s["w1"].data_ptr(), s["y1"].data_ptr(),
            t, width, EPS, stream)
    if dt == "f16":
        p = s["pages"]
        ql.call("ql_rope_paged_kv_append_f16", s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), t, h, hk, hd,
                *strides, None, 0, THETA, c["pairing"], p.k_table.data_ptr(), p.v_table.data_ptr(), p.blocks,
                s["slots"].data_ptr(), LAYER, LAYERS, stream)
        kc, vc = p.k, p.v
    else:
        kc, vc = s["k_cache"], s["v_cache"]
        ql.call("ql_rope_kv_append_f32", s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), t, h, hk, hd,
                *strides, None, 0, THETA, c["pairing"], kc.data_ptr(), vc.data_ptr(), LAYER, 0, t, LAYERS, stream)
    ql.call("ql_add_rmsnorm_" + dt, s["x"].data_ptr(), s["d2"].data_ptr(), s["w2"].data_ptr(), s["y2"].data_ptr(),
            t, width, EPS, stream)
    ql.call("ql_swiglu_" + dt, s["gate"].data_ptr(), s["up"].data_ptr(), s["mid"].data_ptr(), t, c["ffn"], stream)
    return {"x": s["x"], "y1": s["y1"], "q": s["q"], "k": s["k"], "k_cache": kc, "v_cache": vc, "y2": s["y2"],
            "mid": s["mid"]}


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _rope64(x, heads, head_dim, pos, theta, pairing):
    """x [T, heads*head_dim] rotated at the positions pos [T]."""
    x = x.double().reshape(x.shape[0], heads, head_dim)
    i = torch.arange(head_dim // 2, device=DEV, dtype=torch.float64)
    a = pos.double()[:, None] * theta ** (-2.0 * i / head_dim)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    if pairing:
        x0, x1 = x[..., :head_dim // 2], x[..., head_dim // 2:]
        y = torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1)
    else:
        x0, x1 = x[..., 0::2], x[..., 1::2]
        y = torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1)
    return y.reshape(y.shape[0], -1)


def _exact_layer_ops(c, s):
    t, hk, hd = c["tokens"], c["kv_heads"], c["head_dim"]
    pos = torch.arange(t, device=DEV)
    x1 = s["x"].double() + s["d1"].double()
    x2 = x1 + s["d2"].double()
    k, v = _rope64(s["k"], hk, hd, pos, THETA, c["pairing"]), s["v"].double()
    if c["dtype"] == "f16":
        kc, vc = torch.zeros_like(s["pages"].k, dtype=torch.float64), torch.zeros_like(s["pages"].v, dtype=torch.float64)
        at = s["slots"].long()
        kc[at // PAGE, LAYER, at % PAGE] = k.reshape(t, hk, hd)
        vc[at // PAGE, LAYER, at % PAGE] = v.reshape(t, hk, hd)
    else:
        kc, vc = torch.zeros_like(s["k_cache"], dtype=torch.float64), torch.zeros_like(s["v_cache"], dtype=torch.float64)
        kc[LAYER], vc[LAYER] = k.reshape(t, hk, hd), v.reshape(t, hk, hd)
    g = s["gate"].double()
    return {"x": x2, "y1": _norm64(x1, s["w1"]), "q": _rope64(s["q"], c["heads"], hd, pos, THETA, c["pairing"]), "k": k,
            "k_cache": kc, "v_cache": vc, "y2": _norm64(x2, s["w2"]), "mid": g / (1 + torch.exp(-g)) * s["up"].double()}


# ---- softmax ------------------------------------------------------------------------------------
def _prepare_softmax(c, r):
    x = r.normal(c["rows"], c["cols"], scale=2.0, dtype=_dtype(c))
    if c["causal"]:
        x.masked_fill_(torch.ones_like(x, dtype=torch.bool).triu_(max(1, c["cols"] - c["rows"] + 1)), float("-inf"))
    return dict(x=x, y=torch.empty_like(x))


def _run_softmax(s, c, stream):
    ql.call("ql_softmax_" + c["dtype"], s["x"].data_ptr(), s["y"].data_ptr(), c["rows"], c["cols"], stream)
    return s["y"]


def _exact_softmax(c, s):
    return torch.softmax(s["x"].double(), dim=1)


# ---- attention ----------------------------------------------------------------------------------
def _attention64(q, k, v, heads, kv_heads):
    """q [rows, heads, d] at the last positions of k, v [keys, kv_heads, d], causal."""
    rows, keys, d = q.shape[0], k.shape[0], q.shape[2]
    out = torch.empty(rows, heads, d, dtype=torch.float64, device=DEV)
    hidden = None
    if rows > 1:
        hidden = torch.ones(rows, keys, dtype=torch.bool, device=DEV).triu_(keys - rows + 1)
    for h in range(heads):
        g = h * kv_heads // heads
        p = (q[:, h].double() @ k[:, g].double().t().contiguous()) / math.sqrt(d)
        if hidden is not None:
            p.masked_fill_(hidden, float("-inf"))
        out[:, h] = torch.softmax(p, dim=1) @ v[:, g].double().contiguous()
    return out


def _prepare_attn_prefill(c, r):
    t, hd = c["tokens"], c["head_dim"]
    width, kv = c["heads"] * hd, c["kv_heads"] * hd
    out = torch.empty(t, width, dtype=torch.float16, device=DEV)
    if c["fused"]:
        qkv = r.normal(t, width + 2 * kv)
        return dict(q=qkv[:, :width], k=qkv[:, width:width + kv], v=qkv[:, width + kv:], out=out)
    return dict(q=r.normal(t, width), k=r.normal(t, kv), v=r.normal(t, kv), out=out)


def _run_attn_prefill(s, c, stream):
    q, k, v, out, t = s["q"], s["k"], s["v"], s["out"], c["tokens"]
    if c["fused"]:
        ql.call("ql_attention_f16", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), t, t, c["heads"],
                c["kv_heads"], c["head_dim"], q.stride(0), k.stride(0), out.stride(0), 1, stream)
    else:
        ql.call("ql_flash_attention_f16", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), t, c["heads"],
                c["kv_heads"], c["head_dim"], 1, stream)
    return out


def _exact_attn_prefill(c, s):
    t, d = c["tokens"], c["head_dim"]
    return _attention64(s["q"].reshape(t, -1, d), s["k"].reshape(t, -1, d), s["v"].reshape(t, -1, d), c["heads"],
                        c["kv_heads"]).reshape(t, -1)


def _prepare_attn_chunked(c, r):
    lengths = _lengths(c)
    p = Pages(r, lengths, LAYERS, c["kv_heads"], c["head_dim"])
    cu = [0]
    for rows, _ in lengths:
        cu.append(cu[-1] + rows)
    width = c["heads"] * c["head_dim"]
    return dict(pages=p, lengths=lengths, cu=_int32(cu), ctx=_int32([x for _, x in lengths]), rows=cu[-1],
                q=r.normal(cu[-1], width), out=torch.empty(cu[-1], width, dtype=torch.float16, device=DEV))


def _run_attn_chunked(s, c, stream):
    p, width = s["pages"], c["heads"] * c["head_dim"]
    ql.call("ql_paged_attention_f16", s["q"].data_ptr(), s["out"].data_ptr(), width, width, s["rows"], c["seqs"],
            s["cu"].data_ptr(), s["ctx"].data_ptr(), max(n for n, _ in s["lengths"]), p.tables.data_ptr(), p.max_blocks,
            p.k_table.data_ptr(), p.v_table.data_ptr(), p.blocks, LAYER, LAYERS, c["heads"], c["kv_heads"],
            c["head_dim"], 1, stream)
    return s["out"]


def _exact_attn_chunked(c, s):
    p, d, at, out = s["pages"], c["head_dim"], 0, []
    for i, (rows, ctx) in enumerate(s["lengths"]):
        q = s["q"][at:at + rows].reshape(rows, -1, d)
        out.append(_attention64(q, p.rows(p.k, LAYER, i, ctx), p.rows(p.v, LAYER, i, ctx), c["heads"], c["kv_heads"]))
        at += rows
    return torch.cat(out).reshape(at, -1)


def _prepare_attn_decode(c, r):
    h, hk, hd = c["heads"], c["kv_heads"], c["head_dim"]
    s = dict(q=r.normal(c["seqs"], h * hd), out=torch.empty(c["seqs"], h * hd, dtype=torch.float16, device=DEV))
    if c["layout"] == "contiguous":
        s.update(k=r.normal(c["ctx"], hk * hd), v=r.normal(c["ctx"], hk * hd),
                 ws=_workspace(_bytes("ql_decode_attention_workspace_size", h, hk, hd, c["ctx"])))
        return s
    lengths = _lengths(c)
    s.update(pages=Pages(r, lengths, LAYERS, hk, hd), lengths=lengths, ctx=_int32([x for _, x in lengths]),
             ws=_workspace(_bytes("ql_paged_decode_workspace_size", c["seqs"], h, hk, hd, c["ctx"])))
    return s


def _run_attn_decode(s, c, stream):
    h, hk, hd, ws = c["heads"], c["kv_heads"], c["head_dim"], s["ws"]
    if c["layout"] == "contiguous":
        ql.call("ql_decode_attention_f16", s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["out"].data_ptr(),
                c["ctx"], h, hk, hd, hk * hd, ws.data_ptr(), ws.numel(), stream)
    else:
        p = s["pages"]
        ql.call("ql_paged_decode_attention_f16", s["q"].data_ptr(), s["out"].data_ptr(), h * hd, h * hd, c["seqs"],
                s["ctx"].data_ptr(), c["ctx"], p.tables.data_ptr(), p.max_blocks, p.k_table.data_ptr(),
                p.v_table.data_ptr(), p.blocks, LAYER, LAYERS, h, hk, hd, ws.data_ptr(), ws.numel(), stream)
    return s["out"]


def _exact_attn_decode(c, s):
    h, hk, d = c["heads"], c["kv_heads"], c["head_dim"]
    if c["layout"] == "contiguous":
        return _attention64(s["q"].reshape(1, h, d), s["k"].reshape(-1, hk, d), s["v"].reshape(-1, hk, d), h, hk).reshape(1, -1)
    p = s["pages"]
    return torch.cat([_attention64(s["q"][i:i + 1].reshape(1, h, d), p.rows(p.k, LAYER, i, ctx),
                                   p.rows(p.v, LAYER, i, ctx), h, hk) for i, (_, ctx) in enumerate(s["lengths"])]).reshape(c["seqs"], -1)


# ---- FP8 ----------------------------------------------------------------------------------------
def _prepare_fp8_codec(c, r):
    rows, cols = c["rows"], c["cols"]
    n = ctypes.c_int(0)
    ql.call("ql_fp8_num_scales", rows, cols, c["granularity"], c["group"], ctypes.byref(n))
    return dict(w=r.normal(rows, cols, scale=cols ** -0.5), codes=torch.empty(rows, cols, dtype=torch.uint8, device=DEV),
                scales=torch.empty(n.value, device=DEV), back=torch.empty(rows, cols, dtype=torch.float16, device=DEV))


def _run_fp8_codec(s, c, stream):
    how = (c["rows"], c["cols"], c["format"], c["granularity"], c["group"], c["mode"])
    ql.call("ql_fp8_quantize", s["w"].data_ptr(), *how, s["codes"].data_ptr(), s["scales"].data_ptr(), stream)
    ql.call("ql_fp8_dequantize", s["codes"].data_ptr(), s["scales"].data_ptr(), *how, s["back"].data_ptr(), stream)
    return {"codes": s["codes"], "scales": s["scales"], "back": s["back"]}


def _exact_fp8_codec(c, s):
    how = (c["format"], c["granularity"], c["group"])
    codes, scales = _quantize(s["w"], *how, c["mode"])
    return {"codes": None, "scales": scales.double(), "back": _decoded(codes, scales, *how)}


def _prepare_fp8_gemm(c, r):
    codes, scales = _quantize(r.normal(c["n"], c["k"], scale=c["k"] ** -0.5), c["format"], c["granularity"], c["group"],
                              c["mode"])
    return dict(a=r.normal(c["m"], c["k"]), codes=codes, scales=scales,
                c=torch.empty(c["m"], c["n"], dtype=torch.float16, device=DEV),
                ws=_workspace(_bytes("ql_fp8_gemm_workspace_size", c["m"], c["n"], c["k"], c["granularity"], c["group"])))


def _run_fp8_gemm(s, c, stream):
    ql.call("ql_fp8_gemm_f16", s["a"].data_ptr(), s["codes"].data_ptr(), s["scales"].data_ptr(), c["m"], c["n"], c["k"],
            c["format"], c["granularity"], c["group"], c["mode"], s["c"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(),
            stream)
    return s["c"]


def _exact_fp8_gemm(c, s):
    w = _decoded(s["codes"], s["scales"], c["format"], c["granularity"], c["group"])
    return s["a"].double() @ w.t()


# ---- engine -------------------------------------------------------------------------------------
ENGINE_MATRICES = ("wqkv", "wo", "w_gate", "w_up", "w_down")


def _matrices(c):
    hidden, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    return {"wqkv": (hidden + 2 * kv, hidden), "wo": (hidden, hidden), "w_gate": (c["ffn"], hidden),
            "w_up": (c["ffn"], hidden), "w_down": (hidden, c["ffn"])}


def _prepare_engine(c, r):
    hidden, lengths = c["heads"] * c["head_dim"], _lengths(c)
    fp8 = c["weights"] == "fp8"
    p = Pages(r, lengths, c["layers"], c["kv_heads"], c["head_dim"])
    cu, pos, slots = [0], [], []
    for (rows, ctx), at in zip(lengths, p.slots):
        cu.append(cu[-1] + rows)
        pos += range(ctx - rows, ctx)
        slots += at
    t, most = cu[-1], max(ctx for _, ctx in lengths)
    weights, structs = [], []
    for _ in range(c["layers"]):
        w = {"attn_norm": r.uniform(0.5, 1.5, hidden), "ffn_norm": r.uniform(0.5, 1.5, hidden)}
        for name, (n, k) in _matrices(c).items():
            w[name] = r.normal(n, k, scale=k ** -0.5)
            if fp8:
                w[name] = _quantize(w[name], 0, c["granularity"], c["group"], c["mode"])
        weights.append(w)
        at = {n: x.data_ptr() if torch.is_tensor(x) else ql.FP8Weight(x[0].data_ptr(), x[1].data_ptr()) for n, x in w.items()}
        if fp8:
            structs.append(ql.LayerWeightsFP8(at["attn_norm"], at["wqkv"], at["wo"], at["ffn_norm"], at["w_gate"],
                                              at["w_up"], at["w_down"], 0, c["granularity"], c["group"], c["mode"]))
        else:
            structs.append(ql.LayerWeights(at["attn_norm"], at["wqkv"], at["wo"], at["ffn_norm"], at["w_gate"],
                                           at["w_up"], at["w_down"]))
    dims = ql.LayerDims(hidden, c["heads"], c["kv_heads"], c["head_dim"], c["ffn"], THETA, EPS, ql.ROPE_HALF)
    arrays = dict(positions=_int32(pos), slots=_int32(slots), cu=_int32(cu), ctx=_int32([x for _, x in lengths]),
                  sample=_int32([n - 1 for n in cu[1:]]),
                  ids=torch.randint(0, c["vocab"], (t,), generator=r.g, device=DEV, dtype=torch.int32))
    step = ql.StepDevice(t, c["seqs"], max(n for n, _ in lengths), most, p.max_blocks, arrays["positions"].data_ptr(),
                         arrays["slots"].data_ptr(), arrays["cu"].data_ptr(), arrays["ctx"].data_ptr(),
                         p.tables.data_ptr(), p.k_table.data_ptr(), p.v_table.data_ptr(), p.blocks, c["layers"])
    return dict(pages=p, lengths=lengths, weights=weights, structs=structs, arrays=arrays, step=step, tokens=t,
                engine=Engine(dims, t, c["seqs"], most, (c["granularity"], c["group"]) if fp8 else None),
                table=r.normal(c["vocab"], hidden), lm_head=r.normal(c["vocab"], hidden, scale=hidden ** -0.5),
                final_norm=r.uniform(0.5, 1.5, hidden),
                x=torch.empty(t, hidden, dtype=torch.float16, device=DEV),
                deltas=[torch.empty(t, hidden, dtype=torch.float16, device=DEV) for _ in range(2)],
                logits=torch.empty(c["seqs"], c["vocab"], dtype=torch.float16, device=DEV))


def _run_engine(s, c, stream):
    e, a, x, deltas, step = s["engine"].h, s["arrays"], s["x"], s["deltas"], ctypes.byref(s["step"])
    layer = "ql_engine_layer_fp8" if c["weights"] == "fp8" else "ql_engine_layer_f16"
    ql.call("ql_embed_f16", s["table"].data_ptr(), a["ids"].data_ptr(), s["tokens"], c["vocab"], x.shape[1], x.data_ptr(), stream)
    for i, w in enumerate(s["structs"]):
        ql.call(layer, e, ctypes.byref(w), i, x.data_ptr(), deltas[(i + 1) & 1].data_ptr() if i else None,
                deltas[i & 1].data_ptr(), step, stream)
    last = deltas[(c["layers"] - 1) & 1]
    ql.call("ql_engine_logits_f16", e, x.data_ptr(), last.data_ptr(), s["final_norm"].data_ptr(), s["lm_head"].data_ptr(),
            c["vocab"], a["sample"].data_ptr(), c["seqs"], s["tokens"], s["logits"].data_ptr(), None, stream)
    return {"logits": s["logits"], "x": x, "k_cache": s["pages"].k, "v_cache": s["pages"].v}


def _exact_engine(c, s):
    hidden, h, hk, hd = c["heads"] * c["head_dim"], c["heads"], c["kv_heads"], c["head_dim"]
    p, a, kv = s["pages"], s["arrays"], hk * hd
    pos, at = a["positions"], a["slots"].long()
    kc, vc = p.k.double(), p.v.double()
    x = s["table"][a["ids"].long()].double()
    for i, w in enumerate(s["weights"]):
        m = {n: w[n].double() if torch.is_tensor(w[n]) else _decoded(*w[n], 0, c["granularity"], c["group"])
             for n in ENGINE_MATRICES}
        qkv = _norm64(x, w["attn_norm"]) @ m["wqkv"].t()
        q = _rope64(qkv[:, :hidden], h, hd, pos, THETA, 1).reshape(-1, h, hd)
        kc[at // PAGE, i, at % PAGE] = _rope64(qkv[:, hidden:hidden + kv], hk, hd, pos, THETA, 1).reshape(-1, hk, hd)
        vc[at // PAGE, i, at % PAGE] = qkv[:, hidden + kv:].reshape(-1, hk, hd)
        out, row = [], 0
        for n, (rows, ctx) in enumerate(s["lengths"]):
            out.append(_attention64(q[row:row + rows], p.rows(kc, i, n, ctx), p.rows(vc, i, n, ctx), h, hk))
            row += rows
        x = x + torch.cat(out).reshape(-1, hidden) @ m["wo"].t()
        y = _norm64(x, w["ffn_norm"])
        g = y @ m["w_gate"].t()
        x = x + (g / (1 + torch.exp(-g)) * (y @ m["w_up"].t())) @ m["w_down"].t()
    logits = _norm64(x[a["sample"].long()], s["final_norm"]) @ s["lm_head"].double().t()
    return {"logits": logits, "x": x, "k_cache": kc, "v_cache": vc}


# ---- what a pass cannot do without, and how far correct results may lie apart ---------------------
def _visible(lengths):
    """Query-key pairs that causal attention looks at."""
    return sum(rows * ctx - rows * (rows - 1) // 2 for rows, ctx in lengths)


def work(case):
    c, f = case, case["family"]
    if f == "sample":
        return {"bytes": c["seqs"] * (2 * c["vocab"] + 4 * c["hidden"] + 4), "flops": 0}
    if f == "layer_ops":
        size, width, kv = (2 if c["dtype"] == "f16" else 4), c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        # two add + RMSNorm (2 in, 2 out), Q in place, K to its row and the cache, V to the cache, SwiGLU
        per_token = 2 * 4 * width + 2 * width + 3 * kv + 2 * kv + 3 * c["ffn"]
        return {"bytes": size * (c["tokens"] * per_token + 2 * width), "flops": 0}
    if f == "softmax":
        return {"bytes": 2 * (2 if c["dtype"] == "f16" else 4) * c["rows"] * c["cols"], "flops": 0}
    if f == "fp8_codec":
        n = c["rows"] * c["cols"]
        scales = {0: 1, 1: c["rows"], 2: -(-n // c["group"])}[c["granularity"]]
        return {"bytes": 6 * n + 8 * scales, "flops": 0}
    if f == "fp8_gemm":
        scales = {0: 1, 1: c["n"], 2: -(-c["n"] * c["k"] // c["group"])}[c["granularity"]]
        return {"bytes": c["n"] * c["k"] + 4 * scales + 2 * c["m"] * (c["k"] + c["n"]),
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    width, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    if f == "attn_prefill":
        t = c["tokens"]
        return {"bytes": 2 * t * (2 * width + 2 * kv), "flops": 4 * width * _visible([(t, t)])}
    lengths = _lengths(c)
    rows, keys = sum(n for n, _ in lengths), sum(x for _, x in lengths)
    if f in ("attn_chunked", "attn_decode"):
        return {"bytes": 2 * (rows * 2 * width + keys * 2 * kv), "flops": 4 * width * _visible(lengths)}
    each = 1 if c["weights"] == "fp8" else 2
    weights = sum(n * k for n, k in _matrices(c).values())
    old = keys - rows   # keys read from the cache; the new rows are written to it
    per_layer = {"bytes": each * weights + 2 * 2 * kv * (old + rows), "flops": 2 * rows * weights + 4 * width * _visible(lengths)}
    return {"bytes": c["layers"] * per_layer["bytes"] + 2 * c["vocab"] * width + 2 * rows * width + 2 * c["seqs"] * c["vocab"],
            "flops": c["layers"] * per_layer["flops"] + 2 * c["seqs"] * c["vocab"] * width}


def tolerance(case):
    f = case["family"]
    if f in ("sample", "fp8_codec"):   # copies, indices and bytes; elementwise conversions
        return "exact"
    if f in ("layer_ops", "softmax"):
        # one rounding to the stored type (2^-11 in binary16) or a 32-bit sum in another order
        return {"rel": 1.2e-3, "max": 5e-3} if case["dtype"] == "f16" else {"rel": 2e-6, "max": 2e-5}
    if f == "fp8_gemm":
        # binary16 results of 32-bit sums over weights rounded to binary16 before or scaled after
        return {"rel": 1.2e-3, "max": 1e-2}
    if f.startswith("attn"):   # binary16 probabilities and results
        return {"rel": 1.2e-3, "max": 1e-2}
    return {"rel": 3e-3, "max": 2e-2}   # some ten binary16 roundings, one after the other


_PREPARE = {"sample": _prepare_sample, "layer_ops": _prepare_layer_ops, "softmax": _prepare_softmax,
            "attn_prefill": _prepare_attn_prefill, "attn_chunked": _prepare_attn_chunked,
            "attn_decode": _prepare_attn_decode, "fp8_codec": _prepare_fp8_codec, "fp8_gemm": _prepare_fp8_gemm,
            "engine": _prepare_engine}
_RUN = {"sample": _run_sample, "layer_ops": _run_layer_ops, "softmax": _run_softmax, "attn_prefill": _run_attn_prefill,
        "attn_chunked": _run_attn_chunked, "attn_decode": _run_attn_decode, "fp8_codec": _run_fp8_codec,
        "fp8_gemm": _run_fp8_gemm, "engine": _run_engine}
_EXACT = {"sample": _exact_sample, "layer_ops": _exact_layer_ops, "softmax": _exact_softmax,
          "attn_prefill": _exact_attn_prefill, "attn_chunked": _exact_attn_chunked, "attn_decode": _exact_attn_decode,
          "fp8_codec": _exact_fp8_codec, "fp8_gemm": _exact_fp8_gemm, "engine": _exact_engine}
