"""The work this library is used for, as cases that a timing or comparison program can run.

Every case goes through the primitives of `onednn_amd.dnnl` (descriptor, primitive, execute on a stream) on tensors
that are on the GPU.  `prepare` builds what a program holds before the call: seeded inputs with the distributions of
quantized layers (normal activations and weights, scales from the values' maxima), primitives, memory objects and
weights in the layout the primitive descriptor asked for.  `run` executes the primitives once.

  int8      u8 / s8 activations x s8 weights, per-column scales; f32 dst with bias, s8 dst with ReLU and a dst scale,
            or bf16 dst: the layers of an int8 network
  fp8       e4m3 x e4m3 -> bf16 with bias and the feed-forward chains (gelu + residual, swish x gate) or none
  mx        MXFP4 / MXFP8 operands (e8m0 scales per 32 k on both) -> bf16
  linear    a bf16 / f16 linear layer by the inner-product primitives: inference, or forward + backward by data +
            backward by weights (one training step of the layer)
  woq       16-bit activations x 4-bit weights with scales (and zero points) per group of k: decode and prefill
  moe       grouped matmul of a mixture-of-experts layer, fp8 / MXFP8 / MXFP4 / bf16: decode and prefill
  moe_grad  its weights' gradient (both operands grouped along k)
  attention scaled dot-product attention: decode and prefill, causal, masked or plain
  reorder   quantization of activations and weights, layout changes of weights
"""
import ctypes as C
import math

import numpy as np
import torch

from onednn_amd import cabi, dnnl

DT = cabi.DT_NAMES
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "s8": torch.int8, "u8": torch.uint8}
BITS = {name: cabi.DT_BITS[v] for name, v in DT.items() if v in cabi.DT_BITS}

# The largest pass of a kind that is drawn, in operations: what the largest listed cases cost or a little less.
MOST_OPS = {"int8": 1.1e12, "fp8": 1.92e12, "mx": 1.1e12, "linear": 1.2e12, "woq": 4e11, "moe": 4e11, "moe_grad": 6e11,
            "attention": 1.4e11}


def listed():
    return [
        # the first layer of a small int8 network: a few microseconds, latency and launch count
        dict(name="int8-small", kind="int8", M=256, N=1024, K=1024, src="u8", dst="f32", wtag="any"),
        # a large int8 layer, throughput
        dict(name="int8-large", kind="int8", M=8192, N=8192, K=8192, src="s8", dst="s8", wtag="any"),
        # feed-forward up-projection of an fp8 model at prefill, activation and residual fused
        dict(name="fp8-ffn", kind="fp8", M=4096, N=28672, K=8192, chain="gelu_residual"),
        # the block-scaled 4-bit format at the size of a large layer
        dict(name="mxfp4-large", kind="mx", M=8192, N=8192, K=8192, fmt="mxf4"),
        # one training step of a linear layer, three products and the bias gradient
        dict(name="linear-train", kind="linear", M=2048, N=14336, K=4096, dt="bf16", train=True),
        # generating one token: the 4-bit weights are read once, nothing else matters
        dict(name="woq-decode-1", kind="woq", M=1, N=14336, K=4096, group=128, dt="bf16", wdt="u4", wtag="any"),
        # the same layer for a batch of sequences
        dict(name="woq-decode-32", kind="woq", M=32, N=14336, K=4096, group=128, dt="bf16", wdt="u4", wtag="any"),
        # the same layer for a prompt
        dict(name="woq-prefill", kind="woq", M=2048, N=14336, K=4096, group=128, dt="bf16", wdt="u4", wtag="any"),
        # an expert layer at prefill: 512 tokens over 16 experts, short ragged groups
        dict(name="moe-prefill", kind="moe", rows=512, experts=16, N=8192, K=5120, fmt="f8", routing=9),
        # the weights' gradient of the same layer
        dict(name="moe-grad", kind="moe_grad", rows=512, experts=16, M=5120, N=8192, dt="bf16", routing=9),
        # causal self-attention over a prompt
        dict(name="attention-prefill", kind="attention", b=1, h=16, hk=16, sq=4096, sk=4096, d=128, dt="bf16", mask="causal"),
        # quantization of a large tensor with a scale per column
        dict(name="quantize", kind="reorder", rows=8192, cols=8192, src="f32", dst="s8", scales="column", transpose=False),
    ]


def draw(rng):
    """One more case of the ranges above."""

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def tokens(lo, hi):
        n = log(lo, hi)          # any count; a power of two as often as a ragged one
        return 1 << max(0, int(round(math.log2(n)))) if rng.random() < 0.3 else n

    def width(lo, hi, odd=16, step=64):
        n = log(lo, hi)          # a layer's width: mostly multiples of 64, now and then only of `odd`
        s = odd if rng.random() < 0.2 else step
        return max(s, n // s * s)

    while True:
        kind = rng.choice(["int8", "fp8", "mx", "linear", "woq", "woq", "moe", "moe_grad", "attention", "reorder"])
        if kind == "int8":
            src = rng.choice(["u8", "s8"])
            c = dict(kind=kind, M=tokens(16, 8192), N=width(256, 16384), K=width(256, 16384), src=src,
                     dst=rng.choice(["f32", "s8", "bf16"]), wtag=rng.choice(["any", "any", "ab"]))
        elif kind == "fp8":
            c = dict(kind=kind, M=tokens(16, 8192), N=width(512, 28672), K=width(512, 16384),
                     chain=rng.choice(["gelu_residual", "swish_gate", "none"]))
        elif kind == "mx":
            c = dict(kind=kind, M=tokens(64, 8192), N=width(512, 16384), K=width(512, 16384, odd=32),
                     fmt=rng.choice(["mxf4", "mxf8"]))
        elif kind == "linear":
            c = dict(kind=kind, M=tokens(32, 8192), N=width(512, 16384), K=width(512, 16384), dt=rng.choice(["bf16", "bf16", "f16"]),
                     train=rng.random() < 0.6)
        elif kind == "woq":
            decode = rng.random() < 0.5
            c = dict(kind=kind, M=rng.choice([1, 1, 2, 3, 4, 8, 13, 16, 24, 32]) if decode else tokens(33, 4096),
                     N=width(1024, 28672, odd=64, step=256), K=width(1024, 16384, odd=128, step=256), group=rng.choice([128, 128, 64]),
                     dt=rng.choice(["bf16", "bf16", "f16"]), wdt=rng.choice(["u4", "u4", "s4"]), wtag=rng.choice(["any", "any", "ab"]))
        elif kind == "moe":
            fmt = rng.choice(["f8", "f8", "mxf8", "mxf4", "bf16"])
            c = dict(kind=kind, rows=tokens(8, 8192), experts=rng.choice([8, 16, 32, 64, 128, 256]), N=width(512, 8192, odd=64),
                     K=width(512, 7168, odd=512, step=512), fmt=fmt, routing=rng.randrange(1000))
        elif kind == "moe_grad":
            c = dict(kind=kind, rows=tokens(64, 16384), experts=rng.choice([8, 16, 32, 64]), M=width(512, 7168), N=width(512, 8192),
                     dt=rng.choice(["bf16", "bf16", "f16"]), routing=rng.randrange(1000))
        elif kind == "attention":
            h = rng.choice([8, 16, 32])
            c = dict(kind=kind, b=rng.choice([1, 1, 2, 4, 8]), h=h, hk=rng.choice([h, h, 1]), d=rng.choice([64, 128, 128]),
                     dt=rng.choice(["bf16", "bf16", "f16"]))
            if rng.random() < 0.4:       # decode: one query (or a few), a cache of any length
                c.update(sq=rng.choice([1, 1, 4]), sk=tokens(128, 16384), mask="none")
            else:                        # prefill, possibly behind a cached prefix
                sq = tokens(64, 4096)
                c.update(sq=sq, sk=sq + (tokens(64, 2048) if rng.random() < 0.25 else 0), mask=rng.choice(["causal", "causal", "none", "buffer"]))
        else:
            c = dict(kind=kind, rows=tokens(64, 16384), cols=width(512, 16384), src=rng.choice(["f32", "bf16", "s8"]), dst="s8",
                     scales="none", transpose=False)
            if c["src"] == "s8":
                c["transpose"] = True    # weights into the layout that format_tag::any resolves to
            else:
                c.update(dst=rng.choice(["s8", "s8", "f8_e4m3"]), scales=rng.choice(["column", "tensor"]), transpose=rng.random() < 0.25)
        w = _ops_and_bytes(c)
        if w["flops"] <= MOST_OPS.get(kind, 1e12) and w["bytes"] <= 4.0e9 and max(w["flops"] / 5e14, w["bytes"] / 8e12) > 1e-7:
            return c


# ---------------------------------------------------------------------------------------------------- work and tolerance
def _routed(c):
    """Rows of every expert: a router that prefers some experts, the same for every seed of the inputs."""
    r = np.random.default_rng(c["routing"])
    p = r.gamma(4.0, size=c["experts"])
    return r.multinomial(c["rows"], p / p.sum())


def _ops_and_bytes(c):
    kind = c["kind"]
    if kind in ("int8", "fp8", "mx", "linear", "woq"):
        M, N, K = c["M"], c["N"], c["K"]
        ops = 2.0 * M * N * K
        if kind == "int8":
            b = M * K + K * N + M * N * BITS[c["dst"]] // 8 + 8 * N
        elif kind == "fp8":
            b = M * K + K * N + 2 * M * N + 2 * N + (0 if c["chain"] == "none" else 2 * M * N)
        elif kind == "mx":
            e = 4 if c["fmt"] == "mxf4" else 8
            b = (M * K + K * N) * e // 8 + (M + N) * K // 32 + 2 * M * N
        elif kind == "linear":
            b = 2 * (M * K + K * N + M * N + N)
            if c["train"]:   # src, weights, diff_dst in; dst, diff_src, diff_weights, the bias and its gradient out
                b, ops = 2 * (2 * M * K + 2 * K * N + 2 * M * N + 2 * N), 3 * ops
        else:
            g = K // c["group"]
            b = K * N // 2 + g * N * 2 + (g * N // 2 if c["wdt"] == "u4" else 0) + 2 * M * K + 2 * M * N
        return {"bytes": float(b), "flops": ops}
    if kind == "moe":
        sizes = _routed(c)
        active = int((sizes > 0).sum())
        e = {"f8": 8, "mxf8": 8, "mxf4": 4, "bf16": 16}[c["fmt"]]
        rows, N, K = c["rows"], c["N"], c["K"]
        b = (active * K * N + rows * K) * e // 8 + rows * N * 2 + 8 * c["experts"]
        b += {"f8": 4 * (rows + active * N), "bf16": 0}.get(c["fmt"], (rows + active * N) * K // 32)
        return {"bytes": float(b), "flops": 2.0 * rows * N * K}
    if kind == "moe_grad":
        b = 2 * (c["rows"] * (c["M"] + c["N"]) + c["experts"] * c["M"] * c["N"]) + 8 * c["experts"]
        return {"bytes": float(b), "flops": 2.0 * c["rows"] * c["M"] * c["N"]}
    if kind == "attention":
        b, h, hk, sq, sk, d = (c[k] for k in ("b", "h", "hk", "sq", "sk", "d"))
        pairs = sq * sk
        if c["mask"] == "causal":   # query i sees the keys up to i + sk - sq
            pairs = sq * (sk - sq) + sq * (sq + 1) // 2
        nbytes = 2 * b * d * (2 * h * sq + 2 * hk * sk) + (2 * sq * sk if c["mask"] == "buffer" else 0)
        return {"bytes": float(nbytes), "flops": 4.0 * b * h * pairs * d}
    n = c["rows"] * c["cols"]
    return {"bytes": float(n * (BITS[c["src"]] + BITS[c["dst"]]) // 8 + (4 * c["cols"] if c["scales"] == "column" else 0)), "flops": 0.0}


def work(case):
    """Bytes and operations of one pass: every input read once, every output written once."""
    return _ops_and_bytes(case)


def tolerance(case):
    """About four times what the path's results differ by from the same sums in float64 (rel: 1.7e-3 for a bf16 dst,
    2.1e-4 for f16, the rounding of dst; attention and the decompressed weights of a prefill round once more inside)."""
    kind = case["kind"]
    if kind == "reorder" or (kind == "int8" and case["dst"] == "s8"):
        return "exact"
    if kind == "int8" and case["dst"] == "f32":    # exact integer sums, three f32 operations (rel 3.3e-8, max 1.2e-7)
        return {"rel": 2e-7, "max": 5e-7}
    half = case.get("dt") == "f16"
    if kind == "attention":                        # 2.4e-3 / 1.6e-2 and 2.9e-4 / 1.5e-3
        return {"rel": 1.2e-3, "max": 6e-3} if half else {"rel": 9.4e-3, "max": 6e-2}
    if kind == "woq":                              # 2.2e-3 / 8.6e-3 and 2.7e-4 / 1.1e-3
        return {"rel": 1.1e-3, "max": 4.4e-3} if half else {"rel": 8.6e-3, "max": 3.5e-2}
    return {"rel": 8.4e-4, "max": 2e-3} if half else {"rel": 6.6e-3, "max": 1.6e-2}


# ------------------------------------------------------------------------------------------------------------ the inputs
_ENGINE = None


def _engine():
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = dnnl.engine(dnnl.gpu, torch.cuda.current_device())
    return _ENGINE


class _Gen:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


class _Memory:
    """A dnnl memory object over a torch tensor (and a second one for a grouped tensor's offsets)."""

    def __init__(self, md, tensor, offsets=None):
        self.md, self.tensor, self.offsets, self.h = md, tensor, offsets, C.c_void_p()
        if offsets is None:
            st = dnnl.lib().dnnl_memory_create(C.byref(self.h), md.h, _engine().h, C.c_void_p(tensor.data_ptr()))
        else:
            both = (C.c_void_p * 2)(tensor.data_ptr(), offsets.data_ptr())
            st = dnnl.lib().dnnl_memory_create_v2(C.byref(self.h), md.h, _engine().h, 2, both)
        if st != dnnl.success:
            raise dnnl.error(st, "memory_create")

    def __del__(self):
        dnnl.lib().dnnl_memory_destroy(self.h)


class _State:
    """Primitives with their arguments, in the order in which a pass executes them, and the tensors they write."""

    def __init__(self):
        self.stream = dnnl.stream(_engine(), hip_stream=torch.cuda.current_stream().cuda_stream)
        self.steps, self.out = [], {}

    def add(self, prim, args):
        self.steps.append((prim, args))

    def __del__(self):
        for prim, _ in self.steps:
            dnnl.lib().dnnl_primitive_destroy(prim.h)


def _md(dims, dt, tag=None, strides=None):
    if tag is None and strides is None:
        tag = {1: dnnl.tag_a, 2: dnnl.tag_ab, 3: dnnl.tag_abc, 4: dnnl.tag_abcd}[len(dims)]
    return dnnl.memory_desc(list(dims), DT[dt], tag=tag, strides=strides)


def _mem(tensor, dt, dims=None, strides=None):
    return _Memory(_md(dims or tensor.shape, dt, strides=strides), tensor)


def _empty(*shape, dtype):
    return torch.empty(shape, device="cuda", dtype=dtype)


def _in_layout(state, want_md, plain, plain_md):
    """Weights in the layout the primitive descriptor asked for: one reorder when it is not the plain one."""
    if want_md.format_kind() == plain_md.format_kind() and want_md.strides() == plain_md.strides():
        return _Memory(want_md, plain)
    out = torch.empty(want_md.get_size(), device="cuda", dtype=torch.uint8)
    src, dst = _Memory(plain_md, plain), _Memory(want_md, out)
    prim = dnnl.reorder(dnnl.reorder_primitive_desc(_engine(), plain_md, _engine(), want_md))
    prim.execute(state.stream, {dnnl.ARG_FROM: src, dnnl.ARG_TO: dst})
    torch.cuda.current_stream().synchronize()
    dnnl.lib().dnnl_primitive_destroy(prim.h)
    return dst


def _nibbles(codes):
    """Two 4-bit codes of the last dim per byte, the even one in the low half."""
    return (codes[..., 0::2] | (codes[..., 1::2] << 4)).contiguous()


def _u4_groups(w, group, dt, signed):
    """w [K][N] -> 4-bit codes per group of k and column with scales (16-bit) and zero points."""
    K, N = w.shape
    blk = w.view(K // group, group, N)
    if signed:
        scale = (blk.abs().amax(1) / 7).clamp_(min=1e-6).to(dt)
        q = (blk / scale.float()[:, None]).round_().clamp_(-8, 7).to(torch.int8).view(K, N)
        return _nibbles((q & 15).to(torch.uint8)), scale, None
    lo, hi = blk.amin(1), blk.amax(1)
    scale = ((hi - lo) / 15).clamp_(min=1e-6).to(dt)
    zp = (-lo / scale.float()).round_().clamp_(0, 15)
    q = (blk / scale.float()[:, None] + zp[:, None]).round_().clamp_(0, 15).to(torch.uint8).view(K, N)
    return _nibbles(q), scale, _nibbles(zp.to(torch.uint8))


def _e4m3(x, scale):
    return (x / scale).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)


_E2M1 = None


def _mx(x, fmt):
    """x [..., K] in blocks of 32 along K: (codes, e8m0 scales [..., K / 32])."""
    global _E2M1
    blk = x.view(*x.shape[:-1], x.shape[-1] // 32, 32)
    amax = blk.abs().amax(-1)
    e = torch.floor(torch.log2(amax.clamp(min=1e-30))) - (8 if fmt == "mxf8" else 2)
    e = e.clamp_(-127, 127)
    q = blk * torch.exp2(-e)[..., None]
    sc = (e + 127).to(torch.uint8)
    if fmt == "mxf8":
        return _e4m3(q, 1.0).view(x.shape), sc
    if _E2M1 is None:   # the midpoints between the magnitudes 0, 0.5, 1, 1.5, 2, 3, 4, 6
        _E2M1 = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
    codes = torch.bucketize(q.abs(), _E2M1).to(torch.uint8) | ((q < 0).to(torch.uint8) << 3)
    return _nibbles(codes.view(x.shape)), sc


# ------------------------------------------------------------------------------------------------------- one per kind
def _prepare_int8(c, gen, s):
    M, N, K = c["M"], c["N"], c["K"]
    x = gen.normal(M, K)
    if c["src"] == "u8":
        src = (x * 32).round_().add_(128).clamp_(0, 255).to(torch.uint8)
    else:
        src = (x * 32).round_().clamp_(-127, 127).to(torch.int8)
    del x
    w = gen.normal(K, N, std=1 / math.sqrt(K))
    wsc = (w.abs().amax(0) / 127).contiguous()
    wei = (w / wsc).round_().to(torch.int8)
    del w
    scalar = lambda v, dt: torch.tensor([v], device="cuda", dtype=dt)  # noqa: E731
    attr = dnnl.primitive_attr()
    attr.set_scales_mask(dnnl.ARG_SRC, 0)
    attr.set_scales_mask(dnnl.ARG_WEIGHTS, 2)
    args = {dnnl.ARG_SRC: _mem(src, c["src"]),
            dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC: _mem(scalar(1 / 32, torch.float32), "f32"),
            dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS: _mem(wsc, "f32")}
    if c["src"] == "u8":
        attr.set_zero_points_mask(dnnl.ARG_SRC, 0)
        args[dnnl.ARG_ATTR_ZERO_POINTS | dnnl.ARG_SRC] = _mem(scalar(128, torch.int32), "s32")
    bias_md = None
    if c["dst"] == "s8":
        attr.set_scales_mask(dnnl.ARG_DST, 0)
        args[dnnl.ARG_ATTR_SCALES | dnnl.ARG_DST] = _mem(scalar(4 / 127, torch.float32), "f32")
        po = dnnl.post_ops()
        po.append_eltwise(cabi.ELTWISE["relu"])
        attr.set_post_ops(po)
    else:
        bias = gen.normal(1, N)
        bias_md = _md((1, N), "f32")
        args[dnnl.ARG_BIAS] = _Memory(bias_md, bias)
    plain_md = _md((K, N), "s8")
    wei_md = plain_md if c["wtag"] == "ab" else _md((K, N), "s8", tag=dnnl.tag_any)
    dst_md = _md((M, N), c["dst"])
    pd = dnnl.matmul_primitive_desc(_engine(), _md((M, K), c["src"]), wei_md, dst_md, bias_md=bias_md, attr=attr)
    args[dnnl.ARG_WEIGHTS] = _in_layout(s, pd.query_md(dnnl.query_weights_md), wei, plain_md)
    dst = _empty(M, N, dtype=TORCH[c["dst"]])
    args[dnnl.ARG_DST] = _Memory(dst_md, dst)
    s.add(dnnl.matmul(pd), args)
    s.out["dst"] = dst


def _prepare_fp8(c, gen, s):
    M, N, K = c["M"], c["N"], c["K"]
    x = gen.normal(M, K)
    ssc = (x.abs().amax() / 448).reshape(1)
    src = _e4m3(x, ssc)
    del x
    w = gen.normal(N, K, std=1 / math.sqrt(K))     # a linear layer's [out][in], K-contiguous
    wsc = (w.abs().amax() / 448).reshape(1)
    wei = _e4m3(w, wsc)
    del w
    bias = gen.normal(1, N, std=0.1, dtype=torch.bfloat16)
    attr = dnnl.primitive_attr()
    attr.set_scales_mask(dnnl.ARG_SRC, 0)
    attr.set_scales_mask(dnnl.ARG_WEIGHTS, 0)
    dst_md, bias_md = _md((M, N), "bf16"), _md((1, N), "bf16")
    wei_md = _md((K, N), "f8_e4m3", tag=dnnl.tag_ba)
    args = {dnnl.ARG_SRC: _Memory(_md((M, K), "f8_e4m3"), src), dnnl.ARG_WEIGHTS: _Memory(wei_md, wei),
            dnnl.ARG_BIAS: _Memory(bias_md, bias),
            dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC: _mem(ssc, "f32"),
            dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS: _mem(wsc, "f32")}
    if c["chain"] != "none":
        other = gen.normal(M, N, dtype=torch.bfloat16)
        po = dnnl.post_ops()
        if c["chain"] == "gelu_residual":
            po.append_eltwise(cabi.ELTWISE["gelu_tanh"])
            po.append_binary(cabi.BINARY["add"], dst_md)
        else:
            po.append_eltwise(cabi.ELTWISE["swish"], 1.0)
            po.append_binary(cabi.BINARY["mul"], dst_md)
        attr.set_post_ops(po)
        args[dnnl.ARG_ATTR_MULTIPLE_POST_OP(1) | dnnl.ARG_SRC_1] = _Memory(dst_md, other)
    pd = dnnl.matmul_primitive_desc(_engine(), _md((M, K), "f8_e4m3"), wei_md, dst_md, bias_md=bias_md, attr=attr)
    dst = _empty(M, N, dtype=torch.bfloat16)
    args[dnnl.ARG_DST] = _Memory(dst_md, dst)
    s.add(dnnl.matmul(pd), args)
    s.out["dst"] = dst


def _prepare_mx(c, gen, s):
    M, N, K = c["M"], c["N"], c["K"]
    dt = "f4_e2m1" if c["fmt"] == "mxf4" else "f8_e4m3"
    src, ssc = _mx(gen.normal(M, K), c["fmt"])
    wei, wsc = _mx(gen.normal(N, K, std=1 / math.sqrt(K)), c["fmt"])
    wsc = wsc.t().contiguous()                     # [K / 32][N]
    attr = dnnl.primitive_attr()
    attr.set_scales(dnnl.ARG_SRC, 3, (1, 32), DT["e8m0"])
    attr.set_scales(dnnl.ARG_WEIGHTS, 3, (32, 1), DT["e8m0"])
    src_md, wei_md, dst_md = _md((M, K), dt), _md((K, N), dt, tag=dnnl.tag_ba), _md((M, N), "bf16")
    pd = dnnl.matmul_primitive_desc(_engine(), src_md, wei_md, dst_md, attr=attr)
    dst = _empty(M, N, dtype=torch.bfloat16)
    s.add(dnnl.matmul(pd), {
        dnnl.ARG_SRC: _Memory(src_md, src), dnnl.ARG_WEIGHTS: _Memory(wei_md, wei), dnnl.ARG_DST: _Memory(dst_md, dst),
        dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC: _Memory(_md((M, K // 32), "e8m0"), ssc),
        dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS: _Memory(_md((K // 32, N), "e8m0"), wsc)})
    s.out["dst"] = dst


def _prepare_linear(c, gen, s):
    M, N, K, dt = c["M"], c["N"], c["K"], c["dt"]
    t = TORCH[dt]
    src, wei, bias = gen.normal(M, K, dtype=t), gen.normal(N, K, std=1 / math.sqrt(K), dtype=t), gen.normal(N, std=0.1, dtype=t)
    src_md, wei_md, bias_md, dst_md = _md((M, K), dt), _md((N, K), dt), _md((N,), dt), _md((M, N), dt)
    src_m, wei_m = _Memory(src_md, src), _Memory(wei_md, wei)
    dst = _empty(M, N, dtype=t)
    fwd = dnnl.inner_product_forward_primitive_desc(
        _engine(), dnnl.forward_training if c["train"] else dnnl.forward_inference, src_md, wei_md, dst_md, bias_md=bias_md)
    s.add(dnnl.inner_product_forward(fwd), {dnnl.ARG_SRC: src_m, dnnl.ARG_WEIGHTS: wei_m, dnnl.ARG_BIAS: _Memory(bias_md, bias),
                                            dnnl.ARG_DST: _Memory(dst_md, dst)})
    s.out["dst"] = dst
    if not c["train"]:
        return
    dd_m = _Memory(dst_md, gen.normal(M, N, dtype=t))
    dsrc, dwei, dbias = _empty(M, K, dtype=t), _empty(N, K, dtype=t), _empty(N, dtype=t)
    bd = dnnl.inner_product_backward_data_primitive_desc(_engine(), src_md, wei_md, dst_md, hint_fwd_pd=fwd)
    s.add(dnnl.inner_product_backward_data(bd), {dnnl.ARG_DIFF_DST: dd_m, dnnl.ARG_WEIGHTS: wei_m,
                                                 dnnl.ARG_DIFF_SRC: _Memory(src_md, dsrc)})
    bw = dnnl.inner_product_backward_weights_primitive_desc(_engine(), src_md, wei_md, dst_md, diff_bias_md=bias_md, hint_fwd_pd=fwd)
    s.add(dnnl.inner_product_backward_weights(bw), {dnnl.ARG_DIFF_DST: dd_m, dnnl.ARG_SRC: src_m,
                                                    dnnl.ARG_DIFF_WEIGHTS: _Memory(wei_md, dwei),
                                                    dnnl.ARG_DIFF_BIAS: _Memory(bias_md, dbias)})
    s.out.update(diff_src=dsrc, diff_weights=dwei, diff_bias=dbias)


def _prepare_woq(c, gen, s):
    M, N, K, dt, group = c["M"], c["N"], c["K"], c["dt"], c["group"]
    t = TORCH[dt]
    src = gen.normal(M, K, dtype=t)
    wei, sc, zp = _u4_groups(gen.normal(K, N, std=1 / math.sqrt(K)), group, t, c["wdt"] == "s4")
    attr = dnnl.primitive_attr()
    attr.set_scales(dnnl.ARG_WEIGHTS, 3, (group, 1), DT[dt])
    args = {dnnl.ARG_SRC: _mem(src, dt), dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS: _mem(sc, dt)}
    if zp is not None:
        attr.set_zero_points(dnnl.ARG_WEIGHTS, 3, (group, 1), DT["u4"])
        args[dnnl.ARG_ATTR_ZERO_POINTS | dnnl.ARG_WEIGHTS] = _mem(zp, "u4", dims=(K // group, N))
    attr.set_fpmath_mode(dnnl.fpmath_bf16 if dt == "bf16" else dnnl.fpmath_f16, True)
    plain_md = _md((K, N), c["wdt"])
    wei_md = plain_md if c["wtag"] == "ab" else _md((K, N), c["wdt"], tag=dnnl.tag_any)
    dst_md = _md((M, N), dt)
    pd = dnnl.matmul_primitive_desc(_engine(), _md((M, K), dt), wei_md, dst_md, attr=attr)
    args[dnnl.ARG_WEIGHTS] = _in_layout(s, pd.query_md(dnnl.query_weights_md), wei, plain_md)
    dst = _empty(M, N, dtype=t)
    args[dnnl.ARG_DST] = _Memory(dst_md, dst)
    s.add(dnnl.matmul(pd), args)
    s.out["dst"] = dst


def _prepare_moe(c, gen, s):
    rows, G, N, K, fmt = c["rows"], c["experts"], c["N"], c["K"], c["fmt"]
    sizes = _routed(c)
    offs = torch.tensor(np.cumsum(sizes).astype(np.int32), device="cuda")
    dt = {"f8": "f8_e4m3", "mxf8": "f8_e4m3", "mxf4": "f4_e2m1", "bf16": "bf16"}[fmt]
    bits = BITS[dt]
    x = gen.normal(rows, K)
    kb = K * bits // 8
    wei = _empty(G, N, kb // (2 if dt == "bf16" else 1), dtype=torch.bfloat16 if dt == "bf16" else torch.uint8)
    attr, extra = dnnl.primitive_attr(), {}
    ws = None
    if fmt == "f8":
        ss = (x.abs().amax(1) / 448).contiguous()
        src = _e4m3(x, ss[:, None])
        ws = _empty(G, 1, N, dtype=torch.float32)
        attr.set_scales(dnnl.ARG_SRC, 1, (), DT["f32"])
        attr.set_scales(dnnl.ARG_WEIGHTS, 5, (), DT["f32"])
        extra[dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC] = _Memory(_md((rows, 1), "f32"), ss)
    elif fmt == "bf16":
        src = x.to(torch.bfloat16)
    else:
        src, ss = _mx(x, fmt)
        ws = _empty(G, K // 32, N, dtype=torch.uint8)
        attr.set_scales(dnnl.ARG_SRC, 3, (1, 32), DT["e8m0"])
        attr.set_scales(dnnl.ARG_WEIGHTS, 7, (32, 1), DT["e8m0"])
        extra[dnnl.ARG_ATTR_SCALES | dnnl.ARG_SRC] = _Memory(_md((rows, K // 32), "e8m0"), ss)
    del x
    for g in range(G):      # expert by expert: the f32 values of all of them would not be small
        w = gen.normal(N, K, std=1 / math.sqrt(K))
        if fmt == "f8":
            ws[g, 0] = w.abs().amax(1) / 448
            wei[g] = _e4m3(w, ws[g, 0][:, None])
        elif fmt == "bf16":
            wei[g] = w
        else:
            wei[g], sb = _mx(w, fmt)
            ws[g] = sb.t()
    if ws is not None:
        extra[dnnl.ARG_ATTR_SCALES | dnnl.ARG_WEIGHTS] = _Memory(_md(ws.shape, "f32" if fmt == "f8" else "e8m0"), ws)
    src_md, dst_md = dnnl.grouped_memory_desc([rows, K], DT[dt], 0, G), dnnl.grouped_memory_desc([rows, N], DT["bf16"], 0, G)
    wei_md = _md((G, K, N), dt, tag=dnnl.tag_acb)
    pd = dnnl.matmul_primitive_desc(_engine(), src_md, wei_md, dst_md, attr=attr)
    dst = _empty(rows, N, dtype=torch.bfloat16)
    s.add(dnnl.matmul(pd), {dnnl.ARG_SRC: _Memory(src_md, src, offs), dnnl.ARG_WEIGHTS: _Memory(wei_md, wei),
                            dnnl.ARG_DST: _Memory(dst_md, dst, offs), **extra})
    s.out["dst"] = dst


def _prepare_moe_grad(c, gen, s):
    rows, G, M, N, dt = c["rows"], c["experts"], c["M"], c["N"], c["dt"]
    t = TORCH[dt]
    offs = torch.tensor(np.cumsum(_routed(c)).astype(np.int32), device="cuda")
    src, wei = gen.normal(rows, M, dtype=t), gen.normal(rows, N, dtype=t)   # [tokens][features], both
    src_md = dnnl.grouped_memory_desc([M, rows], DT[dt], 1, G)
    wei_md = dnnl.grouped_memory_desc([rows, N], DT[dt], 0, G)
    dst_md = _md((G, M, N), dt)
    pd = dnnl.matmul_primitive_desc(_engine(), src_md, wei_md, dst_md)
    dst = _empty(G, M, N, dtype=t)
    s.add(dnnl.matmul(pd), {dnnl.ARG_SRC: _Memory(src_md, src, offs), dnnl.ARG_WEIGHTS: _Memory(wei_md, wei, offs),
                            dnnl.ARG_DST: _Memory(dst_md, dst)})
    s.out["dst"] = dst


def _prepare_attention(c, gen, s):
    b, h, hk, sq, sk, d, dt = (c[k] for k in ("b", "h", "hk", "sq", "sk", "d", "dt"))
    t = TORCH[dt]
    q, k, v = gen.normal(b, h, sq, d, dtype=t), gen.normal(b, hk, sk, d, dtype=t), gen.normal(b, hk, sk, d, dtype=t)
    q_md, v_md, dst_md = _md((b, h, sq, d), dt), _md((b, hk, sk, d), dt), _md((b, h, sq, d), dt)
    k_md = _md((b, hk, d, sk), dt, strides=[hk * sk * d, sk * d, 1, d])     # keys stored [b][hk][sk][d]
    scale_md = _md((1,), "f32")
    scale = torch.tensor([1 / math.sqrt(d)], device="cuda")
    mask_md, mask = None, None
    if c["mask"] == "buffer":      # an additive mask: a window around the diagonal, shared by all heads
        i, j = torch.arange(sq, device="cuda")[:, None] + (sk - sq), torch.arange(sk, device="cuda")[None]
        width = max(16, sk // 2)
        mask = torch.where((i - j).abs() < width, 0.0, -math.inf).to(t).view(1, 1, sq, sk).contiguous()
        mask_md = _md((1, 1, sq, sk), dt)
    mask_type = {"none": dnnl.attn_mask_undef, "buffer": dnnl.attn_mask_buffer, "causal": dnnl.attn_mask_bottom_right}[c["mask"]]
    pd = dnnl.sdpa_primitive_desc(_engine(), q_md, k_md, v_md, dst_md, mask_md=mask_md, scale_md=scale_md, kv_head_number=hk,
                                  attn_mask_type=mask_type)
    dst = _empty(b, h, sq, d, dtype=t)
    args = {dnnl.ARG_QUERIES: _Memory(q_md, q), dnnl.ARG_KEYS: _Memory(k_md, k), dnnl.ARG_VALUES: _Memory(v_md, v),
            dnnl.ARG_DST: _Memory(dst_md, dst), dnnl.ARG_SCALE: _Memory(scale_md, scale)}
    if mask is not None:
        args[dnnl.ARG_ATTN_MASK] = _Memory(mask_md, mask)
    s.add(dnnl.sdpa(pd), args)
    s.out["dst"] = dst


def _prepare_reorder(c, gen, s):
    R, N = c["rows"], c["cols"]
    x = gen.normal(R, N)
    attr, args = dnnl.primitive_attr(), {}
    if c["src"] == "s8":
        src = (x * 32).round_().clamp_(-127, 127).to(torch.int8)
    else:
        src = x.to(TORCH[c["src"]])
        most = 127 if c["dst"] == "s8" else 448
        sc = ((x.abs().amax(0) if c["scales"] == "column" else x.abs().amax().reshape(1)) / most).contiguous()
        attr.set_scales_mask(dnnl.ARG_DST, 2 if c["scales"] == "column" else 0)
        args[dnnl.ARG_ATTR_SCALES | dnnl.ARG_DST] = _mem(sc, "f32")
    del x
    src_md = _md((R, N), c["src"])
    dst_md = _md((R, N), c["dst"], strides=[1, R]) if c["transpose"] else _md((R, N), c["dst"])
    pd = dnnl.reorder_primitive_desc(_engine(), src_md, _engine(), dst_md, attr=attr)
    dst = _empty(*((N, R) if c["transpose"] else (R, N)), dtype=torch.int8 if c["dst"] == "s8" else torch.uint8)
    args.update({dnnl.ARG_FROM: _Memory(src_md, src), dnnl.ARG_TO: _Memory(dst_md, dst)})
    s.add(dnnl.reorder(pd), args)
    s.out["dst"] = dst


def prepare(case, seed):
    s = _State()
    globals()["_prepare_" + case["kind"]](case, _Gen(seed), s)
    return s


def run(state):
    for prim, args in state.steps:
        prim.execute(state.stream, args)
    return state.out
