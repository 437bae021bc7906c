"""The work the kernel library's speed is measured on: one launch per case, through the public
entry points (`unikern_amd.solve` once, `unikern_amd.launch` per pass), on device tensors that
the caller owns.

listed() is the fixed set, draw(rng) one more case from the ranges the listed ones stand for.
A case names an op spec (op, dims, dtype, layout and the conv's options); prepare() makes its
inputs and the plan a program keeps, run() is one launch, exact() the same result in binary64.
"""
import ctypes
import math

import torch

import unikern_amd as uk

# Sizes: 4096 and 11008 are the weight shapes of the Q8_0 samples, 4096^3 is the f16 sample's, and
# 512x9728x2560, 65536x256 and the 256x256x32 conv are shapes the reference publishes times for.
_LISTED = [
    # The scalar sum (the reference's reduce op) of a short vector: the smallest call, all launches.
    dict(name="reduce_65536", op="reduce", d0=1 << 16),
    # The norm of a 1000-token prefill of width 4096.
    dict(name="rmsnorm_1000x4096", op="rmsnorm", d0=1000, d1=4096),
    # Many short rows (the shape the reference times its softmax at): bound by memory.
    dict(name="softmax_65536x256", op="softmax", d0=65536, d1=256),
    # Rows of an odd length (attention scores over 5003 positions): rows start unaligned.
    dict(name="softmax_2048x5003", op="softmax", d0=2048, d1=5003),
    # The headline f16 GEMM: column-major B, whole tiles. The largest call.
    dict(name="gemm_f16_4096", op="gemm", d0=4096, d1=4096, d2=4096, dtype="fp16", layout="TN"),
    # A 1000-token prefill through a 4096 -> 11008 projection: M is no multiple of a tile.
    dict(name="gemm_f16_1000x11008x4096", op="gemm", d0=1000, d1=11008, d2=4096, dtype="fp16", layout="TN"),
    # A decode batch of 16 through the same projection: bound by reading the weights.
    dict(name="gemm_f16_16x11008x4096", op="gemm", d0=16, d1=11008, d2=4096, dtype="fp16", layout="TN"),
    # f16 in the reference's own layout (row-major B).
    dict(name="gemm_f16_nt_512x9728x2560", op="gemm", d0=512, d1=9728, d2=2560, dtype="fp16", layout="NT"),
    # f32 in the reference's own layout at a size that divides into no tile.
    dict(name="gemm_f32_nt_1000", op="gemm", d0=1000, d1=1000, d2=1000, dtype="fp32", layout="NT"),
    # The reference's conv layout (HWC, valid padding) at the larger of its published shapes.
    dict(name="conv_nt_256x256x32_k3_64", op="conv", d0=256, d1=256, d2=32, d3=3, d4=3, d5=64, dtype="fp32",
         layout="NT"),
    # One decode token through the Q8_0 4096 -> 11008 projection: bound by the weight stream.
    dict(name="q8_0_1x11008x4096", op="gemm", d0=1, d1=11008, d2=4096, dtype="q8_0", layout="TN"),
    # A 512-token prefill through a Q8_0 4096 -> 4096 projection.
    dict(name="q8_0_512x4096x4096", op="gemm", d0=512, d1=4096, d2=4096, dtype="q8_0", layout="TN"),
]

_MAX_ROW_ELEMS = 1 << 24                      # 65536 x 256
_MAX_FLOPS = {"fp16": 2 * 4096 ** 3, "fp32": 2 * 512 * 9728 * 2560, "q8_0": 2 * 512 * 4096 * 4096}
_MAX_CONV_FLOPS = 2 * 254 * 254 * 64 * 288    # the listed conv


def listed():
    return [dict(c) for c in _LISTED]


def _size(rng, lo, hi, step=64):
    """A size spread over the logarithm of [lo, hi]: half of them multiples of `step` where they
    can be (model widths), the others as they fall (odd ones among them)."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= step:
        v = v // step * step
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["rmsnorm", "softmax", "rowsum", "reduce", "channelscale", "gemm_fp16", "gemm_fp16", "gemm_fp32",
                       "conv", "q8_0_decode", "q8_0_prefill"])
    if kind in ("rmsnorm", "softmax", "rowsum", "channelscale"):
        c = _size(rng, 64, 70001)
        rows = _size(rng, 1, max(1, min(65536, _MAX_ROW_ELEMS // c)))
        return dict(op="reduce" if kind == "rowsum" else kind, d0=rows, d1=c)
    if kind == "reduce":
        return dict(op="reduce", d0=_size(rng, 4096, 1 << 25))
    if kind.startswith("gemm"):
        dt = kind[5:]
        n, k = _size(rng, 64, 11008), _size(rng, 64, 4096)
        m = _size(rng, 1, max(1, min(4096, _MAX_FLOPS[dt] // (2 * n * k))))
        return dict(op="gemm", d0=m, d1=n, d2=k, dtype=dt, layout=rng.choice(["TN", "NT"]))
    if kind.startswith("q8_0"):
        n, k = _size(rng, 64, 11008), 64 * rng.randint(1, 172)
        m = rng.randint(1, 16) if kind == "q8_0_decode" else rng.randint(17, 512)
        m = max(1, min(m, _MAX_FLOPS["q8_0"] // (2 * n * k)))
        return dict(op="gemm", d0=m, d1=n, d2=k, dtype="q8_0", layout="TN")
    while True:
        ks, ch, oc = rng.choice([1, 3, 3, 5]), _size(rng, 3, 256, 16), _size(rng, 16, 256, 16)
        h = _size(rng, 7, 256, 4)
        w = _size(rng, 7, 256, 4)
        c = dict(op="conv", d0=h, d1=w, d2=ch, d3=ks, d4=ks, d5=oc, dtype="fp32", layout=rng.choice(["NCHW", "NCHW", "NT"]))
        if c["layout"] == "NCHW":
            c.update(batch=rng.randint(1, 8), pad=rng.choice([0, ks // 2]), stride=rng.choice([1, 1, 2]),
                     epilogue=rng.choice(["none", "channelscale"]))
        if work(c)["flops"] <= _MAX_CONV_FLOPS:
            return c


def _dims(case):
    return [case["d%d" % i] for i in range(6) if "d%d" % i in case]


def _desc(case):
    return uk.make_desc(case["op"], _dims(case), dtype=case.get("dtype", "fp32"), layout=case.get("layout", "NT"),
                        batch=case.get("batch", 1), pad=case.get("pad", 0), stride=case.get("stride", 1),
                        epilogue=case.get("epilogue", "none"))


def _conv_out(case):
    H, W, _, kh, kw, oc = _dims(case)
    p, s = case.get("pad", 0), case.get("stride", 1)
    return case.get("batch", 1), oc, (H + 2 * p - kh) // s + 1, (W + 2 * p - kw) // s + 1


def work(case):
    op, d = case["op"], _dims(case)
    if op == "gemm":
        m, n, k = d
        a, b, c = {"fp16": (2, 2, 2), "fp32": (4, 4, 4), "q8_0": (2, 34 / 32, 4)}[case["dtype"]]
        return {"bytes": a * m * k + b * n * k + c * m * n, "flops": 2 * m * n * k}
    if op == "conv":
        H, W, ch, kh, kw, oc = d
        nb, _, ho, wo = _conv_out(case)
        return {"bytes": 4 * (nb * H * W * ch + oc * ch * kh * kw + nb * oc * ho * wo),
                "flops": 2 * nb * oc * ho * wo * ch * kh * kw}
    if op == "reduce":
        n = math.prod(d)
        return {"bytes": 4 * n + 4 * (d[0] if len(d) == 2 else 1), "flops": n}
    rows, c = d
    return {"bytes": 8 * rows * c + (0 if op == "softmax" else 4 * c),
            "flops": {"softmax": 5, "rmsnorm": 4, "channelscale": 1}[op] * rows * c}


def tolerance(case):
    # About four times what the results measured against exact(), by the type the outputs and sums
    # are held in: f16 outputs (2.1e-4) differ by their last rounding, 32-bit sums by their order
    # (GEMM and conv 1e-7 at short sums to 1.2e-6 at K = 4096, the row family 4e-8 to 1.9e-7).
    if case["op"] == "gemm" and case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 4e-3}
    if case["op"] == "channelscale":
        return "exact"
    if case["op"] in ("gemm", "conv"):
        return {"rel": 5e-6, "max": 5e-5}
    return {"rel": 1e-6, "max": 1e-5}


def _inputs(case, seed):
    """The op's inputs on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    op, d = case["op"], _dims(case)

    def normal(*shape, dtype=torch.float32):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)

    if op == "gemm" and case["dtype"] == "q8_0":
        m, n, k = d
        q = torch.randint(-127, 128, (n, k // 32, 32), generator=g, device="cuda", dtype=torch.int8)
        s = (torch.rand((n, k // 32, 1), generator=g, device="cuda") * 9e-3 + 1e-3).half()
        return [normal(m, k, dtype=torch.float16), torch.cat([s.view(torch.uint8), q.view(torch.uint8)], dim=2).contiguous()]
    if op == "gemm":
        m, n, k = d
        dt = torch.float16 if case["dtype"] == "fp16" else torch.float32
        b = (n, k) if case["layout"] == "TN" else (k, n)
        return [torch.rand((m, k), generator=g, device="cuda").mul_(2).sub_(1).to(dt),
                torch.rand(b, generator=g, device="cuda").mul_(2).sub_(1).to(dt)]
    if op == "conv":
        H, W, ch, kh, kw, oc = d
        nchw = case["layout"] == "NCHW"
        x = normal(case["batch"], ch, H, W) if nchw else normal(H, W, ch)
        w = normal(oc, ch, kh, kw) if nchw else normal(oc, kh, kw, ch)
        return [x, w.mul_(1 / math.sqrt(ch * kh * kw))] + \
            ([normal(oc).mul_(0.1).add_(1)] if case.get("epilogue") == "channelscale" else [])
    if op == "reduce":  # positive values: the sums stay well conditioned
        return [torch.rand(d, generator=g, device="cuda")]
    x = normal(*d)
    if op == "softmax":
        return [x.mul_(8)]
    return [x, normal(d[1]).mul_(0.1).add_(1)]


def _output(case):
    op, d = case["op"], _dims(case)
    if op == "gemm":
        return torch.empty((d[0], d[1]), device="cuda", dtype=torch.float16 if case["dtype"] == "fp16" else torch.float32)
    if op == "conv":
        nb, oc, ho, wo = _conv_out(case)
        return torch.empty((nb, oc, ho, wo) if case["layout"] == "NCHW" else (oc, ho, wo), device="cuda")
    if op == "reduce":
        return torch.empty((d[0] if len(d) == 2 else 1,), device="cuda")
    return torch.empty(d, device="cuda")


class _Operand:
    """A torch tensor as a launch operand: launch() reads .ptr, a device address."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


class _State:
    def __init__(self, case, seed):
        self.desc = _desc(case)
        self.plan = uk.solve(self.desc).plan
        self.ins = [_Operand(t) for t in _inputs(case, seed)]
        self.out = _Operand(_output(case))


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    uk.launch(state.desc, state.ins, state.out, plan=state.plan, sync=False)
    return state.out.tensor


def exact(case, seed):
    op, x = case["op"], _inputs(case, seed)
    if op == "gemm":
        a = x[0].double()
        if case["dtype"] == "q8_0":
            w = x[1][:, :, 2:].view(torch.int8).double() * x[1][:, :, :2].contiguous().view(torch.float16).double()
            return a @ w.reshape(w.shape[0], -1).t().contiguous()
        b = x[1].double()
        return a @ (b.t().contiguous() if case["layout"] == "TN" else b)
    if op == "conv":
        H, W, ch, kh, kw, oc = _dims(case)
        nb, _, ho, wo = _conv_out(case)
        nchw = case["layout"] == "NCHW"
        img = x[0] if nchw else x[0].permute(2, 0, 1)[None]
        w = (x[1] if nchw else x[1].permute(0, 3, 1, 2)).double().reshape(oc, -1)
        y = torch.stack([(w @ torch.nn.functional.unfold(img[i:i + 1].double(), (kh, kw), padding=case.get("pad", 0),
                                                         stride=case.get("stride", 1))[0]).reshape(oc, ho, wo)
                         for i in range(nb)])
        if len(x) == 3:
            y = y * x[2].double()[None, :, None, None]
        return y if nchw else y[0]
    v = x[0].double()
    if op == "reduce":
        return v.sum(dim=-1) if v.dim() == 2 else v.sum().reshape(1)
    if op == "softmax":
        return torch.softmax(v, dim=-1)
    if op == "rmsnorm":
        return v / torch.sqrt(v.square().mean(dim=-1, keepdim=True) + 1e-6) * x[1].double()
    return v * x[1].double()
