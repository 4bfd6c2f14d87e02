"""The work a user of this framework has it do, as measurable cases.

Five kinds, each through the public Python entry points on device tensors:

``awq``         one AWQ int4 linear (``quant.awq.gemm``), decode to prefill;
``moe_w4``      one MoE layer on AWQ experts from router logits
                (``blocks.moe.moe_forward_w4``), decode to prefill;
``moe_fp8``     one MoE layer on 128x128-block FP8 experts
                (``blocks.moe.moe_forward_fp8``);
``moe_fp8row``  one MoE layer on per-row FP8 experts, the checkpoint's own
                format, float32 activations (``topk_softmax`` and
                ``moe_ffn_fp8row``);
``linear``      one float32 Linear through its layer method's ``apply``:
                FP8 per row, MXFP4, MXFP8, INT8 W8A16 and INT8 W8A8.

Weights are what a model keeps after loading (re-packed once, in
``prepare``); a pass takes new activations to outputs."""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "costcut-infer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # decode GEMV of a small model: the smallest call, bound by latency
        dict(name="awq gemv", kind="awq", M=1, K=2048, N=5632, group=128, dtype="f16"),
        # a serving batch of odd size on an 8B model's MLP projection
        dict(name="awq batch 37", kind="awq", M=37, K=4096, N=14336, group=128, dtype="bf16"),
        # prompt processing on the same projection
        dict(name="awq prefill 2048", kind="awq", M=2048, K=4096, N=14336, group=128, dtype="f16"),
        # single-stream decode of an int4 MoE layer
        dict(name="moe int4 decode 1", kind="moe_w4", T=1, E=64, k=6, H=2048, I=1408, skew=0.0),
        # batched decode: the benchmark's headline workload
        dict(name="moe int4 decode 16", kind="moe_w4", T=16, E=64, k=6, H=2048, I=1408, skew=0.0),
        # a large decode batch, or a short prompt, of odd size
        dict(name="moe int4 batch 93", kind="moe_w4", T=93, E=128, k=8, H=2048, I=768, skew=0.0),
        # prefill with a skewed router: hot experts and empty ones
        dict(name="moe int4 prefill 4096", kind="moe_w4", T=4096, E=128, k=8, H=2048, I=768, skew=2.0),
        # prefill of the large block-FP8 MoE layer (11 GB of experts): the largest
        dict(name="moe fp8 prefill 2048", kind="moe_fp8", T=2048, E=256, k=8, H=7168, I=2048, skew=0.0),
        # batched decode on the checkpoint's own expert format
        dict(name="moe fp8row decode 16", kind="moe_fp8row", T=16, E=256, k=8, H=2048, I=512, skew=0.0),
        # prompt processing on a per-row FP8 linear
        dict(name="fp8 row linear 512", kind="linear", fmt="fp8row", M=512, K=4096, N=14336),
        # batched decode on an MXFP4 linear
        dict(name="mxfp4 linear 16", kind="linear", fmt="mxfp4", M=16, K=4096, N=14336),
        # prompt processing on a W8A8 attention projection
        dict(name="int8 w8a8 1024", kind="linear", fmt="w8a8", M=1024, K=4096, N=4096),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("awq", "awq", "moe_w4", "moe_w4", "moe_fp8", "moe_fp8row", "linear", "linear"))
    if kind == "awq":
        return dict(kind=kind, M=_log(rng, 1, 2048), K=128 * _log(rng, 8, 56), N=16 * _log(rng, 64, 896),
                    group=rng.choice((128, 128, 64, 32)), dtype=rng.choice(("f16", "bf16")))
    if kind == "moe_w4":
        E = _log(rng, 8, 128)
        return dict(kind=kind, T=_log(rng, 1, 4096), E=E, k=rng.randint(1, min(8, E)), H=128 * _log(rng, 8, 32),
                    I=128 * _log(rng, 4, 16), skew=rng.choice((0.0, 0.0, 2.0)))
    if kind == "moe_fp8":
        E = _log(rng, 8, 64)
        return dict(kind=kind, T=_log(rng, 1, 2048), E=E, k=rng.randint(1, min(8, E)), H=128 * _log(rng, 8, 56),
                    I=128 * _log(rng, 4, 16), skew=rng.choice((0.0, 0.0, 2.0)))
    if kind == "moe_fp8row":
        E = _log(rng, 8, 256)
        return dict(kind=kind, T=_log(rng, 1, 512), E=E, k=rng.randint(1, min(8, E)), H=256 * _log(rng, 4, 16),
                    I=256 * _log(rng, 1, 6), skew=rng.choice((0.0, 0.0, 2.0)))
    return dict(kind=kind, fmt=rng.choice(("fp8row", "mxfp4", "mxfp8", "w8a16", "w8a8")), M=_log(rng, 1, 512),
                K=128 * _log(rng, 8, 48), N=_log(rng, 512, 14336))


# ------------------------------------------------------------------ inputs --
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _words(g, *shape):
    """int32 words of eight uniform 4-bit codes."""
    return torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, device="cuda", dtype=torch.int64).to(torch.int32)


def _scales(g, *shape):
    return torch.randn(shape, generator=g, device="cuda").abs_().mul_(0.01).add_(1e-3)


def _awq(g, K: int, N: int, group: int, E: int | None = None):
    lead = () if E is None else (E,)
    return (_words(g, *lead, K, N // 8), _words(g, *lead, K // group, N // 8),
            _scales(g, *lead, K // group, N).to(torch.float16))


def _fp8(g, *shape):
    """e4m3fn bytes of N(0, 0.02), one slice of the first axis at a time."""
    w = torch.empty(shape, dtype=torch.uint8, device="cuda")
    for one in w.split(max(1, (1 << 27) // math.prod(shape[1:]))):
        one.copy_(torch.randn(one.shape, generator=g, device="cuda").mul_(0.02).to(torch.float8_e4m3fn).view(torch.uint8))
    return w


def _routed(case, g):
    lg = torch.randn((case["T"], case["E"]), generator=g, device="cuda")
    if case["skew"]:
        lg = lg + torch.randn((1, case["E"]), generator=g, device="cuda") * case["skew"]
    return lg.contiguous()


def _raw(case, seed: int) -> dict:
    """The case's inputs as a checkpoint and a model hold them."""
    g, kind = _gen(seed), case["kind"]
    if kind == "awq":
        return dict(w=_awq(g, case["K"], case["N"], case["group"]),
                    x=torch.randn((case["M"], case["K"]), generator=g, device="cuda").to(_DT[case["dtype"]]))
    if kind == "linear":
        M, K, N, fmt = case["M"], case["K"], case["N"], case["fmt"]
        x = torch.randn((M, K), generator=g, device="cuda")
        if fmt == "fp8row":
            return dict(x=x, w=_fp8(g, N, K), s=_scales(g, N).to(torch.bfloat16).float())
        if fmt in ("w8a8", "w8a16"):
            return dict(x=x, w=torch.randint(-127, 128, (N, K), generator=g, device="cuda", dtype=torch.int8),
                        s=_scales(g, N))
        e8 = torch.randint(117, 124, (N, -(-K // 32)), generator=g, device="cuda").to(torch.uint8)
        w = (_fp8(g, N, K) if fmt == "mxfp8" else
             torch.randint(0, 256, (N, K // 2), generator=g, device="cuda").to(torch.uint8))
        return dict(x=x, w=w, s=e8)
    E, H, I = case["E"], case["H"], case["I"]
    x = torch.randn((case["T"], H), generator=g, device="cuda")
    lg = _routed(case, g)
    if kind == "moe_w4":
        return dict(x=x.to(torch.bfloat16), lg=lg,
                    w=(_awq(g, H, I, 128, E), _awq(g, H, I, 128, E), _awq(g, I, H, 128, E)))
    if kind == "moe_fp8":
        one = lambda N, K: (_fp8(g, E, N, K), _scales(g, E, N // 128, K // 128))  # noqa: E731
        return dict(x=x.to(torch.bfloat16), lg=lg, w=(one(I, H), one(I, H), one(H, I)))
    one = lambda N, K: (_fp8(g, E, N, K), _scales(g, E, N).to(torch.bfloat16))  # noqa: E731
    return dict(x=x, lg=lg, w=(one(I, H), one(I, H), one(H, I)))


_KEY = {"fp8row": "fp8_static_channel_sym", "w8a8": "int8_static_channel_sym", "w8a16": "int8_static_channel_sym",
        "mxfp4": "mxfp4_dynamic", "mxfp8": "mxfp8_dynamic"}


def _method(fmt: str):
    from ccut.quant.int8 import Int8LinearMethod
    from ccut.quant.method import make_method_for_spec
    from ccut.quant.spec import LayerQuantSpec, ScaleDesc, get_quant_key

    spec = LayerQuantSpec(layer_name="mlp.up_proj", weight_key=get_quant_key(_KEY[fmt]),
                          scales=(ScaleDesc(name="weight_scale", dtype="U8" if "mx" in fmt else "F32", shape=(1,)),))
    return Int8LinearMethod(spec, compute_mode="w8a8") if fmt == "w8a8" else make_method_for_spec(spec)


def prepare(case, seed):
    from ccut.blocks import moe
    from ccut.quant import awq

    r, kind = _raw(case, seed), case["kind"]
    if kind == "awq":
        qw, qz, sc = r["w"]
        return dict(kind=kind, x=r["x"], w=awq.prepare(qw, qz, sc, case["group"]))
    if kind == "linear":
        return dict(kind=kind, x=r["x"], w=r["w"], s={"weight_scale": r["s"]}, m=_method(case["fmt"]))
    make = {"moe_w4": moe.W4Experts.from_awq, "moe_fp8": moe.Fp8Experts.from_block,
            "moe_fp8row": moe.Fp8RowExperts.from_rows}[kind]
    return dict(kind=kind, x=r["x"], lg=r["lg"], k=case["k"], ex=make(*r["w"]))


def run(state):
    from ccut.blocks import moe
    from ccut.quant import awq

    kind = state["kind"]
    if kind == "awq":
        return awq.gemm(state["x"], state["w"])
    if kind == "linear":
        return state["m"].apply(state["w"], state["s"], state["x"])
    if kind == "moe_w4":
        return moe.moe_forward_w4(state["x"], state["lg"], state["ex"], state["k"])
    if kind == "moe_fp8":
        return moe.moe_forward_fp8(state["x"], state["lg"], state["ex"], state["k"])
    w, ids = moe.topk_softmax(state["lg"], state["k"])
    return moe.moe_ffn_fp8row(state["x"], ids, w, state["ex"])


# ------------------------------------------------------------ work, bounds --
def _experts_hit(case) -> int:
    """Distinct experts that a batch of the case's routing reaches."""
    g = torch.Generator().manual_seed(1)
    lg = torch.randn((case["T"], case["E"]), generator=g)
    if case["skew"]:
        lg = lg + torch.randn((1, case["E"]), generator=g) * case["skew"]
    return lg.topk(case["k"], dim=1).indices.unique().numel()


def work(case):
    kind = case["kind"]
    if kind in ("awq", "linear"):
        M, K, N = case["M"], case["K"], case["N"]
        if kind == "awq":
            w = K * N // 2 + (K // case["group"]) * (N * 2 + N // 2)
            act = 2 * M * (K + N)
        else:
            w = {"fp8row": K * N + 4 * N, "w8a16": K * N + 4 * N, "w8a8": K * N + 4 * N,
                 "mxfp8": K * N + N * -(-K // 32), "mxfp4": K * N // 2 + N * -(-K // 32)}[case["fmt"]]
            act = 4 * M * (K + N)
        return {"bytes": w + act, "flops": 2 * M * K * N}
    T, H, I = case["T"], case["H"], case["I"]
    one = {"moe_w4": 3 * H * I // 2 + 3 * H * I // 128 * 5 // 2, "moe_fp8": 3 * H * I + 3 * (H // 128) * (I // 128) * 4,
           "moe_fp8row": 3 * H * I + 2 * (2 * I + H)}[kind]
    act = T * H * (8 if kind == "moe_fp8row" else 4) + 4 * T * case["E"]
    return {"bytes": _experts_hit(case) * one + act, "flops": 6 * T * case["k"] * H * I}


def tolerance(case):
    if case["kind"] == "awq":  # float32 sums, one rounding to the 16-bit output
        return {"rel": 1e-3, "max": 1e-2} if case["dtype"] == "f16" else {"rel": 8e-3, "max": 4e-2}
    if case["kind"] in ("moe_w4", "moe_fp8"):  # 16-bit intermediate, down rows and output
        return {"rel": 1.2e-2, "max": 1e-1}
    return {"rel": 1e-5, "max": 2e-4}  # float32 sums in another order


# ---------------------------------------------------------------- 64 bits --
_SHIFTS = (0, 16, 4, 20, 8, 24, 12, 28)  # bit of column j of eight in an AWQ word


def _nibbles(words):
    return torch.stack([(words >> s) & 15 for s in _SHIFTS], -1).reshape(*words.shape[:-1], -1).double()


def _awq_matrix(qw, qz, sc):
    group = qw.shape[0] // qz.shape[0]
    return (_nibbles(qw) - _nibbles(qz).repeat_interleave(group, 0)) * sc.double().repeat_interleave(group, 0)


def _decode8(w):
    return w.view(torch.float8_e4m3fn).double()


def _tensor_div(a: float, b):
    return torch.full_like(b, a) / b


def _quant128(x):
    """The block format's activations: e4m3fn per token per 128 channels."""
    b = x.float().reshape(x.shape[0], -1, 128)
    s = b.abs().amax(2, keepdim=True).clamp_min(1e-12)
    s = s / torch.full_like(s, 448.0)
    q = (b / s).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).reshape(x.shape)


def _blocks(w, s):
    return _decode8(w) * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)


def _moe(case, r):
    x = _quant128(r["x"]) if case["kind"] == "moe_fp8" else r["x"].double()
    v, ids = r["lg"].double().topk(case["k"], dim=1)
    wt = v.softmax(1)

    def matrix(t, e):  # [in, out]
        if case["kind"] == "moe_w4":
            return _awq_matrix(t[0][e], t[1][e], t[2][e])
        if case["kind"] == "moe_fp8":
            return _blocks(t[0][e], t[1][e]).T
        return (_decode8(t[0][e]) * t[1][e].double()[:, None]).T

    y = torch.zeros((case["T"], case["H"]), dtype=torch.float64, device="cuda")
    gate, up, down = r["w"]
    for e in ids.unique().tolist():
        t, slot = (ids == e).nonzero(as_tuple=True)
        a = x[t]
        h = torch.nn.functional.silu(a @ matrix(gate, e)) * (a @ matrix(up, e))
        y.index_add_(0, t, (h @ matrix(down, e)) * wt[t, slot, None])
    return y


def exact(case, seed):
    r, kind = _raw(case, seed), case["kind"]
    if kind == "awq":
        return r["x"].double() @ _awq_matrix(*r["w"])
    if kind != "linear":
        return _moe(case, r)
    x, w, s, fmt = r["x"], r["w"], r["s"], case["fmt"]
    if fmt == "fp8row":
        return x.double() @ (_decode8(w) * s.double()[:, None]).T
    if fmt == "w8a16":
        return x.double() @ (w.double() * s.double()[:, None]).T
    if fmt == "w8a8":  # the per-token factor 127 / (amax / 127), in float32
        xs = x.abs().amax(1, keepdim=True)
        xs = xs / torch.full_like(xs, 127.0)
        q = (x * _tensor_div(127.0, xs)).round().clamp(-127, 127)
        return (q.double() @ w.double().T) * xs.double() * s.double()[None, :]
    scale = torch.exp2(s.double() - 127).repeat_interleave(32, 1)[:, : x.shape[1]]
    if fmt == "mxfp8":
        return x.double() @ (_decode8(w) * scale).T
    lut = torch.tensor([0, 0.5, 1, 1.5, -0.0, -0.5, -1, -1.5] * 2, dtype=torch.float64, device="cuda")
    codes = torch.stack([w & 15, w >> 4], -1).reshape(w.shape[0], -1).long()
    return x.double() @ (lut[codes] * scale).T
