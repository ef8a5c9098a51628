"""Performance cases of the framework: what its users run, through its public entry points.

A case names an entry point ("api"), a shape and the options of the call:
  "vc"      sageattention_local.sageattn_vc: preparation and the fused kernel, fresh inputs
  "fp8"     sageattention_local.vc_fp8.sageattn_vc_fp8: the block-scaled FP8 QK variant
  "step"    vc_attention.attention, one denoising step; "reuse": a step that finds its layer's
            V layout in the request's LayoutCache (three steps in four), else a one-shot call
  "rotate"  vcx.preprocess_qk: binary32 K centring and Hadamard rotation of post-RoPE Q/K

Inputs ("data"): "normal" N(0,1); "outlier" per-channel K offsets and V around 8 centroids per
head, which is what smoothing and grouping are for; "student" heavy-tailed Q/K.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "cake-opt-vc_attention_amd"))

import vcx  # noqa: E402
from sageattention_local import sageattn_vc  # noqa: E402
from sageattention_local.vc_fp8 import sageattn_vc_fp8  # noqa: E402
from vc_attention import Config, LayoutCache, attention  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BASE = dict(api="vc", B=1, H=2, Nq=2048, Nk=2048, D=128, dtype="bf16", layout="HND", expcast=True,
             smooth=False, clusters=8, reuse=False, rotate=False, data="normal")


def _case(name=None, N=None, **options):
    case = dict(_BASE, **options)
    if N is not None:
        case["Nq"] = case["Nk"] = N
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # the smallest configuration of the benchmark: launches and host work decide
        _case("small_2x2048", H=2, N=2048),
        # the replay tool's default call, both VC features on: one-shot layout, input checks
        _case("replay_2x2048", api="step", H=2, N=2048, smooth=True, data="outlier"),
        # a range of queries against all keys, as the replay tool samples them
        _case("queries_4x1024x8192", H=4, Nq=1024, Nk=8192, smooth=True, data="outlier"),
        # a batch of medium sequences of a D64 model, ragged, fp16, token-major as a model holds it
        _case("batch_2x16x4097_d64", B=2, H=16, N=4097, D=64, dtype="f16", layout="NHD"),
        # the headline: one layer of the video model at full length, smoothing off
        _case("main_28x37741", H=28, N=37741),
        # the same layer with grouping and block-mean smoothing (the library's default call)
        _case("smooth_28x37741", H=28, N=37741, smooth=True, data="outlier"),
        # the D64 model's layer
        _case("d64_40x32760", H=40, N=32760, D=64, smooth=True),
        # twice the frames: the largest call, heavy-tailed Q/K
        _case("long_28x75482", H=28, N=75482, smooth=True, data="student"),
        # the FP8 QK variant of the headline layer, token-major
        _case("fp8_28x37741", api="fp8", H=28, N=37741, layout="NHD"),
        # one GPU's share of the layer under 4-way sequence parallelism, a step between two
        # refreshes of the layout, with the Hadamard rotation
        _case("step_7x37741", api="step", H=7, N=37741, smooth=True, reuse=True, rotate=True, data="outlier"),
        # the same share on the Sage FP8 control probabilities, fp16, a finer grouping
        _case("control_7x37741_c16", H=7, N=37741, dtype="f16", expcast=False, smooth=True, clusters=16,
              data="outlier"),
        # Q/K preprocessing for a caller's own attention: centred K, both rotated, binary32 out
        _case("rotate_28x37741", api="rotate", H=28, N=37741, rotate=True, smooth=True, data="outlier"),
    ]


_MOST = 28 * 75482 * 75482 * 128  # query-key-channel products of the largest listed case


def _tokens(rng, low, high):
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return n if rng.random() < 0.25 else n | 1  # mostly odd, so ragged in every tile


def draw(rng):
    api = rng.choice(["vc"] * 6 + ["fp8", "step", "step", "rotate"])
    case = _case(api=api, D=rng.choice([128, 128, 64]), dtype=rng.choice(["bf16", "bf16", "f16"]),
                 H=rng.choice([1, 2, 4, 7, 8, 14, 16, 24, 28, 40]), N=_tokens(rng, 512, 75482))
    if api == "rotate":
        case.update(D=rng.choice([128, 64, 37]), dtype=rng.choice(["bf16", "f16", "f32"]), smooth=rng.random() < 0.75,
                    rotate=rng.random() < 0.75, data=rng.choice(["normal", "outlier"]))
        case["Nq"] = case["Nk"] = min(case["Nk"], 37741)
        return case
    if rng.random() < 0.2:
        case["B"] = 2
    if rng.random() < 0.2:  # a range of queries against all keys
        case["Nq"] = min(case["Nk"], _tokens(rng, 64, 4096))
    if api != "fp8":
        case["smooth"] = rng.random() < 0.6
    if api != "step":
        case["layout"] = rng.choice(["HND", "NHD"])
    case["expcast"] = rng.random() < 0.8
    if case["smooth"]:
        case["clusters"] = rng.choice([8, 8, 8, 8, 4, 16, 32])
    if api == "step":
        case["rotate"] = rng.random() < 0.5
        case["reuse"] = case["smooth"] and rng.random() < 0.75
    case["data"] = rng.choice(["normal", "outlier", "student"])
    while case["B"] * case["H"] * case["Nq"] * case["Nk"] * case["D"] > _MOST:
        if case["B"] > 1:
            case["B"] = 1
        else:
            case["H"] = case["H"] * 3 // 4
    return case


def _normal(shape, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _student(shape, g):
    """0.5 * Student-t with 4 degrees of freedom (a normal over the root of a chi-square mean),
    within the range that a model's Q/K normalization leaves."""
    u = torch.rand(shape, generator=g, device="cuda").clamp_(min=1e-7)
    u.mul_(torch.rand(shape, generator=g, device="cuda").clamp_(min=1e-7))
    return _normal(shape, g).mul_(0.5).div_(u.log_().mul_(-0.5).sqrt_()).clamp_(-4.0, 4.0)


def _clustered(shape, g):
    B, H, N, D = shape
    centroids = _normal((B, H, 8, D), g) * 2.0 ** 0.5
    which = torch.randint(0, 8, (B, H, N, 1), generator=g, device="cuda").expand(B, H, N, D)
    return torch.gather(centroids, 2, which) + _normal(shape, g) * 0.3 ** 0.5


def _inputs(case, seed):
    """Q, K, V as [B,H,N,D] of the case's type (K offsets and V clusters by its "data")."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    qs, ks = (case["B"], case["H"], case["Nq"], case["D"]), (case["B"], case["H"], case["Nk"], case["D"])
    make = _student if case["data"] == "student" else _normal
    dtype = _DTYPES[case["dtype"]]
    q, k = make(qs, g).to(dtype), make(ks, g)
    if case["data"] == "outlier":
        k += _normal((ks[0], ks[1], 1, ks[3]), g) * 2.0
    k = k.to(dtype)
    if case["api"] == "rotate":
        return q, k, None
    v = (_clustered(ks, g) if case["data"] == "outlier" else _normal(ks, g)).to(dtype)
    return q, k, v


def _config(case):
    return Config(backend="hip", qk_format="int8", q_block=64, k_quant_block=128, kv_block=128,
                  expcast=case["expcast"], v_smooth=case["smooth"], qk_hadamard=case["rotate"],
                  clusters=case["clusters"])


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    state = {"case": case, "q": q, "k": k, "v": v}
    if case["layout"] == "NHD":
        for name in "qkv":
            state[name] = state[name].transpose(1, 2).contiguous()
    if case["api"] == "step":
        state["config"] = _config(case)
        if case["reuse"]:
            # the request's cache after the step before, whose V was a little different
            g = torch.Generator(device="cuda").manual_seed(seed + 1000003)
            before = (v + 0.1 * _normal(v.shape, g).to(v.dtype))
            state["cache"] = LayoutCache(state["config"])
            state["cache"].layout(before, step=0, total_steps=8, request_id="request", layer_id=0)
    return state


def run(state):
    case, q, k, v = (state[n] for n in ("case", "q", "k", "v"))
    if case["api"] == "vc":
        return sageattn_vc(q, k, v, tensor_layout=case["layout"], expcast=case["expcast"], v_smooth=case["smooth"],
                           clusters=case["clusters"])
    if case["api"] == "fp8":
        return sageattn_vc_fp8(q, k, v, tensor_layout=case["layout"], expcast=case["expcast"])
    if case["api"] == "rotate":
        return vcx.preprocess_qk(q, k, case["smooth"], case["rotate"])
    if case["reuse"]:
        return attention(q, k, v, state["config"], cache=state["cache"], step=1, total_steps=8,
                         request_id="request", layer_id=0)[0]
    return attention(q, k, v, state["config"])[0]


def _width(case):
    return 1 << (case["D"] - 1).bit_length() if case["rotate"] else case["D"]


def work(case):
    rows_q, rows_k = case["B"] * case["H"] * case["Nq"], case["B"] * case["H"] * case["Nk"]
    size = 4 if case["dtype"] == "f32" else 2
    if case["api"] == "rotate":
        width = _width(case)
        flops = (rows_q + rows_k) * width * (math.log2(width) + 1 if case["rotate"] else 1)
        return {"bytes": (rows_q + rows_k) * (case["D"] * size + width * 4), "flops": flops}
    return {"bytes": (2 * rows_q + 2 * rows_k) * case["D"] * size, "flops": 4 * rows_q * case["Nk"] * case["D"]}


def tolerance(case):
    """Attention: one quantized contract, so two implementations differ by the order of the
    binary32 sums and the rounding of the output. Against 64-bit sums over the same payloads
    and probability bytes the path measures 1.7e-3 (bf16) and 2.1e-4 (fp16), at most 3.9e-3
    and 5.9e-4 on one value; outliers of a row add to that. The FP8 scores are sums whose order
    the contract leaves open, so about 2 in 10^4 probability bytes move by one code. Rotation:
    binary32 sums of at most 128 terms, 1.0e-7 against 64 bits."""
    if case["api"] == "rotate":
        return {"rel": 5e-7, "max": 5e-6}
    if case["api"] == "fp8":
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 4e-3, "max": 4e-2}
    return {"rel": 7e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 5e-3}


def _hadamard(x):
    """Normalized Sylvester-Hadamard rotation of the last axis, zero padded to a power of two."""
    width = 1 << (x.shape[-1] - 1).bit_length()
    x = torch.nn.functional.pad(x, (0, width - x.shape[-1]))
    shape, stride = x.shape, 1
    while stride < width:
        x = x.reshape(*shape[:-1], width // (2 * stride), 2, stride)
        a, b = x[..., 0, :], x[..., 1, :]
        x = torch.stack((a + b, a - b), dim=-2).reshape(shape)
        stride *= 2
    return x / math.sqrt(width)


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    if case["api"] == "rotate":
        out = []
        for x, centre in ((q, False), (k, case["smooth"])):
            y = torch.empty((*x.shape[:-1], _width(case)), dtype=torch.float64, device=x.device)
            for b in range(x.shape[0]):
                for h in range(x.shape[1]):
                    row = x[b, h].double()
                    row = row - row.mean(0) if centre else row
                    y[b, h] = _hadamard(row) if case["rotate"] else row
            out.append(y)
        return tuple(out)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    chunk = max(1, (1 << 28) // case["Nk"])
    for b in range(case["B"]):
        for h in range(case["H"]):
            kt, vd = k[b, h].double().t().contiguous(), v[b, h].double()
            for r in range(0, case["Nq"], chunk):
                logits = torch.mm(q[b, h, r:r + chunk].double() * case["D"] ** -0.5, kt)
                out[b, h, r:r + chunk] = torch.mm(torch.softmax(logits, dim=-1), vd)
    return out.transpose(1, 2).contiguous() if case["layout"] == "NHD" else out
