"""Performance cases of the StripedHyena2 library: the work its users have it do.

Operator cases go through the operator C ABI (``include/evo/hip_ops.h``) at the
shapes of the two model topologies of the repository (7B: width 4096, FFN
11264, 32 heads; 1B: width 1920, FFN 5120, 15 heads); the whole-call cases go
through the evo C ABI on a model with one block of each mixer at 7B width.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs, weights and handles on the GPU
    run(state)           one pass
    work(case)           bytes and operations the pass cannot do without
    tolerance(case)      how far a correct implementation may be off
    exact(case, seed)    the same outputs in 64 bits, in plain torch
"""
import ctypes
import math
import os
import sys
import tempfile
from functools import lru_cache

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "evo.cpp_amd"))

from evo_hip import artifact, capi, native  # noqa: E402

DEVICE = "cuda:0"
WIDTHS = {4096: dict(inner=11264, heads=32, groups=256, rope_scale=128.0),
          1920: dict(inner=5120, heads=15, groups=128, rope_scale=1.0)}
VOCAB = 512
STATE = 16
TAPS = {"hcs": 7, "hcm": 128}
KINDS = {"hcs": native.HYENA_HCS, "hcm": native.HYENA_HCM, "hcl": native.HYENA_HCL}
DTYPES = {"f32": native.DTYPE_F32, "bf16": native.DTYPE_BF16, "f16": native.DTYPE_F16,
          "bf16_f16": native.DTYPE_BF16_F16}
EPS = 1e-6
CODE_SCALE = 448.0 / 8.0  # the fixed activation scale of load-time FP8 conversion
FP8_PROJECTIONS = 1 << 8  # EVO_MODEL_FLAG_HIP_FP8_PROJECTIONS
F16_OUT = 1 << 12         # EVO_CONTEXT_FLAG_HIP_F16_OUT


def listed():
    return [
        # A block's output projection (bias, residual) over a prompt of about
        # a thousand bases in the 1B topology, split-BF16 activations.
        dict(name="out_proj_prompt", op="linear", rows=1000, n=1920, k=1920, planes=2,
             bias=True, residual=True, workspace=True),
        # The gated MLP of a short query sequence (a primer or probe), 7B.
        dict(name="mlp_short", op="mlp", rows=61, width=4096, planes=2, gelu=False),
        # The gated MLP of one full prefill chunk, 7B: where a long prefill
        # spends most of its time.
        dict(name="mlp_chunk", op="mlp", rows=8192, width=4096, planes=2, gelu=False),
        # Norm, E4M3 quantisation and software-FP8 input projection of a
        # Hyena block: an amplicon-sized prompt, and one full chunk.
        dict(name="fp8_projection_prompt", op="fp8", rows=200, width=4096, mode=1),
        dict(name="fp8_projection_chunk", op="fp8", rows=8192, width=4096, mode=1),
        # The three Hyena mixers. HCS on a BF16-projection (F32) model's prompt
        # with its continuation caches, FP16 output; HCM and HCL on one full
        # chunk of an FP8-projection model.
        dict(name="hcs_prompt", op="hyena", kind="hcs", rows=611, width=1920, dtype="f16",
             keep=True),
        dict(name="hcm_chunk", op="hyena", kind="hcm", rows=8192, width=4096,
             dtype="bf16_f16", keep=False),
        dict(name="hcl_chunk", op="hyena", kind="hcl", rows=8192, width=4096, dtype="bf16",
             keep=False),
        # Attention of a gene-sized prompt (1B) and of a later chunk of a
        # long-context prefill (7B).
        dict(name="attention_prompt", op="attention", rows=1500, width=1920, prefix=0),
        dict(name="attention_long", op="attention", rows=4096, width=4096, prefix=28672),
        # Scoring one record of a FASTA file: a fresh context, its prefill with
        # host logits, and the context's end.
        dict(name="score_record", op="score", rows=300),
        # A prompt followed by cached decode steps, tokens and prompt logits
        # in device memory, FP8 projections and FP16 output projections.
        dict(name="generate", op="generate", rows=1024, steps=16),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    op = rng.choice(["linear", "linear", "mlp", "mlp", "fp8", "fp8", "hyena", "hyena",
                     "hyena", "attention", "attention", "score", "generate"])
    width = rng.choice([4096, 1920])
    rows = _log_int(rng, 1, 8192)
    if op == "linear":
        n = rng.choice([width, width, 3 * width, VOCAB])
        out_proj = n == width
        return dict(op=op, rows=rows, n=n, k=width, planes=rng.choice([2, 2, 1]),
                    bias=out_proj, residual=out_proj, workspace=rng.choice([True, False]))
    if op == "mlp":
        return dict(op=op, rows=rows, width=width, planes=rng.choice([2, 2, 1]),
                    gelu=rng.choice([True, False, False]))
    if op == "fp8":
        return dict(op=op, rows=rows, width=width, mode=rng.choice([1, 1, 0]))
    if op == "hyena":
        return dict(op=op, kind=rng.choice(["hcs", "hcm", "hcl"]), rows=rows, width=width,
                    dtype=rng.choice(["f32", "bf16", "f16", "bf16_f16"]),
                    keep=rng.choice([True, False]))
    if op == "attention":
        prefix = rng.choice([0, 0, _log_int(rng, 64, 28672)])
        return dict(op=op, rows=_log_int(rng, 1, 4096), width=width, prefix=prefix)
    if op == "score":
        return dict(op=op, rows=_log_int(rng, 16, 2048))
    return dict(op=op, rows=_log_int(rng, 16, 2048), steps=rng.randint(4, 16))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    generator = torch.Generator(device=DEVICE)
    generator.manual_seed(seed)
    return generator


def _normal(generator, *shape, std=1.0):
    return torch.randn(*shape, generator=generator, device=DEVICE) * std


def _planes(x, planes):
    """The GEMM activation layout: hi = bf16(x), lo = bf16(x - hi)."""
    hi = x.to(torch.bfloat16)
    return hi, (x - hi.float()).to(torch.bfloat16) if planes == 2 else None


def _value(hi, lo):
    return hi.double() if lo is None else hi.double() + lo.double()


def _ptr(tensor):
    return None if tensor is None else tensor.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEVICE)


def _linear_inputs(case, seed):
    g, m, n, k = _gen(seed), case["rows"], case["n"], case["k"]
    hi, lo = _planes(_normal(g, m, k), case["planes"])
    return dict(hi=hi, lo=lo, w=_normal(g, n, k, std=0.02).to(torch.bfloat16),
                bias=_normal(g, n, std=0.02).to(torch.bfloat16) if case["bias"] else None,
                residual=_normal(g, m, n) if case["residual"] else None)


def _prepare_linear(case, seed):
    state = _linear_inputs(case, seed)
    state["out"] = _empty(case["rows"], case["n"])
    state["workspace"] = _empty(16 << 20) if case["workspace"] else None
    return state


def _run_linear(case, s):
    args = (_ptr(s["hi"]), _ptr(s["lo"]), _ptr(s["w"]), _ptr(s["bias"]), _ptr(s["residual"]),
            case["rows"], case["n"], case["k"], _ptr(s["out"]))
    if s["workspace"] is None:
        native.call("evo_hip_linear", *args, _stream())
    else:
        native.call("evo_hip_linear_split", *args, _ptr(s["workspace"]),
                    s["workspace"].numel() * 4, _stream())
    return s["out"]


def _exact_linear(case, seed):
    s = _linear_inputs(case, seed)
    out = _value(s["hi"], s["lo"]) @ s["w"].double().T
    if s["bias"] is not None:
        out += s["bias"].double()
    if s["residual"] is not None:
        out += s["residual"].double()
    return out


def _mlp_inputs(case, seed):
    g, m, width = _gen(seed), case["rows"], case["width"]
    inner = WIDTHS[width]["inner"]
    hi, lo = _planes(_normal(g, m, width), case["planes"])
    l1, l2 = (_normal(g, inner, width, std=0.02).to(torch.bfloat16) for _ in range(2))
    return dict(hi=hi, lo=lo, l1=l1, l2=l2,
                l3=_normal(g, width, inner, std=0.02).to(torch.bfloat16),
                residual=_normal(g, m, width))


def _prepare_mlp(case, seed):
    state = _mlp_inputs(case, seed)
    m, width, inner = case["rows"], case["width"], WIDTHS[case["width"]]["inner"]
    w12 = _empty(2 * inner, width, dtype=torch.bfloat16)
    l1, l2 = state.pop("l1"), state.pop("l2")
    native.call("evo_hip_pack_mlp", _ptr(l1), _ptr(l2), inner, width, _ptr(w12), _stream())
    torch.cuda.synchronize()  # l1 and l2 end here
    state.update(w12=w12, inner=_empty(case["planes"] * m * inner, dtype=torch.bfloat16),
                 out=_empty(m, width))
    return state


def _run_mlp(case, s):
    native.call("evo_hip_gated_mlp", _ptr(s["hi"]), _ptr(s["lo"]), _ptr(s["w12"]),
                _ptr(s["l3"]), case["rows"], case["width"], WIDTHS[case["width"]]["inner"],
                int(case["gelu"]), _ptr(s["inner"]), _ptr(s["residual"]), _ptr(s["out"]),
                _stream())
    return s["out"]


def _exact_mlp(case, seed):
    s = _mlp_inputs(case, seed)
    x = _value(s["hi"], s["lo"])
    first, second = x @ s["l1"].double().T, x @ s["l2"].double().T
    if case["gelu"]:
        first = 0.5 * first * (1 + torch.erf(first / math.sqrt(2)))
    return (first * second) @ s["l3"].double().T + s["residual"].double()


def _fp8_inputs(case, seed):
    g, m, width = _gen(seed), case["rows"], case["width"]
    x = _normal(g, m, width, std=2.0)
    scale = 1 + _normal(g, width, std=0.02)
    weight = _normal(g, 3 * width, width, std=0.02)
    weight_scale = 448.0 / float(weight.abs().max())
    codes = (weight * weight_scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    return dict(x=x, scale=scale, w=codes,
                output_scale=float(np.float32(1.0 / (CODE_SCALE * weight_scale))))


def _prepare_fp8(case, seed):
    state = _fp8_inputs(case, seed)
    m, width = case["rows"], case["width"]
    state.update(codes=_empty(m, width, dtype=torch.uint8),
                 out=_empty(m, 3 * width, dtype=torch.bfloat16))
    return state


def _run_fp8(case, s):
    m, width = case["rows"], case["width"]
    native.call("evo_hip_rms_norm_e4m3", _ptr(s["x"]), m, width, _ptr(s["scale"]), EPS,
                CODE_SCALE, _ptr(s["codes"]), _stream())
    native.call("evo_hip_fp8_linear_bf16", _ptr(s["codes"]), _ptr(s["w"]), _ptr(s["out"]), m,
                3 * width, width, s["output_scale"], case["mode"], _stream())
    return [s["codes"], s["out"]]


def _exact_fp8(case, seed):
    s = _fp8_inputs(case, seed)
    x = s["x"].double()
    y = x / (x.square().mean(1, keepdim=True).sqrt() + EPS) * s["scale"].double()
    codes = (y.float().to(torch.bfloat16).float() * CODE_SCALE).clamp(-448, 448).to(
        torch.float8_e4m3fn)
    return [None, (codes.double() @ s["w"].double().T) * s["output_scale"]]


def _hyena_inputs(case, seed):
    g, length, width, kind = _gen(seed), case["rows"], case["width"], case["kind"]
    projection = _normal(g, length, 3 * width)
    if case["dtype"].startswith("bf16"):
        projection = projection.to(torch.bfloat16)
    s = dict(projection=projection, short=_normal(g, 3 * width, 3, std=0.5).to(torch.bfloat16),
             inner=None, direct=None, poles=None, residues=None)
    if kind != "hcl":
        groups, taps = WIDTHS[width]["groups"], TAPS[kind]
        s["inner"] = _normal(g, groups, taps, std=taps ** -0.5).to(torch.bfloat16).float()
    if kind != "hcs":
        s["direct"] = _normal(g, width, std=0.5).to(torch.bfloat16).float()
    if kind == "hcl":
        s["poles"] = 0.5 + 0.49 * torch.rand(width, STATE, generator=g, device=DEVICE)
        s["residues"] = _normal(g, width, STATE, std=0.1)
    return s


def _prepare_hyena(case, seed):
    s = _hyena_inputs(case, seed)
    length, width, kind = case["rows"], case["width"], case["kind"]
    s["out"] = _empty(length, width, dtype={"f32": torch.float32, "bf16": torch.bfloat16}.get(
        case["dtype"], torch.float16))
    s["workspace"] = _empty(max(16, native.call("evo_hip_hyena_workspace_bytes", KINDS[kind],
                                                length, width, STATE)), dtype=torch.uint8)
    s["caches"] = [None, None, None]
    if case["keep"]:
        s["caches"][0] = _empty(2, 3 * width)
        if kind == "hcl":
            s["caches"][2] = _empty(width, STATE)
        else:
            s["caches"][1] = _empty(TAPS[kind] - 1, width)
    return s


def _run_hyena(case, s):
    kind, width = case["kind"], case["width"]
    for cache in s["caches"]:  # a new sequence starts from empty caches
        if cache is not None:
            cache.zero_()
    native.call("evo_hip_hyena_forward", KINDS[kind],
                DTYPES[case["dtype"]] | native.DTYPE_BF16_TAPS, _ptr(s["projection"]),
                case["rows"], width, _ptr(s["short"]), 3, _ptr(s["inner"]),
                0 if kind == "hcl" else WIDTHS[width]["groups"], TAPS.get(kind, 0),
                _ptr(s["direct"]), _ptr(s["poles"]), _ptr(s["residues"]),
                STATE if kind == "hcl" else 0, *(_ptr(c) for c in s["caches"]),
                _ptr(s["workspace"]), s["workspace"].numel(), _ptr(s["out"]), _stream())
    return [s["out"], *s["caches"]]


def _last_rows(x, count):
    pad = torch.zeros(max(0, count - x.shape[0]), x.shape[1], dtype=x.dtype, device=x.device)
    return torch.cat([pad, x[-count:]])


def _shifted(x, by):
    out = torch.zeros_like(x)
    if by < x.shape[0]:
        out[by:] = x[:x.shape[0] - by]
    return out


def _exact_hyena(case, seed):
    s, kind, length, width = _hyena_inputs(case, seed), case["kind"], case["rows"], case["width"]
    p, short = s["projection"].double(), s["short"].double()
    fir = sum(_shifted(p, 2 - t) * short[:, t] for t in range(3)).view(length, width, 3)
    x2, u = fir[:, :, 0], fir[:, :, 1] * fir[:, :, 2]
    state = None
    if kind == "hcl":
        steps = torch.arange(length, dtype=torch.float64, device=DEVICE)[:, None]
        log_poles, residues = s["poles"].double().log(), s["residues"].double()
        kernel = sum(residues[:, m] * torch.exp(steps * log_poles[:, m]) for m in range(STATE))
        size = 2 * length
        inner = torch.fft.irfft(torch.fft.rfft(u, n=size, dim=0) *
                                torch.fft.rfft(kernel, n=size, dim=0), n=size, dim=0)[:length]
        state = torch.stack([(u * torch.exp((length - 1 - steps) * log_poles[:, m])).sum(0)
                             for m in range(STATE)], 1)
    else:
        taps = TAPS[kind]
        filters = s["inner"].double().repeat_interleave(width // s["inner"].shape[0], 0)
        # HCS taps are stored oldest first, HCM's newest first.
        inner = sum(_shifted(u, t) * filters[:, taps - 1 - t if kind == "hcs" else t]
                    for t in range(min(taps, length)))
    if s["direct"] is not None:
        inner = inner + s["direct"].double() * u
    if not case["keep"]:
        return [inner * x2, None, None, None]
    return [inner * x2, _last_rows(p, 2), None if kind == "hcl" else _last_rows(u, TAPS[kind] - 1),
            state]


def _attention_inputs(case, seed):
    g, rows, width, prefix = _gen(seed), case["rows"], case["width"], case["prefix"]
    dim = width // WIDTHS[width]["heads"]
    inv_freq = (1.0 / (10000.0 ** (np.arange(0, dim, 2, dtype=np.float64) / dim))).astype(
        np.float32)
    capacity = (prefix + rows + 63) // 64 * 64
    keys = torch.zeros(2, capacity, width, dtype=torch.bfloat16, device=DEVICE)
    values = torch.zeros(2, width, capacity, dtype=torch.bfloat16, device=DEVICE)
    # The caches after an earlier prefill of `prefix` positions: split planes,
    # values transposed with position bits 2 and 3 swapped.
    if prefix:
        keys[0, :prefix], keys[1, :prefix] = _planes(_normal(g, prefix, width), 2)
        whole = (prefix + 15) // 16 * 16
        position = torch.arange(whole, device=DEVICE)
        column = ((position & ~15) | (position & 3) | ((position & 4) << 1) |
                  ((position & 8) >> 1))
        v = torch.zeros(width, whole, device=DEVICE)
        v[:, :prefix] = _normal(g, width, prefix)
        values[0][:, :whole], values[1][:, :whole] = _planes(v[:, column], 2)
    return dict(projected=_normal(g, rows, 3 * width), keys=keys, values=values,
                capacity=capacity, inv_freq=torch.from_numpy(inv_freq).to(DEVICE))


def _prepare_attention(case, seed):
    s = _attention_inputs(case, seed)
    rows, width = case["rows"], case["width"]
    s.update(query=_empty(2 * rows * width, dtype=torch.bfloat16), out=_empty(rows, width),
             workspace=_empty(16 << 20))
    return s


def _run_attention(case, s):
    rows, width = case["rows"], case["width"]
    dims = WIDTHS[width]
    native.call("evo_hip_attention_ws", _ptr(s["projected"]), rows, width, dims["heads"], 1,
                _ptr(s["inv_freq"]), dims["rope_scale"], case["prefix"], _ptr(s["query"]),
                _ptr(s["keys"]), _ptr(s["values"]), s["capacity"], _ptr(s["out"]),
                _ptr(s["workspace"]), s["workspace"].numel() * 4, _stream())
    return [s["out"], s["keys"], s["values"]]


def _exact_attention(case, seed):
    s, rows, width, prefix = _attention_inputs(case, seed), case["rows"], case["width"], case["prefix"]
    heads = WIDTHS[width]["heads"]
    dim, half = width // heads, width // heads // 2
    qkv = s["projected"].view(rows, heads, 3, dim)
    position = torch.arange(prefix, prefix + rows, device=DEVICE)
    # The rotation angle is defined in F32: position / scale * inv_freq.
    angle = ((position.float() / WIDTHS[width]["rope_scale"])[:, None] * s["inv_freq"]).double()
    cosine, sine = angle.cos(), angle.sin()

    def rotate(x):
        a, b = x[:, :half].double(), x[:, half:].double()
        return torch.cat([a * cosine - b * sine, b * cosine + a * sine], 1)

    key = torch.arange(prefix + rows, device=DEVICE)
    column = (key & ~15) | (key & 3) | ((key & 4) << 1) | ((key & 8) >> 1)
    out = _empty(rows, width, dtype=torch.float64)
    for h in range(heads):
        at = slice(h * dim, (h + 1) * dim)
        k = _value(s["keys"][0][:prefix + rows, at], s["keys"][1][:prefix + rows, at])
        v = _value(s["values"][0][at, column], s["values"][1][at, column]).T.contiguous()
        k[prefix:], v[prefix:] = rotate(qkv[:, h, 1]), qkv[:, h, 2].double()
        q = rotate(qkv[:, h, 0])
        for first in range(0, rows, 1024):
            last = min(rows, first + 1024)
            scores = (q[first:last] @ k.T) / math.sqrt(dim)
            scores.masked_fill_(key > position[first:last, None], -math.inf)
            out[first:last, at] = torch.softmax(scores, 1) @ v
    return [out, None, None]


# ------------------------------------------------------------- whole calls
@lru_cache(maxsize=None)
def _artifact_path():
    """A seeded model file with one block of each mixer at 7B width."""
    shape = artifact.tiny_shape(width=4096, layers=4, heads=32, inner=11264, groups=256,
                                attn=(3,), rope_scale=128.0,
                                model_id="random-init-evo2-7b-width-4-blocks")
    path = os.path.join(tempfile.mkdtemp(prefix="evo_cases_"), "model.safetensors")
    artifact.random_artifact(shape, seed=4, init="survey").write(path)
    return path


@lru_cache(maxsize=None)
def _model(flags):
    """The loaded model: a program loads it once and keeps it."""
    return capi.EvoLibrary(native.LIBRARY_PATH).load(_artifact_path(), capi.BACKEND_HIP, flags)


def _prepare_score(case, seed):
    return dict(model=_model(0),
                sequence=artifact.acgt_tokens(case["rows"], seed).astype(np.uint8).tobytes())


def _run_score(case, s):
    context = s["model"].context(case["rows"])
    try:
        return context.prefill(s["sequence"])
    finally:
        context.close()


def _prepare_generate(case, seed):
    model, rows, steps = _model(FP8_PROJECTIONS), case["rows"], case["steps"]
    tokens = artifact.acgt_tokens(rows + steps, seed)
    return dict(context=model.context(rows + steps, F16_OUT),
                prompt=torch.from_numpy(tokens[:rows].astype(np.int32)).to(DEVICE),
                next=[int(t) for t in tokens[rows:]], logits=_empty(rows, VOCAB))


def _run_generate(case, s):
    context = s["context"]
    library = context.model.library
    library.check(library.lib.evo_hip_context_prefill_resident(
        context.handle, ctypes.c_void_p(_ptr(s["prompt"])), ctypes.c_size_t(case["rows"]),
        ctypes.c_void_p(_ptr(s["logits"]))))
    return [s["logits"], np.stack([context.decode(token) for token in s["next"]])]


# ------------------------------------------------------------------- entry
_PREPARE = dict(linear=_prepare_linear, mlp=_prepare_mlp, fp8=_prepare_fp8,
                hyena=_prepare_hyena, attention=_prepare_attention, score=_prepare_score,
                generate=_prepare_generate)
_RUN = dict(linear=_run_linear, mlp=_run_mlp, fp8=_run_fp8, hyena=_run_hyena,
            attention=_run_attention, score=_run_score, generate=_run_generate)
_EXACT = dict(linear=_exact_linear, mlp=_exact_mlp, fp8=_exact_fp8, hyena=_exact_hyena,
              attention=_exact_attention)


def prepare(case, seed):
    return dict(_PREPARE[case["op"]](case, seed), case=case)


def run(state):
    case = state["case"]
    return _RUN[case["op"]](case, state)


def exact(case, seed):
    make = _EXACT.get(case["op"])
    return None if make is None else make(case, seed)


def work(case):
    op, m = case["op"], case["rows"]
    if op == "linear":
        n, k = case["n"], case["k"]
        return dict(bytes=2 * case["planes"] * m * k + 2 * n * k + 4 * m * n +
                    (2 * n if case["bias"] else 0) + (4 * m * n if case["residual"] else 0),
                    flops=2 * m * n * k)
    if op in ("score", "generate"):
        # One block of each mixer: four MLPs, output projections and input
        # projections (FP8 for the three Hyena blocks of `generate`), the
        # unembedding, causal attention.
        w, inner = 4096, 11264
        weights = 4 * (3 * w * inner + 4 * w * w) + VOCAB * w
        resident = 2 * weights - (9 * w * w if op == "generate" else 0)
        steps = case.get("steps", 0)
        return dict(bytes=(1 + steps) * resident + 4 * (m + steps) * VOCAB + 8 * steps * m * w,
                    flops=2 * (m + steps) * weights + 2 * m * m * w + 4 * steps * m * w)
    width = case["width"]
    inner = WIDTHS[width]["inner"]
    if op == "mlp":
        return dict(bytes=2 * case["planes"] * m * width + 6 * width * inner + 8 * m * width,
                    flops=6 * m * width * inner)
    if op == "fp8":
        return dict(bytes=4 * m * width + m * width + 3 * width * width + 6 * m * width,
                    flops=6 * m * width * width)
    if op == "hyena":
        size_in = 2 if case["dtype"].startswith("bf16") else 4
        size_out = 4 if case["dtype"] == "f32" else 2
        taps = TAPS.get(case["kind"], 2 * STATE)
        return dict(bytes=m * width * (3 * size_in + size_out),
                    flops=m * width * (18 + 2 * taps + 4))
    keys = case["prefix"] + m
    pairs = m * case["prefix"] + m * (m + 1) / 2
    return dict(bytes=12 * m * width + 8 * keys * width + 4 * m * width,
                flops=4 * pairs * width)


def tolerance(case):
    # About four times each path's distance from its 64-bit result.
    op = case["op"]
    if op == "linear":
        return dict(rel=1e-5, max=1e-4)
    if op == "mlp":  # one plane: the gated activation is rounded to BF16
        return dict(rel=1e-5, max=1e-4) if case["planes"] == 2 else dict(rel=6e-3, max=3e-2)
    if op == "fp8":
        return dict(rel=8e-3 if case["mode"] == 1 else 1.5e-2, max=7e-2, differ=1e-4)
    if op == "hyena":
        return {"f32": dict(rel=2e-5, max=5e-4), "bf16": dict(rel=6.6e-3, max=1.6e-2)}.get(
            case["dtype"], dict(rel=8e-4, max=4e-3))
    if op == "attention":
        return dict(rel=2.4e-5, max=6.5e-4)
    # Whole calls: another split of the rows into chunks (other F32 sums and,
    # with FP8 projections, other codes for about 0.2 % of the activations)
    # moves the logits by 9e-6 (BF16 projections) and 5.4e-5 (FP8).
    return dict(rel=4e-5, max=2e-4) if op == "score" else dict(rel=2e-4, max=1e-3)
