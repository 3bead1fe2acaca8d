"""Workloads of the group quantizer for timing, through the package's public entry points.

Six kinds of work, which is what a program that quantizes a model has this package do:

  tiles    independent 256-weight tiles through the two-pass Viterbi (viterbi_tiles_dev)
  group    one Hessian group by itself (quantize_group_h): rotate, factor, LDLQ, proxy, pack
  groups   several groups through the scheduler (run_groups)
  hessian  token batches of one layer summed into its Hessian, mirrored and scaled (the step before a group)
  nvfp4    the fallback quantizer of a group, from and to host memory (nvfp4_quantize_group)
  dequant  a quantized linear back to its weights on the device (dequantize_linear)

Sizes are the package's benchmark configurations and the sizes of its tests, and ragged ones between them.
"""
import math

import numpy as np
import torch

from __graft_entry__ import _pkg

_handle = None


def _quantizer():
    """The context a worker makes once and keeps."""
    global _handle
    if _handle is None:
        _handle = _pkg().Quantizer(0)
    return _handle


def listed():
    return [
        # Viterbi by itself: a handful of tiles (one tile row of a small layer), and benchmark configuration 1
        dict(name="tiles_24", path="tiles", tiles=24),
        dict(name="tiles_4096", path="tiles", tiles=4096),
        # the reference's end-to-end case: two linears behind one 256-wide Hessian, host memory in and out
        dict(name="group_64+32x256_host", path="group", ms="64,32", n=256, dtype="f32", device=False, feedback=0),
        # benchmark configuration 2: a lone 1024 x 1024 group
        dict(name="group_1024x1024", path="group", ms="1024", n=1024, dtype="f32", device=True, feedback=0),
        # a mid-sized layer's q/k/v behind one Hessian, bf16 checkpoint weights, fp32 feedback (split-bf16 products)
        dict(name="group_qkv_4096_bf16_fb1", path="group", ms="4096,1024,1024", n=4096, dtype="bf16", device=True, feedback=1),
        # small layers of a model in one call, FP8 checkpoint weights in host memory: they share the chip
        dict(name="groups_6_2048x2560_fp8_host", path="groups", count=6, ms="2048", n=2560, dtype="fp8", device=False, feedback=0),
        # benchmark configuration 3: q-proj
        dict(name="group_12288x12288", path="group", ms="12288", n=12288, dtype="f32", device=True, feedback=0),
        # benchmark configuration 5, the headline: down-proj through the scheduler
        dict(name="groups_12288x28672", path="groups", count=1, ms="12288", n=28672, dtype="f32", device=True, feedback=0),
        # calibration: one ragged batch of a small layer; the Hessian of configurations 3 and 4 in batches of 2048 tokens
        dict(name="hessian_1000x2560", path="hessian", rows=1000, batches=1, n=2560),
        dict(name="hessian_4x2048x12288", path="hessian", rows=2048, batches=4, n=12288),
        # the fallback quantizer on the layer shape of its tests, calibrated
        dict(name="nvfp4_4096x4096", path="nvfp4", ms="4096", n=4096, hessian=True),
        # decoding a quantized linear of configuration 3
        dict(name="dequant_12288x12288", path="dequant", m=12288, n=12288),
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(v / multiple + 0.5) * multiple)


# Sizes the Hadamard transform takes: a power of two, or one of its factors times one.
_DIMS = sorted({k << p for k in (1, 12, 20, 28, 36) for p in range(4, 14) if 256 <= k << p <= 12288 and (k << p) % 128 == 0})


def draw(rng):
    path = rng.choice(["tiles", "group", "group", "groups", "hessian", "nvfp4", "dequant"])
    if path == "tiles":
        return dict(path=path, tiles=_log_int(rng, 1, 12288))
    if path == "hessian":
        rows, n = _log_int(rng, 16, 4096), _log_int(rng, 256, 12288, 8)
        return dict(path=path, rows=rows, batches=rng.choice([1, 2, 4]), n=n)
    if path == "nvfp4":
        return dict(path=path, ms=",".join(str(_log_int(rng, 64, 4096)) for _ in range(rng.choice([1, 1, 2, 3]))),
                    n=_log_int(rng, 256, 4096, 16), hessian=rng.random() < 0.75)
    if path == "dequant":
        return dict(path=path, m=rng.choice(_DIMS), n=rng.choice(_DIMS))
    dtype, device, feedback = rng.choice(["f32", "bf16", "fp8"]), rng.random() < 0.5, rng.choice([0, 0, 0, 1])
    if path == "group":
        n = rng.choice(_DIMS)
        ms = [rng.choice([m for m in _DIMS if m * n <= 12288 * 12288]) for _ in range(rng.choice([1, 1, 2, 3]))]
        if sum(ms) > 12288:
            ms = ms[:1]
        return dict(path=path, ms=",".join(map(str, ms)), n=n, dtype=dtype, device=device, feedback=feedback)
    dims = [d for d in _DIMS if d <= 4096]
    return dict(path=path, count=rng.randint(2, 6), ms=str(rng.choice(dims)), n=rng.choice(dims), dtype=dtype, device=device,
                feedback=feedback)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weights(g, m, n):
    """Heavy-tailed weights of a trained layer's scale: N(0, 0.015^2) with one in a hundred ten times as large."""
    w = torch.randn(m, n, device="cuda", generator=g) * 0.015
    return torch.where(torch.rand(m, n, device="cuda", generator=g) < 0.01, w * 10.0, w)


def _activations(g, rows, n):
    """bf16 token vectors whose channels hang together (each is mixed with its neighbours), a few of them large."""
    x = torch.randn(rows, n, device="cuda", generator=g)
    for shift, rho in ((1, 0.8), (2, 0.64), (4, 0.41), (8, 0.17)):
        x = x + rho * torch.roll(x, shift, dims=1)
    x[:, torch.randint(0, n, (max(1, n // 384),), device="cuda", generator=g)] *= 20.0
    return x.to(torch.bfloat16)


def _hessian(g, n):
    rows = min(8192, max(512, 2 * n))
    x = _activations(g, rows, n).float()
    h = x.T @ x / float(rows)
    return ((h + h.T) * 0.5).contiguous()


def _linear(pkg, g, name, m, n, dtype, device):
    w = _weights(g, m, n)
    place = (lambda t: t.contiguous()) if device else (lambda t: t.cpu().numpy())
    if dtype == "f32":
        return pkg.LinearIn(name, m, w_f32=place(w))
    if dtype == "bf16":
        return pkg.LinearIn(name, m, w_bf16=place(w.to(torch.bfloat16).view(torch.int16)))
    scale = (w.abs().amax(dim=1) / 448.0).to(torch.bfloat16)
    codes = (w / scale.float()[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return pkg.LinearIn(name, m, w_fp8=place(codes.view(torch.uint8)), scale_bf16=place(scale.view(torch.int16)))


def _group(pkg, case, seed):
    g = _gen(seed)
    n = case["n"]
    lins = [_linear(pkg, g, "w%d" % i, int(m), n, case["dtype"], case["device"]) for i, m in enumerate(case["ms"].split(","))]
    h = _hessian(g, n)
    return lins, n, h if case["device"] else h.cpu().numpy(), seed % 100003 + 1


def prepare(case, seed):
    pkg, q, path = _pkg(), _quantizer(), case["path"]
    state = dict(case=case, q=q)
    g = _gen(seed)
    if path == "tiles":
        b = case["tiles"]
        # what LDLQ hands the search: rotated weights at nine tenths of the codebook's rms, rounded to fp16
        x = (torch.randn(b, 256, device="cuda", generator=g) * (0.9 * q.lut_rms)).half().float()
        state.update(x=x, states=torch.zeros(b, 128, dtype=torch.int16, device="cuda"),
                     packed=torch.zeros(b, 32, dtype=torch.int16, device="cuda"))
    elif path in ("group", "groups"):
        state.update(opt=pkg.QuantOpts(feedback=case["feedback"]),
                     groups=[_group(pkg, case, seed + 7919 * k) for k in range(case.get("count", 1))])
    elif path == "hessian":
        n, rows = case["n"], case["rows"]
        state.update(x=[_activations(g, rows, n).view(torch.int16) for _ in range(case["batches"])],
                     h=torch.empty(n, n, device="cuda"))
    elif path == "nvfp4":
        n = case["n"]
        state.update(ws=[_weights(g, int(m), n).cpu().numpy() for m in case["ms"].split(",")],
                     h=_hessian(g, n).cpu().numpy() if case["hessian"] else None)
    else:
        m, n = case["m"], case["n"]
        rng = np.random.default_rng(seed)
        su = rng.integers(0, 2, n).astype(np.uint16)
        state.update(lin=pkg.LinearOut(name="w", m=m, n=n, wscale=0.0163,
                                       trellis=rng.integers(0, 65536, (m // 16) * (n // 16) * 32, dtype=np.uint16),
                                       su_bf16=np.where(su, np.uint16(0xBF80), np.uint16(0x3F80)),
                                       sv=np.where(rng.integers(0, 2, m), np.float32(-1), np.float32(1))),
                     hat=torch.empty(m, n, device="cuda"))
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------- one pass
def _outputs(outs):
    return [dict(trellis=o.trellis, su=o.su_bf16, sv=o.sv, wscale=o.wscale, proxy=o.proxy, proxy_rot_reg=o.proxy_rot_reg)
            for o in outs]


def run(state):
    case, q = state["case"], state["q"]
    path = case["path"]
    if path == "tiles":
        q.viterbi_tiles_dev(state["x"], case["tiles"], state["states"], state["packed"])
        q.stream_signal()  # what torch does next with the results comes after them
        return state["states"], state["packed"]
    if path == "group":
        lins, n, h, seed = state["groups"][0]
        return _outputs(q.quantize_group_h(lins, n, h, seed, state["opt"])[0])
    if path == "groups":
        return [_outputs(r[0]) for r in q.run_groups(state["groups"], state["opt"])]
    if path == "hessian":
        h, n = state["h"], case["n"]
        h.zero_()
        for x in state["x"]:
            q.hessian_accumulate_dev(x, case["rows"], n, h)
        q.hessian_finish_dev(h, n, 1.0 / (case["rows"] * case["batches"]))
        q.stream_signal()
        return h
    if path == "nvfp4":
        tensors, calibrated = q.nvfp4_quantize_group(state["ws"], case["n"], state["h"])
        return [dict(packed=t.packed, scales=t.scales, scale=t.global_scale) for t in tensors] + [int(calibrated)]
    return q.dequantize_linear(state["lin"], state["hat"])


# ---------------------------------------------------------------- what a pass cannot do without
_ACS = 65536.0 * 2  # per weight: 2^16 add-compare-selects (two passes of 128 steps over 2^16 states per 256 weights), an add and a minimum each


def work(case):
    path, n = case["path"], float(case.get("n", 0))
    if path == "tiles":
        return dict(bytes=case["tiles"] * (1024.0 + 256 + 64), flops=case["tiles"] * 256 * _ACS)
    if path == "hessian":
        rows = float(case["rows"]) * case["batches"]
        return dict(bytes=2 * rows * n + 4 * n * n, flops=rows * n * (n + 1))
    if path == "dequant":
        m = float(case["m"])
        return dict(bytes=m * n / 4 + 4 * m * n, flops=m * n * (math.log2(m) + math.log2(n)))
    mt = float(sum(int(m) for m in case["ms"].split(",")))
    if path == "nvfp4":
        cal = bool(case["hessian"])
        return dict(bytes=mt * n * (4 + 0.5 + 1 / 16) + (4 * n * n if cal else 0),
                    flops=mt * n * 11 * 20 + (mt * n * n + n ** 3 / 3 if cal else 0))
    size = {"f32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
    # search; feedback of every column from those behind it; the factorization; two quadratic forms (symmetric)
    flops = mt * n * _ACS + mt * n * n + n ** 3 / 3 + 2 * mt * n * n
    return dict(bytes=case.get("count", 1) * (mt * n * (size + 0.25) + 4 * n * n), flops=case.get("count", 1) * flops)


def tolerance(case):
    """What another correct implementation may differ by: four times what each path differs from itself in 64 bits."""
    if case["path"] in ("tiles", "nvfp4"):
        return "exact"
    if case["path"] == "hessian":
        return {"rel": 1e-6, "max": 6e-5}   # fp32 sums of bf16 products: 1.4e-7 to 2.4e-7, largest 1.4e-5
    if case["path"] == "dequant":
        return {"rel": 6e-7, "max": 3e-6}   # fp32 butterflies: 1.4e-7, largest 7.2e-7
    # words and scales to the bit; the two proxies are sums of three bf16 products in fp32: 1.9e-5 to 3e-5
    return {"rel": 1.2e-4, "differ": 0.0}
