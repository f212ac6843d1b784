"""The work that programs give this library: inputs, one pass through the public
calls, the bytes and operations a pass cannot do without, and the result in 64 bits.

A case names an operation ("op") and its sizes.  Inputs are those of the
library's own benchmark: Gaussian or uniform complex signals, images in [0, 1),
block-floating-point signals spread over six decades, and filters given as
natural-order spectra that are planned before the call (or, where new filters
arrive with the signals, in the pass itself).
"""
from __future__ import annotations

import math

import torch

import fufft_amd as ff

DEV = "cuda"

# points per drawn case: from one transform up to a quarter of the largest listed case
MOST_POINTS = 1 << 25


def listed():
    return [
        # The smallest call: a few short signals, as in a control or audio loop that
        # filters each buffer as it arrives.  Launch and call overhead.
        {"name": "conv_256_x3", "op": "conv", "n": 256, "batch": 3, "mid": "mul", "layout": "dr"},
        # A batch of medium signals correlated with one template (matched filter),
        # everything at its default: the benchmark's N = 1024, 8192 signals.
        {"name": "corr_1024_x8192", "op": "conv", "n": 1024, "batch": 8192, "mid": "conj", "layout": "dr"},
        # Long signals, an odd number of them, with the default filter order.
        {"name": "conv_16384_x99", "op": "conv", "n": 16384, "batch": 99, "mid": "mul", "layout": "dr"},
        # The benchmark's headline and the largest case: 2^27 points, N = 4096, the
        # fastest plan and its filter order.
        {"name": "conv_4096_x32768", "op": "conv", "n": 4096, "batch": 32768, "mid": "mul", "layout": "lane"},
        # A filter of its own for every signal, new ones with each batch: the spectra
        # are planned on the device and then convolved, in the radix-16 plan.
        {"name": "plan_conv_4096_x3001", "op": "plan_conv", "n": 4096, "batch": 3001, "mid": "mul", "layout": "dr",
         "variant": "v16"},
        # int16 block floating point, one exponent per 64 points: the benchmark's N = 4096.
        {"name": "bfp_4096_x16384", "op": "bfp", "n": 4096, "batch": 16384, "mid": "mul", "layout": "lane", "block": 64},
        # One signal against a bank of filters: its forward transform, then the apply.
        {"name": "split_8192_x500", "op": "split", "n": 8192, "batch": 500, "mid": "mul", "layout": "dr"},
        # Spectral processing: natural-order transform and its inverse.
        {"name": "c2c_2048_x5001", "op": "c2c", "n": 2048, "batch": 5001},
        # Signals beyond one workgroup: the benchmark's N = 32768, an odd batch.
        {"name": "large_32768_x301", "op": "large", "n": 32768, "batch": 301, "mid": "mul"},
        # The longest signals, a few at a time.
        {"name": "large_1048576_x3", "op": "large", "n": 1 << 20, "batch": 3, "mid": "mul"},
        # Pairs of real images: the benchmark's 512 x 512, a handful of pairs.
        {"name": "real2d_512x512_x9", "op": "real2d", "h": 512, "w": 512, "batch": 9, "layout": "lane"},
        # Small images (tiles, patches), each convolved with the same kernel.
        {"name": "image_64x64_x4000", "op": "image", "h": 64, "w": 64, "batch": 4000, "mid": "mul", "layout": "dr"},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same operations: every power of two the operation takes,
    any batch, from a single transform to MOST_POINTS points."""
    op = rng.choice(("conv", "conv", "conv", "plan_conv", "real1d", "bfp", "bfp_scaled", "split", "c2c", "large",
                     "large", "image", "real2d", "split2d", "image"))
    case = {"op": op}
    if op in ("image", "real2d", "split2d"):
        if op == "image" and rng.random() < 0.5:       # small images: at most 8192 points, sides 8 .. 512
            while True:
                h, w = 1 << rng.randint(3, 9), 1 << rng.randint(3, 9)
                if h * w <= 8192:
                    break
        else:                                          # large ones: 256 .. 2048 rows of 256 .. 4096 points
            h, w = 1 << rng.randint(8, 11), 1 << rng.randint(8, 12)
        case.update(h=h, w=w, batch=_log_uniform(rng, 1, MOST_POINTS // (h * w)))
        case["layout"] = rng.choice(("dr", "lane"))
        if op != "real2d":
            case["mid"] = rng.choice(("mul", "mul", "conj"))
        return case
    if op == "large":
        n = 1 << rng.randint(13, 20)
        case.update(n=n, batch=_log_uniform(rng, 1, MOST_POINTS // n), mid=rng.choice(("mul", "mul", "conj")))
        if rng.random() < 0.25:
            case["own_filters"] = True
        return case
    if op == "conv":
        n = 1 << rng.randint(8, 15)
    elif op == "bfp":
        n = 1 << rng.randint(10, 14)
    else:
        n = 1 << rng.randint(8, 14)
    case.update(n=n, batch=_log_uniform(rng, 1, MOST_POINTS // n))
    if op == "c2c":
        return case
    case["layout"] = rng.choice(("dr", "lane"))
    if op != "real1d":
        case["mid"] = rng.choice(("mul", "mul", "conj"))
    if op == "bfp":
        case["block"] = rng.choice((64, 64, n))
    return case


# ---- inputs ------------------------------------------------------------------------

def _gen(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + 13)
    return g


def _gauss(g, points):
    return torch.randn(points, dtype=torch.complex64, device=DEV, generator=g)


def _uniform(g, points):
    return torch.view_as_complex(torch.rand(points, 2, device=DEV, generator=g) * 2 - 1)


def _inputs(case, seed):
    """The natural-order inputs of a case, from the seed alone: signals and filter spectra."""
    g, op, batch = _gen(case, seed), case["op"], case["batch"]
    if op in ("image", "real2d", "split2d"):
        pts = case["h"] * case["w"]
        if op == "real2d":
            x, y = torch.rand(batch * pts, device=DEV, generator=g), torch.rand(batch * pts, device=DEV, generator=g)
            # a real filter's spectrum
            taps = torch.rand(case["h"], case["w"], device=DEV, generator=g, dtype=torch.float64)
            return {"x": x, "y": y, "spec": torch.fft.fft2(taps).to(torch.complex64).reshape(-1)}
        x = torch.view_as_complex(torch.rand((1 if op == "split2d" else batch) * pts, 2, device=DEV, generator=g))
        return {"x": x, "spec": _gauss(g, pts * (batch if op == "split2d" else 1))}
    n = case["n"]
    if op == "real1d":
        x, y = torch.randn(batch * n, device=DEV, generator=g), torch.randn(batch * n, device=DEV, generator=g)
        taps = torch.randn(n, device=DEV, generator=g, dtype=torch.float64)
        return {"x": x, "y": y, "spec": torch.fft.fft(taps).to(torch.complex64)}
    if op == "large":
        # all-pass filters: the call works in place, and its result is the next pass's signal
        angle = torch.rand(n * (batch if case.get("own_filters") else 1), device=DEV, generator=g) * (2 * math.pi)
        return {"x": _uniform(g, batch * n), "spec": torch.polar(torch.ones_like(angle), angle)}
    if op == "split":
        return {"x": _gauss(g, n), "spec": _gauss(g, batch * n)}
    if op in ("bfp", "bfp_scaled"):
        decades = torch.rand(batch, 1, device=DEV, generator=g) * 6 - 3
        x = (_gauss(g, batch * n).view(batch, n) * torch.pow(10.0, decades)).reshape(-1)
        return {"x": x, "spec": _gauss(g, n)}
    if op == "c2c":
        return {"x": _gauss(g, batch * n)}
    return {"x": _gauss(g, batch * n), "spec": _gauss(g, n * (batch if op == "plan_conv" else 1))}


def _variant(case):
    """The plan a program takes: the default's, the one named, or the fastest for the filter order."""
    if "variant" in case:
        return case["variant"]
    return ff.fastest_variant(case["n"], "lane") if case.get("layout") == "lane" else "auto"


def _quantise_blocks(x, block):
    """int16 pairs and an int8 exponent per block: the smallest e with absmax <= 32767 * 2^e."""
    v = torch.view_as_real(x).reshape(-1, 2 * block)
    top = v.abs().amax(dim=1).double()
    e = torch.ceil(torch.log2(top / 32767.0)).clamp(-128, 127)
    e = torch.where(top <= 32767.0 * torch.exp2(e - 1), e - 1, e)
    e = torch.where(top > 32767.0 * torch.exp2(e), e + 1, e)
    q = torch.empty(v.shape, dtype=torch.int16, device=v.device)
    rows = max(1, (1 << 24) // (2 * block))
    for a in range(0, v.shape[0], rows):
        b = a + rows
        q[a:b] = torch.round(v[a:b].double() * torch.exp2(-e[a:b, None])).to(torch.int16)
    return q.reshape(-1), e.to(torch.int8)


def _quantise_scaled(x, n):
    """int16 pairs and an fp32 scale per n points: absmax / 32767."""
    v = torch.view_as_real(x).reshape(-1, 2 * n)
    top = v.abs().amax(dim=1).clamp_min(1e-30)
    q = torch.round((v * (32767.0 / top)[:, None]).clamp(-32767, 32767)).to(torch.int16)
    return q.reshape(-1), top / 32767.0


def prepare(case, seed):
    case = dict(case)
    s = _inputs(case, seed)
    op, batch, layout = case["op"], case["batch"], case.get("layout", "dr")
    s["case"] = case
    if op in ("image", "real2d", "split2d"):
        h, w = case["h"], case["w"]
        count = batch if op == "split2d" else 1
        s["filt"] = torch.empty_like(s["spec"])
        ff.plan_filter2d_device(s.pop("spec"), s["filt"], h, w, count=count, layout=layout)
        if op == "real2d":
            s["u"], s["v"] = torch.empty_like(s["x"]), torch.empty_like(s["y"])
            s["work"] = torch.empty(batch * h * w, dtype=torch.complex64, device=DEV)
        else:
            s["out"] = torch.empty(batch * h * w, dtype=torch.complex64, device=DEV)
            if op == "split2d":
                s["fx"] = torch.empty_like(s["x"])
        return s
    n = case["n"]
    case["variant"] = _variant(case)
    if op == "c2c":
        s["fx"], s["out"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
        return s
    if op == "large":
        s["filt"] = torch.empty_like(s["spec"])
        ff.plan_filter_large_device(s.pop("spec"), s["filt"], n, count=s["filt"].numel() // n)
        return s
    s["filt"] = torch.empty_like(s["spec"])
    if op != "plan_conv":
        ff.plan_filter_device(s.pop("spec"), s["filt"], n, count=s["filt"].numel() // n, variant=case["variant"],
                              layout=layout)
    if op == "real1d":
        s["u"], s["v"] = torch.empty_like(s["x"]), torch.empty_like(s["y"])
    elif op == "bfp":
        s["q"], s["e"] = _quantise_blocks(s.pop("x"), case["block"])
        s["qo"], s["eo"] = torch.empty_like(s["q"]), torch.empty_like(s["e"])
    elif op == "bfp_scaled":
        s["q"], s["sc"] = _quantise_scaled(s.pop("x"), n)
        s["qf"], s["sf"] = _quantise_scaled(s.pop("filt"), n)
        s["qo"], s["so"] = torch.empty_like(s["q"]), torch.empty_like(s["sc"])
    else:
        s["out"] = torch.empty(batch * n, dtype=torch.complex64, device=DEV)
        if op == "split":
            s["fx"] = torch.empty_like(s["x"])
    return s


# ---- one pass ------------------------------------------------------------------------

def run(s):
    c = s["case"]
    op, batch = c["op"], c["batch"]
    if op == "conv":
        ff.conv(s["x"], s["filt"], s["out"], c["n"], batch, mid=c["mid"], variant=c["variant"], layout=c["layout"])
        return s["out"]
    if op == "plan_conv":
        n = c["n"]
        ff.plan_filter_device(s["spec"], s["filt"], n, count=batch, variant=c["variant"], layout=c["layout"])
        ff.conv(s["x"], s["filt"], s["out"], n, batch, filt_stride=n, mid=c["mid"], variant=c["variant"],
                layout=c["layout"])
        return s["filt"], s["out"]
    if op == "real1d":
        ff.conv_r2(s["x"], s["y"], s["filt"], s["u"], s["v"], c["n"], batch, variant=c["variant"], layout=c["layout"])
        return s["u"], s["v"]
    if op == "bfp":
        ff.conv_bfp16(s["q"], s["e"], s["filt"], s["qo"], s["eo"], c["n"], batch, mid=c["mid"], variant=c["variant"],
                      layout=c["layout"], block=c["block"])
        return s["qo"], s["eo"]
    if op == "bfp_scaled":
        ff.conv_bfp16_scaled(s["q"], s["sc"], s["qf"], s["sf"], s["qo"], s["so"], c["n"], batch, mid=c["mid"],
                             variant=c["variant"], layout=c["layout"])
        return s["qo"], s["so"]
    if op == "split":
        n = c["n"]
        ff.fwd(s["x"], s["fx"], n, 1, variant=c["variant"])
        ff.apply(s["fx"], s["filt"], s["out"], n, batch, spec_stride=0, filt_stride=n, mid=c["mid"],
                 variant=c["variant"], layout=c["layout"])
        return s["fx"], s["out"]
    if op == "c2c":
        ff.c2c(s["x"], s["fx"], c["n"], batch, direction=ff.FORWARD)
        ff.c2c(s["fx"], s["out"], c["n"], batch, direction=ff.INVERSE)
        return s["fx"], s["out"]
    if op == "large":
        n = c["n"]
        ff.conv_large(s["x"], s["filt"], n, batch, filt_stride=n if c.get("own_filters") else 0, mid=c["mid"])
        return s["x"]
    h, w = c["h"], c["w"]
    if op == "image":
        ff.conv2d(s["x"], s["filt"], s["out"], h, w, batch, mid=c["mid"], layout=c["layout"])
        return s["out"]
    if op == "real2d":
        ff.conv2d_r2(s["x"], s["y"], s["filt"], s["u"], s["v"], s["work"], h, w, batch, layout=c["layout"])
        return s["u"], s["v"]
    if op == "split2d":
        ff.fwd2d(s["x"], s["fx"], h, w, 1)
        ff.apply2d(s["fx"], s["filt"], s["out"], h, w, batch, spec_stride=0, filt_stride=h * w, mid=c["mid"],
                   layout=c["layout"])
        return s["fx"], s["out"]
    raise ValueError(op)


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    """Bytes: every input read once, every output written once.  Operations: 5 n log2 n
    per complex transform of n points and 6 per product of two spectra."""
    op, batch = case["op"], case["batch"]
    n = case["h"] * case["w"] if "h" in case else case["n"]
    pts, transform = batch * n, 5 * n * math.log2(n)
    fused = {"bytes": 16 * pts + 8 * n, "flops": batch * (2 * transform + 6 * n)}
    if op == "plan_conv":       # spectra read and filters written, then signals, filters and results
        return {"bytes": 40 * pts, "flops": fused["flops"]}
    if op == "bfp":
        return {"bytes": 8 * pts + 2 * (pts // case["block"]) + 8 * n, "flops": fused["flops"]}
    if op == "bfp_scaled":
        return {"bytes": 8 * pts + 8 * batch + 4 * n + 4, "flops": fused["flops"]}
    if op in ("split", "split2d"):   # one forward; filters read, results written
        return {"bytes": 16 * n + 16 * pts, "flops": transform + batch * (transform + 6 * n)}
    if op == "c2c":
        return {"bytes": 32 * pts, "flops": 2 * batch * transform}
    if op == "large" and case.get("own_filters"):
        return {"bytes": 24 * pts, "flops": fused["flops"]}
    return fused


def tolerance(case):
    """fp32 transforms of 2^8 to 2^22 points are 2e-7 to 8e-7 of the 64-bit result
    (relative 2-norm).  Block-floating-point words round at 2^-15 of their block's largest
    value, and a difference of 1e-6 in the value moves about one word in 500 by one."""
    if case["op"] in ("bfp", "bfp_scaled"):
        return {"rel": 4e-6, "differ": 0.008}
    return {"rel": 3e-6, "max": 3e-5}


# ---- the same in 64 bits ------------------------------------------------------------------

def _digit_order(spec, n, variant):
    """Natural-order spectra (rows of n) in digit order: one leading radix for the bits
    that whole radix-16 (radix-8) digits leave over, the digits then reversed."""
    if variant == "auto":
        variant = "r8" if n in (512, 4096, 8192) else "v16"
    bits, digit = n.bit_length() - 1, 3 if variant == "r8" else 4
    widths = ([bits % digit] if bits % digit else []) + [digit] * (bits // digit)
    # bin = sum of digits, the first pass's digit least significant; slot: most significant
    sizes = [1 << b for b in reversed(widths)]
    v = spec.reshape(-1, *sizes)
    return v.permute(0, *range(len(sizes), 0, -1)).reshape(-1, n)


def _convolved(x, spec, conj, dims):
    """Cyclic convolution (correlation) of rows of x with the filters of spectrum spec."""
    axes = tuple(range(-dims, 0))
    f = torch.fft.fftn(x.to(torch.complex128), dim=axes)
    return torch.fft.ifftn(f * (spec.conj() if conj else spec), dim=axes)


def exact(case, seed):
    op, batch, conj = case["op"], case["batch"], case.get("mid") == "conj"
    if op in ("bfp", "bfp_scaled"):
        return None             # whole words and exponents: the rounding of the result is the result
    s = _inputs(case, seed)
    two_d = "h" in case
    shape = (case["h"], case["w"]) if two_d else (case["n"],)
    x = s["x"].view(-1, *shape)
    if op == "c2c":
        f = torch.fft.fft(x.to(torch.complex128))
        return f, x.to(torch.complex128) * case["n"]
    if op in ("real1d", "real2d"):
        spec = s["spec"].view(shape).to(torch.complex128)
        dims = len(shape)
        return (_convolved(x, spec, False, dims).real, _convolved(s["y"].view(-1, *shape), spec, False, dims).real)
    out = torch.empty(batch, *shape, dtype=torch.complex128, device=DEV)
    spec = s["spec"].view(-1, *shape)
    step = max(1, (1 << 24) // math.prod(shape))
    for a in range(0, batch, step):
        b = min(batch, a + step)
        xs = x if x.shape[0] == 1 else x[a:b]
        fs = spec if spec.shape[0] == 1 else spec[a:b]
        out[a:b] = _convolved(xs, fs.to(torch.complex128), conj, len(shape))
    if op == "split":
        return _digit_order(torch.fft.fft(x.to(torch.complex128)), case["n"], _variant(case)), out
    if op == "plan_conv":
        order = _digit_order(s["spec"].to(torch.complex128) / case["n"], case["n"], _variant(case))
        return order if case["layout"] == "dr" else None, out
    if op == "split2d":
        return None, out        # the 2D spectrum's column order is the library's own
    return out
