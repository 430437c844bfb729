"""The work that users of this framework give it, as cases to be timed.

Every case goes through the public Python entry points (FMMPlan, BatchPlan,
DCTPlan, Leg2Cheb) on device arrays and one HIP stream, as a spectral code
keeps them; Leg2Cheb alone works on host arrays, as its callers do.  Kinds:

  single   one vector through a plan (L2C, C2L, or both: forward and back)
  lines    many vectors of one length, back to back, in one call
  grid     a 2-D or 3-D array, L2C along every axis, then C2L back
  batch    independent vectors of uneven length, packed back to back
  dct      values <-> Chebyshev coefficients of one or several vectors
  host     the drop-in Leg2Cheb class on NumPy arrays

`exact` is the definition of each transform summed in 64 bits.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

L2C, C2L, BOTH = 0, 1, 2
_HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "l2c_amd" in sys.modules:
        return sys.modules["l2c_amd"]
    d = os.path.join(_HERE, "legendre-to-chebyshev_amd")
    if not os.path.isdir(d):
        d = os.path.join(os.getcwd(), "legendre-to-chebyshev_amd")
    spec = importlib.util.spec_from_file_location("l2c_amd", os.path.join(d, "__init__.py"),
                                                  submodule_search_locations=[d])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["l2c_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


_streams = []


def _stream():
    """The one stream a program runs its transforms on."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0].cuda_stream


# ---------------------------------------------------------------------------
# cases

def listed():
    return [
        # the smallest calls: 512 coefficients forward and back (the reference
        # CLI's own example, `l2c -N512 -d2`); launch latency is all there is
        {"name": "roundtrip_512", "kind": "single", "n": 512, "leaf": 64, "direction": BOTH,
         "decay": 1.0, "lagrange": 0},
        # 2^12, 2^16, 2^20: the sizes the single transform is quoted at
        {"name": "single_4096_l2c", "kind": "single", "n": 4096, "leaf": 64, "direction": L2C,
         "decay": 0.0, "lagrange": 0},
        {"name": "single_65536_c2l", "kind": "single", "n": 65536, "leaf": 64, "direction": C2L,
         "decay": 1.5, "lagrange": 0},
        # a length that is no power of two, at the leaf size Leg2Cheb takes by default
        {"name": "single_100000_l2c_leaf36", "kind": "single", "n": 100000, "leaf": 36,
         "direction": L2C, "decay": 1.0, "lagrange": 0},
        # the headline
        {"name": "single_1048576_l2c", "kind": "single", "n": 1 << 20, "leaf": 64,
         "direction": L2C, "decay": 0.0, "lagrange": 0},
        # the largest length that is no power of two
        {"name": "single_1000000_c2l", "kind": "single", "n": 1000000, "leaf": 64,
         "direction": C2L, "decay": 1.5, "lagrange": 0},
        # many long vectors of one length in a call
        {"name": "lines_64x262144_l2c", "kind": "lines", "n": 1 << 18, "lines": 64, "leaf": 64,
         "direction": L2C, "decay": 1.0},
        # a spectral field along its three axes and back, 65,536 lines a pass
        {"name": "grid_256x256x256", "kind": "grid", "n0": 256, "n1": 256, "n2": 256, "leaf": 64},
        # a 2-D array of ordinary, uneven sides
        {"name": "grid_1200x900", "kind": "grid", "n0": 1200, "n1": 900, "n2": 1, "leaf": 64},
        # thousands of independent vectors of lengths 64 .. 8192, tuned plan, graph replay
        {"name": "batch_4096_uneven", "kind": "batch", "count": 4096, "lo": 64, "hi": 8192,
         "direction": L2C},
        # function values at 2^20 Chebyshev points to coefficients
        {"name": "dct2_1048576", "kind": "dct", "n": 1 << 20, "count": 1, "type": 2},
        # the drop-in class on host arrays, with its default leaf size
        {"name": "host_200000_l2c", "kind": "host", "n": 200000, "direction": L2C},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "single", "single", "lines", "lines", "grid", "grid", "batch",
                       "dct", "host"])
    if kind == "single":
        n = _loguniform(rng, 512, 1 << 20)
        if rng.random() < 0.25:
            n = 1 << max(9, min(20, int(round(math.log2(n)))))
        # lengths small enough for a pass of one direction to be over in less
        # than 5 us are taken forward and back
        return {"kind": kind, "n": n, "leaf": rng.choice([64, 64, 36, 32, 50]),
                "direction": BOTH if n < 3000 else rng.choice([L2C, C2L]),
                "decay": rng.choice([0.0, 1.0, 1.5]), "lagrange": int(rng.random() < 0.15)}
    if kind == "lines":
        n = _loguniform(rng, 256, 1 << 18)
        return {"kind": kind, "n": n, "lines": max(2, min(4096, _loguniform(rng, 1 << 17, 1 << 23) // n)),
                "leaf": rng.choice([64, 64, 36, 32]), "direction": rng.choice([L2C, C2L]),
                "decay": rng.choice([0.0, 1.0])}
    if kind == "grid":
        if rng.random() < 0.5:
            return {"kind": kind, "n0": _loguniform(rng, 48, 256), "n1": _loguniform(rng, 48, 256),
                    "n2": _loguniform(rng, 48, 256), "leaf": 64}
        return {"kind": kind, "n0": _loguniform(rng, 200, 2048), "n1": _loguniform(rng, 200, 2048),
                "n2": 1, "leaf": rng.choice([64, 64, 36])}
    if kind == "batch":
        lo = _loguniform(rng, 16, 256)
        return {"kind": kind, "count": _loguniform(rng, 256, 4096), "lo": lo,
                "hi": _loguniform(rng, 4 * lo, 8192), "direction": rng.choice([L2C, C2L])}
    if kind == "dct":
        n = 1 << rng.randint(10, 20)
        return {"kind": kind, "n": n, "count": max(1, _loguniform(rng, 1 << 16, 1 << 21) // n),
                "type": rng.choice([2, 3])}
    return {"kind": kind, "n": _loguniform(rng, 2000, 200000), "direction": rng.choice([L2C, C2L])}


# ---------------------------------------------------------------------------
# inputs

def _uniform(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return 2 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g) - 1


def _weights(n, decay):
    return torch.arange(1, n + 1, dtype=torch.float64, device="cuda") ** -decay


def _lengths(case):
    """The lengths of a batch: the same for every input of the case."""
    r = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    lo, hi = case["lo"], case["hi"]
    x = np.floor(np.exp(r.uniform(math.log(lo), math.log(hi + 1), case["count"])))
    return np.clip(x, lo, hi).astype(np.int64)


def _axes(case):
    return [case["n0"], case["n1"]] + ([case["n2"]] if case["n2"] > 1 else [])


def _input(case, seed):
    """The input of a case, a float64 tensor on the GPU."""
    k = case["kind"]
    if k == "single":
        return _uniform(case["n"], seed) * _weights(case["n"], case["decay"])
    if k == "lines":
        u = _uniform(case["n"] * case["lines"], seed).view(case["lines"], case["n"])
        return (u * _weights(case["n"], case["decay"])).contiguous()
    if k == "grid":
        shape = _axes(case)
        u = _uniform(int(np.prod(shape)), seed).view(*shape)
        for d, n in enumerate(shape):
            u = u * _weights(n, 1.0).view([n if e == d else 1 for e in range(len(shape))])
        return u.contiguous()
    if k == "batch":
        n = _lengths(case)
        first = np.repeat(np.cumsum(n) - n, n)
        place = torch.from_numpy(np.arange(int(n.sum())) - first).cuda().double()
        return _uniform(int(n.sum()), seed) / (place + 1)
    if k == "dct":
        # values of a smooth function with some noise (type 2), or decaying coefficients (type 3)
        u = _uniform(case["n"] * case["count"], seed).view(case["count"], case["n"])
        if case["type"] == 3:
            return (u * _weights(case["n"], 1.0)).contiguous()
        x = torch.cos(math.pi * (torch.arange(case["n"], dtype=torch.float64, device="cuda") + 0.5)
                      / case["n"])
        return (torch.exp(u[:, :1] * x) + 0.01 * u).contiguous()
    return _uniform(case["n"], seed) * _weights(case["n"], 1.0)


def prepare(case, seed):
    amd, k = _package(), case["kind"]
    x = _input(case, seed)
    s = {"case": case, "x": x, "stream": _stream()}
    if k == "host":
        s["x"] = x.cpu().numpy()
        n = case["n"]
        s["plan"] = amd.Leg2Cheb(np.zeros(n), np.zeros(n), direction=case["direction"], verbose=0)
        return s
    if k == "single":
        s["plan"] = amd.FMMPlan(case["n"], case["leaf"], 18, case["direction"],
                                lagrange=case["lagrange"])
        s["out"] = torch.zeros_like(x)
        s["back"] = torch.zeros_like(x)
    elif k == "lines":
        s["plan"] = amd.FMMPlan(case["n"], case["leaf"], 18, case["direction"])
        s["out"] = torch.zeros_like(x)
    elif k == "grid":
        plans = {n: amd.FMMPlan(n, case["leaf"], 18, BOTH) for n in set(_axes(case))}
        s["plan"] = [plans[n] for n in _axes(case)]
        s["out"], s["back"], s["tmp"] = (torch.zeros_like(x) for _ in range(3))
    elif k == "batch":
        s["plan"] = amd.BatchPlan(_lengths(case), 18, case["direction"], tune=True)
        s["plan"].graph(True)
        s["out"] = torch.zeros_like(x)
    elif k == "dct":
        s["plan"] = amd.DCTPlan(case["n"], case["count"])
        s["out"] = torch.zeros_like(x)
    torch.cuda.synchronize()
    return s


def _line_map(shape, axis):
    """(lines, n0, stride0, stride1, element stride) of an axis of a C-ordered array."""
    inner = int(np.prod(shape[axis + 1:]))
    outer = int(np.prod(shape[:axis]))
    if inner == 1:
        return outer, outer, shape[axis], 0, 1
    return outer * inner, inner, 1, inner * shape[axis], inner


def run(s):
    case, st = s["case"], s["stream"]
    k = case["kind"]
    if k == "host":
        return s["plan"](s["x"], direction=case["direction"])
    p, x = s["plan"], s["x"]
    if k == "single":
        if case["direction"] == BOTH:
            p.execute_device(x.data_ptr(), s["out"].data_ptr(), L2C, stream=st)
            p.execute_device(s["out"].data_ptr(), s["back"].data_ptr(), C2L, stream=st)
            return {"forward": s["out"], "back": s["back"]}
        p.execute_device(x.data_ptr(), s["out"].data_ptr(), case["direction"], stream=st)
        return s["out"]
    if k == "lines":
        n, b = case["n"], case["lines"]
        p.execute_lines_device(x.data_ptr(), s["out"].data_ptr(), case["direction"], b, b, n, 0, 1,
                               stream=st)
        return s["out"]
    if k == "grid":
        shape = _axes(case)
        d = len(shape)
        src = x
        for i, axis in enumerate(reversed(range(d))):  # forward, the last axis first
            dst = s["out"] if (d - 1 - i) % 2 == 0 else s["tmp"]
            p[axis].execute_lines_device(src.data_ptr(), dst.data_ptr(), L2C,
                                         *_line_map(shape, axis), stream=st)
            src = dst
        for i, axis in enumerate(range(d)):  # and back
            dst = s["back"] if (d - 1 - i) % 2 == 0 else s["tmp"]
            p[axis].execute_lines_device(src.data_ptr(), dst.data_ptr(), C2L,
                                         *_line_map(shape, axis), stream=st)
            src = dst
        return {"forward": s["out"], "back": s["back"]}
    if k == "batch":
        p.execute_device(x.data_ptr(), s["out"].data_ptr(), case["direction"], stream=st)
        return s["out"]
    p.execute_device(x.data_ptr(), s["out"].data_ptr(), case["type"], stream=st)
    return s["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _transform_flops(n):
    """Floating-point operations of one length-n transform: the direct sum's
    n^2 / 4 terms of two operations each, or, where that is less, the
    reference's own count for the fast multipole form (its ~400 per element at
    leaf size 64)."""
    return min(n * n / 2.0, 400.0 * n)


def work(case):
    k = case["kind"]
    if k == "single":
        passes = 2 if case["direction"] == BOTH else 1
        return {"bytes": passes * 24 * case["n"], "flops": passes * _transform_flops(case["n"])}
    if k == "host":
        return {"bytes": 24 * case["n"], "flops": _transform_flops(case["n"])}
    if k == "lines":
        n, b = case["n"], case["lines"]
        return {"bytes": 16 * n * b + 8 * n, "flops": b * _transform_flops(n)}
    if k == "grid":
        shape = _axes(case)
        total = int(np.prod(shape))
        return {"bytes": 2 * len(shape) * 16 * total,
                "flops": 2 * sum(total // n * _transform_flops(n) for n in shape)}
    if k == "batch":
        n = _lengths(case).astype(float)
        return {"bytes": 16 * float(n.sum()), "flops": float(np.minimum(n * n / 2, 400 * n).sum())}
    total = case["n"] * case["count"]
    return {"bytes": 16 * total, "flops": 2.5 * total * math.log2(case["n"])}


# ---------------------------------------------------------------------------
# the definitions, summed in 64 bits

def _lambda(n):
    """Gamma(k + 1/2) / Gamma(k + 1), k < n."""
    k = np.arange(1, n, dtype=np.longdouble)
    a = np.concatenate([[np.longdouble(1)], np.cumprod((k - np.longdouble(0.5)) / k)])
    return a * np.sqrt(np.longdouble("3.14159265358979323846264338327950288"))


def _tables(n, direction):
    """The factors h[m - r] and p[m + r + par] of the direct sums."""
    a = _lambda(n + 2)
    if direction == L2C:
        return a[:n].astype(np.float64), a[:n].astype(np.float64), None
    i = np.arange(1, n, dtype=np.longdouble)
    an = np.concatenate([[2 / np.sqrt(np.longdouble("3.14159265358979323846264338327950288"))],
                         1 / (2 * a[1:n] * i * (i + np.longdouble(0.5)))])
    j = np.arange(1, n, dtype=np.longdouble)
    dn = np.concatenate([[np.longdouble(0)], a[:n - 1] / (2 * j)])
    return -dn.astype(np.float64), an.astype(np.float64), an


def _direct(x, direction):
    """L2C or C2L of the rows of x (lines, n), by the direct sums."""
    b, n = x.shape
    dev = x.device
    h, p, an = _tables(n, direction)
    h = torch.from_numpy(np.concatenate([np.zeros(n), h])).to(dev)  # h[k] at n + k
    p = torch.from_numpy(np.concatenate([p, np.zeros(n + 1)])).to(dev)
    out = torch.empty_like(x)
    i = torch.arange(n, dtype=torch.float64, device=dev)
    v = x if direction == L2C else x * torch.where(i > 0, i, torch.ones_like(i))
    for par in range(2):
        xp = v[:, par::2].t().contiguous()  # (columns, lines)
        m = xp.shape[0]
        y = torch.zeros_like(xp)
        rows, cols = 2048, 8192
        for r0 in range(0, m, rows):
            r1 = min(m, r0 + rows)
            for c0 in range(r0, m, cols):
                c1 = min(m, c0 + cols)
                # p[c + r + par] and, rows reversed, h[c - r]
                hank = p.as_strided((r1 - r0, c1 - c0), (1, 1), r0 + c0 + par)
                toep = h.as_strided((r1 - r0, c1 - c0), (1, 1), n + c0 - (r1 - 1))
                y[r0:r1] += (toep.flip(0) * hank) @ xp[c0:c1]
        out[:, par::2] = y.t()
    if direction == L2C:
        out *= 2 / math.pi
        out[:, 0] *= 0.5
        return out
    diag = torch.from_numpy((np.sqrt(np.longdouble("3.14159265358979323846264338327950288")) * an)
                            .astype(np.float64)).to(dev)
    return (out + v * diag) * (i + 0.5)


def _dct_exact(x, kind):
    """REDFT10 (kind 2) or REDFT01 (kind 3) of the rows of x, through a
    complex FFT of twice the length in extended precision."""
    x = x.cpu().numpy().astype(np.longdouble)
    b, n = x.shape
    pi = np.longdouble("3.14159265358979323846264338327950288")
    ph = pi * np.arange(n, dtype=np.longdouble) / (2 * n)
    if kind == 2:
        f = np.fft.fft(np.concatenate([x, np.zeros_like(x)], axis=1), axis=1)[:, :n]
        y = 2 * (np.cos(ph) * f.real + np.sin(ph) * f.imag)
    else:
        c = x * (np.cos(ph) + 1j * np.sin(ph))
        c[:, 0] *= 0.5
        f = np.fft.ifft(np.concatenate([c, np.zeros_like(c)], axis=1), axis=1)[:, :n] * (2 * n)
        y = 2 * f.real
    return torch.from_numpy(y.astype(np.float64))


def exact(case, seed):
    k = case["kind"]
    x = _input(case, seed)
    if k == "single":
        x = x[None]
        if case["direction"] == BOTH:
            f = _direct(x, L2C)
            return {"forward": f[0], "back": _direct(f, C2L)[0]}
        return _direct(x, case["direction"])[0]
    if k == "host":
        return _direct(x[None], case["direction"])[0].cpu().numpy()
    if k == "lines":
        return _direct(x, case["direction"])
    if k == "grid":
        d = x.dim()
        out = []
        for direction, axes in ((L2C, reversed(range(d))), (C2L, range(d))):
            for axis in axes:
                t = x.movedim(axis, -1)
                x = _direct(t.reshape(-1, t.shape[-1]), direction).view(t.shape).movedim(-1, axis)
                x = x.contiguous()
            out.append(x)
        return {"forward": out[0], "back": out[1]}
    if k == "batch":
        n = _lengths(case)
        out = torch.empty_like(x)
        o = 0
        for m in n.tolist():
            out[o:o + m] = _direct(x[None, o:o + m], case["direction"])[0]
            o += m
        return out
    return _dct_exact(x, case["type"])
