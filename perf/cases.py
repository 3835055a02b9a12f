"""Performance cases: the analyses that users of this framework run, through
its public entry points.

Each case is a plain dict; ``prepare`` makes what a program holds before the
call (frames on the device, a plan and its buffers, or host frames), ``run``
makes one pass, ``exact`` gives the same outputs in 64 bits with plain torch.
Single-precision analyses (``fp32c``) return float32 and double-precision ones
float64, the two result types of the front end.
"""

import ctypes
import math

import numpy as np
import torch

import fastddm_amd as fddm
from fastddm_amd import _core_hip as core
from fastddm_amd import next_fast_len
from fastddm_amd.azimuthalaverage import azimuthal_average_device
from fastddm_amd.lags import logspace_int
from fastddm_amd.window import blackman_harris

# image formats of the uneven batches, and the most pixels a drawn stack has
BATCH_SHAPES = ((96, 96), (150, 200), (384, 384), (480, 640))
MOST_PIXELS = 4000 * 1024 * 1024
PIXELS = {"uint8": np.uint8, "uint16": np.uint16, "float32": np.float32}
SPECKLE = {  # mean, standard deviation of the frames
    "uint8": (120.0, 25.0),
    "uint16": (1000.0, 150.0),
    "float32": (1000.0, 150.0),
}


def _plan(name, mode, L, H, W, dtype, precision, lags, window):
    """lags: 0 for every lag, else that many logarithmically spaced ones."""
    return {"name": name, "kind": "plan", "mode": mode, "L": L, "H": H, "W": W, "dtype": dtype,
            "precision": precision, "lags": lags, "window": window}


def listed():
    return [
        # the smallest analysis: a short clip of a small region of interest
        _plan("fft_64x128x128_fp32c", "fft", 64, 128, 128, "uint16", "fp32c", 0, False),
        # the ordinary movie: a 512^2 camera, every lag, windowed, in both precisions
        _plan("fft_2000x512x512_fp32c", "fft", 2000, 512, 512, "uint16", "fp32c", 0, True),
        _plan("fft_2000x512x512_fp64", "fft", 2000, 512, 512, "uint16", "fp64", 0, True),
        # a shorter 8-bit movie at logarithmically spaced lags, an odd frame count
        _plan("fft_1003x512x512_fp32c_log", "fft", 1003, 512, 512, "uint8", "fp32c", 80, True),
        # a camera format that is no power of two, float frames (already corrected or normalised)
        _plan("fft_997x480x640_fp32c", "fft", 997, 480, 640, "float32", "fp32c", 0, False),
        # an odd-sized crop in double precision; the transform is padded
        _plan("fft_271x147x201_fp64", "fft", 271, 147, 201, "uint16", "fp64", 0, False),
        # the largest movie
        _plan("fft_4000x1024x1024_fp32c", "fft", 4000, 1024, 1024, "uint16", "fp32c", 0, True),
        # direct differences at a few lags: a short movie, and a larger one in double precision
        _plan("diff_300x256x256_fp32c", "diff", 300, 256, 256, "uint8", "fp32c", 50, False),
        _plan("diff_1200x512x512_fp64", "diff", 1200, 512, 512, "uint16", "fp64", 60, True),
        # many stacks of uneven sizes and lengths in one launch
        {"name": "batch_16_stacks_fp32c", "kind": "batch", "stacks": 16, "longest": 1500},
        # one blocking call from host frames to a host result, in the front end's default precision
        {"name": "ddm_500x256x256_host", "kind": "host", "mode": "fft", "L": 500, "H": 256, "W": 256,
         "dtype": "uint16", "precision": "fp64", "lags": 60, "window": True},
        # azimuthal average with errors of a result on the device
        {"name": "azimuthal_502x512x512", "kind": "azimuthal", "rows": 502, "H": 512, "W": 512, "bins": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("plan", "host", "azimuthal", "batch"), (78, 8, 7, 7))[0]
    if kind == "batch":
        return {"kind": kind, "stacks": rng.randint(3, 16), "longest": _log_int(rng, 80, 1500)}
    square = rng.random() < 0.4
    H = rng.choice((64, 128, 256, 512, 1024)) if square else _log_int(rng, 60, 1030)
    W = H if square else _log_int(rng, 60, 1030)
    if kind == "azimuthal":
        return {"kind": kind, "rows": _log_int(rng, 20, 700), "H": min(H, 600), "W": min(W, 600), "bins": rng.randint(10, 80)}
    mode = "fft" if rng.random() < 0.75 else "diff"
    precision = "fp64" if kind == "host" or rng.random() < 0.35 else "fp32c"
    most = MOST_PIXELS // (32 if kind == "host" else 4 if precision == "fp64" or mode == "diff" else 1)
    L = _log_int(rng, 20, min(4000, max(40, most // (H * W))))
    lags = 0 if mode == "fft" and kind == "plan" and rng.random() < 0.6 else _log_int(rng, 8, 80)
    return {"kind": kind, "mode": mode, "L": L, "H": H, "W": W, "dtype": rng.choice(("uint16", "uint16", "uint8", "float32")),
            "precision": precision, "lags": min(lags, L // 2), "window": rng.random() < 0.5}


# ---- inputs ----
def _speckle(L, H, W, dtype, seed):
    """(L, H, W) frames on the device: AR(1) speckle (each wavevector relaxes
    at D q^2, as for Brownian particles), shot noise, the camera's type.
    uint16 frames come as an int16 tensor of the same bits (values < 2^15)."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    mean, std = SPECKLE[dtype]
    ky = 2 * math.pi * torch.fft.fftfreq(H, device="cuda")
    kx = 2 * math.pi * torch.fft.rfftfreq(W, device="cuda")
    q2 = ky[:, None] ** 2 + kx[None, :] ** 2
    env = torch.exp(-0.5 * q2 * 1.5 ** 2)
    rho = torch.exp(-0.2 * q2)
    kick = torch.sqrt(1 - rho * rho) * env
    # standard deviation of one frame: each half-plane amplitude has unit complex variance
    full = torch.full_like(env, 2.0)
    full[:, 0] = 1.0
    scale = std / math.sqrt(float((full * env * env).sum()))

    def noise():
        return torch.randn((H, W // 2 + 1), generator=g, device="cuda", dtype=torch.complex64)

    out = torch.empty((L, H, W), device="cuda", dtype={"uint8": torch.uint8, "uint16": torch.int16, "float32": torch.float32}[dtype])
    amp = noise() * env
    step = max(1, min(64, (1 << 26) // (H * W)))
    for t0 in range(0, L, step):
        n = min(step, L - t0)
        block = torch.empty((n, H, W // 2 + 1), device="cuda", dtype=torch.complex64)
        for i in range(n):
            block[i] = amp
            amp = rho * amp + kick * noise()
        x = torch.fft.irfft2(block, s=(H, W), norm="forward") * scale + mean
        x = x + torch.sqrt(x.clamp(min=0)) * torch.randn(x.shape, generator=g, device="cuda")
        out[t0:t0 + n] = x if dtype == "float32" else x.round().clamp(0, 255 if dtype == "uint8" else 32000).to(out.dtype)
    return out


def _lags(case):
    L, n = case["L"], case["lags"]
    return np.arange(1, L) if n == 0 else logspace_int(L - 1, num=n)


def _window(case):
    return blackman_harris((case["H"], case["W"])) if case["window"] else None


class _Buffer:
    """A tensor's memory in the shape of the library's device buffers."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())
        self.nbytes = tensor.numel() * tensor.element_size()


def _out_type(precision):
    return (np.float64, torch.float64) if precision == "fp64" else (np.float32, torch.float32)


def _batch_stacks(case, seed):
    """(L, H, W) of every stack: frames log-uniform in [50, longest], the shapes in turn."""
    lengths = np.exp(np.linspace(math.log(50), math.log(case["longest"]), case["stacks"])).round().astype(int)
    order = np.random.default_rng(4).permutation(case["stacks"])
    return [(int(lengths[order[k]]),) + BATCH_SHAPES[k % 4] for k in range(case["stacks"])]


def _result(case, seed):
    """A (rows, ny, nxh) analysis result on the device: saturating D(q, dt) with counting noise."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    rows, ny, nx = case["rows"], next_fast_len(case["H"], "hip"), next_fast_len(case["W"], "hip")
    ky = 2 * math.pi * torch.fft.fftshift(torch.fft.fftfreq(ny, device="cuda", dtype=torch.float64))
    kx = 2 * math.pi * torch.fft.fftfreq(nx, device="cuda", dtype=torch.float64)[: nx // 2 + 1]
    q2 = ky[:, None] ** 2 + kx.abs()[None, :] ** 2
    data = torch.empty((rows, ny, nx // 2 + 1), device="cuda", dtype=torch.float64)
    for i in range(rows):
        rise = 1 - torch.exp(-0.2 * q2 * (i + 1)) if i < rows - 2 else torch.ones_like(q2)
        noise = 1 + 0.1 * torch.randn(q2.shape, generator=g, device="cuda", dtype=torch.float64)
        data[i] = (2e4 * torch.exp(-2.25 * q2) * rise + 2000.0) * noise
    return data, kx.cpu().numpy(), ky.cpu().numpy(), nx


def prepare(case, seed):
    kind = case["kind"]
    core.set_device(0)
    if kind == "azimuthal":
        data, kx, ky, nx = _result(case, seed)
        return {"kind": kind, "data": _Buffer(data), "shape": tuple(data.shape), "kx": kx, "ky": ky, "width": nx,
                "tau": np.arange(1, case["rows"] - 1, dtype=np.float64), "bins": case["bins"]}
    if kind == "batch":
        items = []
        for k, (L, H, W) in enumerate(_batch_stacks(case, seed)):
            img = _speckle(L, H, W, "uint16", seed * 1000 + k)
            out = torch.empty((L + 1, H, W // 2 + 1), device="cuda", dtype=torch.float32)
            items.append(dict(mode="fft", img=_Buffer(img), shape=(L, H, W), dtype=np.uint16, lags=np.arange(1, L), nx=W, ny=H,
                              nt=next_fast_len(2 * L, "hip"), precision="fp32c", out_dtype=np.float32, out=_Buffer(out)))
        torch.cuda.synchronize()
        return {"kind": kind, "batch": core.Batch(items), "outs": [it["out"].tensor for it in items]}
    L, H, W = case["L"], case["H"], case["W"]
    img = _speckle(L, H, W, case["dtype"], seed)
    if kind == "host":
        return {"kind": kind, "img": img.cpu().numpy().view(PIXELS[case["dtype"]]), "lags": _lags(case), "mode": case["mode"],
                "window": _window(case), "precision": case["precision"]}
    nx, ny, nt = next_fast_len(W, "hip"), next_fast_len(H, "hip"), next_fast_len(2 * L, "hip")
    np_out, torch_out = _out_type(case["precision"])
    plan = core.Plan(case["mode"], PIXELS[case["dtype"]], (L, H, W), _lags(case), nx, ny, nt, _window(case),
                     case["precision"], np_out)
    out = torch.empty(plan.out_shape, device="cuda", dtype=torch_out)
    work_space = torch.empty(plan.workspace_size(), device="cuda", dtype=torch.uint8)
    return {"kind": kind, "plan": plan, "img": _Buffer(img), "out": _Buffer(out), "ws": _Buffer(work_space)}


def _parts(out):
    """D, the power spectrum and the variance of a (NL+2, ny, nxh) result."""
    return [out[:-2], out[-2], out[-1]]


def run(state):
    kind = state["kind"]
    if kind == "plan":
        state["plan"].execute(state["img"], state["out"], state["ws"])
        return _parts(state["out"].tensor)
    if kind == "batch":
        state["batch"].launch()
        return [_parts(o) for o in state["outs"]]
    if kind == "host":
        isf = fddm.ddm(state["img"], state["lags"], core="hip", mode=state["mode"], window=state["window"],
                       precision=state["precision"])
        return [isf.data, isf.power_spec, isf.var]
    avg = azimuthal_average_device(state["data"], state["shape"], state["kx"], state["ky"], state["tau"], state["width"],
                                   np.float64, bins=state["bins"])
    return [avg.data, avg.err, avg.power_spec, avg.power_spec_err, avg.var, avg.var_err, avg.k]


# ---- what a pass cannot do without ----
def _stack_work(L, H, W, b_in, nl, b_out, mode, window):
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    nq = ny * (nx // 2 + 1)
    flops = L * 2.5 * nx * ny * math.log2(nx * ny)
    if mode == "fft":
        n = 2 * L
        flops += nq * (5 * n * math.log2(n) + 2.5 * n * math.log2(n) + 4 * n)
    else:
        flops += nq * 6.0 * (nl * L if nl < L else L * L / 2)
    return L * H * W * b_in + (nl + 2) * nq * b_out + (H * W * 8 if window else 0), flops


def work(case):
    kind = case["kind"]
    if kind == "azimuthal":
        n = case["rows"] * next_fast_len(case["H"], "hip") * (next_fast_len(case["W"], "hip") // 2 + 1)
        return {"bytes": 8 * n + 16 * case["rows"] * case["bins"], "flops": 6 * n}
    if kind == "batch":
        parts = [_stack_work(L, H, W, 2, L - 1, 4, "fft", False) for L, H, W in _batch_stacks(case, 0)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    b_in = np.dtype(PIXELS[case["dtype"]]).itemsize
    b_out = 8 if case["precision"] == "fp64" else 4
    b, f = _stack_work(case["L"], case["H"], case["W"], b_in, len(_lags(case)), b_out, case["mode"], case["window"])
    return {"bytes": b, "flops": f}


# ---- the same in 64 bits ----
def _exact_stack(img, lags, window, mode):
    """(NL+2, ny, nxh) float64: D = <|F(t+dt) - F(t)|^2>, <|F|^2> and the
    variance of F, fftshifted along y.  D from the time FFT of the series
    without its mean (D does not depend on it), or from the differences."""
    L, H, W = img.shape
    nx, ny = next_fast_len(W, "hip"), next_fast_len(H, "hip")
    nxh = nx // 2 + 1
    win = None if window is None else torch.from_numpy(np.asarray(window, dtype=np.float64)).cuda()
    F = torch.empty((L, ny * nxh), device="cuda", dtype=torch.complex128)
    step = max(1, (1 << 26) // (nx * ny))
    for t in range(0, L, step):
        x = img[t:t + step].to(torch.float64)
        if win is not None:
            x = x * win
        F[t:t + step] = torch.fft.rfft2(x, s=(ny, nx), norm="ortho").reshape(x.shape[0], -1)
    lag = torch.as_tensor(np.asarray(lags), device="cuda", dtype=torch.int64)
    out = torch.empty((len(lags) + 2, ny * nxh), device="cuda", dtype=torch.float64)
    n = 1 << (2 * L - 1).bit_length()
    cols = max(1, (1 << 27) // n)
    for c in range(0, ny * nxh, cols):
        f = F[:, c:c + cols].T.contiguous()
        m = f.mean(dim=1, keepdim=True)
        f = f - m
        p = f.real ** 2 + f.imag ** 2
        var = p.mean(dim=1)
        out[-2, c:c + cols] = var + (m.real ** 2 + m.imag ** 2)[:, 0]
        out[-1, c:c + cols] = var
        if mode == "diff":
            for i, d in enumerate(lags):
                e = f[:, d:] - f[:, : L - d]
                out[i, c:c + cols] = (e.real ** 2 + e.imag ** 2).mean(dim=1)
            continue
        s = torch.fft.fft(f, n=n, dim=1)
        corr = torch.fft.ifft(s.real ** 2 + s.imag ** 2, dim=1).real
        head = torch.cumsum(p, dim=1)
        num = head[:, L - 1 - lag] + (head[:, -1:] - head[:, lag - 1]) - 2 * corr[:, lag]
        out[:-2, c:c + cols] = (num / (L - lag)).T
    return torch.fft.fftshift(out.reshape(-1, ny, nxh), dim=1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "azimuthal":
        return _exact_average(case, seed)
    if kind == "batch":
        return [_parts(_exact_stack(_speckle(L, H, W, "uint16", seed * 1000 + k), np.arange(1, L), None, "fft"))
                for k, (L, H, W) in enumerate(_batch_stacks(case, seed))]
    img = _speckle(case["L"], case["H"], case["W"], case["dtype"], seed)
    return _parts(_exact_stack(img, _lags(case), _window(case), case["mode"]))


def _exact_average(case, seed):
    """Weighted mean and its error per ring of |k|; each half-plane pixel
    counts for itself and its mirror image."""
    data, kx, ky, nx = _result(case, seed)
    rows, ny, nxh = data.shape
    X, Y = np.meshgrid(kx, ky)
    dist = np.sqrt(X ** 2 + Y ** 2)
    edges = np.linspace(dist.min(), dist.max(), case["bins"])
    counts = np.full(dist.shape, 2.0)
    counts[:, 0] = 1.0
    if nx % 2 == 0:
        counts[:, -1] = 1.0
    ring = np.searchsorted(edges, dist)
    flat = data.reshape(rows, -1)
    avg = torch.full((case["bins"], rows), float("nan"), dtype=torch.float64)
    err = torch.full((case["bins"], rows), float("nan"), dtype=torch.float64)
    k = np.empty(case["bins"])
    for b in range(case["bins"]):
        at = np.flatnonzero(ring.ravel() == b)
        if not len(at):
            k[b] = 0.5 * (edges[b - 1] + edges[b]) if b else edges[0]
            continue
        w = torch.from_numpy(counts.ravel()[at]).cuda()
        x = flat[:, torch.from_numpy(at).cuda()]
        sw = w.sum()
        mean = (x * w).sum(dim=1) / sw
        avg[b] = mean.cpu()
        err[b] = torch.sqrt((w * (x - mean[:, None]) ** 2).sum(dim=1) / (sw - w.sum() / sw)).cpu()
        k[b] = float((counts.ravel()[at] * dist.ravel()[at]).sum() / counts.ravel()[at].sum())
    return [avg[:, :-2], err[:, :-2], avg[:, -2], err[:, -2], avg[:, -1], err[:, -1], k]
