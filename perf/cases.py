"""What is timed: the SOI transforms a program has this library do, through its public calls.

A case is one transform shape (or a batch of them) with its options.  The transform works in
place, so a program that keeps its samples copies them into the work buffer and transforms that:
run() does the same.  Sizes are the ones the tests, the benchmark and its batching workload use,
their neighbours with other odd factors, and the sizes between.

  kind   "device"  compute_soi_async on device memory, on the program's stream
         "call"    compute_soi on device memory: the blocking call, one transform at a time
         "host"    compute_soi on host memory, as a program written for the CPU library calls it
         "batch"   soi_batch_run: one graph of many transforms
  window "default" mu = 5/4, B = 72; "b76", "b64", "b44", "b30": the other rows of the accuracy
         table (fewer taps, less accuracy); "mu87": mu = 8/7, which exchanges less data
  vlc    the exchanged data go through the VLC codec
"""
import math

import numpy as np
import torch

import soi_fft_amd as soi

WINDOWS = {
    "default": dict(),
    "b76": dict(B=76, tau=872 / 1024, sigma=313.1715),
    "b64": dict(B=64, tau=818 / 1024, sigma=267.4513),
    "b44": dict(B=44, tau=512 / 1024, sigma=121.0936),
    "b30": dict(B=30, tau=0.154, sigma=73.2102363),
    "mu87": dict(n_mu=8, d_mu=7, tau=0.7, sigma=360.0),
}

BATCH_SIZES = (2 ** 16, 3 * 2 ** 15, 2 ** 18, 5 * 2 ** 16, 2 ** 20)
BATCH_P = (8, 16, 32)


def _one(name, kind, N, P, k=1, single=False, window="default", vlc=False):
    c = dict(kind=kind, N=N, P=P, k=k, single=single, window=window, vlc=vlc)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one small block at a time, each waited for: latency and launches
        _one("call_2e13", "call", 2 ** 13, 4),
        # a small uneven block in single precision, one of a stream of them
        _one("c64_3x2e15", "device", 3 * 2 ** 15, 16, single=True),
        # the reference driver's default run: host memory, 8 ranks
        _one("host_2e20", "host", 2 ** 20, 8),
        # an ordinary block whose length has a factor 9 (frames, sample rates in decimal units)
        _one("c128_45x2e16", "device", 45 * 2 ** 16, 8),
        # a narrow window: less accuracy asked for, fewer taps
        _one("c128_b44_2e22", "device", 2 ** 22, 16, window="b44"),
        # little oversampling: less data between the steps
        _one("c128_mu87_7x2e20", "device", 7 * 2 ** 20, 32, window="mu87"),
        # several segments per rank: 64 in all
        _one("c128_k2_2e24", "device", 2 ** 24, 32, k=2),
        # a long block with an odd factor, single precision
        _one("c64_27x2e20", "device", 27 * 2 ** 20, 16, single=True),
        # many independent blocks of uneven lengths and ranks, one launch
        dict(name="batch_c128_192", kind="batch", count=192, single=False, pick=2028),
        # a banded spectrum exchanged through the VLC codec
        _one("c128_vlc_7x2e23", "device", 7 * 2 ** 23, 64, window="mu87", vlc=True),
        # the largest transforms, in both precisions
        _one("c64_2e27", "device", 2 ** 27, 32, single=True),
        _one("c128_2e27", "device", 2 ** 27, 32),
    ]


def _valid(c):
    kw = WINDOWS[c["window"]]
    S, B, d, n = c["k"] * c["P"], kw.get("B", 72), kw.get("d_mu", 4), kw.get("n_mu", 5)
    if c["N"] % S or not 4 <= S <= 64:
        return False
    M = c["N"] // S
    # the library's own conditions (P*d_mu divides M, M/P >= B), and segments of 2^10 to 2^22
    # rows
    return M % (c["P"] * d) == 0 and M // c["P"] >= B and 1024 <= M <= 2 ** 22 and n * M // d <= 5 * 2 ** 20


def draw(rng):
    """One more case: lengths odd * 2^e spread over their logarithm; the odd factors are the ones
    blocks come in (1, 3, 5, 9, 15, 25, 27, 45, 75)."""
    what = rng.choice(["device"] * 7 + ["call", "host", "batch"])
    if what == "batch":
        return dict(kind="batch", count=rng.randrange(24, 193), single=rng.random() < 0.5,
                    pick=rng.randrange(1 << 20))
    while True:
        single = rng.random() < 0.45
        # single precision goes with the wide windows: the others' gain at the segments' edges
        # leaves it too few digits
        window = rng.choice(["default"] * 6 + ["b76", "b64"] +
                            ([] if single else ["b44", "b30", "mu87", "mu87"]))
        odd = rng.choice([1, 1, 3, 5, 9, 15, 25, 27, 45, 75])
        vlc = not single and what == "device" and rng.random() < 0.2
        top = {"device": 26.5, "call": 18, "host": 21}[what]
        if window != "default" or odd != 1 or vlc:
            top = min(top, 25.0)  # no more work than the largest listed case
        want = 2.0 ** rng.uniform(13, top)
        if window == "mu87":
            odd *= 7
        N = odd * 2 ** max(6, round(math.log2(want / odd)))
        c = _one(None, what, N, rng.choice([4, 8, 8, 16, 16, 32, 32, 64]), rng.choice([1, 1, 1, 2]),
                 single, window, vlc)
        if N <= 2.0 ** (top + 0.5) and _valid(c):
            return c


def _batch_shapes(case):
    """(N, P) of the members: uniform over the sizes and ranks, as a queue of requests fills."""
    r = np.random.default_rng(case["pick"])
    shapes = []
    while len(shapes) < case["count"]:
        n, p = int(r.choice(BATCH_SIZES)), int(r.choice(BATCH_P))
        if (n, p) != (2 ** 16, 32):  # M/P < B
            shapes.append((n, p))
    return shapes


def _dtype(case):
    return torch.complex64 if case["single"] else torch.complex128


def _samples(case, seed):
    """The samples: uniform noise in [-1, 1]; long blocks and VLC blocks are tones over a noise
    floor, the VLC ones all in one band of width N/P."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    N = sum(n for n, _ in _batch_shapes(case)) if case["kind"] == "batch" else case["N"]
    x = torch.rand((N, 2), generator=g, device="cuda", dtype=torch.float64)
    x = torch.view_as_complex(x.mul_(2).sub_(1))
    tones = 0 if case["kind"] == "batch" else 24 if case["vlc"] else 8 if N >= 2 ** 24 else 0
    if tones:
        x.mul_(1e-3)
        r = np.random.default_rng(seed)
        lo, width = (int(r.integers(0, case["P"])) * (N // case["P"]), N // case["P"]) if case["vlc"] else (0, N)
        t = torch.arange(N, device="cuda", dtype=torch.float64).mul_(2 * math.pi / N)
        for _ in range(tones):
            f, a = lo + float(r.uniform(0, width)), float(r.uniform(0, 2 * math.pi))
            ang = t * f + a
            part = torch.view_as_real(x)
            part[:, 0] += torch.cos(ang)
            part[:, 1] += torch.sin(ang)
            del ang
    return x.to(_dtype(case))


class _Transform:
    """One descriptor and its buffers; released with the object."""

    def __init__(self, case, x):
        self.desc = None
        self.kind, self.x = case["kind"], x
        if self.kind == "host":
            self.x = x.cpu().numpy()
            self.buf = np.empty_like(self.x)
        else:
            self.buf = torch.empty_like(x)
        self.desc = soi.make_descriptor(
            case["N"], case["P"], case["k"], use_vlc=case["vlc"],
            precision=soi.SOI_PREC_FP32 if case["single"] else soi.SOI_PREC_FP64,
            **WINDOWS[case["window"]])
        self.ptr = self.buf.ctypes.data if self.kind == "host" else self.buf.data_ptr()
        self.handle = soi.stream_of(self.desc)
        self.stream = torch.cuda.ExternalStream(self.handle)

    def run(self):
        if self.kind == "host":
            np.copyto(self.buf, self.x)
            soi.compute_soi(self.desc, self.ptr)
            return self.buf
        with torch.cuda.stream(self.stream):
            self.buf.copy_(self.x)
        if self.kind == "call":
            soi.compute_soi(self.desc, self.ptr)
        else:
            soi.compute_soi_async(self.desc, self.ptr, self.handle)
        return self.buf

    def __del__(self):
        if self.desc is not None:
            torch.cuda.synchronize()
            soi.free_soi_descriptor(self.desc)


class _Batch:
    """Many descriptors over one allocation, captured into one graph."""

    def __init__(self, case, x):
        self.descs, self.batch = [], None
        self.x, self.buf = x, torch.empty_like(x)
        prec = soi.SOI_PREC_FP32 if case["single"] else soi.SOI_PREC_FP64
        ptrs, at = [], 0
        for n, p in _batch_shapes(case):
            self.descs.append(soi.make_descriptor(n, p, precision=prec))
            ptrs.append(self.buf.data_ptr() + at * x.element_size())
            at += n
        self.batch = soi.Batch(self.descs, ptrs, autotune=False)
        self.stream = torch.cuda.ExternalStream(self.batch.stream)

    def run(self):
        with torch.cuda.stream(self.stream):
            self.buf.copy_(self.x)
        self.batch.run()
        return self.buf

    def __del__(self):
        torch.cuda.synchronize()
        if self.batch is not None:
            self.batch.close()
        for d in self.descs:
            soi.free_soi_descriptor(d)


def prepare(case, seed):
    x = _samples(case, seed)
    state = (_Batch if case["kind"] == "batch" else _Transform)(case, x)
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()


def work(case):
    shapes = _batch_shapes(case) if case["kind"] == "batch" else [(case["N"], case["P"])]
    size = 8 if case["single"] else 16
    return {"bytes": sum(2.0 * size * n for n, _ in shapes),
            "flops": sum(5.0 * n * math.log2(n) for n, _ in shapes)}


def exact(case, seed):
    """The DFT itself, in 64 bits."""
    x = _samples(case, seed).to(torch.complex128)
    if case["kind"] != "batch":
        y = torch.fft.fft(x)
        return y.cpu().numpy() if case["kind"] == "host" else y
    parts, at = [], 0
    for n, _ in _batch_shapes(case):
        parts.append(torch.fft.fft(x[at:at + n]))
        at += n
    return torch.cat(parts)
