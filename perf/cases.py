"""The work that users of this library have it do, as measurable cases.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program
holds before the call (matrices and right-hand sides on the GPU, the plan, batch or requests),
run() is one pass through the public entry points and returns its whole result, work() the
bytes and operations of a pass that no implementation can do without, exact() the result in
64 bits by plain torch.

The step runs in place and a time-stepping program applies it to the result of its last pass,
so the matrices here are those of a step that neither blows up nor dies out: the fused step's
V = D (I - A) M and T = D (I + A) with a skew-symmetric tridiagonal A (a Crank-Nicolson step of
a rotation) make M^-1 T^-1 V similar to an orthogonal matrix, the bidiagonal step multiplies
by a product of plane rotations, the tridiagonal solve is an implicit diffusion step.
"""
import math
import random

import numpy as np
import torch

import pfsolve_amd as pf

DEV = "cuda"


# ---------------------------------------------------------------- cases

def listed():
    return [
        # the smallest step in use: 1024 short real systems, one launch, latency
        dict(name="small", kind="fused", N=64, nsys=1024, stride=64, natural=False),
        # a truncation that is odd, systems packed one after the other (no 16-byte alignment)
        dict(name="odd_packed", kind="fused", N=333, nsys=30000, stride=333, natural=False),
        # long radial expansions, complex fields (pairs of real systems)
        dict(name="rows_1000", kind="fused", N=1000, nsys=16384, stride=1000, natural=False),
        # the longest a wavefront holds, matrices in natural order
        dict(name="rows_2000", kind="fused", N=2000, nsys=8192, stride=2000, natural=True),
        # throughput: complex strided input scaled on the way in, rows [480, 512) kept, real systems out
        dict(name="throughput", kind="blocks", N=512, ncx=65536, in_op=1, out_op=-1, keep_lo=480, keep_hi=512),
        # complex in and out around the step, added to a field already there
        dict(name="blocks_accumulate", kind="blocks", N=384, ncx=16384, in_op=2, out_op=0, keep_lo=0, keep_hi=384),
        # one plain bidiagonal step (multiply by one connection matrix, solve another) at runtime offsets
        dict(name="connection", kind="mode", jw=10, ub=1, N=256, nsys=8192, runtime=True),
        # one matrix set and 32 complex fields for each harmonic degree, sizes falling with the degree
        dict(name="degrees", kind="batch", degrees=1024, nmax=1024, halving=2, nsys=64, resident=False),
        # extended precision
        dict(name="double_double", kind="dd", N=256, nsys=16384),
        # four connection steps of falling size in one call
        dict(name="chain", kind="chain", N=512, K=4, nsys=65536),
        # few very long systems
        dict(name="long", kind="long", N=100000, nsys=512),
        # a burst of requests from host memory, every one with its own size and matrices
        dict(name="burst", kind="serve", requests=48, nmax=2048, cmax=1024, mix=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fused", "fused", "fused", "fused", "blocks", "blocks", "mode", "mode", "batch", "batch",
                       "dd", "chain", "long", "serve"])
    rows = math.exp(rng.uniform(math.log(1 << 16), math.log(40 << 20)))   # rows of all systems together
    if kind == "fused":
        N = _log(rng, 17, 2048)
        stride = N if rng.random() < 0.5 else N + N % 2
        return dict(kind=kind, N=N, nsys=max(2, int(rows / N)), stride=stride, natural=rng.random() < 0.3)
    if kind == "blocks":
        N = _log(rng, 17, 512)
        hi = N if rng.random() < 0.5 else rng.randint(N // 2, N)
        return dict(kind=kind, N=N, ncx=max(1, int(rows / N / 2)), in_op=rng.choice([1, 2]),
                    out_op=rng.choice([-1, 0, 1]), keep_lo=0, keep_hi=hi)
    if kind == "mode":
        jw, ub = rng.choice([(10, 0), (10, 1), (13, 2)])
        N = _log(rng, 17, 1024)
        return dict(kind=kind, jw=jw, ub=ub, N=N, nsys=max(2, int(rows / N)), runtime=jw == 10 and rng.random() < 0.5)
    if kind == "batch":
        degrees, nmax = _log(rng, 16, 1024), _log(rng, 64, 1024)
        halving = max(2, -(-2 * degrees // nmax))     # the smallest system keeps about half the rows
        nsys = 2 * rng.randint(1, 32)
        return dict(kind=kind, degrees=degrees, nmax=nmax, halving=halving, nsys=nsys, resident=rng.random() < 0.5)
    if kind == "dd":
        N = _log(rng, 17, 512)
        return dict(kind=kind, N=N, nsys=max(2, int(rows / N / 8)))
    if kind == "chain":
        N, K = _log(rng, 32, 1024), rng.choice([2, 3, 4, 8])
        return dict(kind=kind, N=N, K=K, nsys=2 * max(1, int(rows / N / 2)))
    if kind == "long":
        N = _log(rng, 2049, 100000)
        return dict(kind=kind, N=N, nsys=max(2, min(4096, int(rows / N))))
    return dict(kind=kind, requests=rng.randint(4, 40), nmax=_log(rng, 64, 2048), cmax=_log(rng, 80, 1024),
                mix=rng.randrange(1 << 20))


# ---------------------------------------------------------------- matrices

def storage_order(N, layout=None):
    """Position of row i of a stored diagonal: registers of the layout one after the other, each
    over the lanes; beyond 3840 rows in blocks of 704."""
    block = N if N <= 3840 else 704
    size = (layout or N) if N <= 3840 else 704
    lanes = 64 if size < 512 else (size + 1023) // 1024 * 64
    R = -(-size // lanes)
    R += R % 2 == 0
    out = np.empty(N, dtype=np.int64)
    for base in range(0, N, block):
        n = min(block, N - base)
        i = np.arange(n)
        k, q = i % R, i // R
        big = n % R
        out[base:base + n] = base + q + np.where(k < big, k * (-(-n // R)), big * (-(-n // R)) + (k - big) * (n // R))
    return out


def fused_parts(N, rng):
    """V [5, N] by column (entry [j, c] in row c - 2 + j), and the stored diagonals of T and M:
    a/b, 1/b, c/b and 1/d, e/d, in natural order."""
    a, D = rng.uniform(-0.5, 0.5, N + 2), rng.uniform(2, 3, N)
    d, e = rng.uniform(1, 2, N + 2), rng.uniform(-0.5, 0.5, N + 2)
    a[0] = 0.0
    a[N:] = 0.0
    e[N - 1:] = 0.0
    r = np.arange(N)
    rows = np.zeros((5, N))              # [4 - (column - row + 2), row]
    rows[4] = 1e-9 * rng.uniform(-1, 1, N)
    rows[3] = -D * a[r] * d[r - 1]
    rows[2] = D * (d[r] - a[r] * e[r - 1] * (r > 0))
    rows[1] = D * (e[r] + a[r + 1] * d[r + 1])
    rows[0] = D * a[r + 1] * e[r + 1]
    V = np.zeros((5, N))
    for j in range(5):                   # row c - 2 + j
        c = np.arange(max(0, 2 - j), min(N, N + 2 - j))
        V[j, c] = rows[j, c - 2 + j]
    ld, md, ud = D * a[:N], D, -D * a[1:N + 1]
    return V, ld / md, 1.0 / md, ud / md, 1.0 / d[:N], e[:N] / d[:N]


def pack_fused(parts, natural, pad=0):
    V, ld, md, ud, dm, em = parts
    N = V.shape[1]
    P = np.arange(N) if natural or N <= 64 else storage_order(N)
    buf = np.zeros(10 * N + pad)
    buf[:5 * N] = V.ravel()
    for k, x in enumerate((ld, md, ud, dm, em)):
        buf[(5 + k) * N + P] = x
    return buf


def mode_parts(case, rng):
    """Diagonals of one reference step. jw 10: (D + off) then the unit bidiagonal solve, whose
    product is a chain of plane rotations; jw 13: a tridiagonal solve (I + weighted Laplacian)."""
    N = case["N"]
    if case["jw"] == 13:
        w = np.concatenate([[0.0], rng.uniform(0, 0.5, N - 1), [0.0]])
        b = 1.0 + w[:-1] + w[1:]
        return -w[:-1] / b, 1.0 / b, -w[1:] / b
    t = rng.uniform(-0.6, 0.6, N - 1)
    c, s = np.concatenate([[1.0], np.cos(t), [1.0]]), np.sin(t)
    D = c[1:] / c[:-1]
    off = np.concatenate([-s, [0.0]])                      # upper: row r couples with r + 1
    low = np.concatenate([[0.0], -s * c[2:] / c[1:-1]])    # lower solve: row r with r - 1
    if case["ub"] == 0:                                    # the same step on the rows in reverse
        return D[::-1].copy(), off[::-1].copy(), low[::-1].copy()
    return D, off, low


def chain_parts(N, K, l):
    """Connection matrices of degree l, normalised by row: (I + up) then the solve of (I + low),
    for N - i rows; the first multiply scales the rows as well."""
    beta = l + 0.5

    def mu(n):
        return np.sqrt(2 * (n + beta) * (n - 0.5 + beta) / (2 * n - 0.5 + beta) / (2 * n + 0.5 + beta))

    def nu(n):
        return np.sqrt(2 * (n + 1) * (n + 0.5) / (2 * n + 0.5 + beta) / (2 * n + 1.5 + beta))
    out = []
    for i in range(K):
        r = np.arange(N - i, dtype=np.float64)
        up, low = nu(r + 1) / mu(r), nu(r) / mu(r)
        low[0] = 0.0
        scale = 0.9 * mu(r) / mu(r[:1]) if i == 0 else np.ones(N - i)
        if i == 0:
            up[-1] = 0.0
            up *= scale
        out.append((scale, up, low))
    return out


def degree_sizes(case):
    return [case["nmax"] - l // case["halving"] for l in range(case["degrees"])]


def request_sizes(case):
    r = random.Random(case["mix"])
    return [(_log(r, 32, case["nmax"]), 2 * _log(r, 64, case["cmax"])) for _ in range(case["requests"])]


def _rng(seed, salt):
    return np.random.default_rng([seed, salt])


def uniform(shape, seed, salt=0):
    g = torch.Generator(device=DEV).manual_seed((seed << 8) + salt)
    return torch.rand(shape, dtype=torch.float64, device=DEV, generator=g).mul_(2).sub_(1)


# ---------------------------------------------------------------- prepare

def _fused_fields(N):
    return dict(jw_type=14, offsetV=0, offsetT=5 * N, offsetM=8 * N, scaleC=1.0)


def prepare(case, seed):
    k = case["kind"]
    if k in ("fused", "long"):
        N, nsys = case["N"], case["nsys"]
        stride, natural = case.get("stride", N), case.get("natural", False)
        mat = torch.from_numpy(pack_fused(fused_parts(N, _rng(seed, 1)), natural)).to(DEV)
        x = uniform((nsys, stride), seed)
        fields = dict(_fused_fields(N), jw_type=1014 if natural else 14)
        plan = pf.Plan(mat.data_ptr(), x.data_ptr(), size=[N, nsys, 1], doublePrecision=1,
                       outputBufferStride=[stride], **fields)
        return dict(kind=k, plan=plan, mat=mat, out=x)
    if k == "dd":
        N, nsys = case["N"], case["nsys"]
        hi = pack_fused(fused_parts(N, _rng(seed, 1)), False)
        lo = _rng(seed, 2).uniform(-1, 1, hi.size) * 2.0 ** -60 * np.abs(hi)
        mat = torch.from_numpy(np.stack([hi, lo], -1)).to(DEV)
        xh = uniform((nsys, N), seed)
        x = torch.stack([xh, uniform((nsys, N), seed, 3) * 2.0 ** -60 * xh.abs()], -1).contiguous()
        plan = pf.Plan(mat.data_ptr(), x.data_ptr(), size=[N, nsys, 1], quadDoubleDoublePrecision=1, **_fused_fields(N))
        return dict(kind=k, plan=plan, mat=mat, out=x)
    if k == "blocks":
        N, ncx = case["N"], case["ncx"]
        mat = torch.from_numpy(pack_fused(fused_parts(N, _rng(seed, 1)), False)).to(DEV)
        field = uniform((ncx, N, 2), seed)
        fields = dict(_fused_fields(N), inputBlock=100 * case["in_op"] + 4, inputBlockLshift=1,
                      inputBlockScale=_in_scale(case), inputBufferStride=[N],
                      inputZeropad=[case["keep_lo"], case["keep_hi"]])
        if case["out_op"] >= 0:
            fields.update(outputBlock=100 * case["out_op"] + 27, outputBlockScale=0.5)
            out = uniform((ncx, N, 2), seed, 4)
        else:
            out = torch.zeros((2 * ncx, N), dtype=torch.float64, device=DEV)
        plan = pf.Plan(mat.data_ptr(), out.data_ptr(), size=[N, 2 * ncx, 1], doublePrecision=1, **fields)
        return dict(kind=k, plan=plan, mat=mat, field=field, out=out)
    if k == "mode":
        N, nsys, ub = case["N"], case["nsys"], case["ub"]
        p = mode_parts(case, _rng(seed, 1))
        P = np.arange(N) if N <= 64 else storage_order(N)
        buf = np.zeros(3 * N)
        launch, mask = {}, 0
        if case["jw"] == 13:                                  # [low | 1/b | up]
            at = (0, N, 2 * N)
        elif case["runtime"]:                                 # upper [up | diag], lower [diag | low], then the solve
            at = (N, 0, 2 * N) if ub else (0, N, 2 * N)
            mask = pf.RUNTIME_OFFSETM | pf.RUNTIME_OFFSETV
            launch = dict(offsetM=0, offsetV=2 * N)
        else:                                                 # upper [diag | up], lower [low | diag], then the solve
            at = (0, N, 2 * N) if ub else (N, 0, 2 * N)
        for base, x in zip(at, p):
            buf[base + P] = x
        mat = torch.from_numpy(buf).to(DEV)
        x = uniform((nsys, N), seed)
        plan = pf.Plan(mat.data_ptr(), x.data_ptr(), size=[N, nsys, 1], doublePrecision=1, jw_type=case["jw"],
                       upperBanded=ub, scaleC=1.0, jw_control_bitmask=mask)
        return dict(kind=k, plan=plan, mat=mat, out=x, launch=launch)
    if k == "chain":
        N, K, nsys = case["N"], case["K"], case["nsys"]
        mats = []
        for i, (scale, up, low) in enumerate(chain_parts(N, K, _degree(seed, N))):
            n = N - i
            P = storage_order(n, N)
            buf = np.zeros(3 * n)
            for base, x in zip((0, n, 2 * n), (scale, up, low) if i == 0 else (up, low)):
                buf[base + P] = x
            mats.append(torch.from_numpy(buf).to(DEV))
        stride = N + N % 2
        x = uniform((nsys, stride), seed)
        plan = pf.Plan([m.data_ptr() for m in mats], x.data_ptr(), size=[N, nsys, 1], doublePrecision=1, jw_type=10,
                       upperBanded=1, scaleC=1.0, numConsecutiveJWIterations=K, useMultipleInputBuffers=K,
                       outputBufferStride=[stride])
        return dict(kind=k, plan=plan, mat=mats, out=x)
    if k == "batch":
        sizes, nsys = degree_sizes(case), case["nsys"]
        bufs = [pack_fused(fused_parts(N, _rng(seed, 10 + l)), False) for l, N in enumerate(sizes)]
        mat = torch.from_numpy(np.concatenate(bufs)).to(DEV)
        total = sum(nsys * (N + N % 2) for N in sizes)
        x = uniform((total,), seed)
        sets, mo, ro = [], 0, 0
        for N in sizes:
            stride = N + N % 2
            sets.append(dict(N=N, nsys=nsys, matrices=mat.data_ptr(), offsetV=mo, offsetT=mo + 5 * N,
                             offsetM=mo + 8 * N, rhs=x.data_ptr() + 8 * ro, stride=stride))
            mo += 10 * N
            ro += nsys * stride
        b = pf.Batch(sets)
        if case["resident"]:
            b.prepare()
        return dict(kind=k, batch=b, mat=mat, out=x, resident=case["resident"])
    # serve
    sizes = request_sizes(case)
    total = sum(N * nsys for N, nsys in sizes)
    rhs_in = torch.empty(total, dtype=torch.float64, pin_memory=True)
    rhs_in.copy_(uniform((total,), seed))
    out = torch.zeros(total, dtype=torch.float64, pin_memory=True)
    reqs, keep, at = [], [], 0
    for i, (N, nsys) in enumerate(sizes):
        buf = pack_fused(fused_parts(N, _rng(seed, 10 + i)), False)
        keep.append(buf)
        reqs.append(dict(N=N, nsys=nsys, matrix_key=i, matrices=buf.ctypes.data, offsetV=0, offsetT=5 * N,
                         offsetM=8 * N, rhs_in=rhs_in.data_ptr() + 8 * at, rhs_out=out.data_ptr() + 8 * at,
                         arrival_s=0.0))
        at += N * nsys
    return dict(kind=k, requests=reqs, keep=keep, rhs_in=rhs_in, out=out)


def _in_scale(case):
    return 0.75 if case["in_op"] == 1 else 0.5


def _degree(seed, N):
    return 2 * N + seed % 97


# ---------------------------------------------------------------- run

def run(state):
    k = state["kind"]
    if k == "blocks":
        state["plan"].append(inputBuffer=state["field"].data_ptr())
    elif k == "mode":
        state["plan"].append(**state["launch"])
    elif k == "batch":
        if state["resident"]:
            state["batch"].solve()
        else:
            state["batch"].run()
    elif k == "serve":
        stats, results = pf.serve(state["requests"], hbm_budget=2 << 30, max_inflight=64, streams=4, max_batch=16)
        if any(status for _, _, status in results):
            raise RuntimeError("a request failed")
    else:
        state["plan"].append()
    x = state["out"]
    return {"hi": x[..., 0], "lo": x[..., 1]} if k == "dd" else x


# ---------------------------------------------------------------- work

def _fused_work(N, nsys, read=None, elt=8):
    read = N if read is None else read
    return elt * (nsys * (read + N) + 10 * N), 18.0 * nsys * N


def work(case):
    k = case["kind"]
    if k in ("fused", "long"):
        b, f = _fused_work(case["N"], case["nsys"])
    elif k == "dd":
        b, f = _fused_work(case["N"], case["nsys"], elt=16)
        f *= 7.5          # a double-double multiply-add: 15 operations
    elif k == "blocks":
        N, n = case["N"], 2 * case["ncx"]
        b, f = _fused_work(N, n, case["keep_hi"] - case["keep_lo"])
        if case["out_op"] >= 0:
            b += 8 * n * N
    elif k == "mode":
        N, n = case["N"], case["nsys"]
        b, f = 8 * (2 * n * N + 3 * N), 5.0 * n * N
    elif k == "chain":
        N, K, n = case["N"], case["K"], case["nsys"]
        b, f = 8 * n * (2 * N - K + 1) + 8 * (2 * K + 1) * N, 4.0 * K * n * N
    else:
        sizes = [(N, case["nsys"]) for N in degree_sizes(case)] if k == "batch" else request_sizes(case)
        parts = [_fused_work(N, n) for N, n in sizes]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------- exact

def _solve_fused(parts, x):
    """x: rows first, [N, ..., systems]; parts' arrays [N, ...] (V: [5, N, ...])."""
    V, ld, md, ud, dm, em = (torch.as_tensor(p, dtype=torch.float64, device=x.device).unsqueeze(-1) for p in parts)
    N = x.shape[0]
    y = torch.zeros_like(x)
    for j in range(5):
        lo, hi = max(0, 2 - j), min(N, N + 2 - j)
        y[lo - 2 + j:hi - 2 + j].addcmul_(V[j, lo:hi], x[lo:hi])
    y *= md
    _tridiagonal(ld, ud, y)
    y *= dm
    for r in range(N - 2, -1, -1):
        y[r].addcmul_(em[r], y[r + 1], value=-1)
    return y


def _tridiagonal(ld, ud, y):
    """y <- (I + low + up)^-1 y, rows first."""
    N = y.shape[0]
    lo, up = ld.squeeze(-1).cpu().numpy(), ud.squeeze(-1).cpu().numpy()
    g, p = np.zeros_like(up), np.ones(lo.shape[1:])
    ip = np.ones_like(lo)
    for r in range(N):
        if r:
            p = 1.0 - lo[r] * g[r - 1]
        ip[r] = 1.0 / p
        g[r] = up[r] / p
    ip, g = (torch.from_numpy(v).to(y.device).unsqueeze(-1) for v in (ip, g))
    for r in range(N):
        if r:
            y[r].addcmul_(ld[r], y[r - 1], value=-1)
        y[r].mul_(ip[r])
    for r in range(N - 2, -1, -1):
        y[r].addcmul_(g[r], y[r + 1], value=-1)


def _rows(x):
    return x.transpose(0, 1).contiguous()


def exact(case, seed):
    k = case["kind"]
    if k in ("fused", "long", "dd"):
        N, nsys = case["N"], case["nsys"]
        x = uniform((nsys, case.get("stride", N)), seed)
        x[:, :N] = _solve_fused(fused_parts(N, _rng(seed, 1)), _rows(x[:, :N])).transpose(0, 1)
        return {"hi": x, "lo": None} if k == "dd" else x
    if k == "blocks":
        N, ncx = case["N"], case["ncx"]
        n = torch.arange(N, dtype=torch.float64, device=DEV)
        s = _in_scale(case)
        row = s if case["in_op"] == 1 else 2 * (n + 2) * torch.sqrt((n + 1) / (n + s + 2.5))
        keep = (n >= case["keep_lo"]) & (n < case["keep_hi"])
        x = uniform((ncx, N, 2), seed).permute(1, 0, 2).reshape(N, 2 * ncx)
        x *= (row * keep).unsqueeze(-1)
        y = _solve_fused(fused_parts(N, _rng(seed, 1)), x)
        if case["out_op"] < 0:
            return y.transpose(0, 1).contiguous()
        if case["out_op"] == 1:
            y *= 0.5
        return uniform((ncx, N, 2), seed, 4) + y.reshape(N, ncx, 2).permute(1, 0, 2)
    if k == "mode":
        N = case["N"]
        p = [torch.from_numpy(v).to(DEV).unsqueeze(-1) for v in mode_parts(case, _rng(seed, 1))]
        x = _rows(uniform((case["nsys"], N), seed))
        if case["jw"] == 13:
            y = x * p[1]
            _tridiagonal(p[0], p[2], y)
            return y.transpose(0, 1).contiguous()
        D, off, solve = p
        y = D * x
        if case["ub"]:
            y[:-1] += off[:-1] * x[1:]
            for r in range(1, N):
                y[r].addcmul_(solve[r], y[r - 1], value=-1)
        else:
            y[1:] += off[1:] * x[:-1]
            for r in range(N - 2, -1, -1):
                y[r].addcmul_(solve[r], y[r + 1], value=-1)
        return y.transpose(0, 1).contiguous()
    if k == "chain":
        N, K = case["N"], case["K"]
        x = uniform((case["nsys"], N + N % 2), seed)
        y = _rows(x[:, :N])
        for i, (scale, up, low) in enumerate(chain_parts(N, K, _degree(seed, N))):
            n = N - i
            scale, up, low = (torch.from_numpy(v).to(DEV).unsqueeze(-1) for v in (scale, up, low))
            nxt = torch.zeros_like(y[:n])
            m = min(n, y.shape[0] - 1)
            nxt[:m] = up[:m] * y[1:m + 1]
            nxt += scale * y[:n]
            y = nxt
            for r in range(1, n):
                y[r].addcmul_(low[r], y[r - 1], value=-1)
        x[:, :N - K + 1] = y.transpose(0, 1)
        return x
    if k == "batch":
        # every set at once, padded with rows that stay zero
        sizes, nsys = degree_sizes(case), case["nsys"]
        nmax, S = max(sizes), len(sizes)
        parts = [np.zeros((5, nmax, S))] + [np.zeros((nmax, S)) for _ in range(5)]
        flat = uniform((sum(nsys * (N + N % 2) for N in sizes),), seed)
        x = torch.zeros((nmax, S, nsys), dtype=torch.float64, device=DEV)
        at = 0
        for l, N in enumerate(sizes):
            p = fused_parts(N, _rng(seed, 10 + l))
            parts[0][:, :N, l] = p[0]
            for q, v in zip(parts[1:], p[1:]):
                q[:N, l] = v
            stride = N + N % 2
            x[:N, l] = flat[at:at + nsys * stride].view(nsys, stride)[:, :N].t()
            at += nsys * stride
        y = _solve_fused(parts, x)
        at = 0
        for l, N in enumerate(sizes):
            stride = N + N % 2
            flat[at:at + nsys * stride].view(nsys, stride)[:, :N] = y[:N, l].t()
            at += nsys * stride
        return flat
    sizes = request_sizes(case)
    flat = uniform((sum(N * n for N, n in sizes),), seed)
    at = 0
    for i, (N, n) in enumerate(sizes):
        v = flat[at:at + N * n].view(n, N)
        v.copy_(_solve_fused(fused_parts(N, _rng(seed, 10 + i)), _rows(v)).t())
        at += N * n
    return flat.cpu()
