"""The work this library is used for, as cases of one list.

Coefficients in, coefficients or grid values out: the rotation executors
(sphere, FP64 and FP32), the whole harmonic transforms around them (sphere with
its grid, triangle, disk), the spin-weighted sphere, batches of transforms of
uneven degree and the drop-in call on a host array, from degree 24, where a
call is its launches, to degree 2048.  Every case goes through the package's
public functions; device matrices are torch tensors of shape (M, n), row j the
column j of the n x M column-major matrix.  The library transforms in place,
so a pass copies the coefficients it keeps into a work buffer first, as a
program that goes on using them does.

``exact`` restates each operation from the mathematics in extended precision:
the Givens rotations from their closed forms, the 1D connection matrices by
Gauss quadrature, the trigonometric transforms by long double FFTs.
"""
import math

import numpy as np
import torch

import fasttransforms_amd as ft

LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288420")


# ------------------------------------------------------------------- cases --

def _full_M(geometry, n):
    return {"tri": n, "disk": 4 * n - 3}.get(geometry, 2 * n - 1)


def listed():
    return [
        # one small transform, as inside a time step of a coarse model: launches and latency
        {"name": "rot_sph_n64", "kind": "rot", "geometry": "sph", "dir": "hi2lo", "fp32": False, "n": 64, "M": 127},
        # the headline size of the sphere's rotations (bench.py's default workload)
        {"name": "rot_sph_n1024", "kind": "rot", "geometry": "sph", "dir": "hi2lo", "fp32": False, "n": 1024,
         "M": 2047},
        # a truncated, odd-sized FP32 analysis direction
        {"name": "rot_sph_fp32_n733", "kind": "rot", "geometry": "sph", "dir": "lo2hi", "fp32": True, "n": 733,
         "M": 1001},
        # the largest transform of the benchmark
        {"name": "rot_sph_n2048", "kind": "rot", "geometry": "sph", "dir": "lo2hi", "fp32": False, "n": 2048,
         "M": 4095},
        # spherical harmonic coefficients to grid values at the headline size
        {"name": "sht_n1024", "kind": "sht", "dir": "synthesis", "n": 1024},
        # grid values to coefficients, a size that is no power of two
        {"name": "sht_inv_n600", "kind": "sht", "dir": "analysis", "n": 600},
        # the grid step alone (sph2fourier done elsewhere or kept), an odd number of rows
        {"name": "grid_n451", "kind": "grid", "n": 451, "M": 901},
        # Zernike coefficients to Chebyshev x Fourier
        {"name": "disk2cxf_n400", "kind": "harmonic", "transform": "disk2cxf", "n": 400, "M": 1597},
        # bivariate Chebyshev coefficients to Proriol's on the triangle
        {"name": "cheb2tri_n511", "kind": "harmonic", "transform": "cheb2tri", "n": 511, "M": 511},
        # spin-2 coefficients (polarization, gravitational waves), analysis direction
        {"name": "spin2_n512", "kind": "spin", "dir": "lo2hi", "s": 2, "n": 512, "M": 1023},
        # many transforms of uneven degree in one call (adaptive grids, serving)
        {"name": "batch48", "kind": "batch", "dir": "hi2lo", "count": 48, "nmin": 32, "nmax": 512, "sizes": 7},
        # the C entry point a program of the reference calls, on a host array
        {"name": "host_sph2fourier_n384", "kind": "host", "transform": "sph2fourier", "n": 384, "M": 767},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rot", "rot", "sht", "sht", "grid", "harmonic", "harmonic", "spin", "batch", "host"])
    if kind == "rot":
        geometry = rng.choice(["sph", "sph", "tri", "disk"])
        n = _log_int(rng, 24, {"sph": 2047, "tri": 1400, "disk": 900}[geometry])
        full = _full_M(geometry, n)
        M = full if rng.random() < 0.6 else rng.randint(full // 3, full)
        if geometry != "tri":
            M -= 1 - M % 2
        return {"kind": kind, "geometry": geometry, "dir": rng.choice(["hi2lo", "lo2hi"]),
                "fp32": rng.random() < 0.25, "n": n, "M": M}
    if kind == "sht":
        return {"kind": kind, "dir": rng.choice(["synthesis", "analysis"]), "n": _log_int(rng, 24, 1100)}
    if kind == "grid":
        n = _log_int(rng, 24, 1100)
        M = 2 * n - 1 if rng.random() < 0.5 else 2 * rng.randint(n // 2, n) + 1
        return {"kind": kind, "n": n, "M": M}
    if kind == "harmonic":
        transform = rng.choice(["tri2cheb", "cheb2tri", "disk2cxf", "cxf2disk"])
        disk = "disk" in transform
        n = _log_int(rng, 24, 560 if disk else 1000)
        return {"kind": kind, "transform": transform, "n": n, "M": _full_M("disk" if disk else "tri", n)}
    if kind == "spin":
        n = _log_int(rng, 24, 900)
        return {"kind": kind, "dir": rng.choice(["hi2lo", "lo2hi"]), "s": rng.choice([-2, -1, 1, 2, 4]), "n": n,
                "M": 2 * n - 1}
    if kind == "batch":
        return {"kind": kind, "dir": rng.choice(["hi2lo", "lo2hi"]), "count": rng.randint(8, 64), "nmin": 24,
                "nmax": _log_int(rng, 96, 600), "sizes": rng.randint(0, 10 ** 6)}
    n = _log_int(rng, 24, 600)
    return {"kind": "host", "transform": rng.choice(["sph2fourier", "fourier2sph"]), "n": n, "M": 2 * n - 1}


def _batch_sizes(case):
    rng = np.random.default_rng(case["sizes"])
    u = rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]), case["count"])
    return [int(round(math.exp(v))) for v in u]


# ------------------------------------------------------------------ inputs --

def _orders(geometry, M):
    """Order of every column."""
    j = np.arange(M)
    return j if geometry == "tri" else (j + 1) // 2


def _rows(geometry, n, M):
    """Coefficients every column holds; the rows below are zero."""
    m = _orders(geometry, M)
    return n - (m + 1) // 2 if geometry == "disk" else n - m


def _coefficients(rng, geometry, n, M):
    """Coefficients of a smooth function: random signs and sizes, falling with the degree, (M, n)."""
    l = np.arange(n)[None, :]
    A = rng.standard_normal((M, n)) / (1.0 + l + _orders(geometry, M)[:, None])
    return np.where(l < _rows(geometry, n, M)[:, None], A, 0.0)


def _field(rng, N, M):
    """A smooth function on the sphere's grid, (M, N): a sum of plane waves."""
    th = (np.arange(N) + 0.5) * np.pi / N
    ph = np.arange(M) * 2.0 * np.pi / M
    x = np.cos(ph)[:, None] * np.sin(th)[None, :]
    y = np.sin(ph)[:, None] * np.sin(th)[None, :]
    z = np.broadcast_to(np.cos(th)[None, :], (M, N))
    F = np.zeros((M, N))
    for _ in range(8):
        k = rng.standard_normal(3)
        k *= rng.uniform(0.0, N / 3.0) / np.linalg.norm(k)
        F += rng.standard_normal() * np.cos(k[0] * x + k[1] * y + k[2] * z + rng.uniform(0, 2 * np.pi))
    return F


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    kind, n = case["kind"], case.get("n")
    if kind == "rot":
        A = _coefficients(rng, case["geometry"], n, case["M"])
        return A.astype(np.float32) if case["fp32"] else A
    if kind == "sht":
        return _coefficients(rng, "sph", n, 2 * n - 1) if case["dir"] == "synthesis" else _field(rng, n, 2 * n - 1)
    if kind in ("grid", "host"):
        # Fourier coefficients: order m's row is a frequency
        A = _coefficients(rng, "sph", n, case["M"])
        return A
    if kind == "harmonic":
        return _coefficients(rng, "disk" if "disk" in case["transform"] else "tri", n, case["M"])
    if kind == "spin":
        A = _coefficients(rng, "sph", n, case["M"]) + 1j * _coefficients(rng, "sph", n, case["M"])
        # order m has rows max(|m|, |s|) .. n-1
        m = _orders("sph", case["M"])
        return np.where(np.arange(n)[None, :] < (n - np.maximum(m, abs(case["s"])))[:, None], A, 0.0)
    return [_coefficients(rng, "sph", k, 2 * k - 1) for k in _batch_sizes(case)]


def _harmonic_plan(transform, n):
    if transform in ("sph2fourier", "fourier2sph"):
        return ft.plan_sph2fourier(n)
    if transform in ("tri2cheb", "cheb2tri"):
        return ft.plan_tri2cheb(n, 0.0, 0.0, 0.0)
    return ft.plan_disk2cxf(n, 0.0, 0.0)


def prepare(case, seed):
    kind, n = case["kind"], case.get("n")
    A = _inputs(case, seed)
    st = {"case": case}
    if kind == "batch":
        sizes = _batch_sizes(case)
        plans = {k: ft.plan_rotsphere(k) for k in set(sizes)}
        st["plans"] = [plans[k] for k in sizes]
        st["coef"] = [torch.from_numpy(a).cuda() for a in A]
        st["work"] = [torch.empty_like(a) for a in st["coef"]]
        return st
    if kind == "host":
        st["plan"] = _harmonic_plan(case["transform"], n)
        st["coef"] = np.asfortranarray(A.T)
        st["work"] = np.empty_like(st["coef"])
        return st
    if kind == "rot":
        st["plan"] = {"sph": lambda: ft.plan_rotsphere(n), "tri": lambda: ft.plan_rottriangle(n, 0.0, 0.0, 0.0),
                      "disk": lambda: ft.plan_rotdisk(n, 0.0, 0.0)}[case["geometry"]]()
    elif kind == "sht":
        st["plan"] = ft.plan_sph2fourier(n)
        st["grid"] = (ft.plan_sph_synthesis if case["dir"] == "synthesis" else ft.plan_sph_analysis)(n, 2 * n - 1)
    elif kind == "grid":
        st["grid"] = ft.plan_sph_synthesis(n, case["M"])
    elif kind == "harmonic":
        st["plan"] = _harmonic_plan(case["transform"], n)
    else:
        st["plan"] = ft.plan_rotspinsphere(n, case["s"])
    st["coef"] = torch.from_numpy(A).cuda()
    st["work"] = torch.empty_like(st["coef"])
    return st


def run(st):
    case, work = st["case"], st["work"]
    kind = case["kind"]
    if kind == "batch":
        for w, a in zip(work, st["coef"]):
            w.copy_(a)
        ft.gpu_execute_batch(st["plans"], case["dir"], work)
        return work
    if kind == "host":
        np.copyto(work, st["coef"])
        getattr(ft, "execute_" + case["transform"])("N", st["plan"], work)
        return work
    work.copy_(st["coef"])
    if kind == "rot":
        ft.gpu_execute(st["plan"], case["dir"], work, precision=ft.FP32 if case["fp32"] else ft.FP64)
    elif kind == "sht" and case["dir"] == "synthesis":
        ft.gpu_execute_harmonic("sph2fourier", "N", st["plan"], work)
        ft.gpu_execute_sph_grid("sph_synthesis", "N", st["grid"], work)
    elif kind == "sht":
        ft.gpu_execute_sph_grid("sph_analysis", "N", st["grid"], work)
        ft.gpu_execute_harmonic("fourier2sph", "N", st["plan"], work)
    elif kind == "grid":
        ft.gpu_execute_sph_grid("sph_synthesis", "N", st["grid"], work)
    elif kind == "harmonic":
        ft.gpu_execute_harmonic(case["transform"], "N", st["plan"], work)
    else:
        ft.gpu_execute_spinsph(st["plan"], case["dir"], work)
    return work


# -------------------------------------------------------------------- work --

def _top(geometry, n, j):
    """Last row of sequence j's rotations (below 0: none)."""
    return {"sph": n - 3 - j, "tri": n - 2 - j, "disk": n - 2 - (j + 1) // 2}[geometry]


def _rotations(geometry, n, orders):
    step = 1 if geometry == "tri" else 2
    total, per_order = 0, {}
    for m in orders:
        m = int(m)
        if m not in per_order:
            j = np.arange(m % step, m - step + 1, step)
            top = n - 2 - (j + 1) // 2 if geometry == "disk" else n - (3 if geometry == "sph" else 2) - j
            per_order[m] = int(np.maximum(top + 1, 0).sum())
        total += per_order[m]
    return total


def _tables(geometry, n):
    """Bytes of the rotations' sines and cosines, once each."""
    return 16 * (n * n if geometry == "disk" else n * (n + 1) // 2)


def _fft_flops(N, M):
    """A real transform of length N per column and one of length M per row, 2.5 L log2 L each."""
    return 2.5 * N * M * (math.log2(max(N, 2)) + math.log2(max(M, 2)))


def work(case):
    kind, n = case["kind"], case.get("n")
    if kind == "batch":
        sizes = _batch_sizes(case)
        return {"bytes": sum(16 * k * (2 * k - 1) for k in sizes) + _tables("sph", max(sizes)),
                "flops": 6 * sum(_rotations("sph", k, _orders("sph", 2 * k - 1)) for k in sizes)}
    M = case.get("M", 2 * n - 1 if n else 0)
    size = n * M
    if kind == "rot":
        item = 4 if case["fp32"] else 8
        return {"bytes": 2 * item * size + _tables(case["geometry"], n) * item // 8,
                "flops": 6 * _rotations(case["geometry"], n, _orders(case["geometry"], M))}
    if kind == "grid":
        return {"bytes": 16 * size, "flops": _fft_flops(n, M)}
    if kind == "spin":
        s = abs(case["s"])
        m = _orders("sph", M)
        d = np.abs(m - s)
        first = sum(max(n - 1 - int(dd) - j, 0) for mm, dd in zip(m, d) for j in range(min(int(mm), s)))
        return {"bytes": 32 * size + _tables("sph", n) + 16 * s * n * (n + 1) // 2,
                "flops": 12 * (_rotations("sph", n, d) + first)}
    # both triangles of a harmonic transform, multiply and add
    if kind in ("sht", "host"):
        geometry, products, matrices = "sph", n * (n + 1) * M, 2
    elif "disk" in case["transform"]:
        geometry, products, matrices = "disk", n * (n + 1) * M, 2
    else:
        geometry, products, matrices = "tri", 2 * n * (n + 1) * M, 2
    w = {"bytes": 16 * size + _tables(geometry, n) + matrices * 4 * n * (n + 1),
         "flops": 6 * _rotations(geometry, n, _orders(geometry, M)) + products}
    if kind == "sht":
        w["flops"] += _fft_flops(n, M)
    return w


# ------------------------------------------------------------------- exact --

def _sc(geometry, n, j):
    """Sines and cosines of sequence j, rows 0 .. top, in long double."""
    l = np.arange(max(_top(geometry, n, j), -1) + 1).astype(LD)
    j = LD(j)
    if geometry == "sph":
        num, numc, den = (l + 1) * (l + 2), (2 * j + 2) * (2 * l + 2 * j + 5), (l + 2 * j + 3) * (l + 2 * j + 4)
    elif geometry == "tri":
        num, numc, den = (l + 1) * (l + 1), (2 * j + 2) * (2 * l + 2 * j + 4), (l + 2 * j + 3) * (l + 2 * j + 3)
    else:
        num, numc, den = (l + 1) * (l + 1), (j + 1) * (2 * l + j + 3), (l + j + 2) * (l + j + 2)
    s = np.sqrt(num / den)
    return (-s if geometry == "disk" else s), np.sqrt(numc / den)


def _rotate(A, geometry, orders, hi2lo):
    """The rotation sequences of every column of A (n x columns, long double), in place."""
    n = A.shape[0]
    step, gap = (1 if geometry == "tri" else 2), (2 if geometry == "sph" else 1)
    for parity in range(step):
        idx = np.nonzero((orders % step == parity) & (orders >= step + parity))[0]
        if not len(idx):
            continue
        idx = idx[np.argsort(-orders[idx], kind="stable")]
        m = orders[idx]
        G = np.ascontiguousarray(A[:, idx])
        seqs = range(parity, int(m[0]) - step + 1, step)
        for j in (reversed(seqs) if hi2lo else seqs):
            top = _top(geometry, n, j)
            if top < 0:
                continue
            cnt = int(np.searchsorted(-m, -j, side="left"))  # columns of order above j
            s, c = _sc(geometry, n, j)
            if not hi2lo:
                s = -s
            H = G[:, :cnt]
            # rows of one residue mod gap are chains of their own: gap of them at once
            blocks = [(max(k - gap + 1, 0), k + 1) for k in range(top, -1, -gap)]
            for a, b in (blocks if hi2lo else reversed(blocks)):
                x, y = H[a:b], H[a + gap:b + gap]
                sk, ck = s[a:b, None], c[a:b, None]
                new = ck * x + sk * y
                H[a + gap:b + gap] = ck * y - sk * x
                H[a:b] = new
        A[:, idx] = G
    return A


def _spin_first(A, orders, spin, hi2lo):
    """The spin-weighted sphere's sequences of adjacent rows (A: n x columns, complex long double)."""
    n, as_ = A.shape[0], abs(spin)
    am = np.abs(orders)
    for sign in (True, False):
        for lo in range(as_ + 1):  # columns of order lo < |s| one by one, the others together
            sel = (am == lo) if lo < as_ else (am >= as_)
            idx = np.nonzero(sel & ((orders * spin >= 0) == sign))[0]
            if not len(idx):
                continue
            d = np.abs(am[idx] - as_)
            idx, d = idx[np.argsort(d, kind="stable")], np.sort(d)
            dl = d.astype(LD)
            G = np.ascontiguousarray(A[:, idx])
            seqs = range(min(lo, as_))
            for j in (reversed(seqs) if hi2lo else seqs):
                rows = range(n - 2 - j - int(d[0]), -1, -1)
                for k in (rows if hi2lo else reversed(rows)):
                    cnt = int(np.searchsorted(d, n - 2 - j - k, side="right"))
                    if cnt == 0:
                        continue
                    e, l = dl[:cnt], LD(k)
                    den = (l + 2 * j + e + 2) * (l + 2 * j + 2 * e + 2)
                    s = np.sqrt((l + 1) * (l + e + 1) / den)
                    c = np.sqrt((2 * j + e + 1) * (2 * l + 2 * j + 2 * e + 3) / den)
                    if sign != hi2lo:
                        s = -s
                    x, y = G[k, :cnt].copy(), G[k + 1, :cnt].copy()
                    G[k, :cnt], G[k + 1, :cnt] = c * x + s * y, c * y - s * x
            A[:, idx] = G
    return A


def _dot(U, X):
    """U @ X to about 2^-63 of the row and column maxima: products of 20-bit slices are exact in FP64."""
    def slices(V, axis):
        scale = np.abs(V).max(axis=axis, keepdims=True)
        scale = np.where(scale > 0, LD(2) ** np.ceil(np.log2(np.where(scale > 0, scale, 1)).astype(np.float64)), LD(1))
        r, out = V / scale, []
        for i in range(1, 5):
            q = LD(2) ** (20 * i)
            part = np.rint(r * q) / q
            out.append(part.astype(np.float64))
            r = r - part
        return out, scale
    us, su = slices(np.asarray(U, LD), 1)
    xs, sx = slices(np.asarray(X, LD), 0)
    acc = np.zeros((U.shape[0], X.shape[1]), LD)
    for i in range(4):
        for k in range(4 - i):
            acc += us[i] @ xs[k]
    return acc * su * sx


def _jacobi(n, a, b, x):
    """Orthonormal Jacobi polynomials of weight (1-x)^a (1+x)^b at x, (len(x), n)."""
    a, b = LD(a), LD(b)
    k = np.arange(1, n + 1).astype(LD)
    s = 2 * k + a + b
    off = 2 * np.sqrt(k * (k + a) * (k + b) * (k + a + b) / ((s - 1) * s * s * (s + 1)))
    diag = np.concatenate([[(b - a) / (a + b + 2)], (b - a) * (a + b) / (s * (s + 2))])
    mu = LD(2) ** (a + b + 1) / (a + b + 1)  # a, b in {0, 1}, not both 1
    if a == 1 and b == 1:
        mu = LD(4) / 3
    P = np.empty((len(x), n), LD)
    P[:, 0] = 1 / np.sqrt(mu)
    for i in range(1, n):
        P[:, i] = (x - diag[i - 1]) * P[:, i - 1]
        if i > 1:
            P[:, i] -= off[i - 2] * P[:, i - 2]
        P[:, i] /= off[i - 1]
    return P


def _connection(n, a, b, family):
    """Upper triangular: orthonormal Jacobi(a, b) of degree j in cos k theta ("T"), normalized T_k ("Tn"),
    sin (k+1) theta / sin theta ("U") or the normalized cos (k+1/2) theta / cos theta/2 ("V")."""
    N = n + 1
    i, k = np.arange(N), np.arange(n)
    th = (2 * i + 1).astype(LD) * PI / (2 * N)

    def trig(f, num, den):  # f(pi num / den), the argument reduced exactly
        return f((num % (2 * den)).astype(LD) * PI / den)

    P = _jacobi(n, a, b, np.cos(th))
    w = 1 / LD(N)
    if family in ("T", "Tn"):
        C = trig(np.cos, np.outer(k, 2 * i + 1), 2 * N) * np.where(k == 0, w, 2 * w)[:, None]
        if family == "Tn":
            C *= np.where(k == 0, np.sqrt(PI), np.sqrt(PI / 2))[:, None]
    elif family == "U":
        C = trig(np.sin, np.outer(k + 1, 2 * i + 1), 2 * N) * (2 * w)
        P = P * np.sin(th)[:, None]
    else:
        C = trig(np.cos, np.outer(2 * k + 1, 2 * i + 1), 4 * N) * (2 * w * np.sqrt(PI))
        P = P * np.cos(th / 2)[:, None]
    return np.triu(_dot(C, P))


def _solve(U, F):
    """U^{-1} F for the upper triangular U, long double."""
    F = F.copy()
    for j in range(U.shape[0] - 1, -1, -1):
        F[j] /= U[j, j]
        if j:
            F[:j] -= U[:j, j:j + 1] * F[j]
    return F


def _harmonic_exact(transform, A):
    """The harmonic transform of the n x M long double matrix A."""
    n, M = A.shape
    inverse = transform in ("fourier2sph", "cxf2disk", "cheb2tri")
    geometry = {"sph2fourier": "sph", "fourier2sph": "sph", "disk2cxf": "disk", "cxf2disk": "disk"}.get(transform, "tri")
    apply = _solve if inverse else _dot
    orders = _orders(geometry, M)
    if not inverse:
        A = _rotate(A.copy(), geometry, orders, True)
    if geometry == "tri":
        U0, U1 = _connection(n, 1, 0, "Tn"), _connection(n, 0, 0, "Tn")[:M, :M]
        if not inverse:
            A = apply(U1, apply(U0, A).T).T.copy()
        root, scale = (np.sqrt(LD(2)), PI / 2) if inverse else (1 / np.sqrt(LD(2)), 2 / PI)
        A = A * scale
        A[:, 0] *= root
        A[0] *= root
        if inverse:
            A = apply(U0, apply(U1, A.T.copy()).T.copy())
    else:
        if geometry == "sph":
            U = [_connection(n, 0, 0, "T"), _connection(n, 1, 1, "U")]
        else:
            U = [2 * _connection(n, 0, 0, "T"), 2 * np.sqrt(2 / PI) * _connection(n, 0, 1, "V")]
        out = np.empty_like(A)
        for odd in (0, 1):
            idx = np.nonzero(orders % 2 == odd)[0]
            if len(idx):
                out[:, idx] = apply(U[odd], A[:, idx])
        A = out
    if inverse:
        A = _rotate(np.ascontiguousarray(A), geometry, orders, False)
    return A


def _cis(num, den):
    """e^{i pi num / den} in long double."""
    t = (num % (2 * den)).astype(LD) * PI / den
    return np.cos(t) + 1j * np.sin(t)


def _fft(Z, axis, inverse=False):
    Z = np.asarray(Z, np.clongdouble)
    return np.fft.ifft(Z, axis=axis, norm="forward") if inverse else np.fft.fft(Z, axis=axis)


def _synthesis_exact(A):
    """Bivariate Fourier coefficients (n x M) to values on the sphere's grid."""
    N, M = A.shape
    m = _orders("sph", M)
    k = np.arange(N)
    V = np.empty((N, M), LD)
    for odd, shift in ((0, 0), (1, 1)):
        idx = np.nonzero(m % 2 == odd)[0]
        Z = np.zeros((2 * N, len(idx)), np.clongdouble)
        Z[:N] = A[:, idx] * _cis(k + shift, 2 * N)[:, None]
        # sum_k a_k e^{i (k + shift) theta_r}, theta_r = pi (2 r + 1) / 2N
        W = _fft(Z, 0, True)[:N] * _cis(2 * k * shift, 2 * N)[:, None]
        V[:, idx] = W.imag if odd else W.real
    V *= 1 / (2 * np.sqrt(PI))  # cos 0 and the frequencies above it: 1 / sqrt(4 pi) and sqrt(2) below
    V[:, 0] *= np.sqrt(LD(2))
    Y = np.zeros((N, M), np.clongdouble)
    Y[:, 0] = V[:, 0]
    if M > 1:
        # value = c0 + sum_q 2 (a_q cos q phi + b_q sin q phi)
        half = V[:, 2::2] - 1j * V[:, 1::2]
        Y[:, 1:M // 2 + 1] = half
        Y[:, M - M // 2:] = np.conj(half[:, ::-1])
    return _fft(Y, 1, True).real


def _analysis_exact(F):
    """Values on the sphere's grid (n x M) to bivariate Fourier coefficients."""
    N, M = F.shape
    Y = _fft(F, 1)
    X = np.empty((N, M), LD)
    X[:, 0] = Y[:, 0].real
    X[:, 2::2] = Y[:, 1:M // 2 + 1].real
    X[:, 1::2] = -Y[:, 1:M // 2 + 1].imag
    X *= 4 * np.sqrt(PI) / (2 * N * M)
    X[:, 0] /= np.sqrt(LD(2))
    m = _orders("sph", M)
    k = np.arange(N)
    A = np.empty((N, M), LD)
    for odd, shift in ((0, 0), (1, 1)):
        idx = np.nonzero(m % 2 == odd)[0]
        Z = np.zeros((2 * N, len(idx)), np.clongdouble)
        Z[:N] = X[:, idx] * _cis(-2 * k * shift, 2 * N)[:, None]
        W = _fft(Z, 0)[:N] * _cis(-(k + shift), 2 * N)[:, None]
        A[:, idx] = -2 * W.imag if odd else 2 * W.real
    A[0, m % 2 == 0] /= 2
    return A


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    # long double on one core: about 7 s for 1e9 rotation flops
    if kind != "grid" and work(case)["flops"] > {"sht": 4.6e9}.get(kind, 2.4e9):
        return None

    def tensor(A):
        return torch.from_numpy(np.ascontiguousarray(A.T.astype(np.float64)))

    X = _inputs(case, seed)
    if kind == "batch":
        return [tensor(_rotate(a.T.astype(LD).copy(), "sph", _orders("sph", a.shape[0]), case["dir"] == "hi2lo"))
                for a in X]
    if kind == "spin":
        A = np.ascontiguousarray(X.T).astype(np.clongdouble)
        m = _orders("sph", case["M"]) * np.where(np.arange(case["M"]) % 2 == 1, -1, 1)
        d = np.abs(np.abs(m) - abs(case["s"]))
        if case["dir"] == "hi2lo":
            A = _rotate(_spin_first(A, m, case["s"], True), "sph", d, True)
        else:
            A = _spin_first(_rotate(A, "sph", d, False), m, case["s"], False)
        return torch.from_numpy(np.ascontiguousarray(A.T.astype(np.complex128)))
    A = np.ascontiguousarray(X.T).astype(LD)
    if kind == "rot":
        return tensor(_rotate(A, case["geometry"], _orders(case["geometry"], case["M"]), case["dir"] == "hi2lo"))
    if kind == "sht":
        if case["dir"] == "synthesis":
            return tensor(_synthesis_exact(_harmonic_exact("sph2fourier", A)))
        return tensor(_harmonic_exact("fourier2sph", _analysis_exact(A)))
    if kind == "grid":
        return tensor(_synthesis_exact(A))
    A = _harmonic_exact(case["transform"], A)
    if kind == "host":
        return np.asfortranarray(A.astype(np.float64))
    return tensor(A)
