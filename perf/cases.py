"""Performance cases of the mBSR path: what a solver built on this package has it do.

Every case is one call sequence through the public entry points (``amgt_amd.mbsr``,
``amgt_amd.hypre``, ``amgt_amd.coarsen``, ``amgt_amd.amg``) on diffusion problems of the kinds
the package is tested and benchmarked on: 5-, 7- and 27-point operators on 2D and 3D grids with
constant or random-field coefficients, their prolongations, and dense-row coarse operators.

* ``matvec``    y = A x, f - A u, or the restriction P^T r through the transposed product, in
                FP64 / FP32 / FP16 values: the solve phase, a few dozen calls per V-cycle
* ``spmm``      several right-hand sides at once, column-major or interleaved
* ``convert``   CSR -> mBSR, paid once per matrix of a hierarchy
* ``galerkin``  R (A P) of one level, at the CSR boundary HYPRE calls or on mBSR handles
* ``coarsen``   strength, C/F splitting and extended+i interpolation of one level
* ``boomer``    the whole algebraic setup, graph capture and PCG solve
* ``batch``     many independent 2D problems as one geometric setup, capture and solve

All inputs are made on the device from the seed.
"""
from __future__ import annotations

import math

import torch

from amgt_amd import amg as AMG
from amgt_amd import coarsen as CO
from amgt_amd import hypre as H
from amgt_amd.mbsr import MBSRMatrix

_DEV = "cuda"


# ---- the cases ----------------------------------------------------------------------------
def listed():
    return [
        # the residual of a small 2D problem or of a coarse level: launch latency
        {"name": "residual_5pt_128x128", "op": "matvec", "form": "residual", "kind": 5,
         "nx": 128, "ny": 128, "nz": 1, "prec": 0},
        # A p of the finest level in PCG
        {"name": "spmv_7pt_128", "op": "matvec", "form": "plain", "kind": 7,
         "nx": 128, "ny": 128, "nz": 128, "prec": 0},
        # residual with a coarse algebraic operator (30 to 125 entries a row, ragged grid) in
        # the precision the mixed schedule gives to coarse levels
        {"name": "residual_coarse_fp16", "op": "matvec", "form": "residual", "kind": 125,
         "nx": 47, "ny": 41, "nz": 39, "prec": 2},
        # restriction by the transposed product with P, as BoomerAMG restricts
        {"name": "restrict_trans_7pt_128", "op": "matvec", "form": "restrict", "kind": 7,
         "nx": 128, "ny": 128, "nz": 128, "prec": 0},
        # 32 right-hand sides of a 27-point problem
        {"name": "spmm_27pt_64_k32", "op": "spmm", "kind": 27, "nx": 64, "ny": 64, "nz": 64,
         "k": 32, "layout": "columns"},
        # the finest matrix entering the library
        {"name": "convert_7pt_128", "op": "convert", "kind": 7, "nx": 128, "ny": 128, "nz": 128},
        # finest-level Galerkin product with trilinear P at the CSR boundary (P and R are new
        # matrices, A has been used before)
        {"name": "galerkin_7pt_128", "op": "galerkin", "kind": 7, "nx": 128, "ny": 128,
         "nz": 128, "interp": "trilinear", "api": "csr", "prec": 0},
        # Galerkin product with a ragged algebraic P on handles, odd sizes
        {"name": "galerkin_algebraic_101", "op": "galerkin", "kind": 7, "nx": 101, "ny": 99,
         "nz": 97, "interp": "direct", "api": "handles", "prec": 0},
        # coarse-level product of the mixed schedule
        {"name": "galerkin_27pt_fp32", "op": "galerkin", "kind": 27, "nx": 49, "ny": 45,
         "nz": 51, "interp": "trilinear", "api": "handles", "prec": 1},
        # one level of the device setup, finest level
        {"name": "coarsen_pmis_7pt_128", "op": "coarsen", "kind": 7, "nx": 128, "ny": 128,
         "nz": 128, "splitting": "pmis"},
        # a whole solve with the default options (HMIS): 2D random-field diffusion
        {"name": "boomer_solve_5pt_512", "op": "boomer", "kind": 5, "nx": 512, "ny": 512,
         "nz": 1, "splitting": "hmis"},
        # 48 independent 2D problems of 32 to 512 points a side
        {"name": "batch_solve_48", "op": "batch", "count": 48, "lo": 32, "hi": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, kind, lo, hi):
    """A grid of about lo..hi points (over the logarithm), sides within a factor of two."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if kind == 5:
        a = n ** 0.5 * math.exp(rng.uniform(-0.35, 0.35))
        nx = max(3, int(round(a)))
        return nx, max(3, int(n / nx)), 1
    s = n ** (1.0 / 3.0)
    nx = max(3, int(round(s * math.exp(rng.uniform(-0.25, 0.25)))))
    ny = max(3, int(round(s * math.exp(rng.uniform(-0.25, 0.25)))))
    return nx, ny, max(3, int(n / (nx * ny)))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "matvec", "spmm", "spmm", "convert", "galerkin",
                     "galerkin", "coarsen", "boomer", "batch"])
    if op == "batch":
        lo = rng.randint(16, 200)
        return {"op": op, "count": rng.randint(2, 48), "lo": lo, "hi": rng.randint(lo, 512)}
    if op == "matvec":
        form = rng.choice(["plain", "residual", "restrict"])
        kind = rng.choice([5, 7] if form == "restrict" else [5, 7, 27, 125])
        hi = {5: 2_000_000, 7: 2_000_000, 27: 500_000, 125: 100_000}[kind]
        nx, ny, nz = _grid(rng, kind, 2_000, hi)
        prec = 0 if form == "restrict" else rng.choice([0, 0, 1, 2])
        return {"op": op, "form": form, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "prec": prec}
    if op == "spmm":
        kind = rng.choice([7, 27])
        nx, ny, nz = _grid(rng, kind, 4_000, 262_144)
        return {"op": op, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "k": _log_int(rng, 2, 32),
                "layout": rng.choice(["columns", "interleaved"])}
    if op == "convert":
        kind = rng.choice([5, 7, 27, 125])
        hi = {5: 2_000_000, 7: 2_000_000, 27: 500_000, 125: 100_000}[kind]
        nx, ny, nz = _grid(rng, kind, 2_000, hi)
        return {"op": op, "kind": kind, "nx": nx, "ny": ny, "nz": nz}
    if op == "galerkin":
        kind = rng.choice([5, 7, 27])
        nx, ny, nz = _grid(rng, kind, 4_000, 150_000 if kind == 27 else 2_000_000)
        interp = "trilinear" if kind == 27 else rng.choice(["trilinear", "direct"])
        prec = rng.choice([0, 0, 1])
        return {"op": op, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "interp": interp,
                "api": "handles" if prec else rng.choice(["csr", "handles"]), "prec": prec}
    if op == "coarsen":
        kind = rng.choice([5, 7, 27])
        nx, ny, nz = _grid(rng, kind, 4_000, 100_000 if kind == 27 else 2_000_000)
        splitting = rng.choice(["pmis", "hmis"]) if nx * ny * nz < 200_000 else "pmis"
        return {"op": op, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "splitting": splitting}
    kind = rng.choice([5, 7])
    splitting = rng.choice(["pmis", "hmis"])
    nx, ny, nz = _grid(rng, kind, 4_000, 500_000 if splitting == "pmis" else 150_000)
    return {"op": op, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "splitting": splitting}


# ---- inputs -------------------------------------------------------------------------------
def _gen(seed, stream=0):
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed) * 1009 + stream)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float64, device=_DEV)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device=_DEV)


def _field(g, nz, ny, nx):
    """Positive cell coefficients exp(smooth random field), spread about e^+-1.5, smooth enough
    that every coupling of a row is a strong one at the default threshold."""
    w = torch.fft.rfftn(_normal(g, nz, ny, nx))
    k2 = 0.0
    for d, n in enumerate((nz, ny, nx)):
        f = torch.fft.fftfreq(n, device=_DEV, dtype=torch.float64)
        if d == 2:
            f = torch.fft.rfftfreq(n, device=_DEV, dtype=torch.float64)
        k2 = k2 + (f * f).view([-1 if e == d else 1 for e in range(3)])
    v = torch.fft.irfftn(w * torch.exp(-200.0 * k2), s=(nz, ny, nx))
    return torch.exp(v * (0.5 / v.std().clamp_min(1e-30)))


def _offsets(kind):
    if kind == 5:
        return [(0, -1, 0), (-1, 0, 0), (1, 0, 0), (0, 1, 0)]
    if kind == 7:
        return [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
    r = 1 if kind == 27 else 2
    s = range(-r, r + 1)
    return [(i, j, l) for l in s for j in s for i in s if i or j or l]


def _shifted(t, dx, dy, dz, fill):
    """t[z + dz, y + dy, x + dx], `fill` outside the grid."""
    nz, ny, nx = t.shape
    out = torch.full_like(t, fill)
    lo = [max(0, -d) for d in (dz, dy, dx)]
    hi = [n - max(0, d) for n, d in zip((nz, ny, nx), (dz, dy, dx))]
    if all(a < b for a, b in zip(lo, hi)):
        out[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] = \
            t[lo[0] + dz:hi[0] + dz, lo[1] + dy:hi[1] + dy, lo[2] + dx:hi[2] + dx]
    return out


def _matrix(case, seed, constant=False):
    """CSR (I, J, V) of the case's operator, rows diagonal first, then ascending columns.

    5- and 7-point: finite volumes with random-field coefficients (constant: the Poisson
    operator); 27-point: the same couplings to all neighbours; 125-point: a coarse operator,
    couplings over two neighbours each way that decay with the distance, each row keeping a
    share of them of its own (which ones does not depend on the seed)."""
    kind, nx, ny, nz = case["kind"], case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    g = _gen(seed)
    row = torch.arange(n, dtype=torch.int64, device=_DEV).view(nz, ny, nx)
    one = torch.ones(nz, ny, nx, dtype=torch.float64, device=_DEV)
    kf = one if constant else _field(g, nz, ny, nx)
    gk = _gen(0, 4)
    keep = 0.3 + 0.7 * _uniform(gk, nz, ny, nx) if kind == 125 else None
    cols, vals, here = [row.reshape(-1)], [None], [torch.ones(n, dtype=torch.bool, device=_DEV)]
    diag = torch.zeros(nz, ny, nx, dtype=torch.float64, device=_DEV)
    for dx, dy, dz in _offsets(kind):
        inside = _shifted(one, dx, dy, dz, 0.0) > 0
        k2 = _shifted(kf, dx, dy, dz, 0.0)
        v = torch.where(inside, 2.0 * kf * k2 / (kf + k2), kf)  # Dirichlet beyond the boundary
        if kind == 125:
            v = v / float(dx * dx + dy * dy + dz * dz)
            inside = inside & (_uniform(gk, nz, ny, nx) < keep)
        diag += v
        cols.append((row + (dz * ny + dy) * nx + dx).reshape(-1))
        vals.append((-v).reshape(-1))
        here.append(inside.reshape(-1))
    vals[0] = diag.reshape(-1)
    here = torch.stack(here, 1)
    I = torch.zeros(n + 1, dtype=torch.int32, device=_DEV)
    I[1:] = torch.cumsum(here.sum(1), 0)
    J = torch.stack(cols, 1)[here].to(torch.int32)
    V = torch.stack(vals, 1)[here]
    return I, J, V


def _from_coo(r, c, v, nrows, ncols):
    """CSR of distinct (row, column) entries, ascending columns."""
    order = torch.argsort(r * ncols + c)
    I = torch.zeros(nrows + 1, dtype=torch.int32, device=r.device)
    I[1:] = torch.cumsum(torch.bincount(r, minlength=nrows), 0)
    return I, c[order].to(torch.int32), v[order]


def _rows_of(I):
    I = I.to(torch.int64)
    return torch.repeat_interleave(torch.arange(I.numel() - 1, device=I.device), I[1:] - I[:-1])


def _trilinear(nx, ny, nz):
    """Linear interpolation per direction from the even-index points (COO, coarse count)."""
    r = torch.zeros(1, dtype=torch.int64, device=_DEV)
    c, v, ncoarse = r, torch.ones(1, dtype=torch.float64, device=_DEV), 1
    for n in (nz, ny, nx):
        nc = (n + 1) // 2
        f = torch.arange(n, device=_DEV)
        odd = f % 2 == 1
        hi = odd & (f // 2 + 1 < nc)
        r1 = torch.cat([f, f[hi]])
        c1 = torch.cat([f // 2, f[hi] // 2 + 1])
        v1 = torch.cat([torch.where(odd, 0.5, 1.0).to(torch.float64),
                        torch.full((int(hi.sum()),), 0.5, dtype=torch.float64, device=_DEV)])
        r = (r[:, None] * n + r1[None, :]).reshape(-1)
        c = (c[:, None] * nc + c1[None, :]).reshape(-1)
        v = (v[:, None] * v1[None, :]).reshape(-1)
        ncoarse *= nc
    return r, c, v, ncoarse


def _direct(I, J, V):
    """Direct interpolation from a maximal independent set: at most four coarse neighbours a
    row, rows without one empty (COO, coarse count).  The set depends on the sizes alone."""
    n = I.numel() - 1
    r, c = _rows_of(I), J.to(torch.int64)
    off = r != c
    r, c, a = r[off], c[off], V[off]
    w = _uniform(_gen(0, 1), n)
    state = torch.zeros(n, dtype=torch.int8, device=_DEV)  # 0 undecided, 1 coarse, 2 fine
    for _ in range(60):
        live = torch.where(state == 0, w, torch.full_like(w, -1.0))
        best = torch.full_like(w, -1.0).scatter_reduce_(0, r, live[c], "amax")
        new = (state == 0) & (w > best)
        state[new] = 1
        near = torch.zeros(n, dtype=torch.bool, device=_DEV)
        near[r[new[c]]] = True
        state[near & (state == 0)] = 2
        if not bool((state == 0).any()):
            break
    coarse = state == 1
    cidx = torch.cumsum(coarse, 0) - 1
    pick = coarse[c] & ~coarse[r]
    r, c, a = r[pick], c[pick], -a[pick]
    first = torch.cumsum(torch.bincount(r, minlength=n), 0) - torch.bincount(r, minlength=n)
    top = torch.arange(r.numel(), device=_DEV) - first[r] < 4
    r, c, a = r[top], c[top], a[top]
    s = _row_sums(torch.bincount(r, minlength=n), a)
    p = torch.nonzero(coarse).reshape(-1)
    return (torch.cat([r, p]), torch.cat([cidx[c], cidx[p]]),
            torch.cat([a / s[r], torch.ones(p.numel(), dtype=torch.float64, device=_DEV)]),
            int(coarse.sum()))


def _interp(case, I, J, V):
    n = I.numel() - 1
    if case.get("interp", "trilinear") == "trilinear":
        r, c, v, nc = _trilinear(case["nx"], case["ny"], case["nz"])
    else:
        r, c, v, nc = _direct(I, J, V)
    return _from_coo(r, c, v, n, nc), _from_coo(c, r, v, nc, n), n, nc


def _batch_problem(case, seed):
    """Block-diagonal 5-point Poisson problems of random sides (the case's), b = A x*."""
    sides = torch.randint(case["lo"], case["hi"] + 1, (case["count"],), generator=_gen(0, 2),
                          device=_DEV).tolist()
    Is, Js, Vs, seg = [torch.zeros(1, dtype=torch.int32, device=_DEV)], [], [], []
    rows = nnz = 0
    for k, s in enumerate(sides):
        I, J, V = _matrix({"kind": 5, "nx": s, "ny": s, "nz": 1}, seed, constant=True)
        Is.append(I[1:] + nnz)
        Js.append(J + rows)
        Vs.append(V)
        seg.append(torch.full((s * s,), k, dtype=torch.int64, device=_DEV))
        rows += s * s
        nnz += J.numel()
    I, J, V = torch.cat(Is), torch.cat(Js), torch.cat(Vs)
    return I, J, V, [(s, s, 1) for s in sides], torch.cat(seg), _normal(_gen(seed, 3), rows)


def _row_sums(lengths, t):
    """Sums of consecutive runs of t's rows (the same bits every time)."""
    return torch.segment_reduce(t, "sum", lengths=lengths, initial=0)


def _times(I, J, V, x):
    """A x in FP64 (x: (n,) or (n, k))."""
    t = V.view(-1, *([1] * (x.dim() - 1))) * x[J.to(torch.int64)]
    return _row_sums((I[1:] - I[:-1]).to(torch.int64), t)


def prepare(case, seed):
    op = case["op"]
    st = {"case": case}
    if op == "batch":
        I, J, V, grids, seg, xs = _batch_problem(case, seed)
        st.update(I=I, J=J, V=V, grids=grids, seg=seg, b=_times(I, J, V, xs))
        return st
    g = _gen(seed, 3)
    # the finest-level product of the Poisson benchmark has constant coefficients
    constant = op == "matvec" and case["form"] == "plain" and case["kind"] in (5, 7)
    I, J, V = _matrix(case, seed, constant)
    n = I.numel() - 1
    if op == "matvec" and case["form"] == "restrict":
        (PI, PJ, PV), _, n, nc = _interp(case, I, J, V)
        st.update(A=H.CSRMatrix(PI, PJ, PV, n, nc), x=_normal(g, n),
                  y=torch.empty(nc, dtype=torch.float64, device=_DEV))
    elif op == "matvec":
        A = MBSRMatrix.from_csr(I, J, V, n, n)
        A.set_precision(case["prec"])
        st.update(A=A, x=_normal(g, n), f=_normal(g, n),
                  y=torch.empty(n, dtype=torch.float64, device=_DEV))
    elif op == "spmm":
        A = MBSRMatrix.from_csr(I, J, V, n, n)
        shape = (n, case["k"]) if case["layout"] == "interleaved" else (case["k"], n)
        st.update(A=A, X=_normal(g, *shape),
                  Y=torch.empty(shape, dtype=torch.float64, device=_DEV))
    elif op in ("convert", "coarsen"):
        st.update(I=I, J=J, V=V, n=n)
    elif op == "boomer":
        st.update(I=I, J=J, V=V, n=n, b=_times(I, J, V, _normal(g, n)))
    elif op == "galerkin":
        P, R, n, nc = _interp(case, I, J, V)
        if case["api"] == "csr":
            A = H.CSRMatrix(I, J, V, n, n)
            H.CSR2BSR_GPU(A)
            st.update(A=A, P=P, R=R, n=n, nc=nc)
        else:
            A = MBSRMatrix.from_csr(I, J, V, n, n)
            P = MBSRMatrix.from_csr(*P, n, nc)
            R = MBSRMatrix.from_csr(*R, nc, n)
            for M in (A, P, R):
                M.set_precision(case["prec"])
            st.update(A=A, P=P, R=R)
    return st


# ---- one pass -----------------------------------------------------------------------------
def run(st):
    case = st["case"]
    op = case["op"]
    if op == "matvec":
        if case["form"] == "plain":
            return st["A"].spmv(st["x"], st["y"])
        if case["form"] == "residual":
            return st["A"].spmv(st["x"], st["y"], alpha=-1.0, beta=1.0, b=st["f"])
        H.hypre_CSRMatrixMatvecDevice(1, 1.0, st["A"], st["x"], 0.0, st["y"], st["y"])
        return st["y"]
    if op == "spmm":
        if case["layout"] == "interleaved":
            return st["A"].spmm_interleaved(st["X"], st["Y"])
        return st["A"].spmm(st["X"], st["Y"])
    if op == "convert":
        return MBSRMatrix.from_csr(st["I"], st["J"], st["V"], st["n"], st["n"]).arrays()
    if op == "galerkin":
        if case["api"] == "csr":
            P = H.CSRMatrix(*st["P"], st["n"], st["nc"])
            R = H.CSRMatrix(*st["R"], st["nc"], st["n"])
            C = H.hypreDevice_CSRSpGemm(R, H.hypreDevice_CSRSpGemm(st["A"], P))
            return {"i": C.i, "j": C.j, "data": C.data}
        return st["R"].spgemm(st["A"].spgemm(st["P"])).to_csr()
    if op == "coarsen":
        n, I, J, V = st["n"], st["I"], st["J"], st["V"]
        SI, SJ = CO.strength(n, I, J, V, 0.25, 1.0)
        cf, _ = CO.pmis(n, SI, SJ) if case["splitting"] == "pmis" else CO.hmis(n, SI, SJ)
        PI, PJ, PV, _ = CO.extpi_interp(n, I, J, V, SI, SJ, cf, 4)
        return {"SI": SI, "SJ": SJ, "cf": cf, "PI": PI, "PJ": PJ, "PV": PV}
    if op == "boomer":
        amg = AMG.BoomerAMG(st["I"], st["J"], st["V"], st["n"], torch.device(_DEV),
                            coarsen=case["splitting"])
        amg.capture()
        x, iters, _ = amg.pcg(st["b"], tol=1e-8)
        return x, iters
    amg = AMG.GeometricAMG(st["I"], st["J"], st["V"], st["grids"], torch.device(_DEV))
    amg.capture()
    x, iters, _ = amg.pcg(st["b"], tol=1e-8, segments=st["seg"])
    return x, iters


# ---- the same in 64 bits ------------------------------------------------------------------
def _product(A, B, ncols):
    """A B in FP64 over all products of entries (CSR triples, ascending columns)."""
    I, J, V = A
    BI, BJ, BV = B
    J = J.to(torch.int64)
    BI = BI.to(torch.int64)
    cnt = BI[J + 1] - BI[J]
    src = torch.repeat_interleave(torch.arange(J.numel(), device=J.device), cnt)
    at = torch.arange(src.numel(), device=J.device) - (torch.cumsum(cnt, 0) - cnt)[src]
    at += BI[J[src]]
    key = _rows_of(I)[src] * ncols + BJ.to(torch.int64)[at]
    val = V[src] * BV[at]
    del src
    keys, inv = torch.unique(key, return_inverse=True)
    out = torch.zeros(keys.numel(), dtype=torch.float64, device=J.device)
    out.index_add_(0, inv, val)
    CI = torch.zeros(I.numel(), dtype=torch.int32, device=J.device)
    CI[1:] = torch.cumsum(torch.bincount(keys // ncols, minlength=I.numel() - 1), 0)
    return CI, (keys % ncols).to(torch.int32), out


def exact(case, seed):
    op = case["op"]
    if op == "coarsen":
        # which entries the truncation keeps among equal ones is HYPRE's order of operations
        return None
    if op == "batch":
        return _batch_problem(case, seed)[5], None
    g = _gen(seed, 3)
    constant = op == "matvec" and case["form"] == "plain" and case["kind"] in (5, 7)
    I, J, V = _matrix(case, seed, constant)
    n = I.numel() - 1
    if op == "matvec" and case["form"] == "restrict":
        _, R, n, nc = _interp(case, I, J, V)
        return _times(*R, _normal(g, n))
    if op == "matvec":
        x, f = _normal(g, n), _normal(g, n)
        y = _times(I, J, V, x)
        return y if case["form"] == "plain" else f - y
    if op == "spmm":
        if case["layout"] == "interleaved":
            return _times(I, J, V, _normal(g, n, case["k"]))
        X = _normal(g, case["k"], n)
        return torch.stack([_times(I, J, V, x) for x in X])
    if op == "convert":
        # values in (block row, block column, position in the block) order
        r, c = _rows_of(I), J.to(torch.int64)
        bc = (n + 3) // 4
        order = torch.argsort(((r // 4) * bc + c // 4) * 16 + (r % 4) * 4 + c % 4)
        return {"blk_ptr": None, "blk_col": None, "blk_map": None, "val_ptr": None,
                "val": V[order]}
    if op == "boomer":
        return _normal(g, n), None
    P, R, n, nc = _interp(case, I, J, V)
    C = _product(R, _product((I, J, V), P, nc), nc)
    return {"i": None, "j": None, "data": C[2]} if case["api"] == "csr" else (None, None, C[2])


# ---- what a pass cannot do without ----------------------------------------------------------
def _stencil_nnz(kind, nx, ny, nz):
    if kind == 125:
        return int(0.65 * _stencil_nnz_box(2, nx, ny, nz))
    if kind == 27:
        return _stencil_nnz_box(1, nx, ny, nz)
    n = nx * ny * nz
    return 7 * n - 2 * (nx * ny + ny * nz + nx * nz) if nz > 1 else 5 * n - 2 * (nx + ny)


def _stencil_nnz_box(r, nx, ny, nz):
    def one(n):
        return sum(n - abs(d) for d in range(-r, r + 1) if abs(d) < n)
    return one(nx) * one(ny) * one(nz)


def _csr_bytes(rows, nnz):
    return 12 * nnz + 4 * (rows + 1)


def _triple(case):
    """(nnz of P, AP, RAP, products of AP, of R(AP)) of a case."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    nnz = _stencil_nnz(case["kind"], nx, ny, nz)
    if case.get("interp", "trilinear") == "direct":
        # about 0.3 of the points are coarse, 1.8 entries in an average row of P
        p = 1.8 * n
        ap, c = 6.3 * n, 0.3 * n * 20
        return p, ap, c, 1.8 * nnz, 1.8 * ap
    d = 3 if nz > 1 else 2
    p = n * 1.5 ** d
    if case["kind"] == 27:  # per direction: an even point reaches 3 coarse ones, an odd one 2
        ap = n * 2.5 ** d
    else:                   # corner points of the union of the neighbours' cells are missing
        ap = n * (7.75 if d == 3 else 4.75)
    return p, ap, n / 2 ** d * 3 ** d, nnz * 1.5 ** d, ap * 1.5 ** d


def work(case):
    op = case["op"]
    if op == "batch":
        m = sum(s * s for s in (case["lo"], (case["lo"] + case["hi"]) // 2, case["hi"])) / 3
        n = case["count"] * m
        # levels of n, n/4, ...; about 12 iterations of a cycle of five products
        return {"bytes": 12 * 6 * 80 * n * 4 / 3, "flops": 12 * 6 * 12 * n * 4 / 3}
    kind, nx, ny, nz = case["kind"], case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    nnz = _stencil_nnz(kind, nx, ny, nz)
    if op == "matvec":
        if case["form"] == "restrict":
            p, nc = _triple(case)[0], n / (8 if nz > 1 else 4)
            return {"bytes": 8 * p + 1.5 * p + 8 * (n + nc), "flops": 2 * p}
        blocks = nnz / {5: 2.9, 7: 4.0, 27: 5.0, 125: 5.5}[kind]
        value = {0: 8, 1: 4, 2: 2}[case["prec"]]
        vecs = 2 if case["form"] == "plain" else 3
        return {"bytes": value * nnz + 6 * blocks + n + 8 * vecs * n, "flops": 2 * nnz}
    if op == "spmm":
        return {"bytes": 8 * nnz + 6 * nnz / 4.5 + n + 16 * n * case["k"],
                "flops": 2 * nnz * case["k"]}
    if op == "convert":
        return {"bytes": _csr_bytes(n, nnz) + 8 * nnz + 6 * nnz / 4 + 2 * n, "flops": nnz}
    if op == "galerkin":
        p, ap, c, f1, f2 = _triple(case)
        nc = n / (8 if nz > 1 else 4)
        return {"bytes": _csr_bytes(n, nnz) + 2 * _csr_bytes(n, p) + 2 * _csr_bytes(n, ap)
                + _csr_bytes(nc, c), "flops": 2 * (f1 + f2)}
    if op == "coarsen":
        return {"bytes": 2 * _csr_bytes(n, nnz) + 3 * 4 * nnz + 12 * 2.5 * n + 12 * n,
                "flops": 20 * nnz}
    # the whole solve: setup passes over a hierarchy of 2.5 times the finest operator, then
    # about 10 iterations of five products on it
    return {"bytes": 2.5 * 60 * (12 * nnz + 24 * n), "flops": 2.5 * 120 * nnz}
