"""Performance cases: the work that a user of this library has it do.

Each case is a dict of plain values; `prepare` makes its inputs on the GPU
from a seed, `run` is one pass through the public entry points, `work` what
that pass cannot do without, `exact` the same result in 64 bits from plain
torch.  The structure of a matrix (its diagonal offsets) belongs to the case;
its values, and the vectors, come from the seed.

Kinds:
  spmv       y = H x on a Recon matrix (spmv_recon), y kept by the caller
  krylov     psi(t) = exp(-i t H) psi_0 (expm_krylov), workspace kept
  spgemm     C = A B on HM operands with a kept plan (SpgemmPlan.numeric)
  gemm_diag  C = A B on row-packed operands, plan and product (gemm_diag)
  power      H^k, every plan built in the call (chain.power)
  taylor     sum_k (t H)^k / k!, every plan built in the call (taylor_expm)
  propagator the same for exp(-i dt H), complex (chain.propagator)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from diagpu_amd import chain, workloads
from diagpu_amd.krylov import KrylovWorkspace, expm_krylov
from diagpu_amd.spgemm import SpgemmPlan, gemm_diag
from diagpu_amd.spmv import spmv_recon

_DEV = "cuda"
_F32, _F64, _C64, _C128 = torch.float32, torch.float64, torch.complex64, torch.complex128

# option -> (matrix dtype, vector dtype)
_DTYPES = {"f32": (_F32, _F32), "f64": (_F64, _F64), "c64": (_C64, _C64), "f32c64": (_F32, _C64)}
_SIZE = {_F32: 4, _F64: 8, _C64: 8}

HASH_BAND = [-9, -5, -2, -1, 0, 1, 2, 5, 9]


def listed():
    return [
        # One application of the 9-diagonal band of the SpMV tests at their
        # size: what a small call costs.
        {"name": "spmv_small", "kind": "spmv", "dtype": "f32", "n": 1000, "band": "hash"},
        # A band of 64 diagonals in an ordinary size that is no power of two.
        {"name": "spmv_band_f64", "kind": "spmv", "dtype": "f64", "n": 100_003, "band": "random",
         "count": 64, "half": 512, "structure": 1},
        # 2-D 5-point stencil on 2048 x 2048 (the benchmark's headline).
        {"name": "spmv_poisson", "kind": "spmv", "dtype": "f32", "n": 2048 * 2048,
         "band": "stencil5", "side": 2048},
        # 64 random diagonals over +-512 at n = 2^22: the largest SpMV.
        {"name": "spmv_band_large", "kind": "spmv", "dtype": "f32", "n": 1 << 22,
         "band": "random", "count": 64, "half": 512, "structure": 0},
        # A complex propagator's 85 diagonals applied to a complex state.
        {"name": "spmv_propagator", "kind": "spmv", "dtype": "c64", "n": 300_007,
         "band": "random", "count": 85, "half": 6144, "structure": 2},
        # One time step of a small real Hamiltonian on a 141 x 141 lattice.
        {"name": "krylov_small", "kind": "krylov", "dtype": "f32", "side": 141, "m": 30, "t": 0.8},
        # The same on 2048 x 2048 sites.
        {"name": "krylov_large", "kind": "krylov", "dtype": "f32", "side": 2048, "m": 30,
         "t": 0.8},
        # The SpGEMM benchmark's product: two bands of 33 diagonals.
        {"name": "spgemm_banded", "kind": "spgemm", "dtype": "f32", "n": 100_000, "a": "full",
         "a_half": 16, "b": "full", "b_half": 16},
        # 128 x 128 random diagonals over +-4096: the largest SpGEMM.
        {"name": "spgemm_random", "kind": "spgemm", "dtype": "f32", "n": 262_144, "a": "random",
         "a_count": 128, "a_half": 4096, "b": "random", "b_count": 128, "b_half": 4096,
         "structure": 3},
        # gemm_diag's defaults: plan and product of one small call.
        {"name": "gemm_diag", "kind": "gemm_diag", "n": 4096, "half": 10},
        # Order-6 series of the 3-D 7-point stencil on 128 x 128 x 64.
        {"name": "taylor_stencil", "kind": "taylor", "nx": 128, "ny": 128, "nz": 64, "t": 0.05,
         "order": 6},
        # Order-5 complex propagator of a ragged 3-D grid.
        {"name": "propagator_ragged", "kind": "propagator", "nx": 61, "ny": 47, "nz": 53,
         "t": 0.02, "order": 5},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "krylov", "spgemm", "spgemm", "spgemm",
                       "gemm_diag", "power", "taylor", "propagator"])
    if kind == "spmv":
        c = {"kind": kind, "dtype": rng.choice(list(_DTYPES))}
        n = _log_uniform(rng, 1000, 1 << 22)
        if rng.random() < 0.3:
            side = max(8, math.isqrt(n))
            c.update(n=side * side, band="stencil5", side=side)
            return c
        count = _log_uniform(rng, 3, 96)
        # at most the largest listed SpMV's bytes
        most = (64 * 4 << 22) // (max(_SIZE[t] for t in _DTYPES[c["dtype"]]) * count)
        n = max(1000, min(n, most))
        half = min(n // 2, max(count, _log_uniform(rng, 64, 8192)))
        c.update(n=n, band="random", count=count, half=half, structure=rng.randrange(1 << 20))
        return c
    if kind == "krylov":
        return {"kind": kind, "dtype": rng.choice(["f32", "c64"]),
                "side": _log_uniform(rng, 32, 1500), "m": rng.randint(12, 30),
                "t": round(rng.uniform(0.1, 0.3), 3)}
    if kind == "spgemm":
        c = {"kind": kind, "dtype": rng.choice(["f32", "f32", "c64"]),
             "n": _log_uniform(rng, 4000, 1 << 20)}
        if rng.random() < 0.4:
            c.update(a="full", a_half=rng.randint(1, 24), b="full", b_half=rng.randint(1, 24))
            return c
        ca, cb = _log_uniform(rng, 3, 128), _log_uniform(rng, 3, 128)
        half = _log_uniform(rng, 512, 4096)
        # at most a third of the largest listed product's C
        most = (3 << 30) // (8 * min(ca * cb, 4 * half + 1))
        c["n"] = max(2 * half + 1, min(c["n"], most))
        c.update(a="random", a_count=ca, a_half=half, b="random", b_count=cb, b_half=half,
                 structure=rng.randrange(1 << 20))
        if rng.random() < 0.3:
            c.update(a="full", a_half=rng.randint(1, 8))
            del c["a_count"]
        return c
    if kind == "gemm_diag":
        return {"kind": kind, "n": _log_uniform(rng, 2000, 1 << 20), "half": rng.randint(2, 16)}
    c = {"kind": kind, "nx": rng.randint(16, 96), "ny": rng.randint(16, 96),
         "nz": rng.randint(16, 96)}
    if kind == "power":
        c["k"] = rng.randint(2, 5)
    else:
        c.update(t=round(rng.uniform(0.01, 0.05), 4), order=rng.randint(2, 6 if kind == "taylor"
                                                                         else 5))
    return c


# --------------------------------------------------------------------------
# Structure
# --------------------------------------------------------------------------

def _random_offsets(count, half, structure):
    """0 and count - 1 other distinct offsets within +-half."""
    rng = np.random.default_rng(structure)
    pool = np.array([d for d in range(-half, half + 1) if d])
    return sorted({0, *map(int, rng.choice(pool, size=min(count - 1, pool.size), replace=False))})


def _spmv_offsets(case):
    if case["band"] == "hash":
        return list(HASH_BAND)
    if case["band"] == "stencil5":
        return [-case["side"], -1, 0, 1, case["side"]]
    return _random_offsets(case["count"], case["half"], case["structure"])


def _operand_offsets(case, which):
    half = case[which + "_half"]
    if case[which] == "full":
        return list(range(-half, half + 1))
    return _random_offsets(case[which + "_count"], half, 2 * case["structure"] + (which == "b"))


def _product_offsets(n, a, b):
    s = np.unique(np.add.outer(np.array(a, dtype=np.int64), np.array(b, dtype=np.int64)))
    return s[(s > -n) & (s < n)].tolist()


def _stencil7_offsets(case):
    nx, ny = case["nx"], case["ny"]
    return sorted({0, 1, -1, nx, -nx, nx * ny, -nx * ny})


def _sites(case):
    return case["nx"] * case["ny"] * case["nz"]


def _starts(n, offsets):
    return np.concatenate([[0], np.cumsum([n - abs(d) for d in offsets])]).astype(np.int64)


# --------------------------------------------------------------------------
# Values (torch only: prepare and exact share them)
# --------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    return g


def _uniform(shape, g, dtype, lo=-1.0, hi=1.0):
    if dtype.is_complex:
        parts = torch.rand(*shape, 2, generator=g, device=_DEV, dtype=_F32) * (hi - lo) + lo
        return torch.view_as_complex(parts)
    return torch.rand(*shape, generator=g, device=_DEV, dtype=dtype) * (hi - lo) + lo


def _clear_padding(offsets, v):
    n = v.shape[1]
    for k, d in enumerate(offsets):
        if d > 0:
            v[k, :d] = 0
        elif d < 0:
            v[k, n + d:] = 0


def _lattice(side, dtype, g):
    """The tight-binding Hamiltonian of a side x side lattice, Recon rows for
    offsets {side, 1, 0, -1, -side}: hoppings -1 (complex: a magnetic
    field's phase along x), an on-site energy of 4 + U(-1/2, 1/2)."""
    n = side * side
    v = torch.full((5, n), -1.0, device=_DEV, dtype=dtype)
    c = torch.arange(n, device=_DEV)
    if dtype.is_complex:
        angle = (c // side).to(_F32) * (2 * math.pi / 16)
        v[1] = -torch.polar(torch.ones_like(angle), angle)
        v[3] = v[1].conj()
    v[1].masked_fill_(c % side == 0, 0)
    v[3].masked_fill_(c % side == side - 1, 0)
    v[2] = _uniform((n,), g, _F32, 3.5, 4.5).to(dtype)
    _clear_padding([side, 1, 0, -1, -side], v)
    return [side, 1, 0, -1, -side], v


def _spmv_inputs(case, seed):
    mat, vec = _DTYPES[case["dtype"]]
    n, g = case["n"], _gen(seed)
    offsets = sorted(_spmv_offsets(case), reverse=True)
    if case["band"] == "stencil5":
        offsets, v = _lattice(case["side"], mat, g)
    else:
        v = _uniform((len(offsets), n), g, mat)
        _clear_padding(offsets, v)
    return offsets, v, torch.randn(n, generator=g, device=_DEV, dtype=vec)


def _krylov_inputs(case, seed):
    g = _gen(seed)
    offsets, v = _lattice(case["side"], _DTYPES[case["dtype"]][0], g)
    return offsets, v, torch.randn(case["side"] ** 2, generator=g, device=_DEV, dtype=_C64)


def _spgemm_inputs(case, seed):
    """Compact values of A and B, diagonal after diagonal."""
    g, dt = _gen(seed), _DTYPES[case["dtype"]][0]
    out = []
    for which in "ab":
        offs = _operand_offsets(case, which)
        out.append((offs, _uniform((int(_starts(case["n"], offs)[-1]),), g, dt)))
    return out


def _gemm_diag_inputs(case, seed):
    """Row-packed values: [i][t] = M[t, t + d_i], U(0.5, 1.5), zero outside."""
    g, n = _gen(seed), case["n"]
    offs = list(range(-case["half"], case["half"] + 1))
    out = []
    for _ in range(2):
        v = _uniform((len(offs), n), g, _F32, 0.5, 1.5)
        _clear_padding([-d for d in offs], v)
        out.append(v)
    return offs, out


def _stencil7_rows(case, seed):
    """offset -> values by row of the 3-D 7-point stencil: hoppings -1, an
    on-site energy of 6 + U(-1/2, 1/2)."""
    nx, ny, n = case["nx"], case["ny"], _sites(case)
    i = torch.arange(n, device=_DEV)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    inside = {1: x < nx - 1, -1: x > 0, nx: y < ny - 1, -nx: y > 0,
              nx * ny: z < case["nz"] - 1, -nx * ny: z > 0}
    rows = {d: -ok.to(_F32) for d, ok in inside.items()}
    rows[0] = _uniform((n,), _gen(seed), _F32, 5.5, 6.5)
    return rows


def _pack(rows, n):
    """HM values of {offset: values by row}."""
    return torch.cat([rows[d][max(0, -d): n - max(0, d)] for d in sorted(rows)])


# --------------------------------------------------------------------------
# prepare, run
# --------------------------------------------------------------------------

def _ints(v, dtype=torch.int32):
    return torch.tensor(v, dtype=dtype, device=_DEV)


def _hm(n, offsets, values):
    st = _starts(n, offsets)
    return workloads.HM(n, _ints(offsets), _ints([n - abs(d) for d in offsets]),
                        _ints(st[:-1].tolist(), torch.int64), values, list(offsets))


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "spmv":
        offsets, v, x = _spmv_inputs(case, seed)
        s.update(offsets=_ints(offsets), values=v.reshape(-1), n=case["n"], x=x,
                 y=torch.empty_like(x))
    elif kind == "krylov":
        offsets, v, psi = _krylov_inputs(case, seed)
        n = psi.numel()
        s.update(offsets=_ints(offsets), values=v.reshape(-1), n=n, psi=psi,
                 out=torch.empty_like(psi), ws=KrylovWorkspace(n, case["m"]))
    elif kind == "spgemm":
        A, B = (_hm(case["n"], offs, v) for offs, v in _spgemm_inputs(case, seed))
        plan = SpgemmPlan(A, B)
        plan.prepare(A.values.dtype)
        s.update(A=A, B=B, plan=plan,
                 C=torch.empty(plan.info.c_nnz, dtype=A.values.dtype, device=_DEV))
    elif kind == "gemm_diag":
        offs, (va, vb) = _gemm_diag_inputs(case, seed)
        s.update(n=case["n"], offsets=_ints(offs), a=va.reshape(-1), b=vb.reshape(-1))
    else:
        n = _sites(case)
        s["H"] = _hm(n, _stencil7_offsets(case), _pack(_stencil7_rows(case, seed), n))
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "spmv":
        return spmv_recon(s["offsets"], s["values"], s["n"], s["n"], s["x"], s["y"])
    if kind == "krylov":
        r = expm_krylov(s["offsets"], s["values"], s["n"], s["psi"], case["t"], case["m"],
                        out=s["out"], workspace=s["ws"])
        return {"psi": r.psi, "psi0_norm": r.psi0_norm}
    if kind == "spgemm":
        s["plan"].numeric(s["A"].values, s["B"].values, s["C"])
        return s["C"]
    if kind == "gemm_diag":
        plan, c = gemm_diag(s["n"], s["offsets"], s["a"], s["offsets"], s["b"])
        return {"offsets": plan.c_offsets(), "values": c}
    if kind == "power":
        M = chain.power(s["H"], case["k"])
    elif kind == "taylor":
        M = chain.taylor_expm(s["H"], case["t"], case["order"])
    else:
        M = chain.propagator(s["H"], case["t"], case["order"])
    return {"offsets": M.offsets, "starts": M.starts, "values": M.values}


# --------------------------------------------------------------------------
# work, tolerance
# --------------------------------------------------------------------------

def _nnz(n, offsets):
    return sum(n - abs(d) for d in offsets)


def _terms(n, a, b):
    """Multiply-adds of the product: rows i with i, i + da, i + da + db inside."""
    da, db = np.array(a, dtype=np.int64)[:, None], np.array(b, dtype=np.int64)[None, :]
    lo = np.maximum(0, np.maximum(-da, -da - db))
    hi = np.minimum(n, np.minimum(n - da, n - da - db))
    return int(np.maximum(0, hi - lo).sum())


def work(case):
    kind = case["kind"]
    if kind == "spmv":
        mat, vec = _DTYPES[case["dtype"]]
        n, nnz = case["n"], _nnz(case["n"], _spmv_offsets(case))
        per = 2 if not vec.is_complex else 8 if mat.is_complex else 4
        return {"bytes": nnz * _SIZE[mat] + 2 * n * _SIZE[vec], "flops": per * nnz}
    if kind == "krylov":
        mat, side, m = _DTYPES[case["dtype"]][0], case["side"], case["m"]
        n = side * side
        nnz = _nnz(n, [side, 1, 0, -1, -side])
        per = 8 if mat.is_complex else 4
        # per step the product, the dot, the three-term update and its norm;
        # then the combination of the m basis vectors
        return {"bytes": nnz * _SIZE[mat] + 2 * n * 8, "flops": m * (per * nnz + (4 + 10 + 4 + 8) * n)}
    if kind == "spgemm":
        n, a, b = case["n"], _operand_offsets(case, "a"), _operand_offsets(case, "b")
        dt = _DTYPES[case["dtype"]][0]
        nnz = _nnz(n, a) + _nnz(n, b) + _nnz(n, _product_offsets(n, a, b))
        return {"bytes": nnz * _SIZE[dt], "flops": (8 if dt.is_complex else 2) * _terms(n, a, b)}
    if kind == "gemm_diag":
        n, a = case["n"], list(range(-case["half"], case["half"] + 1))
        return {"bytes": 4 * (2 * _nnz(n, a) + _nnz(n, _product_offsets(n, a, a))),
                "flops": 2 * _terms(n, a, a)}
    n, h = _sites(case), _stencil7_offsets(case)
    if kind == "power":
        steps, s = case["k"] - 1, h
    else:
        steps, s = case["order"] - 1, h
    flops = 0
    for _ in range(steps):
        flops += _terms(n, h, s)
        s = sorted({*_product_offsets(n, h, s)})
    cplx = kind == "propagator"
    return {"bytes": 4 * _nnz(n, h) + (8 if cplx else 4) * _nnz(n, s),
            "flops": (8 if cplx else 2) * flops}


def tolerance(case):
    """About four times the distance from the 64-bit result measured on each
    kind (relative 2-norm: SpMV 2e-16 in fp64 and up to 2.3e-7 in fp32 with
    85 terms, Krylov 2.1e-7, products 2e-8 to 9e-8)."""
    if case.get("dtype") == "f64":
        return {"rel": 1e-15, "max": 1e-13}
    if case["kind"] in ("spmv", "krylov"):
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 4e-7, "max": 2e-5}


# --------------------------------------------------------------------------
# exact
# --------------------------------------------------------------------------

def _wide(t):
    return t.to(_C128 if t.is_complex() else _F64)


def _apply(offsets, v, x):
    """H x for Recon rows v."""
    n = x.numel()
    y = torch.zeros(n, dtype=torch.promote_types(v.dtype, x.dtype), device=_DEV)
    for k, d in enumerate(offsets):
        lo, hi = max(0, -d), min(n, n - d)
        y[lo:hi] += v[k, lo + d: hi + d] * x[lo + d: hi + d]
    return y


def _multiply_rows(n, A, B):
    """{offset: values by row} of A B."""
    C = {}
    for db in sorted(B):
        for da in sorted(A):
            dc = da + db
            lo, hi = max(0, -da, -dc), min(n, n - da, n - dc)
            if abs(dc) >= n or lo >= hi:
                continue
            if dc not in C:
                C[dc] = torch.zeros(n, dtype=A[da].dtype, device=_DEV)
            C[dc][lo:hi] += A[da][lo:hi] * B[db][lo + da: hi + da]
    return C


def _result(n, rows):
    offs = sorted(rows)
    return {"offsets": None, "starts": None, "values": _pack(rows, n)} if offs else None


def exact(case, seed):
    kind = case["kind"]
    if kind == "spmv":
        offsets, v, x = _spmv_inputs(case, seed)
        y = torch.zeros(case["n"], dtype=_wide(x).dtype, device=_DEV)
        for k, d in enumerate(offsets):
            lo, hi = max(0, -d), min(x.numel(), x.numel() - d)
            y[lo:hi] += _wide(v[k, lo + d: hi + d]) * _wide(x[lo + d: hi + d])
        return y
    if kind == "krylov":
        offsets, v, psi = _krylov_inputs(case, seed)
        v, psi = _wide(v), _wide(psi)
        norm = float(torch.linalg.vector_norm(psi))
        parts = max(1, math.ceil(9 * case["t"] / 2))    # ||H|| <= 9
        for _ in range(parts):
            term = psi
            for k in range(1, 30):
                term = _apply(offsets, v, term) * (-1j * case["t"] / (parts * k))
                psi = psi + term
        return {"psi": psi, "psi0_norm": norm}
    if kind == "spgemm":
        n = case["n"]
        (a, va), (b, vb) = _spgemm_inputs(case, seed)
        c = _product_offsets(n, a, b)
        sa, sb, sc = _starts(n, a), _starts(n, b), _starts(n, c)
        at = {d: k for k, d in enumerate(c)}
        va, vb = _wide(va), _wide(vb)
        out = torch.zeros(int(sc[-1]), dtype=va.dtype, device=_DEV)
        for i, da in enumerate(a):
            for j, db in enumerate(b):
                dc = da + db
                lo, hi = max(0, -da, -dc), min(n, n - da, n - dc)
                if dc not in at or lo >= hi:
                    continue
                pa, pb = int(sa[i]) + min(da, 0), int(sb[j]) + da + min(db, 0)
                pc = int(sc[at[dc]]) + min(dc, 0)
                out[pc + lo: pc + hi].addcmul_(va[pa + lo: pa + hi], vb[pb + lo: pb + hi])
        return out
    if kind == "gemm_diag":
        n = case["n"]
        offs, (va, vb) = _gemm_diag_inputs(case, seed)
        C = _multiply_rows(n, *({d: _wide(m[k]) for k, d in enumerate(offs)} for m in (va, vb)))
        return {"offsets": None, "values": _pack(C, n)}
    n = _sites(case)
    H = {d: v.to(_C128 if kind == "propagator" else _F64)
         for d, v in _stencil7_rows(case, seed).items()}
    if kind == "power":
        P = H
        for _ in range(case["k"] - 1):
            P = _multiply_rows(n, H, P)
        return _result(n, P)
    t = complex(0.0, -case["t"]) if kind == "propagator" else case["t"]
    S = {d: v * (t / case["order"]) for d, v in H.items()}
    S[0] = S[0] + 1
    for j in range(case["order"] - 1, 0, -1):
        S = {d: v * (t / j) for d, v in _multiply_rows(n, H, S).items()}
        S[0] = S[0] + 1
    return _result(n, S)
