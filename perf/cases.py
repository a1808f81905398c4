"""The work that a program using vcp_amd has it do, as cases that can be timed.

Matrices are column-major AoS pairs ({inf, sup} or {hi, lo}); on the GPU they
are float64 tensors of shape (cols, rows, 2), so a column is contiguous and
the leading dimension is the number of rows.  Each state keeps a Context, as a
program does for the life of its thread.

Kinds:
  host    C = IA * IB from host arrays to a host array (the call that the C++
          policy's operator* makes)
  plain   the FP64 directed-rounding products on device arrays; form "ii"
          (interval x interval), "ip" / "pi" (one point operand), "pp" (RU and
          RD product of two point matrices)
  tn      IA^T IA, the Gram matrices of the verified eigenproblems
  ozaki   the int8 interval product, untuned (nmod = radius = 0) or with the
          moduli count and radius scheme that the tuner gave
  dd      the double-double product
  lss     verified solution of one system with the caller's R ~ inv(mid A)
  lssb    the same for many systems of uneven order in one call
  galerkin  the Galerkin matrix of a 2D Legendre basis of order p at q x q points
"""
import math

import numpy as np
import torch

import vcp_amd
from vcp_amd import workloads

DEV = "cuda"


def listed():
    return [
        # a small block's product through the policy: host in, host out
        {"name": "host_96", "kind": "host", "m": 96, "n": 80, "k": 160},
        # the interval product of an ordinary verification (n = 1024, radius 2^-40 |mid|)
        {"name": "plain_1024", "kind": "plain", "form": "ii", "m": 1024, "n": 1024, "k": 1024},
        # interval matrix times a few vectors: residuals of approximate solutions
        {"name": "thin_4000", "kind": "plain", "form": "ip", "m": 4000, "n": 4, "k": 4000},
        # Gram matrix of an interval basis, ragged
        {"name": "tn_1500", "kind": "tn", "n": 1500, "k": 2900},
        # int8 interval product where the device is not filled, odd size, untuned
        {"name": "ozaki_500", "kind": "ozaki", "m": 500, "n": 500, "k": 500, "wide": False, "nmod": 0, "radius": 0},
        # the size at which the interval products are usually compared, untuned
        {"name": "ozaki_2000", "kind": "ozaki", "m": 2000, "n": 2000, "k": 2000, "wide": False, "nmod": 0,
         "radius": 0},
        # the headline product: exponents over 41 binades, the tuner's 15 moduli and half radius scheme
        {"name": "ozaki_8192", "kind": "ozaki", "m": 8192, "n": 8192, "k": 8192, "wide": True, "nmod": 15,
         "radius": 3},
        # dd products of a refinement step: a small system, and the full size
        {"name": "dd_600", "kind": "dd", "m": 600, "n": 600, "k": 600},
        {"name": "dd_4096", "kind": "dd", "m": 4096, "n": 4096, "k": 4096},
        # one verified solve, and a verification run's set of them
        {"name": "lss_2000", "kind": "lss", "n": 2000, "nrhs": 1},
        {"name": "lssb_64", "kind": "lssb", "count": 64, "nmin": 64, "nmax": 1024, "sizes": 5},
        # the producer of the Galerkin matrices
        {"name": "galerkin_30", "kind": "galerkin", "p": 30, "q": 60},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["host", "plain", "plain", "thin", "tn", "ozaki", "ozaki", "dd", "dd", "lss", "lssb", "galerkin"])
    if kind == "host":
        return {"kind": kind, "m": _log(rng, 2, 400), "n": _log(rng, 2, 400), "k": _log(rng, 2, 400)}
    if kind == "plain":
        return {"kind": kind, "form": rng.choice(["ii", "ip", "pi", "pp"]), "m": _log(rng, 32, 2600),
                "n": _log(rng, 32, 2600), "k": _log(rng, 32, 2600)}
    if kind == "thin":
        # few columns on the right: vectors; the point operand on either side
        return {"kind": "plain", "form": rng.choice(["ip", "ip", "pi", "ii"]), "m": _log(rng, 400, 6000),
                "n": _log(rng, 1, 24), "k": _log(rng, 400, 6000)}
    if kind == "tn":
        return {"kind": kind, "n": _log(rng, 60, 2000), "k": _log(rng, 100, 4000)}
    if kind == "ozaki":
        tuned = rng.random() < 0.4
        return {"kind": kind, "m": _log(rng, 100, 5000), "n": _log(rng, 100, 5000), "k": _log(rng, 100, 5000),
                "wide": rng.random() < 0.3, "nmod": rng.choice([14, 15, 16, 18]) if tuned else 0,
                "radius": rng.choice([1, 2, 3]) if tuned else 0}
    if kind == "dd":
        return {"kind": kind, "m": _log(rng, 100, 3000), "n": _log(rng, 100, 3000), "k": _log(rng, 100, 3000)}
    if kind == "lss":
        return {"kind": kind, "n": _log(rng, 100, 2200), "nrhs": _log(rng, 1, 8)}
    if kind == "lssb":
        return {"kind": kind, "count": _log(rng, 4, 64), "nmin": 64, "nmax": _log(rng, 200, 1024),
                "sizes": rng.randrange(1000)}
    p = rng.randrange(6, 37)
    return {"kind": kind, "p": p, "q": 2 * p + rng.randrange(0, 5)}


# ---- inputs ---------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, rows, cols):
    return torch.rand((cols, rows), dtype=torch.float64, device=DEV, generator=g) * 2.0 - 1.0


def _intervals(mid, rad):
    """[mid - rad, mid + rad], an end moved outward by one ulp where its sum is inexact"""
    lo, hi = mid - rad, mid + rad
    out = torch.empty((*mid.shape, 2), dtype=torch.float64, device=mid.device)
    inf = torch.full((), math.inf, dtype=torch.float64, device=mid.device)
    out[..., 0] = torch.where(lo + rad != mid, torch.nextafter(lo, -inf), lo)
    out[..., 1] = torch.where(hi - rad != mid, torch.nextafter(hi, inf), hi)
    return out


def _interval_matrix(g, rows, cols, wide=False):
    if not wide:
        mid = _uniform(g, rows, cols)
        return _intervals(mid, mid.abs() * 2.0 ** -40)
    mid = torch.rand((cols, rows), dtype=torch.float64, device=DEV, generator=g) + 1.0
    mid *= torch.randint(0, 2, (cols, rows), device=DEV, generator=g) * 2 - 1
    mid *= torch.exp2(torch.randint(-20, 21, (cols, rows), device=DEV, generator=g).double())
    return _intervals(mid, mid.abs() * 2.0 ** -45)


def _dd_matrix(g, rows, cols):
    hi = _uniform(g, rows, cols)
    lo = hi * 2.0 ** -53 * _uniform(g, rows, cols)
    s = hi + lo
    return torch.stack((s, lo - (s - hi)), dim=-1)


def _system(rng, n, nrhs):
    """(R, IA, Ib) of one verified solve, host arrays: workloads.residual_problem and right-hand sides"""
    R, IA = workloads.residual_problem(rng, n)
    return R, IA, workloads.uniform_intervals(rng, n, nrhs, -45)


def _to_dev(x):
    """a column-major host array (pairs or points) on the GPU, columns contiguous"""
    return torch.from_numpy(np.ascontiguousarray(x.swapaxes(0, 1))).to(DEV)


def _sizes(case):
    rng = np.random.default_rng(case["sizes"])
    return [int(round(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))))
            for _ in range(case["count"])]


def _galerkin_inputs(case, seed):
    phi, w, _ = workloads.galerkin(case["p"], case["q"])
    # a smooth positive coefficient function, another one for each seed
    x, _wt = np.polynomial.legendre.leggauss(case["q"])
    c = np.random.default_rng(seed).uniform(-1.0, 1.0, (2, 3))
    f = [sum(c[d][j] * np.cos((j + 1) * np.pi * x / 2) for j in range(3)) for d in range(2)]
    v = (np.outer(f[0], f[1]) / 9.0 + 2.0).reshape(-1, 1)
    u = workloads.interval_from_midrad(v, np.ldexp(np.abs(v), -50)).reshape(-1, 2)
    return phi, w, np.ascontiguousarray(u)


def _inputs(case, seed):
    """every input of a case, on the GPU (host arrays for "host")"""
    kind, g = case["kind"], _gen(seed)
    if kind == "host":
        rng = np.random.default_rng(seed)
        return {"A": workloads.uniform_intervals(rng, case["m"], case["k"], -40),
                "B": workloads.uniform_intervals(rng, case["k"], case["n"], -40)}
    if kind == "plain":
        f, m, n, k = case["form"], case["m"], case["n"], case["k"]
        return {"A": _interval_matrix(g, m, k) if f[0] == "i" else _uniform(g, m, k),
                "B": _interval_matrix(g, k, n) if f[1] == "i" else _uniform(g, k, n)}
    if kind == "tn":
        return {"A": _interval_matrix(g, case["k"], case["n"])}
    if kind == "ozaki":
        return {"A": _interval_matrix(g, case["m"], case["k"], case["wide"]),
                "B": _interval_matrix(g, case["k"], case["n"], case["wide"])}
    if kind == "dd":
        return {"A": _dd_matrix(g, case["m"], case["k"]), "B": _dd_matrix(g, case["k"], case["n"])}
    if kind == "galerkin":
        phi, w, u = _galerkin_inputs(case, seed)
        return {"phi": _to_dev(phi), "w": torch.from_numpy(w).to(DEV), "u": torch.from_numpy(u).to(DEV)}
    rng = np.random.default_rng(seed)
    if kind == "lss":
        R, IA, Ib = _system(rng, case["n"], case["nrhs"])
        return {"R": _to_dev(R), "A": _to_dev(IA), "b": _to_dev(Ib)}
    systems = [_system(rng, n, 1) for n in _sizes(case)]
    return {"R": [_to_dev(s[0]) for s in systems], "A": [_to_dev(s[1]) for s in systems],
            "b": [_to_dev(s[2]) for s in systems]}


def _pairs(rows, cols):
    return torch.zeros((cols, rows, 2), dtype=torch.float64, device=DEV)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], s["ctx"], kind = case, vcp_amd.Context(), case["kind"]
    if kind == "plain":
        if case["form"] == "pp":
            s["C"], s["C2"] = (torch.zeros((case["n"], case["m"]), dtype=torch.float64, device=DEV) for _ in range(2))
        else:
            s["C"] = _pairs(case["m"], case["n"])
    elif kind == "tn":
        s["C"] = _pairs(case["n"], case["n"])
    elif kind == "ozaki":
        s["ctx"].set_param(vcp_amd.PARAM_OZ_NMOD, case["nmod"])
        s["ctx"].set_param(vcp_amd.PARAM_OZ_RADIUS, case["radius"])
        s["C"] = _pairs(case["m"], case["n"])
    elif kind == "dd":
        s["C"] = _pairs(case["m"], case["n"])
    elif kind == "galerkin":
        s["C"] = _pairs(case["p"] ** 2, case["p"] ** 2)
    elif kind == "lss":
        s["X"] = _pairs(case["n"], case["nrhs"])
    elif kind == "lssb":
        n = _sizes(case)
        s["n"], s["X"] = n, torch.zeros((sum(n), 2), dtype=torch.float64, device=DEV)
        starts = np.concatenate(([0], np.cumsum(n)))[:-1]
        s["args"] = (n, [1] * len(n), [t.data_ptr() for t in s["A"]], n, [t.data_ptr() for t in s["b"]], n,
                     [t.data_ptr() for t in s["R"]], n, [s["X"].data_ptr() + 16 * int(o) for o in starts], n)
    torch.cuda.synchronize()   # the context has a stream of its own
    return s


# ---- one pass ---------------------------------------------------------------
def _call(name, ctx, *args):
    rc = getattr(vcp_amd.lib(), name)(ctx.handle, *args)
    if rc:
        raise vcp_amd.VcphipError(rc, name)


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "host":
        return ctx.igemm(s["A"], s["B"])
    if kind == "plain":
        f, m, n, k = case["form"], case["m"], case["n"], case["k"]
        A, B, C = s["A"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr()
        if f == "ii":
            ctx.igemm_dev(vcp_amd.FORM_PLAIN, m, n, k, A, m, B, k, C, m)
        elif f == "ip":
            _call("vcphip_igemm_ip_dev", ctx, m, n, k, A, m, B, k, C, m)
        elif f == "pi":
            ctx.igemm_pi_dev(m, n, k, A, m, B, k, C, m)
        else:
            ctx.gemm_rurd_dev(m, n, k, A, m, B, k, C, s["C2"].data_ptr(), m)
            return {"up": s["C"], "down": s["C2"]}
        return s["C"]
    if kind == "tn":
        _call("vcphip_igemm_tn_dev", ctx, case["k"], case["n"], s["A"].data_ptr(), case["k"], s["C"].data_ptr(),
              case["n"])
        return s["C"]
    if kind == "ozaki":
        m, n, k = case["m"], case["n"], case["k"]
        ctx.igemm_dev(vcp_amd.FORM_OZAKI, m, n, k, s["A"].data_ptr(), m, s["B"].data_ptr(), k, s["C"].data_ptr(), m)
        return s["C"]
    if kind == "dd":
        m, n, k = case["m"], case["n"], case["k"]
        ctx.ddgemm_dev(m, n, k, s["A"].data_ptr(), m, s["B"].data_ptr(), k, s["C"].data_ptr(), m)
        return {"hi": s["C"][..., 0], "lo": s["C"][..., 1]}
    if kind == "lss":
        n, nrhs = case["n"], case["nrhs"]
        g = ctx.lss_dev(n, nrhs, s["A"].data_ptr(), n, s["b"].data_ptr(), n, s["R"].data_ptr(), n, s["X"].data_ptr(),
                        n)
        return {"X": s["X"], "g": g}
    if kind == "lssb":
        g = ctx.lss_batched_dev(*s["args"])
        return {"X": s["X"], "g": np.array(g)}
    p, q = case["p"], case["q"]
    _call("vcphip_uhphiphi_dev", ctx, p * p, q * q, s["phi"].data_ptr(), p * p, s["w"].data_ptr(), s["u"].data_ptr(),
          s["C"].data_ptr(), p * p)
    return s["C"]


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    """each operand read once and each result written once; FP64 operations of
    the product's chains (2 per multiply-add and chain), for the int8 and dd
    products those of the same result by the plain chains (4 and 1)"""
    kind = case["kind"]
    if kind == "galerkin":
        m, pts = case["p"] ** 2, case["q"] ** 2
        return {"bytes": 16 * (m * pts + 2 * pts + m * m), "flops": 8.0 * m * (m + 1) / 2 * pts}
    if kind == "tn":
        n, k = case["n"], case["k"]
        return {"bytes": 16 * (n * k + n * n), "flops": 10.0 * n * (n + 1) / 2 * k}
    if kind == "lss":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 24 * n * n + 32 * n * r, "flops": 6.0 * n ** 3 + 20.0 * n * n * r}
    if kind == "lssb":
        s = _sizes(case)
        return {"bytes": sum(24 * n * n + 32 * n for n in s), "flops": sum(6.0 * n ** 3 + 20.0 * n * n for n in s)}
    m, n, k = case["m"], case["n"], case["k"]
    f = case.get("form", "ii")
    a, b = (16 if x == "i" else 8 for x in f)
    chains = {"ii": 4, "ip": 3, "pi": 3, "pp": 2}[f]
    if kind == "dd":
        chains = 1
    return {"bytes": a * m * k + b * k * n + 16 * m * n, "flops": 2.0 * chains * m * n * k}


# ---- the results in plain 64-bit arithmetic -----------------------------------
def _mr(x):
    """midpoint and radius, rows x cols, of an operand (a point operand: radius 0)"""
    if x.dim() == 2:
        return x.T, torch.zeros_like(x).T
    return (0.5 * (x[..., 0] + x[..., 1])).T, (0.5 * (x[..., 1] - x[..., 0])).T


def _product(A, B):
    am, ar = _mr(A)
    bm, br = _mr(B)
    mid, rad = am @ bm, (am.abs() + ar) @ br + ar @ bm.abs()
    return torch.stack((mid - rad, mid + rad), dim=-1).transpose(0, 1)


def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "host":
        return _product(_to_dev(x["A"]), _to_dev(x["B"])).transpose(0, 1).cpu().numpy()
    if kind == "plain" and case["form"] == "pp":
        c = (x["A"].T @ x["B"].T).T
        return {"up": c, "down": c}
    if kind in ("plain", "ozaki"):
        return _product(x["A"], x["B"])
    if kind == "tn":
        return _product(x["A"].transpose(0, 1), x["A"])
    if kind == "dd":
        # the high part; the low part is below what 64 bits hold
        return {"hi": (x["A"][..., 0].T @ x["B"][..., 0].T).T, "lo": None}
    if kind == "galerkin":
        phi, w, u = _mr(x["phi"])[0], x["w"].mean(dim=-1), x["u"].mean(dim=-1)
        c = (phi * (w * u)) @ phi.T
        return torch.stack((c, c), dim=-1)
    if kind == "lss":
        v = torch.linalg.solve(_mr(x["A"])[0], _mr(x["b"])[0]).T
        return {"X": torch.stack((v, v), dim=-1), "g": None}
    v = torch.cat([torch.linalg.solve(_mr(A)[0], _mr(b)[0])[:, 0] for A, b in zip(x["A"], x["b"])])
    return {"X": torch.stack((v, v), dim=-1), "g": None}
