"""The work that programs have this library do, as cases with inputs, one pass each and the 64-bit values.

A case is a dict of plain values.  ``kind`` says which call it is:

* ``rmp2``       closed-shell MP2 energy, ``jues_rmp2`` on a context that holds the AO integrals
* ``rmp2_grad``  the MP2 adjoint (dE/dC, dE/deps and, for ``dg``, dE/dg), ``jues_rmp2_grad``, likewise
* ``rccd``       a whole closed-shell CCD solve, ``RCCD.do_rccd``, energy and amplitudes
* ``rccsd``      a whole closed-shell CCSD solve, ``RCCSD.do_rccsd``, energy and amplitudes
* ``df_rccd``    ten CCD sweeps with the ladder rebuilt from the factors, ``DFRCCD.do_df_rccd``
* ``triples``    the (T) correction from given CCSD amplitudes, ``PerturbativeTriples.rccsd_pT``

``o`` and ``v`` are the occupied and virtual orbitals, ``naux`` the auxiliary functions (0: the dense
n^4 AO tensor).  The MP2 calls go through the C ABI with a context of their own, as a program that
keeps its integrals on the device does; the solves take a ``Wfn``, whose integrals are uploaded with it.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "jues.jl_amd"))

import jues  # noqa: E402,F401
from jues import CoupledCluster, MollerPlesset, _lib  # noqa: E402
from jues.Wavefunction import FactoredERI, Wfn, prec_code  # noqa: E402

DEVICE = "cuda"

# How strong the integrals are: the largest eigenvalue of (ia|jb) is about this, against orbital
# energy differences of 1 and more, so that the solves take the 10 to 20 iterations of a molecule
# near its equilibrium.
STRENGTH = 0.35

SWEEPS = 10   # sweeps of a df_rccd case
CYCLES = 12   # iterations of a solve, for work(): what such a solve takes at the least


def case(name, kind, o, v, naux, prec="fp64", **more):
    return dict(name=name, kind=kind, o=o, v=v, naux=naux, prec=prec, **more)


def listed():
    return [
        # a small molecule in a minimal basis (water, STO-3G): one call of a scan over geometries
        case("mp2_water", "rmp2", 5, 2, 0),
        # the same molecule's CCSD, all of it: a few dozen numbers an iteration
        case("ccsd_water", "rccsd", 5, 2, 0),
        # a small molecule in a double-zeta basis, CCD from the dense tensor
        case("ccd_n24", "rccd", 5, 19, 0),
        # a dense AO tensor of ordinary size: the four-index transform and the energy
        case("mp2_n128", "rmp2", 20, 108, 0),
        # its orbital gradient, for orbital optimisation and response
        case("mp2_grad_n96", "rmp2_grad", 15, 81, 0, dg=False),
        # density-fitted MP2 and its gradient at the size of a drug-like fragment
        case("df_mp2_n256", "rmp2", 40, 216, 768),
        case("df_mp2_grad_n256", "rmp2_grad", 40, 216, 768, dg=False),
        # CCSD in a triple-zeta basis, plain FP64
        case("ccsd_n120", "rccsd", 20, 100, 360),
        # CCD with FP32 contractions and FP64 refinement, at a size where both stages count; odd sizes
        case("ccd_mixed_n157", "rccd", 23, 134, 471, "fp32_mixed"),
        # the largest: CCD on split-FP16 products with defect correction
        case("ccd_fp16x3_n224", "rccd", 34, 190, 672, "fp16x3_mixed"),
        # (T) after a CCSD of a small molecule in a triple-zeta basis; odd sizes
        case("triples_n61", "triples", 10, 51, 183),
        # CCD without a stored ladder, as it is run where v^4 does not fit
        case("df_ccd_n90", "df_rccd", 15, 75, 270),
    ]


def _span(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _orbitals(rng, lo, hi):
    """(o, v) with n = o + v spread over [lo, hi]; between a twelfth and a third of the orbitals occupied
    (a minimal basis has more)."""
    n = _span(rng, lo, hi)
    o = max(2, min(n - 2, int(round(n * rng.uniform(1 / 12, 1 / 3 if n > 12 else 0.7)))))
    return o, n - o


def _naux(rng, n):
    return int(round(n * rng.uniform(2.4, 3.3)))


def draw(rng):
    kind = rng.choice(["rmp2", "rmp2", "rmp2_grad", "rmp2_grad", "rccd", "rccd", "rccd", "rccsd", "rccsd",
                       "df_rccd", "triples"])
    dense = rng.random() < 0.5
    if kind == "rmp2":
        o, v = _orbitals(rng, 7, 120) if dense else _orbitals(rng, 40, 250)
        return dict(kind=kind, o=o, v=v, naux=0 if dense else _naux(rng, o + v), prec="fp64")
    if kind == "rmp2_grad":
        o, v = _orbitals(rng, 10, 90) if dense else _orbitals(rng, 40, 250)
        return dict(kind=kind, o=o, v=v, naux=0 if dense else _naux(rng, o + v), prec="fp64",
                    dg=dense and o + v <= 32)
    if kind == "rccd":
        o, v = _orbitals(rng, 8, 40) if dense else _orbitals(rng, 40, 160)
        prec = rng.choice(["fp64", "fp32_mixed", "fp16x3_mixed"])
        return dict(kind=kind, o=o, v=v, naux=0 if dense else _naux(rng, o + v), prec=prec)
    if kind == "rccsd":
        o, v = _orbitals(rng, 7, 40) if dense else _orbitals(rng, 40, 110)
        return dict(kind=kind, o=o, v=v, naux=0 if dense else _naux(rng, o + v), prec="fp64")
    if kind == "df_rccd":
        o, v = _orbitals(rng, 20, 90)
        return dict(kind=kind, o=o, v=v, naux=_naux(rng, o + v), prec="fp64")
    o, v = rng.randint(3, 11), _span(rng, 8, 56)
    return dict(kind=kind, o=o, v=v, naux=0 if o + v <= 40 and dense else _naux(rng, o + v), prec="fp64")


# ---- inputs ----------------------------------------------------------------------------------------

def _system(case, seed):
    """Factors b[P, mu, nu] (symmetric in mu, nu), orbitals C (orthonormal columns, occupied first) and
    orbital energies, as CUDA FP64 tensors."""
    o, v = case["o"], case["v"]
    n = o + v
    naux = case["naux"] or 3 * n
    g = torch.Generator(device=DEVICE).manual_seed(1000003 * int(seed) + 7919 * n + o)
    x = torch.randn((naux, n, n), generator=g, device=DEVICE, dtype=torch.float64)
    b = x + x.transpose(1, 2)
    # (ia|jb) of such factors has a largest eigenvalue near 2 (sqrt(ov) + sqrt(naux))^2
    b *= math.sqrt(STRENGTH / 2.0) / (math.sqrt(o * v) + math.sqrt(naux))
    h = np.random.default_rng([int(seed), n, o])
    q, r = np.linalg.qr(h.standard_normal((n, n)))
    C = torch.from_numpy(q * np.sign(np.diag(r))).to(DEVICE)
    eps = np.concatenate([np.sort(h.uniform(-1.5, -0.5, o)), np.sort(h.uniform(0.5, 3.0, v))])
    return b, C, torch.from_numpy(eps).to(DEVICE)


def _amplitudes(case, seed, b, C, eps):
    """T1 [i,a] and T2 [i,j,a,b] of the size that a CCSD leaves: the first-order doubles and small singles."""
    o, v = case["o"], case["v"]
    L = _mo(b, C[:, :o], C[:, o:]).reshape(-1, o * v)
    t2 = (L.T @ L).reshape(o, v, o, v).permute(0, 2, 1, 3) / _d2(eps, o)
    g = torch.Generator(device=DEVICE).manual_seed(1000003 * int(seed) + 13)
    t1 = 0.01 * torch.randn((o, v), generator=g, device=DEVICE, dtype=torch.float64)
    return t1, t2.contiguous()


def _eri(case, b):
    """The AO integrals as a program holds them: b[mu, nu, P] or the dense tensor, in Fortran order."""
    if case["naux"]:
        return FactoredERI(b.cpu().numpy().T)
    n = b.shape[1]
    f = b.reshape(b.shape[0], n * n)
    return (f.T @ f).reshape(n, n, n, n).cpu().numpy().T


def prepare(case, seed):
    b, C, eps = _system(case, seed)
    o, v = case["o"], case["v"]
    n = o + v
    wfn = Wfn.from_orbitals(C.cpu().numpy(), eps.cpu().numpy(), o, _eri(case, b))
    state = dict(case=case, wfn=wfn)
    if case["kind"] == "triples":
        t1, t2 = _amplitudes(case, seed, b, C, eps)
        state.update(T1=np.asfortranarray(t1.cpu().numpy()), T2=np.asfortranarray(t2.cpu().numpy()))
    if case["kind"] in ("rmp2", "rmp2_grad"):
        ctx = _lib.Context(0)
        if case["naux"]:
            ctx.set_ao_factors(wfn.ao_eri.B)
        else:
            ctx.set_ao_eri(wfn.ao_eri)
        wfn.ao_eri = None
        state.update(ctx=ctx, E=np.zeros(1))
        if case["kind"] == "rmp2_grad":
            state.update(dC=np.zeros((n, n), order="F"), deps=np.zeros(n),
                         dg=np.zeros((n, n, n, n), order="F") if case["dg"] else None)
    return state


# ---- one pass --------------------------------------------------------------------------------------

def run(state):
    case, wfn = state["case"], state["wfn"]
    kind, o, v, p = case["kind"], case["o"], case["v"], _lib.ptr
    n = o + v
    if kind == "rmp2":
        ctx, E = state["ctx"], state["E"]
        ctx.check(ctx.lib.jues_rmp2(ctx.h, prec_code(case["prec"]), p(wfn.Cao), o, p(wfn.Cav), v, n, p(wfn.epsa), p(E)))
        return float(E[0])
    if kind == "rmp2_grad":
        ctx, E, dC, deps, dg = (state[k] for k in ("ctx", "E", "dC", "deps", "dg"))
        ctx.check(ctx.lib.jues_rmp2_grad(ctx.h, prec_code(case["prec"]), p(wfn.Ca), o, n, p(wfn.epsa), p(E), p(dC),
                                         p(dg), p(deps)))
        return [float(E[0]), dC, deps] + ([dg] if dg is not None else [])
    if kind == "rccd":
        # the fast forms hand over to FP64 by a restart (FP32) or by defect correction (split FP16)
        refine = "defect" if case["prec"] == "fp16x3_mixed" else "restart"
        return CoupledCluster.RCCD.do_rccd(wfn, prec=case["prec"], refine=refine, return_T2=True, cc_max_rms=1e-10,
                                           cc_e_conv=1e-11)
    if kind == "rccsd":
        return CoupledCluster.RCCSD.do_rccsd(wfn, prec=case["prec"], return_T=True, cc_max_rms=1e-10, cc_e_conv=1e-11)
    if kind == "df_rccd":
        return CoupledCluster.DFRCCD.do_df_rccd(wfn, SWEEPS, return_T2=True, prec=case["prec"])
    return CoupledCluster.PerturbativeTriples.rccsd_pT(wfn, state["T1"], state["T2"], prec=case["prec"])


def work(case):
    o, v, x = case["o"], case["v"], case["naux"]
    n, N2 = o + v, (case["o"] * case["v"]) ** 2
    ints = 8.0 * (n * n * x if x else n ** 4)
    small = 8.0 * (2 * n * n + n)
    # the blocks of MO integrals that the amplitude equations read
    if x:
        xform = 2.0 * n * n * o * x + 2.0 * n * o * v * x + 2.0 * N2 * x
    else:
        xform = 2.0 * n ** 4 * o + 2.0 * n ** 3 * o * o + 2.0 * n * n * o * o * v + 2.0 * n * o * o * v * v
    if case["kind"] == "rmp2":
        return {"bytes": ints + small, "flops": xform + 6.0 * N2}
    if case["kind"] == "rmp2_grad":
        back = 2.0 * xform
        return {"bytes": ints + 2 * small + (8.0 * n ** 4 if case["dg"] else 0.0),
                "flops": xform + back + (2.0 * n ** 4 * o if case["dg"] else 0.0)}
    if case["kind"] == "triples":
        trip = o * (o + 1) * (o + 2) // 6
        return {"bytes": ints + small + 8.0 * N2, "flops": trip * 12.0 * v ** 3 * (v + o)}
    npv, nmv, npo, nmo = v * (v + 1) // 2, v * (v - 1) // 2, o * (o + 1) // 2, o * (o - 1) // 2
    ladder = 2.0 * npo * npv * npv + 2.0 * nmo * nmv * nmv
    if case["kind"] == "df_rccd":
        ladder += 2.0 * v ** 4 * x
    cycle = 10.0 * N2 * o * v + (4.0 * N2 * x if x else 2.0 * N2 * o * v) + ladder
    if case["kind"] == "rccsd":
        cycle += 2.0 * o ** 3 * v ** 3
    k = SWEEPS if case["kind"] == "df_rccd" else CYCLES
    return {"bytes": ints + small + 8.0 * N2, "flops": xform + k * cycle}


# ---- the values in 64 bits -------------------------------------------------------------------------

def _mo(b, C1, C2):
    """L[P, p, q] = sum C1[mu, p] b[P, mu, nu] C2[nu, q]."""
    return torch.matmul(C1.T.contiguous(), torch.matmul(b, C2.contiguous()))


def _d2(eps, o):
    eo, ev = eps[:o], eps[o:]
    return eo[:, None, None, None] + eo[None, :, None, None] - ev[None, None, :, None] - ev[None, None, None, :]


def _pair(A, B):
    """(pq|rs) = sum_P A[P, p, q] B[P, r, s]."""
    m = A.reshape(A.shape[0], -1).T @ B.reshape(B.shape[0], -1)
    return m.reshape(*A.shape[1:], *B.shape[1:])


def _mm(A, B, na, nb):
    """The last na indices of A against the first na of B, nb free indices left in B."""
    sa, sb = A.shape[:A.dim() - na], B.shape[na:]
    assert len(sb) == nb
    return (A.reshape(math.prod(sa), -1) @ B.reshape(-1, math.prod(sb))).reshape(*sa, *sb)


def _mp2(b, C, eps, o):
    """E and its derivatives by autograd, with every entry of C and eps independent."""
    L = _mo(b, C[:, :o], C[:, o:])
    K = _pair(L, L).permute(0, 2, 1, 3)
    return (K * (2.0 * K - K.transpose(2, 3)) / _d2(eps, o)).sum()


def _omega(b, C, eps, o, t1, t2):
    """The closed-shell CCSD vector function in T1-transformed integrals (Helgaker, Jorgensen and Olsen,
    Molecular Electronic-Structure Theory, section 13.7.4), with t1 None for CCD.  t2[i, a, j, b]."""
    n = C.shape[0]
    v = n - o
    Co, Cv = C[:, :o], C[:, o:]
    f = torch.diag(eps)
    X = Y = torch.eye(n, dtype=C.dtype, device=C.device)
    if t1 is not None:
        X, Y = X.clone(), Y.clone()
        X[o:, :o] = -t1.T   # left (bra) orbitals: particles take -t1 of the holes
        Y[:o, o:] = t1      # right (ket) orbitals, transposed below: holes take t1 of the particles
    Cx, Cy = C @ X.T, C @ Y.T
    xo, xv, yo, yv = Cx[:, :o], Cx[:, o:], Cy[:, :o], Cy[:, o:]
    Lov = _mo(b, Co, Cv)
    Lvo, Loo, Lvv = _mo(b, xv, yo), _mo(b, xo, yo), _mo(b, xv, yv)
    F = X @ f @ Y.T
    if t1 is not None:
        Lpq = _mo(b, Cx, Cy)
        w = (Lov * t1).sum((1, 2))
        F = F + 2.0 * torch.tensordot(w, Lpq, 1)
        Lpc, Lkq = Lpq[:, :, o:], Lpq[:, :o, :]      # L[P, p, c], L[P, k, q]
        h = torch.matmul(Lpc, t1.T.contiguous())      # [P, p, k]
        F = F - h.permute(1, 0, 2).reshape(n, -1) @ Lkq.reshape(-1, n)
    Foo, Fov, Fvo, Fvv = F[:o, :o], F[:o, o:], F[o:, :o], F[o:, o:]
    g = _pair(Lov, Lov)                                # (kc|ld)
    u2 = 2.0 * t2 - t2.permute(0, 3, 2, 1)             # u[i, a, j, b]
    Lg = 2.0 * g - g.permute(0, 3, 2, 1)               # 2 (ld|kc) - (lc|kd)
    tij = t2.permute(0, 2, 1, 3).reshape(o * o, v * v)  # t[(ij), (cd)]
    O2 = _pair(Lvo, Lvo).permute(1, 0, 3, 2).clone()   # (ai|bj) at [i, a, j, b]
    # particle-particle ladder, one a at a time: (ac|bd)
    pp = torch.empty((v, o * o, v), dtype=C.dtype, device=C.device)
    Lbd = Lvv.reshape(Lvv.shape[0], v * v)
    for a in range(v):
        ac = (Lvv[:, a, :].T @ Lbd).reshape(v, v, v).permute(0, 2, 1).reshape(v * v, v)  # [(c, d), b]
        pp[a] = tij @ ac
    O2 += pp.reshape(v, o, o, v).permute(1, 0, 2, 3)
    # hole-hole ladder
    kilj = _pair(Loo, Loo).permute(0, 2, 1, 3).reshape(o * o, o * o)                     # [(k, l), (i, j)]
    kcld = g.permute(0, 2, 1, 3).reshape(o * o, v * v)
    B = kilj + kcld @ tij.T
    O2 += (B.T @ tij).reshape(o, o, v, v).permute(0, 2, 1, 3)
    # exchange ring: x[a, i, b, j] = -sum t[k, j, b, c] ((ki|ac) - 1/2 sum t[l, i, a, d] (kd|lc))
    kiac = _pair(Loo, Lvv).permute(0, 3, 1, 2)         # [k, c, i, a]
    kdlc = g.permute(0, 3, 2, 1).contiguous()          # (kd|lc) at [k, c, l, d]
    tli = t2.permute(0, 3, 2, 1).contiguous()          # t_li^ad at [l, d, i, a]
    c2 = kiac - 0.5 * _mm(kdlc, tli, 2, 2)             # [k, c, i, a]
    tkj = t2.permute(2, 1, 0, 3).contiguous()          # t_kj^bc at [j, b, k, c]
    x = -_mm(tkj, c2.contiguous(), 2, 2).permute(2, 3, 0, 1)  # [i, a, j, b]
    y = 0.5 * x + x.permute(2, 1, 0, 3)
    # direct ring
    aikc = 2.0 * _pair(Lvo, Lov) - _pair(_mo(b, xv, yv), _mo(b, xo, yo)).permute(0, 3, 2, 1)  # 2 (ai|kc) - (ac|ki)
    dr = aikc.permute(1, 0, 2, 3) + 0.5 * _mm(u2.contiguous(), Lg.contiguous(), 2, 2)          # [i, a, k, c]
    y = y + 0.5 * _mm(dr.contiguous(), u2.contiguous(), 2, 2)
    # one-electron-like terms
    Fb = Fvv - _fvv(u2, g)
    Fj = Foo + _foo(u2, g)
    y = y + torch.matmul(t2, Fb.T.contiguous())
    y = y - torch.matmul(t2.permute(0, 1, 3, 2), Fj).permute(0, 1, 3, 2)
    O2 += y + y.permute(2, 3, 0, 1)
    O1 = None
    if t1 is not None:
        O1 = Fvo.T.clone()
        O1 += _mm(u2.contiguous(), Fov.contiguous(), 2, 0)
        # sum u[k, c, i, d] (ad|kc) and - sum u[k, a, l, c] (ki|lc)
        w = torch.matmul(u2.permute(2, 3, 0, 1).reshape(o * v, o * v), Lov.reshape(-1, o * v).T)  # [(i, d), P]
        O1 += _mm(w.reshape(o, v, -1), Lvv.permute(2, 0, 1).contiguous(), 2, 1)
        z = w.reshape(o, v, -1)                        # sum_lc u[k, a, l, c] L[P, l, c] at [k, a, P]
        O1 -= _mm(Loo.permute(2, 1, 0).contiguous(), z.permute(0, 2, 1).contiguous(), 2, 1)
    return O1, O2


def _fvv(u2, g):
    """sum u[k, b, l, d] (ld|kc) at [b, c]."""
    o, v = u2.shape[:2]
    A = u2.permute(1, 0, 2, 3).reshape(v, -1)          # [b, (k, l, d)]
    B = g.permute(2, 0, 1, 3).reshape(-1, v)           # g[l, d, k, c] at [(k, l, d), c]
    return A @ B


def _foo(u2, g):
    """sum u[l, c, j, d] (kd|lc) at [k, j]."""
    o = u2.shape[0]
    A = g.permute(0, 2, 3, 1).reshape(o, -1)           # g[k, d, l, c] at [k, (l, c, d)]
    B = u2.permute(0, 1, 3, 2).reshape(-1, o)          # u[l, c, j, d] at [(l, c, d), j]
    return A @ B


def _solve(case, b, C, eps, singles, sweeps=None):
    """(E, t1, t2[i, j, a, b]): the fixed point, or the given number of plain updates from the MP2 guess."""
    o, v = case["o"], case["v"]
    D = _d2(eps, o).permute(0, 2, 1, 3)                # [i, a, j, b]
    d1 = eps[:o, None] - eps[None, o:]
    L = _mo(b, C[:, :o], C[:, o:])
    g = _pair(L, L)
    w = 2.0 * g - g.permute(0, 3, 2, 1)
    t2 = g / D
    t1 = torch.zeros((o, v), dtype=C.dtype, device=C.device) if singles else None
    past = []
    for k in range(sweeps or 80):
        o1, o2 = _omega(b, C, eps, o, t1, t2)
        n2 = t2 + o2 / D
        n1 = t1 + o1 / d1 if singles else None
        e = torch.cat([(n2 - t2).reshape(-1)] + ([(n1 - t1).reshape(-1)] if singles else []))
        t1, t2 = n1, n2
        if sweeps:
            continue
        if float(e.norm()) < 1e-13:
            break
        past = (past + [(torch.cat([n2.reshape(-1)] + ([n1.reshape(-1)] if singles else [])), e)])[-6:]
        m = len(past)
        if m > 1:                                      # least-squares extrapolation over the last updates
            G = torch.stack([torch.stack([torch.dot(p[1], q[1]) for q in past]) for p in past])
            G = G / G.diagonal().max()
            c = torch.linalg.lstsq(G.cpu(), torch.ones(m, 1, dtype=C.dtype)).solution[:, 0]
            c = c / c.sum()
            s = sum(float(ck) * p[0] for ck, p in zip(c, past))
            t2 = s[:t2.numel()].reshape(t2.shape)
            t1 = s[t2.numel():].reshape(t1.shape) if singles else None
    E = (w * t2).sum()
    if singles:
        E = E + torch.dot(t1.reshape(-1), (w.reshape(o * v, o * v) @ t1.reshape(-1)))
    return E, t1, t2.permute(0, 2, 1, 3)


def _triples(case, b, C, eps, t1, t2):
    """E(T) = 1/3 sum (4 W_abc + W_bca + W_cab) (V_abc - V_cba) / D over all i, j, k and a, b, c."""
    o, v = case["o"], case["v"]
    Co, Cv = C[:, :o], C[:, o:]
    Lov, Loo, Lvv = _mo(b, Co, Cv), _mo(b, Co, Co), _mo(b, Cv, Cv)
    iabd = _pair(Lov, Lvv)                             # (ia|bd)
    kcjl = _pair(Lov, Loo)                             # (kc|jl)
    iajb = _pair(Lov, Lov)
    ev = eps[o:]
    dv = ev[:, None, None] + ev[None, :, None] + ev[None, None, :]

    def term(i, j, k):
        # sum_d (ia|bd) t_kj^cd - sum_l (kc|jl) t_il^ab
        x = torch.matmul(iabd[i].reshape(v * v, v), t2[k, j].T).reshape(v, v, v)
        return x - torch.matmul(t2[i].permute(1, 2, 0).reshape(v * v, o), kcjl[k, :, j, :].T).reshape(v, v, v)

    E = torch.zeros((), dtype=C.dtype, device=C.device)
    for i in range(o):
        for j in range(i + 1):
            for k in range(j + 1):
                W = (term(i, j, k) + term(i, k, j).permute(0, 2, 1) + term(j, i, k).permute(1, 0, 2)
                     + term(j, k, i).permute(2, 0, 1) + term(k, i, j).permute(1, 2, 0)
                     + term(k, j, i).permute(2, 1, 0))
                V = (W + t1[i][:, None, None] * iajb[j, :, k, :][None] + t1[j][None, :, None] * iajb[i, :, k, :][:, None, :]
                     + t1[k][None, None, :] * iajb[i, :, j, :][:, :, None])
                D = eps[i] + eps[j] + eps[k] - dv
                weight = 1.0 if i == j == k else (3.0 if i == j or j == k else 6.0)
                # the six orders of (i, j, k) give the same sum over a, b, c when it is symmetrised
                S = torch.zeros((), dtype=C.dtype, device=C.device)
                for p in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
                    w, x = W.permute(*p), V.permute(*p)
                    S = S + ((4.0 * w + w.permute(2, 0, 1) + w.permute(1, 2, 0)) * (x - x.permute(2, 1, 0))
                             / D.permute(*p)).sum()
                E = E + weight * S / 18.0
    return E


def exact(case, seed):
    b, C, eps = _system(case, seed)
    o, kind = case["o"], case["kind"]
    if kind == "rmp2":
        return float(_mp2(b, C, eps, o))
    if kind == "rmp2_grad":
        C, eps = C.requires_grad_(), eps.requires_grad_()
        if case["dg"]:
            n = b.shape[1]
            f = b.reshape(-1, n * n)
            G = (f.T @ f).reshape(n, n, n, n).requires_grad_()
            K = G
            for M in (C[:, :o], C[:, o:], C[:, :o], C[:, o:]):   # each contraction moves its index to the back
                K = torch.tensordot(K, M, dims=([0], [0]))
            K = K.permute(0, 2, 1, 3)
            E = (K * (2.0 * K - K.transpose(2, 3)) / _d2(eps, o)).sum()
            dC, deps, dG = torch.autograd.grad(E, (C, eps, G))
            return [float(E.detach()), dC, deps, dG]
        E = _mp2(b, C, eps, o)
        dC, deps = torch.autograd.grad(E, (C, eps))
        return [float(E.detach()), dC, deps]
    if kind in ("rccd", "df_rccd"):
        E, _, t2 = _solve(case, b, C, eps, False, SWEEPS if kind == "df_rccd" else None)
        return [float(E), t2]
    if kind == "rccsd":
        E, t1, t2 = _solve(case, b, C, eps, True)
        return [float(E), t1, t2]
    t1, t2 = _amplitudes(case, seed, b, C, eps)
    return float(_triples(case, b, C, eps, t1, t2))
