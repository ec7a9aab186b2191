"""The work that is measured: calls of this library as a quantum-chemistry program makes them.

A program that has a converged closed-shell CCSD wavefunction of `no` occupied and `nu` virtual
orbitals has the orbital energies, T1, T2 and the integral blocks VM, VOE and VVVO in hand and
wants E(T) = E[T] + E_ST with v1, or the gradients of E(T) with respect to all of them.  The
problem sizes span those of this repository's configurations and benchmark (no=4, nu=36 up to
no=24, nu=216) and of the water restart files of the reference (no=4, nu=36, 87 and 167), with
odd sizes between, since a basis set makes no promise about multiples of 16.

Kinds of a case:
  energy    TriplesContext.load of device-resident arrays, then TriplesContext.energy: a solver that
            keeps its context and brings new amplitudes (the bench's step)
  gradient  TriplesContext.load, then TriplesContext.gradient with the results on the device
  driver    the Fortran entry cc_triples_acc_ on host arrays, packed VVVO: the drop-in for GAMESS
  tuples    the reference driver's loop over ddcc_t_ijk_acc_ / ddcc_t_ijj_acc_ / ddcc_t_iij_acc_
  virtual   E[T] summed over virtual triples and the cube of one triple (energy_abc, w_abc)

`form` is the arithmetic of the contraction, `packed` whether VVVO comes in the distributed
lower-packed layout.
"""

import ctypes
import math

import numpy as np
import torch

# ---------------------------------------------------------------------------- the cases


def _case(name, kind, no, nu, form="fp64", packed=False):
    c = {"kind": kind, "no": no, "nu": nu, "form": form, "packed": packed}
    return {"name": name, **c} if name else c


def listed():
    return [
        # water in the smallest basis of the reference's files: launches and waits count
        _case("energy fp64 4x36", "energy", 4, 36),
        # water in the largest basis of the reference's files, VVVO as GAMESS distributes it
        _case("energy fp64 4x167 packed", "energy", 4, 167, packed=True),
        # the middle configuration
        _case("energy fp64 8x120", "energy", 8, 120),
        # an ordinary molecule with nothing a multiple of anything
        _case("energy fp64 15x163", "energy", 15, 163),
        # the headline size
        _case("energy fp64 24x216", "energy", 24, 216),
        # the fastest reduced form, at the headline size
        _case("energy fp32 24x216", "energy", 24, 216, form="fp32"),
        # the split form, at an ordinary odd size
        _case("energy bf16x3 16x181", "energy", 16, 181, form="bf16x3"),
        # all five gradients at the size the adjoint is checked at
        _case("gradient fp64 8x120", "gradient", 8, 120),
        # gradients with W in FP32, the faster way to them, at an ordinary size
        _case("gradient fp32 14x150", "gradient", 14, 150, form="fp32"),
        # a Fortran program that links this library in place of the reference
        _case("driver 8x120 host", "driver", 8, 120, packed=True),
        # a program that keeps the reference's own loop over tuples
        _case("tuples 4x87 host", "tuples", 4, 87),
        # a virtual-triple caller
        _case("virtual 6x64", "virtual", 6, 64),
    ]


# What draw() takes: kind, form, least and most no and nu, share of the draws.
_RANGES = [
    ("energy", "fp64", (2, 30), (16, 400), 6),
    ("energy", "fp32", (4, 30), (36, 400), 2),
    ("energy", "bf16x3", (4, 30), (36, 400), 2),
    ("gradient", "fp64", (4, 14), (36, 150), 2),
    ("gradient", "fp32", (4, 14), (36, 150), 2),
    ("driver", "fp64", (2, 12), (16, 160), 1),
    ("tuples", "fp64", (3, 6), (20, 110), 1),
    ("virtual", "fp64", (3, 8), (20, 80), 1),
]
# FLOPs of the contraction a drawn case may have: a solve of the headline size has 6.7e13, an
# adjoint three times its energy's, the virtual-triple route two orders of magnitude less rate.
_MOST = {"energy": 2.5e13, "gradient": 2.5e12, "driver": 1.0e12, "tuples": 3.0e10, "virtual": 1.2e10}


def _spread(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind, form, nos, nus, _ = rng.choices(_RANGES, weights=[r[4] for r in _RANGES])[0]
    while True:
        no, nu = _spread(rng, *nos), _spread(rng, *nus)
        if _contraction(no, nu) <= _MOST[kind]:
            break
    packed = kind == "driver" or (kind == "energy" and rng.random() < 0.3)
    return _case(None, kind, no, nu, form, packed)


# ---------------------------------------------------------------------------- inputs


def _inputs(no, nu, seed):
    """Synthetic density-fitted inputs on the GPU, each tensor in the reversed (C) order of the
    Fortran array, so its buffer is the Fortran one: (pq|rs) = sum_Q B[Q,p,q] B[Q,r,s] with entries
    N(0, 0.05^2) and naux = 3 (no + nu), T2 MP2-like, T1 N(0, 1e-6)."""
    g = torch.Generator(device="cuda").manual_seed(1_000_003 * (no * 4096 + nu) + seed)
    opt = {"dtype": torch.float64, "device": "cuda", "generator": g}
    eh = torch.sort(torch.rand(no, **opt) * 1.2 - 1.5)[0]
    ep = torch.sort(torch.rand(nu, **opt) * 2.9 + 0.1)[0]
    n = no + nu
    naux = 3 * n
    b = torch.randn(naux, n, n, **opt).mul_(0.05)
    b = torch.triu(b) + torch.triu(b, 1).transpose(1, 2)
    t1 = torch.randn(nu, no, **opt).mul_(1e-3)                          # T1(i,a)
    vv = b[:, no:, no:].reshape(naux, nu * nu)
    vo = b[:, :no, no:].reshape(naux, no * nu)                          # (Q, i c)
    oo = b[:, :no, :no].reshape(naux, no * no)
    vvvo = (vo.t() @ vv).view(no, nu, nu, nu)                           # [i][c][b][a]
    vm = (vo.t() @ oo).view(no, nu, no, no).permute(2, 0, 1, 3).contiguous()    # [j][k][c][l]
    voe = (vo.t() @ vo).view(no, nu, no, nu).permute(0, 2, 1, 3).contiguous()   # [k][j][c][b]
    d = eh[:, None, None, None] + eh[None, :, None, None] - ep[:, None] - ep[None, :]
    t2 = voe.transpose(0, 1) / d                                        # [j][i][b][a]
    return {"eh": eh, "ep": ep, "t1": t1, "t2": t2, "vm": vm, "voe": voe, "vvvo": vvvo}


def _packed(vvvo):
    """Row p(p+1)/2 + q (q <= p) of column c + nu x holds VVVO(p,q,c,x)."""
    nu = vvvo.shape[1]
    p, q = torch.tril_indices(nu, nu, device=vvvo.device)
    return vvvo[:, :, p, q].contiguous()


_D = ctypes.POINTER(ctypes.c_double)


def _ptr(t):
    return ctypes.cast(t.data_ptr(), _D)


def _int(v):
    return ctypes.byref(ctypes.c_int64(v))


def prepare(case, seed):
    from libcc_amd.triples import TriplesContext

    kind, no, nu = case["kind"], case["no"], case["nu"]
    x = _inputs(no, nu, seed)
    if case["packed"]:
        x["vvvo"] = _packed(x["vvvo"])
    s = {"case": case, "no": no, "nu": nu}
    if kind in ("energy", "gradient", "virtual"):
        s["inp"] = {k: v.contiguous().reshape(-1) for k, v in x.items()}
        s["ctx"] = TriplesContext(no, nu)
        return s
    if kind == "tuples":
        # the cubes the driver's fetch leaves, VE_x(d,p,q) = VVVO(d,q,p,x)
        x["ve"] = x.pop("vvvo").transpose(1, 2).contiguous()
        s["v3"] = torch.zeros(nu, nu, nu, dtype=torch.float64)
    s["host"] = {k: v.cpu().contiguous() for k, v in x.items()}
    s["t1"] = torch.empty_like(s["host"]["t1"])
    s["v1"] = torch.zeros(no, nu, dtype=torch.float64)
    return s


# ---------------------------------------------------------------------------- one pass


def _status(L, what):
    if L.ccx_last_status() != 0:
        raise RuntimeError("%s: status %d" % (what, L.ccx_last_status()))


def _run_driver(s):
    from libcc_amd import lib

    L, h = lib(), s["host"]
    s["t1"].copy_(h["t1"])   # the call leaves t1 transposed, as the reference does
    ets, etd = ctypes.c_double(), ctypes.c_double()
    L.common_cc_init_(_int(s["no"]), _int(s["nu"]))
    L.ccx_register_vvvo_(_int(1), _ptr(h["vvvo"]), _int(1))
    L.cc_triples_acc_(_ptr(h["eh"]), _ptr(h["ep"]), _ptr(s["v1"]), _ptr(s["t1"]), _ptr(h["t2"]), None, None,
                      _ptr(h["vm"]), _ptr(h["voe"]), _int(1), ctypes.byref(ets), ctypes.byref(etd))
    _status(L, "cc_triples_acc_")
    return {"ets": np.float64(ets.value), "etd": np.float64(etd.value), "v1": s["v1"]}


def _run_tuples(s):
    from libcc_amd import lib

    L, h, no, nu = lib(), s["host"], s["no"], s["nu"]
    n, u = _int(no), _int(nu)
    t2, vm, voe, eh, ep = (_ptr(h[k]) for k in ("t2", "vm", "voe", "eh", "ep"))
    ve = [_ptr(h["ve"][i]) for i in range(no)]
    v1, v3 = _ptr(s["v1"].zero_()), _ptr(s["v3"])
    L.common_cc_init_(n, u)
    for i in range(no):
        for j in range(i):
            for k in range(j):
                L.ddcc_t_ijk_acc_(n, u, _int(i + 1), _int(j + 1), _int(k + 1), v1, t2, vm, v3, voe, eh, ep, ve[i],
                                  ve[j], ve[k])
                _status(L, "ddcc_t_ijk_acc_")
    for i in range(no):
        for j in range(i):
            for call in (L.ddcc_t_ijj_acc_, L.ddcc_t_iij_acc_):
                call(n, u, _int(i + 1), _int(j + 1), v1, t2, vm, v3, None, voe, None, eh, ep, None, ve[i], ve[j])
                _status(L, "ddcc_t_ijj_acc_ / ddcc_t_iij_acc_")
    return {"etd": np.float64(L.ccx_get_etd_()), "v1": s["v1"], "w": s["v3"]}   # W of the last tuple


def _triple(nu):
    """The virtual triple whose cube is asked for (1-based)."""
    return nu, max(1, nu // 2), max(1, nu // 3)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "driver":
        return _run_driver(s)
    if kind == "tuples":
        return _run_tuples(s)
    s["ctx"].load(s["inp"], packed_vvvo=case["packed"])
    if kind == "energy":
        r = s["ctx"].energy(case["form"])
        return {"ets": np.float64(r["ets"]), "etd": np.float64(r["etd"]), "v1": r["v1"]}
    if kind == "gradient":
        r = s["ctx"].gradient(device=True, form=case["form"])
        return {k: np.float64(v) if isinstance(v, float) else v for k, v in r.items()}
    return {"etd": np.float64(s["ctx"].energy_abc()), "w": s["ctx"].w_abc(*_triple(s["nu"]))}


# ---------------------------------------------------------------------------- what a pass needs


def _contraction(no, nu):
    """FLOPs of W for all tuples: 12 nu^3 (no+nu) per distinct tuple, 6 nu^3 (no+nu) per (i,j,j), (i,i,j)."""
    return 2.0 * (no ** 3 - no) * nu ** 3 * (no + nu)


def work(case):
    no, nu, kind = case["no"], case["nu"], case["kind"]
    vvvo = nu * (nu + 1) // 2 * nu * no if case["packed"] else nu ** 3 * no
    small = no + nu + no * nu + 2 * nu * nu * no * no + nu * no ** 3
    out = no * nu
    flops = _contraction(no, nu)
    if kind == "gradient":      # W again and two back-contractions of its size; five gradients
        flops *= 3
        out = nu ** 3 * no + small
    elif kind == "tuples":      # every call takes its tuple's cubes and gives W back
        deg = no * (no - 1)
        dis = deg * (no - 2) // 6
        vvvo = nu ** 3 * (3 * dis + 2 * deg)
        out += nu ** 3 * (dis + deg)
    elif kind == "virtual":
        out = no ** 3
    return {"bytes": 8.0 * (vvvo + small + out), "flops": flops}


def tolerance(case):
    """From the largest differences seen from exact() over the ranges above.  FP64: 3e-15 in E[T], v1
    and the gradients, 5e-15 in E_ST, which is a sum of terms of both signs and so can lose a few
    digits more.  Reduced forms carry W to about 24 bits an element: 3e-7 in E_ST, 6e-7 in dVOE (the
    T1 W contraction averages least), 2e-7 and less in the rest."""
    return {"rel": 3e-6} if case["form"] != "fp64" else {"rel": 1e-12}


# ---------------------------------------------------------------------------- the same in 64 bits


def _operands(x):
    """AX[x] (a b, K) = VVVO(K,b,a,x) then T2(a,b,l,x); BX(y,z) (K, c) = T2(c,K,y,z) then -VM(l,c,z,y)."""
    v, t, m = x["vvvo"], x["t2"], x["vm"]
    no, nu = v.shape[0], v.shape[1]
    ax = [torch.cat([v[i], t[i].permute(2, 1, 0)], 2).reshape(nu * nu, nu + no) for i in range(no)]
    return ax, lambda y, z: torch.cat([t[z, y], -m[y, z].t()], 0)


_SIGMA = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))


def _back(s):
    """The permutation that takes axes (p_s0, p_s1, p_s2) back to (p_0, p_1, p_2)."""
    return tuple(s.index(m) for m in range(3))


def _w(ax, bx, t, nu):
    w = 0
    for s in _SIGMA:
        p = (ax[t[s[0]]] @ bx(t[s[1]], t[s[2]])).view(nu, nu, nu)
        w = w + p.permute(*_back(s))
    return w


def _tuples(no):
    for i in range(no):
        for j in range(i):
            for k in range(j):
                yield (i, j, k), 1.0
    for i in range(no):
        for j in range(i):
            yield (i, j, j), 0.5
            yield (i, i, j), 0.5


def _tuple_energy(w, voe, eh, ep, t):
    """E[T] of a tuple before its weight and its three v1 rows, from W."""
    d = eh[t[0]] + eh[t[1]] + eh[t[2]] - ep[:, None, None] - ep[:, None] - ep
    acb, bac, cba = w.permute(0, 2, 1), w.permute(1, 0, 2), w.permute(2, 1, 0)
    bca, cab = w.permute(2, 0, 1), w.permute(1, 2, 0)   # [a,b,c] -> W(b,c,a), W(c,a,b)
    e = (w * (8 * w - 4 * (acb + cba + bac) + 2 * (bca + cab)) / d).sum()
    z = 2 * (w - bac) - acb + bca
    rows = []
    for r in range(3):
        q = [m for m in range(3) if m != r]
        row = 0
        for y, zz in ((q[0], q[1]), (q[1], q[0])):
            # Z of the ordering (r, y, zz): the cube read at W(e_r, e_y, e_zz)
            zp = z if (r, y, zz) == (0, 1, 2) else _ordered_z(w, (r, y, zz))
            o = voe[t[zz], t[y]].t()                     # VOE(b,c,t_y,t_zz) as [b,c]
            row = row + (zp * o / d).sum((1, 2))
        rows.append(row)
    return e, rows


def _ordered_z(w, s):
    """2(W_P(abc) - W_P(bac)) - W_P(acb) + W_P(bca), W_P the cube of the tuple in ordering P = s."""
    u = w.permute(*s)     # u(a,b,c) = W of the reordered tuple: index m of u is index s[m] of w
    return 2 * (u - u.permute(1, 0, 2)) - u.permute(0, 2, 1) + u.permute(2, 0, 1)


def _exact_energy(x, no, nu):
    ax, bx = _operands(x)
    etd, v1 = 0.0, torch.zeros_like(x["t1"]).t().contiguous()
    for t, wt in _tuples(no):
        e, rows = _tuple_energy(_w(ax, bx, t, nu), x["voe"], x["eh"], x["ep"], t)
        etd = etd + wt * e
        for r in range(3):
            v1[t[r]] += wt * rows[r]
    return etd, 2 * (x["t1"].t() * v1).sum(), v1


def _exact_gradient(x, no, nu):
    ax, bx = _operands(x)
    gax = [torch.zeros_like(a) for a in ax]
    gbx = torch.zeros(no, no, nu + no, nu, dtype=torch.float64, device=x["t2"].device)
    t1 = x["t1"].clone().requires_grad_()
    gvoe, gt1 = torch.zeros_like(x["voe"]), torch.zeros_like(x["t1"])
    etd = ets = 0.0
    for t, wt in _tuples(no):
        w = _w(ax, bx, t, nu).requires_grad_()
        pairs = sorted({(t[a], t[b]) for a in range(3) for b in range(3) if a != b})
        voe = {(z, y): x["voe"][z, y].clone().requires_grad_() for z, y in pairs}
        e, rows = _tuple_energy(w, voe, x["eh"], x["ep"], t)
        st = sum((t1[:, t[r]] * rows[r]).sum() for r in range(3)) * (2 * wt)
        etd, ets = etd + wt * e.detach(), ets + st.detach()
        got = torch.autograd.grad(wt * e + st, [w, t1] + [voe[p] for p in pairs], allow_unused=True)
        gt1 += got[1]
        for p, q in zip(pairs, got[2:]):
            if q is not None:
                gvoe[p] += q
        for s in _SIGMA:
            a, y, z = (t[m] for m in s)
            gp = got[0].permute(*s).reshape(nu * nu, nu)
            gax[a] += gp @ bx(y, z).t()
            gbx[y, z] += ax[a].t() @ gp
    gax = torch.stack(gax).view(no, nu, nu, nu + no)
    f = lambda v: v.permute(*reversed(range(v.dim())))   # noqa: E731  Fortran index order
    t2 = gax[..., nu:].permute(0, 3, 2, 1) + gbx[:, :, :nu].transpose(0, 1)
    return {"etd": etd, "ets": ets, "e": etd + ets, "t1": f(gt1), "t2": f(t2), "vm": f(-gbx[:, :, nu:].transpose(2, 3)),
            "voe": f(gvoe), "vvvo": f(gax[..., :nu])}


def exact(case, seed):
    no, nu, kind = case["no"], case["nu"], case["kind"]
    if _contraction(no, nu) > 7e13 or no > 30:
        return None
    x = _inputs(no, nu, seed)
    if kind == "gradient":
        return _exact_gradient(x, no, nu)
    etd, ets, v1 = _exact_energy(x, no, nu)
    if kind == "tuples":   # W(a,a,a) of the last tuple, (i,i,j), is left 0
        ax, bx = _operands(x)
        w = _w(ax, bx, (no - 1, no - 1, no - 2), nu)
        a = torch.arange(nu, device=w.device)
        w[a, a, a] = 0.0
        return {"etd": etd, "v1": v1, "w": w.permute(2, 1, 0)}
    if kind == "virtual":
        ax, bx = _operands(x)
        a, b, c = (v - 1 for v in _triple(nu))
        w = torch.zeros(no, no, no, dtype=torch.float64, device=etd.device)
        vir = (a, b, c)
        for s in _SIGMA:
            g = torch.stack([u.view(nu, nu, -1)[vir[s[0]], vir[s[1]]] for u in ax])     # (x, K)
            h = torch.stack([torch.stack([bx(y, z)[:, vir[s[2]]] for z in range(no)]) for y in range(no)])
            w += (h.reshape(no * no, -1) @ g.t()).view(no, no, no).permute(2, 0, 1).permute(*_back(s))
        i = torch.arange(no, device=w.device)
        w[i, i, i] = 0.0
        return {"etd": etd, "w": w}
    if kind == "energy":
        v1 = v1.t()        # v1(nu,no) as numpy indexes it
    return {"ets": ets, "etd": etd, "v1": v1}
