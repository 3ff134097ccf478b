"""The calls that a program using this engine makes, for timing.

Every case goes through the Python binding (`dmrg_amd.Ops`, `dmrg_amd.DMRG`) or the C-ABI
itself, on device buffers, with inputs made from a seed:

  matvec      one two-site H_eff product (real FP64, complex128, FP32, split-BF16), the call
              that a sweep makes most often
  site        one single-site H_eff product
  env         a left and a right environment update, one of each as the two half-sweeps make
  eigensolve  one Lanczos ground-state solve of a bond
  split       the truncation of a two-site tensor and the truncated tensor put together again
  solve       a short chain from nothing: engine, MPO, random state, sweeps, energy
  sweep       one more sweep of a chain that is already being swept

The MPOs are the engine's own models (transverse-field Ising, Heisenberg, J1-J2, two-leg
ladder, Josephson array).  Environments come from random isometries, so that H_eff is Hermitian
and scaled as in a sweep; a two-site tensor to split has a decaying Schmidt spectrum.

Tensors are held column-major as the engine wants them: the torch tensor behind a logical
(a, b, c) array has shape (c, b, a).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dmrg-implementations_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import dmrg_amd  # noqa: E402

# model -> (d, D, complex)
MODELS = {"tfim": (2, 3, False), "heisenberg": (2, 5, False), "j1j2": (2, 11, False),
          "ladder": (4, 8, False), "josephson": (5, 4, True)}
PRECISION = {"f64": dmrg_amd.PREC_FP64, "f32": dmrg_amd.PREC_FP32, "bf16x3": dmrg_amd.PREC_BF16X3}


def listed():
    return [
        # a bond next to the end of a chain, where bonds are still small: a call is launch latency
        {"name": "matvec-edge", "kind": "matvec", "model": "heisenberg", "cL": 16, "cR": 32, "precision": "f64"},
        # the centre bond of the L=128, chi=512 Heisenberg chain in each arithmetic that it runs in
        {"name": "matvec-f64-512", "kind": "matvec", "model": "heisenberg", "cL": 512, "cR": 512, "precision": "f64"},
        {"name": "matvec-f32-512", "kind": "matvec", "model": "heisenberg", "cL": 512, "cR": 512, "precision": "f32"},
        # a bond whose dimensions a cutoff has made ragged, split-BF16 products
        {"name": "matvec-bf16x3-ragged", "kind": "matvec", "model": "heisenberg", "cL": 389, "cR": 451,
         "precision": "bf16x3"},
        # the centre bond of the L=32, chi=256 Josephson array (complex, d=5)
        {"name": "matvec-c128-256", "kind": "matvec", "model": "josephson", "cL": 256, "cR": 256, "precision": "f64"},
        # the single-site engine on a frustrated chain (MPO bond 11), ragged bonds
        {"name": "site-j1j2-ragged", "kind": "site", "model": "j1j2", "cL": 243, "cR": 317},
        # what both half-sweeps do after each bond of the chi=512 chain
        {"name": "env-f64-512", "kind": "env", "model": "heisenberg", "ci": 512, "co": 512},
        # one bond of the L=64, chi=256 chain, from a vector that is not yet converged
        {"name": "eigensolve-f64-256", "kind": "eigensolve", "model": "heisenberg", "cL": 256, "cR": 256},
        # the truncation of a chi=256 bond's tensor, no earlier basis at hand
        {"name": "split-f64-512", "kind": "split", "m": 512, "n": 512, "k": 256, "complex": False, "left": False},
        # a short random-field chain solved from nothing, as in a disorder average
        {"name": "solve-chain-16", "kind": "solve", "L": 16, "chi": 32, "sweeps": 4, "precision": "f64"},
        # the steady state of a long run, FP64 and mixed
        {"name": "sweep-f64-256", "kind": "sweep", "L": 32, "chi": 256, "precision": "f64"},
        {"name": "sweep-f32-512", "kind": "sweep", "L": 24, "chi": 512, "precision": "f32"},
    ]


def _size(rng, lo, hi):
    """A size in [lo, hi], even in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "matvec", "site", "env", "eigensolve", "split", "solve", "sweep"])
    if kind in ("solve", "sweep"):
        L, chi = rng.randint(10, 20), _size(rng, 16, 64)
        c = {"kind": kind, "L": L, "chi": chi, "precision": rng.choice(["f64", "f64", "f32"])}
        if kind == "solve":
            c["sweeps"] = rng.randint(2, 4)
        return c
    if kind == "split":
        cplx = rng.random() < 0.3
        m = _size(rng, 24, 400 if cplx else 700)
        n = max(16, min(2 * m, int(m * rng.uniform(0.6, 1.4))))
        return {"kind": kind, "m": m, "n": n, "k": max(8, int(min(m, n) * rng.uniform(0.4, 0.7))),
                "complex": cplx, "left": rng.random() < 0.5}
    model = rng.choice(["tfim", "heisenberg", "heisenberg", "j1j2", "ladder", "josephson"])
    top = {"tfim": 512, "heisenberg": 512, "j1j2": 400, "ladder": 256, "josephson": 200}[model]
    a = _size(rng, 8, top)
    b = max(8, min(top, int(a * rng.uniform(0.5, 2.0))))
    if kind == "matvec":
        precision = "f64" if MODELS[model][2] else rng.choice(["f64", "f64", "f32", "bf16x3"])
        return {"kind": kind, "model": model, "cL": a, "cR": b, "precision": precision}
    if kind == "env":
        return {"kind": kind, "model": model, "ci": a, "co": b}
    if kind == "eigensolve":
        a, b = min(a, 320), min(b, 320)
    return {"kind": kind, "model": model, "cL": a, "cR": b}


# --------------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------------
class _Buffer:
    """A torch tensor on the GPU as the binding's device array: shape, dtype and address."""

    def __init__(self, t, shape=None):
        self.t = t
        self.shape = tuple(shape) if shape else tuple(reversed(t.shape))
        self.dtype = np.dtype({torch.float64: "f8", torch.float32: "f4", torch.complex128: "c16"}[t.dtype])
        self.ptr = ctypes.c_void_p(t.data_ptr())


def _spin_mpo(reach):
    """Bulk tensor of the spin-1/2 chain with exchange 1, 1/2, ... up to `reach` neighbours."""
    Sp = np.array([[0.0, 1.0], [0.0, 0.0]])
    ops = [(Sp, 0.5 * Sp.T), (Sp.T, 0.5 * Sp), (np.diag([0.5, -0.5]), np.diag([0.5, -0.5]))]
    D = 2 + 3 * reach * (reach + 1) // 2
    W = np.zeros((D, 2, 2, D))
    W[0, :, :, 0] = W[D - 1, :, :, D - 1] = np.eye(2)
    at = 1
    for r in range(1, reach + 1):
        for o, close in ops:
            W[0, :, :, at] = o.T
            for _ in range(r - 1):
                W[at, :, :, at + 1] = np.eye(2)
                at += 1
            W[at, :, :, D - 1] = close.T / r
            at += 1
    return W


def _mpo(model):
    """Bulk MPO tensor W[w, s, sp, wp]; row 0 starts the operator, column D-1 has completed it."""
    if model in ("heisenberg", "j1j2"):
        return _spin_mpo(1 if model == "heisenberg" else 2)
    d, D, cplx = MODELS[model]
    W = np.zeros((D, d, d, D), complex if cplx else float)
    W[0, :, :, 0] = W[D - 1, :, :, D - 1] = np.eye(d)
    if model == "tfim":
        W[0, :, :, 1] = W[1, :, :, 2] = np.diag([1.0, -1.0])
        W[1, :, :, 2] *= -1.0
        W[0, :, :, 2] = np.array([[0.0, -1.0], [-1.0, 0.0]])
    elif model == "ladder":
        Sp, Sz, one = np.array([[0.0, 1.0], [0.0, 0.0]]), np.diag([0.5, -0.5]), np.eye(2)
        at = 1
        for leg in (0, 1):
            for o, close in ((Sp, 0.5 * Sp.T), (Sp.T, 0.5 * Sp), (Sz, Sz)):
                on = (lambda x: np.kron(x, one)) if leg == 0 else (lambda x: np.kron(one, x))
                W[0, :, :, at], W[at, :, :, D - 1] = on(o).T, on(close).T
                at += 1
        W[0, :, :, D - 1] = sum(np.kron(a, b) for a, b in ((Sp, 0.5 * Sp.T), (Sp.T, 0.5 * Sp), (Sz, Sz))).T
    else:
        up = np.diag(np.ones(d - 1), -1)
        a = -np.exp(1j * math.pi / 3)
        W[0, :, :, 1], W[0, :, :, 2] = (a * up).T, (np.conj(a) * up.T).T
        W[1, :, :, 3], W[2, :, :, 3] = up, up.T
        W[0, :, :, 3] = np.diag((np.arange(d) - d // 2.0) ** 2)
    return W


def _normal(gen, shape, cplx):
    x = gen.standard_normal(shape)
    return x + 1j * gen.standard_normal(shape) if cplx else x


def _isometry(gen, rows, cols, cplx):
    return np.linalg.qr(_normal(gen, (rows, cols), cplx))[0]


def _gpu(a):
    """Logical array -> column-major torch tensor on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()


def _environment(gen, W, c, left):
    """Environment (c, D, c) of a block of random isometries, logical axes (ket, mpo, bra)."""
    D, d, cplx = W.shape[0], W.shape[1], np.iscomplexobj(W)
    kind = torch.complex128 if cplx else torch.float64
    w = torch.from_numpy(W if left else np.ascontiguousarray(W.transpose(3, 1, 2, 0))).to("cuda", kind)
    E = torch.zeros((1, D, 1), dtype=kind, device="cuda")
    E[0, 0 if left else D - 1, 0] = 1
    dims = [1]
    while dims[-1] < c:
        dims.append(min(c, dims[-1] * d))
    for a, b in zip(dims, dims[1:] + [c]):
        A = torch.from_numpy(_isometry(gen, a * d, b, cplx).reshape(a, d, b)).cuda()
        x = torch.tensordot(E, A, ([0], [0]))                 # mpo, bra, s, ket'
        x = torch.tensordot(x, w, ([0, 2], [0, 1]))           # bra, ket', sp, mpo'
        E = torch.tensordot(x, A.conj(), ([0, 2], [0, 1]))    # ket', mpo', bra'
    return E.contiguous()


def _columns(t):
    """Logical torch array -> column-major storage."""
    return t.permute(*reversed(range(t.dim()))).contiguous()


def _fields(seed, L):
    return np.random.default_rng(seed).uniform(-0.5, 0.5, L)


def _chain(case, seed):
    """MPO of the random-field Heisenberg chain."""
    Ws = []
    for h in _fields(seed, case["L"]):
        W = _spin_mpo(1)
        W[0, :, :, 4] += h * np.diag([0.5, -0.5])
        Ws.append(W)
    return Ws


def _problem(case, seed):
    """Environments and two-site (or site) tensor of a matvec, site or eigensolve case, in 64 bits."""
    gen = np.random.default_rng(seed)
    W = _mpo(case["model"])
    d, cplx = W.shape[1], np.iscomplexobj(W)
    L, R = (_environment(gen, W, c, left) for c, left in ((case["cL"], True), (case["cR"], False)))
    shape = (case["cL"], d, case["cR"]) if case["kind"] == "site" else (case["cL"], d, d, case["cR"])
    theta = _normal(gen, shape, cplx)
    theta = torch.from_numpy(theta / np.linalg.norm(theta)).cuda()
    if case.get("precision", "f64") != "f64":  # the mixed modes hold environments scaled to unit size
        L, R, theta = ((x / x.abs().max()).float() if x.dim() == 3 else x.float() for x in (L, R, theta))
    return W, L, R, theta


def _engine(case):
    return dmrg_amd.DMRG(case["L"], 2, case["chi"], 5, tol=0.0, krylov_max=20,
                         precision=PRECISION[case["precision"]])


def _spectrum(k, n):
    """Schmidt values that fall to 1e-3 at k and go on falling."""
    return 10.0 ** (-3.0 * (np.arange(n) / k) ** 0.7)


def _two_site(case, seed):
    gen = np.random.default_rng(seed)
    m, n, cplx = case["m"], case["n"], case["complex"]
    r = min(m, n)
    s = _spectrum(case["k"], r) * gen.uniform(0.9, 1.1, r)
    U, V = _isometry(gen, m, r, cplx), _isometry(gen, n, r, cplx)
    return (U * (s / np.linalg.norm(s))) @ V.conj().T


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("solve", "sweep"):
        s = {"case": case, "seed": seed, "Ws": _chain(case, seed)}
        if kind == "sweep":
            s["engine"] = _engine(case)
            s["engine"].set_mpo(s["Ws"])
            s["engine"].initialize_mps_random(seed=seed + 1, scale=0.1)
            s["engine"].run(3)
        return s
    s = {"case": case, "ops": dmrg_amd.Ops(0)}
    if kind == "split":
        M = _gpu(_two_site(case, seed))
        m, n, k = case["m"], case["n"], case["k"]
        ctx = ctypes.c_void_p()
        assert dmrg_amd.lib().dmrg_ctx_create(0, ctypes.byref(ctx)) == dmrg_amd.OK
        new = lambda *shape: torch.zeros(shape, dtype=M.dtype, device="cuda")  # noqa: E731
        s.update(M=M, ctx=_Context(ctx), left=new(k, m), right=new(n, k), both=new(n, m),
                 sigma=torch.zeros(k, dtype=torch.float64, device="cuda"))
    elif kind == "env":
        gen = np.random.default_rng(seed)
        W = _mpo(case["model"])
        d, cplx, ci, co = W.shape[1], np.iscomplexobj(W), case["ci"], case["co"]
        L, R = (_environment(gen, W, ci, left) for left in (True, False))
        A = _isometry(gen, ci * d, co, cplx) if co <= ci * d else _normal(gen, (ci * d, co), cplx) / math.sqrt(co)
        B = _isometry(gen, d * ci, co, cplx).conj().T if co <= ci * d else _normal(gen, (co, d * ci), cplx) / math.sqrt(co)
        A, B = A.reshape(ci, d, co), np.ascontiguousarray(B).reshape(co, d, ci)
        out = lambda: torch.zeros((co, W.shape[0], co), dtype=L.dtype, device="cuda")  # noqa: E731
        s.update({k: _Buffer(v) for k, v in dict(L=_columns(L), R=_columns(R), A=_gpu(A), B=_gpu(B), W=_gpu(W),
                                                  Lnew=out(), Rnew=out()).items()})
    else:
        W, L, R, theta = _problem(case, seed)
        s.update({k: _Buffer(v) for k, v in dict(L=_columns(L), R=_columns(R), theta=_columns(theta), W=_gpu(W)).items()})
        s["out"] = _Buffer(torch.zeros_like(s["theta"].t))
    return s


class _Context:
    """An op context of the C-ABI, destroyed with the state that holds it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        if self.handle:
            dmrg_amd.lib().dmrg_ctx_destroy(self.handle)
            self.handle = None


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "matvec":
        if case["precision"] == "f64":
            s["ops"].heff2(s["L"], s["R"], s["W"], s["W"], s["theta"], s["out"])
        else:
            s["ops"].heff2_f32(s["L"], s["R"], s["W"], s["W"], s["theta"], s["out"],
                               prec=PRECISION[case["precision"]])
        return s["out"].t
    if kind == "site":
        s["ops"].heff1(s["L"], s["R"], s["W"], s["theta"], s["out"])
        return s["out"].t
    if kind == "env":
        s["ops"].env_left(s["L"], s["A"], s["W"], s["Lnew"])
        s["ops"].env_right(s["R"], s["B"], s["W"], s["Rnew"])
        return s["Lnew"].t, s["Rnew"].t
    if kind == "eigensolve":
        s["out"].t.copy_(s["theta"].t)  # the solve overwrites the vector that it starts from
        energy, steps = s["ops"].lanczos2(s["L"], s["R"], s["W"], s["W"], s["out"], krylov_max=20)
        return s["out"].t, energy, steps
    if kind == "split":
        # The factors are fixed only up to a phase of each pair of vectors, so the truncated tensor
        # is put together again, as a program that goes on with it does; the spectrum and the kept
        # rank are the split's own.
        m, n, k = case["m"], case["n"], case["k"]
        dt = dmrg_amd.DTYPE_C128 if case["complex"] else dmrg_amd.DTYPE_F64
        nk = ctypes.c_int(0)
        rc = dmrg_amd.lib().dmrg_op_svd_split(
            s["ctx"].handle, None, dt, m, n, k, 1e-14, 0.0, 1 if case["left"] else 0, s["M"].data_ptr(),
            s["left"].data_ptr(), s["right"].data_ptr(), s["sigma"].data_ptr(), ctypes.byref(nk))
        if rc != dmrg_amd.OK:
            raise RuntimeError(dmrg_amd.lib().dmrg_last_error().decode())
        s["ops"].gemm(0, 0, _Buffer(s["left"], (m, nk.value)), _Buffer(s["right"], (nk.value, n)), _Buffer(s["both"]))
        return s["both"], s["sigma"], nk.value
    if kind == "solve":
        # The state is fixed only up to the gauge of its bonds: the energy, the expectation value
        # and norm of the returned state and its bond dimensions are what a gauge leaves alone.
        with _engine(case) as eng:
            eng.set_mpo(s["Ws"])
            eng.initialize_mps_random(seed=s["seed"] + 1, scale=0.1)
            energy = eng.run(case["sweeps"])
            return [energy, *eng.expectation(), *eng.sweep_energies()], np.array(eng.bond_dims())
    eng = s["engine"]
    energy = eng.run(1)
    return [energy, *eng.expectation()], np.array(eng.bond_dims())


# --------------------------------------------------------------------------------------------
# what a pass cannot do without, and its outputs in 64 bits
# --------------------------------------------------------------------------------------------
def _heff2_work(cL, cR, d, D, cplx, item):
    dd, x = d * d, 4 if cplx else 1
    flops = x * (2.0 * D * dd * cL * cR * (cL + cR) + 2.0 * cL * cR * (D * dd) ** 2)
    return {"bytes": float(item * (D * (cL * cL + cR * cR) + 2 * dd * cL * cR) + 16 * x * D * d * d * D), "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("solve", "sweep"):
        # each bond at least once per half-sweep: 7 products (the first convergence check), one
        # environment update, the density matrix and the product factor of the split
        L, chi, d, D = case["L"], case["chi"], 2, 5
        b = [min(d ** min(i, L - i), chi) for i in range(L + 1)]
        flops = size = 0.0
        for i in range(L - 1):
            w = _heff2_work(b[i], b[i + 2], d, D, False, 8)
            m, n = b[i] * d, b[i + 2] * d
            flops += 7 * w["flops"] + 2.0 * m * n * (min(m, n) + b[i + 1]) + 2.0 * D * d * b[i] * b[i + 1] * (b[i] + b[i + 1])
            size += w["bytes"] + 8.0 * (D * b[i + 1] ** 2 + d * b[i + 1] * (b[i] + b[i + 2]))
        n = 2 * case.get("sweeps", 1)
        return {"bytes": n * size, "flops": n * flops}
    if kind == "split":
        m, n, k, x, item = case["m"], case["n"], case["k"], 4 if case["complex"] else 1, 16 if case["complex"] else 8
        N = n if case["left"] else m
        # density matrix, its reduction to tridiagonal form and back, the product factor, the tensor
        return {"bytes": float(item * 2 * m * n), "flops": x * (m * n * N + (4.0 / 3 + 2) * N ** 3 + 4.0 * m * n * k)}
    d, D, cplx = MODELS[case["model"]]
    x, item = (4, 16) if cplx else (1, 8)
    if kind == "env":
        ci, co = case["ci"], case["co"]
        flops = x * (2.0 * D * d * ci * co * (ci + co) + 2.0 * ci * co * (D * d) ** 2)
        return {"bytes": 2.0 * item * (D * (ci * ci + co * co) + d * ci * co + D * d * d * D), "flops": 2 * flops}
    cL, cR = case["cL"], case["cR"]
    if kind == "site":
        flops = x * (2.0 * D * d * cL * cR * (cL + cR) + 2.0 * cL * cR * (D * d) ** 2)
        return {"bytes": float(item * (D * (cL * cL + cR * cR) + 2 * d * cL * cR + D * d * d * D)), "flops": flops}
    one = _heff2_work(cL, cR, d, D, cplx, item if case.get("precision", "f64") == "f64" else 4)
    if kind == "matvec":
        return one
    n, it = cL * d * d * cR, 20  # 20 products; each new vector against all earlier ones, twice over
    return {"bytes": one["bytes"] + float(item * n * it), "flops": it * one["flops"] + x * 4.0 * n * it * it / 2}


def _times_h(L, R, W, theta):
    """H_eff theta for a site tensor or a two-site tensor, logical axes."""
    x = torch.tensordot(L, theta, ([0], [0]))           # w, a', s..., b
    x = torch.tensordot(x, W, ([0, 2], [0, 1]))         # a', (s2,) b, sp, w'
    if theta.dim() == 4:
        x = torch.tensordot(x, W, ([1, 4], [1, 0]))     # a', b, sp1, sp2, n
        return torch.tensordot(x, R, ([1, 4], [0, 1]))  # a', sp1, sp2, b'
    return torch.tensordot(x, R, ([1, 3], [0, 1]))      # a', sp, b'


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "sweep"):
        return None
    if kind == "split":
        M, k = _two_site(case, seed), case["k"]
        U, S, V = np.linalg.svd(M, full_matrices=False)
        both = (U[:, :k] * S[:k]) @ V[:k]
        return torch.from_numpy(np.ascontiguousarray(both.T)), torch.from_numpy(S[:k].copy()), None
    if kind == "env":
        s = prepare(case, seed)
        L, R, A, B, W = (s[k].t.permute(*reversed(range(s[k].t.dim()))) for k in "LRABW")
        x = torch.tensordot(torch.tensordot(L, A, ([0], [0])), W, ([0, 2], [0, 1]))   # bra, ket', sp, w'
        Ln = torch.tensordot(x, A.conj(), ([0, 2], [0, 1]))
        y = torch.tensordot(torch.tensordot(R, B, ([0], [2])), W, ([0, 3], [3, 1]))   # bra, ket', w, sp
        Rn = torch.tensordot(y, B.conj(), ([0, 3], [2, 1]))
        return _columns(Ln), _columns(Rn)
    W, L, R, theta = _problem(case, seed)
    kind64 = torch.complex128 if MODELS[case["model"]][2] else torch.float64
    W = torch.from_numpy(W).to("cuda", kind64)
    L, R, theta = L.to(kind64), R.to(kind64), theta.to(kind64)
    if kind != "eigensolve":
        return _columns(_times_h(L, R, W, theta))
    it = min(20, theta.numel())
    V = torch.zeros((it, theta.numel()), dtype=kind64, device="cuda")
    V[0] = (theta / theta.norm()).reshape(-1)
    T = torch.zeros((it, it), dtype=torch.float64)
    for j in range(it):
        w = _times_h(L, R, W, V[j].reshape(theta.shape)).reshape(-1)
        T[j, j] = torch.vdot(V[j], w).real.item()
        for _ in range(2):
            w = w - V[: j + 1].T @ (V[: j + 1].conj() @ w)
        if j + 1 < it:
            T[j, j + 1] = T[j + 1, j] = w.norm().item()
            V[j + 1] = w / w.norm()
    lam, Y = torch.linalg.eigh(T)
    y = Y[:, 0] * torch.sign(Y[:, 0][Y[:, 0].abs().argmax()])
    x = (V.T @ y.to("cuda", kind64)).reshape(theta.shape)
    return _columns(x / x.norm()), float(lam[0]), None
