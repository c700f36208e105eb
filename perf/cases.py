"""The work a user of the library has it do, as measurable cases.

Each case is one call (or one short run) through the public Python entry
points on tensors of the sizes this repository's tests and benchmark use:

  matvec   the two-vertex effective-Hamiltonian product on device vectors
           (FP64, or FP32 split complex as the mixed eigensolver runs it)
  eigs     the growth-step eigensolve on a device vector
  adjoint  gradient of the Rayleigh quotient, host vector in and out
  gate     one iTEBD bond update and the evolved pair, downloaded
  idmrg    iDMRG growth from an empty chain
  itebd    an iTEBD quench from a product state

Three models: "spin" (spin-1/2 XXZ chain, U(1), d=2, MPO bond 5), "chain"
(d-level Z2 coupled chain, MPO bond 3) and "u1" (d levels with U(1) charges
-3..3, MPO bond 6, 21 bond sectors).
"""
import math

import numpy as np
import torch

import chainamps_amd as cam
from chainamps_amd.capi import IndexDesc

_CTX = None


def context():
    """One context for the process, as a program holds it."""
    global _CTX
    if _CTX is None:
        _CTX = cam.Context(0)
    return _CTX


# ---- cases ------------------------------------------------------------------

def listed():
    return [
        # the smallest products: a spin chain early in its growth, where the
        # four launches are all there is
        {"name": "matvec_spin_chi16", "kind": "matvec", "model": "spin", "d": 2, "chi": 16, "fp32": False},
        # a production spin-chain bond: many small, uneven U(1) blocks
        {"name": "matvec_spin_chi200", "kind": "matvec", "model": "spin", "d": 2, "chi": 200, "fp32": False},
        # the coupled chain at an odd, ordinary bond dimension
        {"name": "matvec_chain_chi97", "kind": "matvec", "model": "chain", "d": 64, "chi": 97, "fp32": False},
        # the largest bond at which a whole DMRG step fits one GPU
        {"name": "matvec_chain_chi500", "kind": "matvec", "model": "chain", "d": 64, "chi": 500, "fp32": False},
        # the mixed-precision solver's product
        {"name": "matvec_chain_chi256_fp32", "kind": "matvec", "model": "chain", "d": 64, "chi": 256, "fp32": True},
        # many charge sectors of very different sizes
        {"name": "matvec_u1_chi1024", "kind": "matvec", "model": "u1", "d": 32, "chi": 1024, "fp32": False},
        # a growth step's eigensolve (20 Krylov vectors, loose tolerance)
        {"name": "eigs_chain_chi64", "kind": "eigs", "model": "chain", "d": 64, "chi": 64},
        # the backward direction: dE/dpsi and dE/dW
        {"name": "adjoint_chain_chi32", "kind": "adjoint", "model": "chain", "d": 64, "chi": 32},
        # one bond update of a time evolution, spin chain and coupled chain
        {"name": "gate_spin_chi100", "kind": "gate", "model": "spin", "d": 2, "chi": 100},
        {"name": "gate_chain_chi12", "kind": "gate", "model": "chain", "d": 64, "chi": 12},
        # whole runs: growth of a chain, and a quench
        {"name": "idmrg_spin_chi48", "kind": "idmrg", "model": "spin", "d": 2, "chi": 48, "steps": 8},
        {"name": "itebd_spin_chi32", "kind": "itebd", "model": "spin", "d": 2, "chi": 32, "steps": 6},
    ]


def draw(rng):
    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return min(hi, n | 1 if rng.random() < 0.5 else n)

    pick = rng.random()
    if pick < 0.14:
        return {"kind": "matvec", "model": "spin", "d": 2, "chi": size(12, 400), "fp32": rng.random() < 0.25}
    if pick < 0.40:
        return {"kind": "matvec", "model": "chain", "d": rng.choice([8, 16, 24, 33, 64]), "chi": size(16, 400),
                "fp32": rng.random() < 0.4}
    if pick < 0.52:
        return {"kind": "matvec", "model": "u1", "d": rng.choice([8, 20, 32]), "chi": size(64, 900),
                "fp32": rng.random() < 0.25}
    if pick < 0.62:
        return {"kind": "eigs", "model": "chain", "d": rng.choice([16, 32, 64]), "chi": size(20, 96)}
    if pick < 0.72:
        return {"kind": "adjoint", "model": "chain", "d": rng.choice([8, 16, 33, 64]), "chi": size(8, 40)}
    if pick < 0.80:
        return {"kind": "gate", "model": "spin", "d": 2, "chi": size(16, 128)}
    if pick < 0.88:
        return {"kind": "gate", "model": "chain", "d": rng.choice([8, 16, 32]), "chi": size(6, 24)}
    if pick < 0.94:
        return {"kind": "idmrg", "model": "spin", "d": 2, "chi": size(12, 60), "steps": rng.randint(5, 8)}
    return {"kind": "itebd", "model": "spin", "d": 2, "chi": size(8, 40), "steps": rng.randint(3, 6)}


# ---- models: charges and dense host tensors -----------------------------------

def _rules(model):
    return [2] if model == "chain" else [0]


def _profile(chi, qs, sigma):
    """chi states over the charges qs, Gaussian sector sizes."""
    w = np.exp(-np.asarray(qs, float) ** 2 / (2 * sigma * sigma))
    w = w / w.sum() * chi
    n = np.floor(w).astype(int)
    for k in np.argsort(n - w, kind="stable")[:chi - n.sum()]:
        n[k] += 1
    return np.repeat(np.asarray(qs), n)


def _bond(case, odd=False):
    """Charges of a bond after an even (odd) number of vertices."""
    chi = case["chi"]
    if case["model"] == "chain":
        return np.arange(chi) % 2
    if case["model"] == "spin":
        return _profile(chi, range(-11, 12, 2) if odd else range(-10, 11, 2), 2.5)
    return _profile(chi, range(-10, 11), 4.0)


def _phys(case):
    if case["model"] == "spin":
        return np.array([1, -1])
    if case["model"] == "chain":
        return np.arange(case["d"]) % 2
    return np.arange(case["d"]) % 7 - 3


def _mpo(case, rng):
    """(bond charges, dense W[s', b_l, s, b_r])."""
    d = case["d"]
    if case["model"] == "spin":
        # XXZ chain: J/2 (S+ S- + S- S+) + Jz Sz Sz
        sp = np.array([[0, 1], [0, 0]], complex)
        sz = np.diag([0.5, -0.5]).astype(complex)
        J, Jz = rng.uniform(0.8, 1.2), rng.uniform(0.4, 1.6)
        bq = np.array([0, 2, -2, 0, 0])
        T = np.zeros((2, 5, 2, 5), complex)
        T[:, 0, :, 0] = T[:, 4, :, 4] = np.eye(2)
        for k, a, b in ((1, sp, 0.5 * J * sp.T), (2, sp.T, 0.5 * J * sp), (3, sz, Jz * sz)):
            T[:, 4, :, k] = a
            T[:, k, :, 0] = b
        q = _flux([_phys(case), bq, _phys(case), bq], (1, 1, -1, -1))
        if np.any(T[q != 0]):           # the raising channel carries charge -2
            bq = -bq
        return bq, T
    if case["model"] == "chain":
        par = _phys(case)
        E = np.sort(rng.uniform(0.0, 8.0, d))
        sig = rng.standard_normal((d, d))
        sig = np.where(par[:, None] != par[None, :], 0.5 * (sig + sig.T), 0.0)
        T = np.zeros((d, 3, d, 3), complex)
        T[:, 0, :, 0] = T[:, 2, :, 2] = np.eye(d)
        T[:, 2, :, 0] = np.diag(E)
        T[:, 1, :, 0] = 0.1 * sig
        T[:, 2, :, 1] = sig
        return np.array([0, 1, 0]), T
    bq = np.array([0, 1, -1, 2, -2, 0])
    ch = [_phys(case), bq, _phys(case), bq]
    T = rng.standard_normal((d, 6, d, 6)) + 1j * rng.standard_normal((d, 6, d, 6))
    return bq, np.where(_flux(ch, (1, 1, -1, -1)) == 0, T, 0)


def _flux(charges, signs):
    f = np.zeros((1,) * len(charges), np.int16)
    for k, (q, s) in enumerate(zip(charges, signs)):
        shape = [1] * len(charges)
        shape[k] = len(q)
        f = f + (s * np.asarray(q, np.int16)).reshape(shape)
    return f


def _allowed(model, charges, signs):
    f = _flux(charges, signs)
    return f % 2 == 0 if model == "chain" else f == 0


def _randn(rng, shape, mask):
    """Complex normal entries where the charges allow one."""
    T = np.zeros(shape, complex)
    n = int(mask.sum())
    T[mask] = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return T


def _environment(case, rng, aq, bq, left):
    """Block tensor over (a', b, a): Hermitian in (a', a) for the chain, whose
    channels are self-conjugate."""
    signs = (1, -1, -1) if left else (-1, 1, 1)
    mask = _allowed(case["model"], [aq, bq, aq], signs)
    T = _randn(rng, mask.shape, mask)
    if case["model"] == "chain":
        T = 0.5 * (T + np.conj(T.transpose(2, 1, 0)))
    return T


# ---- tensors on the device ---------------------------------------------------------

def _upload(case, T, charges, inward, physical, numrows):
    """Dense host tensor (zeros outside the allowed entries) as a library
    tensor: CSC of the mixed radix, first index fastest."""
    rows = int(np.prod(T.shape[:numrows]))
    m = T.transpose(range(T.ndim)[::-1]).reshape(-1, rows)       # (columns, rows)
    c, r = np.nonzero(m)
    p = np.concatenate([[0], np.cumsum(np.bincount(c, minlength=m.shape[0]))])
    idx = [IndexDesc(i, ph, np.asarray(q).reshape(-1, 1)) for q, i, ph in zip(charges, inward, physical)]
    return cam.Tensor.from_csc(context(), _rules(case["model"]), idx, numrows, rows, m.shape[0], p, r, m[c, r])


def _upload_mpo(case, bq, T):
    ph = _phys(case)
    return _upload(case, T, [ph, bq, ph, bq], [True, True, False, False], [True, False, True, False], 2)


def _upload_heff(case, parts):
    aq, bq, L, W, R = parts
    z = np.zeros(1, int)
    n = len(aq)
    Lt = _upload(case, L.reshape(1, n, 1, len(bq), 1, n), [z, aq, z, bq, z, aq],
                 [False, True, True, False, True, False], [False] * 6, 3)
    Rt = _upload(case, R.reshape(n, 1, len(bq), 1, n, 1), [aq, z, bq, z, aq, z],
                 [False, True, True, False, True, False], [False] * 6, 2)
    return cam.Heff(Lt, _upload_mpo(case, bq, W), Rt)


def _heff_parts(case, seed):
    rng = np.random.default_rng([seed, 1])
    bq, W = _mpo(case, rng)
    aq = _bond(case)
    return aq, bq, _environment(case, rng, aq, bq, True), W, _environment(case, rng, aq, bq, False)


def _heff_size(case):
    """Entries of a wavefunction."""
    ph, aq = _phys(case), _bond(case)
    two, ends = {}, {}
    for x in ph:
        for y in ph:
            two[x + y] = two.get(x + y, 0) + 1
    values, counts = np.unique(aq, return_counts=True)
    for a, m in zip(values, counts):
        for b, n in zip(values, counts):
            ends[int(b - a)] = ends.get(int(b - a), 0) + int(m) * int(n)
    if case["model"] == "chain":
        fold = lambda t: {k: sum(v for q, v in t.items() if q % 2 == k) for k in (0, 1)}  # noqa: E731
        two, ends = fold(two), fold(ends)
    return sum(v * ends.get(k, 0) for k, v in two.items())


def _vector(n, seed, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 5)
    real = torch.float64 if dtype == torch.complex128 else torch.float32
    return torch.view_as_complex(torch.randn(n, 2, dtype=real, device="cuda", generator=g))


def _host_vector(n, seed):
    rng = np.random.default_rng([seed, 2])
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def _cell(case, seed):
    """Two-vertex unit cell with decaying weights on both bonds, and the
    chain's MPO: (W with its bond charges, bonds, A0, A1, lambdas)."""
    rng = np.random.default_rng([seed, 3])
    bq, W = _mpo(case, rng)
    ph, even, odd = _phys(case), _bond(case), _bond(case, odd=True)
    lam = lambda q: np.exp(-rng.permutation(len(q)) * (9.0 / len(q)) - rng.uniform(0, 0.1, len(q)))  # noqa: E731
    l0, l1 = lam(even), lam(odd)
    l0, l1 = l0 / np.linalg.norm(l0), l1 / np.linalg.norm(l1)

    def site(ql, qr):
        mask = _allowed(case["model"], [ph, ql, qr], (1, 1, -1))
        return _randn(rng, mask.shape, mask) / math.sqrt(len(ph) * len(ql))

    return (bq, W), even, odd, site(even, odd), l1[:, None] * site(odd, even), l0, l1


def _upload_cell(case, cell):
    (bq, W), even, odd, A0, A1, l0, l1 = cell
    ph = _phys(case)
    up = lambda T, ql, qr: _upload(case, T, [ph, ql, qr], [True, True, False], [True, False, False], 2)  # noqa: E731
    return _upload_mpo(case, bq, W), up(A0, even, odd), up(A1, odd, even)


GATE_DT = 0.05


def _padded(values, n):
    """The bond weights in an array of fixed length (how many are kept
    depends on the spectrum)."""
    out = np.zeros(max(n, len(values)))
    out[:len(values)] = values
    return out


def _dense(t):
    """A tensor as its dense matrix, columns outer."""
    rows, cols, p, i, x = t.to_csc()
    out = np.zeros((cols, rows), complex)
    out[np.repeat(np.arange(cols), np.diff(p)), i] = x
    return out


# ---- prepare / run ---------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": dict(case)}
    if kind in ("matvec", "eigs", "adjoint"):
        parts = _heff_parts(case, seed)
        s["H"] = _upload_heff(case, parts)
        n = s["H"].n
        if kind == "matvec":
            s["fp32"] = case["fp32"]
            s["x"] = _vector(n, seed, torch.complex64 if case["fp32"] else torch.complex128)
            s["y"] = torch.empty_like(s["x"])
        elif kind == "eigs":
            s["start"] = _vector(n, seed, torch.complex128)
            s["x"] = torch.empty_like(s["start"])
            s["stream"] = torch.cuda.ExternalStream(context().stream())
        else:
            s["psi"] = _host_vector(n, seed)
            s["nnzW"] = int(np.count_nonzero(parts[3]))
    elif kind == "gate":
        cell = _cell(case, seed)
        W, s["A0"], s["A1"] = _upload_cell(case, cell)
        s["l0"] = cell[5]
        s["G"] = cam.bond_evolution_operator(cam.bond_hamiltonian(W, True), GATE_DT)
        s["D"] = case["chi"]
    else:
        rng = np.random.default_rng([seed, 4])
        bq, T = _mpo(case, rng)
        s["W"] = _upload_mpo(case, bq, T)
        s["D"], s["steps"] = case["chi"], case["steps"]
        if kind == "itebd":
            # Neel product state: up on the first vertex, down on the second
            ph, z, up = _phys(case), np.zeros(1, int), np.ones(1, int)
            A = np.zeros((2, 2, 1, 1), complex)
            A[0, 0], A[1, 1] = 1.0, 1.0
            io, po = [True, True, False], [True, False, False]
            s["A0"] = _upload(case, A[0], [ph, z, up], io, po, 2)
            s["A1"] = _upload(case, A[1], [ph, up, z], io, po, 2)
    return s


def run(s):
    kind = s["kind"]
    if kind == "matvec":
        if s["fp32"]:
            s["H"].apply_device32(s["x"].data_ptr(), s["y"].data_ptr())
        else:
            s["H"].apply_device(s["x"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    if kind == "eigs":
        with torch.cuda.stream(s["stream"]):
            s["x"].copy_(s["start"])
        e, _ = s["H"].lowest_device(s["x"].data_ptr(), have_start=True, converge=False)
        return {"energy": e, "vector": s["x"]}
    if kind == "adjoint":
        dpsi, dW = s["H"].vjp(s["psi"], s["nnzW"])
        return {"dpsi": dpsi, "dW": dW}
    if kind == "gate":
        B, U, lam, trunc = cam.tebd_gate(s["G"], s["A0"], s["A1"], s["l0"], s["D"])
        # the evolved pair over the new bond, as a measurement reads it
        pair = cam.contract(U, False, B, False, [(2, 1)])
        return {"lambda": _padded(lam, 2 * s["D"]), "truncation": trunc, "pair": _dense(pair)}
    if kind == "idmrg":
        g = cam.IDMRG(s["W"])
        rec = [g.grow(s["D"], 1e-12) for _ in range(s["steps"])]
        return {"records": np.array([[r["energy"], r["entropy"], r["truncation"]] for r in rec]),
                "chi": np.array([r["chi"] for r in rec]), "values": _padded(g.values(), 2 * s["D"])}
    t = cam.ITEBD(s["W"], s["A0"], s["A1"], np.ones(1), np.ones(1), 0.1, 2)
    rec = t.evolve(s["steps"], s["D"], 1e-12)
    return {"record": np.array([rec["time"], rec["truncation"], rec["entropy"]]), "chi": rec["chi"],
            "lambda0": _padded(t.lam(0), 2 * s["D"]), "lambda1": _padded(t.lam(1), 2 * s["D"])}


# ---- work ------------------------------------------------------------------------------

def _matvec_work(case, element):
    """Four stages over the allowed, structurally non-zero blocks: L, W, W, R;
    operands once each."""
    n = _heff_size(case)
    chi, d = case["chi"], case["d"]
    env = 2 * {"chain": 1.5, "spin": 5 / 4.0, "u1": 6 / 12.0}[case["model"]] * chi * chi
    if case["model"] == "chain":
        flops = 12.0 * chi ** 3 * d * d + 20.0 * chi * chi * d ** 3
    else:
        w = 5 if case["model"] == "spin" else 6
        sectors = np.unique(_bond(case), return_counts=True)[1]
        per = float((sectors.astype(float) ** 2).sum()) / chi        # mean rows of a block
        flops = 8.0 * n * w * per * 2
        phys = np.unique(_phys(case), return_counts=True)[1]
        flops += 8.0 * n * (8 if w == 5 else w * w) * float((phys.astype(float) ** 2).sum()) / d * 2
    return element * (2.0 * n + env), flops


def work(case):
    kind, chi, d = case["kind"], case["chi"], case["d"]
    if kind == "matvec":
        b, f = _matvec_work(case, 8.0 if case["fp32"] else 16.0)
        return {"bytes": b, "flops": f}
    if kind == "eigs":
        # 21 products, and per product the basis so far read for the
        # projections and again for their removal
        b, f = _matvec_work(case, 16.0)
        n = _heff_size(case)
        return {"bytes": 21 * b + 16.0 * n * 20 * 21, "flops": 21 * f + 8.0 * n * 2 * 20 * 21}
    if kind == "adjoint":
        b, f = _matvec_work(case, 16.0)
        return {"bytes": 2 * b, "flops": 3 * f}
    # a bond update: theta = G A0 A1, its decomposition (about 22 n^3 complex
    # multiply-adds per block at half the dimension for Z2, thirds for U(1)),
    # and the new right tensor
    parts = 2.0 if case["model"] == "chain" else 5.0
    m = d * chi / parts
    gate = 8.0 * parts * (m ** 3 * 3 + 2 * m * m * d) + 4 * 22.0 * parts * m ** 3
    byts = 16.0 * (2 * d * chi * chi / parts * 2 + 3 * parts * m * m)
    if kind == "gate":
        return {"bytes": byts, "flops": gate}
    if kind == "itebd":
        return {"bytes": byts * 2 * case["steps"], "flops": gate * 2 * case["steps"]}
    b, f = _matvec_work(case, 16.0)
    return {"bytes": case["steps"] * (21 * b + byts), "flops": case["steps"] * (21 * f + gate)}


# ---- exact -----------------------------------------------------------------------------

def _sorted_parts(case, seed):
    """The effective Hamiltonian's dense parts with every index ordered by
    charge, and the sectors' ranges."""
    aq, bq, L, W, R = _heff_parts(case, seed)
    ph = _phys(case)
    oa, op = np.argsort(aq, kind="stable"), np.argsort(ph, kind="stable")
    cu = lambda T: torch.from_numpy(np.ascontiguousarray(T)).cuda()  # noqa: E731
    L, R = cu(L[oa][:, :, oa]), cu(R[oa][:, :, oa])
    W = cu(W[op][:, :, op])

    def ranges(q):
        v, first, n = np.unique(np.sort(q), return_index=True, return_counts=True)
        return [(int(x), int(i), int(i + k)) for x, i, k in zip(v, first, n)]

    return L, W, R, ranges(aq), ranges(ph), (oa, op)


def _blocks(case, sa, sp):
    """(s0, s3, s1, s2) ranges of the allowed blocks in the library's vector
    order: right bond, second vertex, first vertex, left bond, ascending."""
    for q3, *r3 in sa:
        for q2, *r2 in sp:
            for q1, *r1 in sp:
                for q0, *r0 in sa:
                    f = q0 + q1 + q2 - q3
                    if (f % 2 if case["model"] == "chain" else f) == 0:
                        yield r0, r3, r1, r2


def _unpack(case, x, sa, sp):
    """Block vector -> dense psi[s2, s1, a2, a0], indices ordered by charge."""
    chi, d = case["chi"], case["d"]
    psi = torch.zeros(d, d, chi, chi, dtype=torch.complex128, device="cuda")
    at = 0
    for r0, r3, r1, r2 in _blocks(case, sa, sp):
        shape = (r2[1] - r2[0], r1[1] - r1[0], r3[1] - r3[0], r0[1] - r0[0])
        n = math.prod(shape)
        psi[r2[0]:r2[1], r1[0]:r1[1], r3[0]:r3[1], r0[0]:r0[1]] = x[at:at + n].reshape(shape)
        at += n
    return psi


def _pack(case, psi, sa, sp):
    return torch.cat([psi[r2[0]:r2[1], r1[0]:r1[1], r3[0]:r3[1], r0[0]:r0[1]].reshape(-1)
                      for r0, r3, r1, r2 in _blocks(case, sa, sp)])


def _stages(psi, L, W, R, grad=False):
    """H psi for psi[s2, s1, a2, a0], a few left rows at a time; with grad
    also the gradient of <psi|H|psi> with respect to W[s', b_l, s, b_r]."""
    d, _, chi, _ = psi.shape
    w = W.shape[1]
    out = torch.empty_like(psi)
    dW = torch.zeros(w, d, w, d, dtype=psi.dtype, device=psi.device) if grad else None   # [b_l, s', b_r, s]
    W1 = W.permute(3, 0, 1, 2).reshape(w * d, w * d).contiguous()       # (b_r, s') x (b_l, s)
    Rm = R.permute(2, 1, 0).reshape(chi * w, chi).contiguous()          # (a2, b) x a2'
    flat = psi.reshape(-1, chi)
    step = max(1, min(chi, int(2e8 // (w * d * d * chi))))
    for lo in range(0, chi, step):
        k = min(step, chi - lo)
        Lm = L[lo:lo + k].reshape(k * w, chi).t().contiguous()          # a0 x (a', b)
        t1 = (flat @ Lm).reshape(d, d, chi, k, w)                       # s2 s1 a2 a' b
        t1 = t1.permute(4, 1, 0, 2, 3).reshape(w * d, -1)               # (b, s1) x (s2, a2, a')
        t2 = (W1 @ t1).reshape(w, d, d, chi, k)                         # b1 s1' s2 a2 a'
        t2 = t2.permute(0, 2, 1, 3, 4).reshape(w * d, -1)               # (b1, s2) x (s1', a2, a')
        t3 = (W1 @ t2).reshape(w, d, d, chi, k)                         # bR s2' s1' a2 a'
        o = t3.permute(1, 2, 4, 3, 0).reshape(-1, chi * w) @ Rm         # (s2' s1' a') x a2'
        out[..., lo:lo + k] = o.reshape(d, d, k, chi).transpose(2, 3)
        if grad:
            c = psi[..., lo:lo + k].conj().transpose(2, 3).reshape(-1, chi)          # (s2' s1' a') x a2'
            b3 = (c @ Rm.t().contiguous()).reshape(d, d, k, chi, w)                  # s2' s1' a' a2 bR
            b3 = b3.permute(4, 0, 1, 3, 2).reshape(w * d, -1)                        # (bR, s2') x (s1', a2, a')
            dW += (b3 @ t2.t().contiguous()).reshape(w, d, w, d).permute(2, 1, 0, 3)
            b2 = (W1.t().contiguous() @ b3).reshape(w, d, d, chi, k)                 # b1 s2 s1' a2 a'
            b2 = b2.permute(0, 2, 1, 3, 4).reshape(w * d, -1)                        # (b1, s1') x (s2, a2, a')
            dW += (b2 @ t1.t().contiguous()).reshape(w, d, w, d).permute(2, 1, 0, 3)
    return out, dW


def _exact_matvec(case, seed):
    L, W, R, sa, sp, _ = _sorted_parts(case, seed)
    n = _heff_size(case)
    x = _vector(n, seed, torch.complex64 if case["fp32"] else torch.complex128)
    if case["fp32"]:
        # the FP32 product is defined on the rounded operands
        x = x.to(torch.complex128)
    psi = _unpack(case, x, sa, sp)
    del x
    out, _ = _stages(psi, L, W, R)
    del psi
    return _pack(case, out, sa, sp)


def _exact_adjoint(case, seed):
    L, W, R, sa, sp, (oa, op) = _sorted_parts(case, seed)
    ph, aq = _phys(case), _bond(case)
    # the caller's order: (s1, a0, s2, a2) with the first fastest, allowed entries only
    allowed = _allowed(case["model"], [aq, ph, aq, ph], (-1, 1, 1, 1))      # [a2, s2, a0, s1]
    dense = np.zeros(allowed.shape, complex)
    dense[allowed] = _host_vector(int(allowed.sum()), seed)
    dense = dense[oa][:, op][:, :, oa][..., op].transpose(1, 3, 0, 2)         # s2 s1 a2 a0
    psi = torch.from_numpy(np.ascontiguousarray(dense)).cuda()
    h, dW = _stages(psi, L, W, R, grad=True)
    n2 = float(torch.vdot(psi.reshape(-1), psi.reshape(-1)).real)
    e = float(torch.vdot(psi.reshape(-1), h.reshape(-1)).real) / n2
    g = ((h - e * psi) / n2).permute(2, 0, 3, 1).cpu().numpy()               # a2 s2 a0 s1
    ia, ip = np.argsort(oa), np.argsort(op)
    g = g[ia][:, ip][:, :, ia][..., ip]
    dW = (dW / n2).cpu().numpy()[:, ip][..., ip]                             # b_l s' b_r s
    Wd = _heff_parts(case, seed)[3]
    keep = Wd.transpose(3, 2, 1, 0) != 0                                     # b_r s b_l s'
    return {"dpsi": g[allowed], "dW": dW.transpose(2, 3, 0, 1)[keep]}


def _exact_gate(case, seed):
    (bq, W), even, odd, A0, A1, l0, _ = _cell(case, seed)
    d, chi = case["d"], case["chi"]
    w = W.shape[1]
    # odd bond Hamiltonian: both vertices' on-site terms and the couplings
    # (half of neither is shared: the two-vertex chain's own Hamiltonian)
    H = np.zeros((d, d, d, d), complex)                                      # s1' s2' s1 s2
    for b in range(w):
        H += np.einsum("ij,kl->ikjl", W[:, w - 1, :, b], W[:, b, :, 0])
    M = H.transpose(1, 0, 3, 2).reshape(d * d, d * d)
    e, v = np.linalg.eigh(0.5 * (M + M.conj().T))
    G = torch.from_numpy((v * np.exp(-1j * GATE_DT * e)) @ v.conj().T).cuda()  # (s2' s1') x (s2 s1)
    cu = lambda T: torch.from_numpy(np.ascontiguousarray(T)).cuda()  # noqa: E731
    X = cu(A0.transpose(0, 1, 2).reshape(d * chi, chi)) @ cu(A1.transpose(1, 0, 2).reshape(chi, d * chi))
    X = X.reshape(d, chi, d, chi).permute(2, 0, 1, 3).reshape(d * d, chi * chi)
    C = (G @ X).reshape(d, d, chi, chi).permute(1, 2, 0, 3).reshape(d * chi, d * chi)  # (s1 al) x (s2 ar)
    lam = cu(l0)
    theta = (C.reshape(-1, d, chi) * lam).reshape(d * chi, d * chi)
    ph = _phys(case)
    rq = (ph[:, None] + even[None, :]).reshape(-1)
    cq = (even[None, :] - ph[:, None]).reshape(-1)
    if case["model"] == "chain":
        rq, cq = rq % 2, cq % 2
    vals, found = [], {}
    for q in np.unique(rq):
        r, c = np.nonzero(rq == q)[0], np.nonzero(cq == q)[0]
        if not len(c):
            continue
        u, s, _ = torch.linalg.svd(theta[torch.from_numpy(r).cuda()][:, torch.from_numpy(c).cuda()].cpu(),
                                   full_matrices=False)
        found[q] = (r, c, u.cuda(), s.numpy())
        vals += [(x, q) for x in s.numpy()]
    vals.sort(key=lambda t: -t[0])
    n = min(chi, len(vals))
    while n < len(vals) and (vals[n - 1][0] - vals[n][0]) / vals[n - 1][0] < 1e-3:
        n += 1
    pair = np.zeros((d * chi, d * chi), complex)
    for q, (r, c, u, s) in found.items():
        k = sum(1 for x, p in vals[:n] if p == q)
        if not k:
            continue
        block = C[torch.from_numpy(r).cuda()][:, torch.from_numpy(c).cuda()]
        u = u[:, :k]
        pair[np.ix_(r, c)] = (u @ (u.conj().t().contiguous() @ block)).cpu().numpy()
    pair /= math.sqrt(float((l0 ** 2).sum()))
    # columns (s2 + d ar) x rows (s1 + d al)
    pair = pair.reshape(d, chi, d, chi).transpose(3, 2, 1, 0).reshape(d * chi, d * chi)
    return {"lambda": _padded([x for x, _ in vals[:n]], 2 * chi),
            "truncation": float(sum(x * x for x, _ in vals[n:])), "pair": pair}


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        return _exact_matvec(case, seed)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "gate":
        return _exact_gate(case, seed)
    return None
