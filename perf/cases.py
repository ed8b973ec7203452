"""What the quaternion-Hermitian eigensolver is asked to do, as measurable cases.

Kinds of case, each through the package's public entry points:

* ``solve``: one matrix resident on the GPU (``solve_torch``), with
  eigenvectors (jobz ``V``) or eigenvalues only (``N``);
* ``batch``: many matrices of uneven sizes in one call
  (``Context.zquatev_batched_device``);
* ``serve``: a burst of requests through the continuous-batching ``Server``;
* ``host``: the drop-in entry on host memory (``zquatev``);
* ``qgemm``: the quaternion GEMM (``Context.qgemm_device``).

Matrices are the package's two synthetic distributions: ``uniform`` (dense
random, the single-solve workload) and ``fock`` (banded decay around a spread
diagonal, the batched and serving workloads).  All arithmetic is FP64.

Eigenvectors.  A Kramers pair is defined only up to a unit quaternion (an
SU(2) rotation of the pair), so a program that uses the vectors fixes that
phase; ``fix_phase`` makes a fixed real combination of each vector's
components real and positive.  ``run`` returns the whole 2n x 2n matrix after
that step.
"""

import math

import numpy as np
import torch

import zquatev_amd as zq
from zquatev_amd import gen


def listed():
    return [
        # a model Hamiltonian or small molecule: all latency, the serving stream's smallest size
        {"name": "solve_128", "kind": "solve", "n2": 128, "jobz": "V", "matrix": "fock", "pad": 0},
        # a small SCF step, odd half-dimension, matrix inside a larger array
        {"name": "solve_510", "kind": "solve", "n2": 510, "jobz": "V", "matrix": "uniform", "pad": 2},
        # an ordinary SCF step, the largest size of the batched workload
        {"name": "solve_1024", "kind": "solve", "n2": 1024, "jobz": "V", "matrix": "fock", "pad": 0},
        # a mid-size molecule, ragged in every tile size
        {"name": "solve_2730", "kind": "solve", "n2": 2730, "jobz": "V", "matrix": "fock", "pad": 0},
        # the largest request of the serving workload
        {"name": "solve_4096", "kind": "solve", "n2": 4096, "jobz": "V", "matrix": "uniform", "pad": 0},
        # the large single solve
        {"name": "solve_8192", "kind": "solve", "n2": 8192, "jobz": "V", "matrix": "uniform", "pad": 0},
        # orbital energies only: a small and a large spectrum
        {"name": "values_1000", "kind": "solve", "n2": 1000, "jobz": "N", "matrix": "fock", "pad": 0},
        {"name": "values_4096", "kind": "solve", "n2": 4096, "jobz": "N", "matrix": "uniform", "pad": 0},
        # many fragments at once: 512 problems, sizes over [64, 1024]
        {"name": "batch_512", "kind": "batch", "count": 512, "lo": 64, "hi": 1024, "jobz": "V", "sizes_seed": 1002},
        # a burst of mixed requests to a server
        {"name": "serve_32", "kind": "serve", "count": 32, "lo": 128, "hi": 2048, "sizes_seed": 1003},
        # a host program's drop-in call
        {"name": "host_512", "kind": "host", "n2": 512, "matrix": "uniform"},
        # the matrix product of the updates on its own
        {"name": "qgemm_4096", "kind": "qgemm", "m": 4096, "n": 4096, "k": 1024, "ta": "N", "tb": "N", "lower": False},
    ]


def _log_even(rng, lo, hi):
    """An even number, log-uniform over [lo, hi]."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return 2 * min(max(int(round(v / 2.0)), lo // 2), hi // 2)


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "values", "values", "batch", "serve", "host", "qgemm"])
    if kind in ("solve", "values"):
        hi = 6000 if kind == "solve" else 8192
        return {"kind": "solve", "n2": _log_even(rng, 64, hi), "jobz": "V" if kind == "solve" else "N",
                "matrix": rng.choice(["uniform", "fock"]), "pad": rng.choice([0, 0, 1, 6])}
    if kind == "batch":
        lo = _log_even(rng, 16, 256)
        hi = _log_even(rng, 2 * lo, 1024)
        return {"kind": "batch", "count": int(round(math.exp(rng.uniform(math.log(8), math.log(400))))), "lo": lo,
                "hi": hi, "jobz": rng.choice(["V", "V", "N"]), "sizes_seed": rng.randrange(1 << 30)}
    if kind == "serve":
        return {"kind": "serve", "count": rng.randint(8, 40), "lo": 128, "hi": _log_even(rng, 512, 2048),
                "sizes_seed": rng.randrange(1 << 30)}
    if kind == "host":
        return {"kind": "host", "n2": _log_even(rng, 64, 1024), "matrix": "uniform"}
    ta, tb = rng.choice([("N", "N"), ("N", "C"), ("C", "N")])
    lower = rng.random() < 0.3
    m = int(round(math.exp(rng.uniform(math.log(64), math.log(4096)))))
    n = m if lower else int(round(math.exp(rng.uniform(math.log(64), math.log(4096)))))
    k = int(round(math.exp(rng.uniform(math.log(16), math.log(1024)))))
    return {"kind": "qgemm", "m": m, "n": n, "k": k, "ta": ta, "tb": tb, "lower": lower}


# ---------------------------------------------------------------- inputs

def _sizes(case):
    """Orders 2n of a batch or a burst.  A batch has 16 distinct orders spread
    over its range (fragments of a few kinds), a burst is log-uniform over 8."""
    rng = np.random.default_rng(case["sizes_seed"])
    lo, hi = case["lo"] // 2, case["hi"] // 2
    if case["kind"] == "batch":
        kinds = np.unique(np.round(lo + (hi - lo) * (np.arange(16) + rng.random(16)) / 16.0).astype(int))
    else:
        t = (np.arange(8) + rng.random(8)) / 8.0
        kinds = np.unique(np.round(np.exp(np.log(lo) + (np.log(hi) - np.log(lo)) * t)).astype(int))
    return [int(2 * v) for v in rng.choice(kinds, case["count"])]


def _jobs(case):
    """jobz of each request of a burst: 70% ask for eigenvectors."""
    rng = np.random.default_rng(case["sizes_seed"] + 1)
    return ["V" if u < 0.7 else "N" for u in rng.random(case["count"])]


def _fill(out, matrix, seed):
    """The left half of D: out[j] is column j (out: n columns of 2n rows or more)."""
    make = gen.uniform_case_device if matrix == "uniform" else gen.fock_case_device
    make(out.shape[0], seed, out)


def _weights(n, device):
    """Fixed real weights of the phase convention."""
    k = torch.arange(n, dtype=torch.float64, device=device)
    return torch.cos(1.0 + 0.7 * k * k).to(torch.complex128)


def fix_phase(X, c):
    """Right-multiplies every eigenvector (a quaternion column) by the unit
    quaternion that makes sum_r c_r x_r real and positive.  X: (..., 2n, 2n),
    X[..., j, :] column j; in place."""
    n = c.shape[0]
    L = X[..., :n, :]
    qa = torch.matmul(L[..., :n], c)
    qb = torch.matmul(L[..., n:], c)
    r = torch.rsqrt(qa.real ** 2 + qa.imag ** 2 + qb.real ** 2 + qb.imag ** 2)
    new = L * (qa.conj() * r).unsqueeze(-1)
    new.addcmul_(X[..., n:, :], (qb * -r).unsqueeze(-1))
    L.copy_(new)
    X[..., n:, :n] = -new[..., n:].conj()
    X[..., n:, n:] = new[..., :n].conj()
    return X


def prepare(case, seed):
    dev = torch.device("cuda")
    kind = case["kind"]
    st = {"case": case}
    if kind == "solve":
        n2 = case["n2"]
        n = n2 // 2
        st["H"] = torch.zeros((n if case["jobz"] == "V" else n2, n2 + case["pad"]), dtype=torch.complex128, device=dev)
        _fill(st["H"][:n], case["matrix"], seed)
        st["D"] = torch.zeros((n2, n2 + case["pad"]), dtype=torch.complex128, device=dev) if case["jobz"] == "V" else st["H"]
        st["c"] = _weights(n, dev)
        st["ctx"] = zq.Context(0)
    elif kind == "batch":
        sizes = sorted(_sizes(case), reverse=True)
        st["sizes"] = sizes
        st["H"], st["D"], st["eig"], st["c"] = [], [], [], []
        ptr, eptr = [], []
        for n2 in sorted(set(sizes), reverse=True):      # the matrices of one order, stacked
            k, n = sizes.count(n2), n2 // 2
            H = torch.zeros((k, n, n2), dtype=torch.complex128, device=dev)
            for i in range(k):
                _fill(H[i], "fock", seed + 7919 * len(ptr))
                ptr.append(0)
            D = torch.zeros((k, n2, n2), dtype=torch.complex128, device=dev)
            eig = torch.zeros((k, n), dtype=torch.float64, device=dev)
            st["H"].append(H)
            st["D"].append(D)
            st["eig"].append(eig)
            st["c"].append(_weights(n, dev))
            eptr += [eig[i].data_ptr() for i in range(k)]
        st["ptr"] = [D[i].data_ptr() for D in st["D"] for i in range(D.shape[0])]
        st["eptr"] = eptr
        st["ctx"] = zq.Context(0)
    elif kind == "serve":
        st["sizes"], st["jobs"] = _sizes(case), _jobs(case)
        st["H"], st["D"], st["eig"], st["c"] = [], [], [], []
        for i, n2 in enumerate(st["sizes"]):
            H = torch.zeros((n2 // 2, n2), dtype=torch.complex128, device=dev)
            _fill(H, "fock", seed + 7919 * i)
            st["H"].append(H)
            st["D"].append(torch.zeros((n2, n2), dtype=torch.complex128, device=dev))
            st["eig"].append(torch.zeros(n2 // 2, dtype=torch.float64, device=dev))
            st["c"].append(_weights(n2 // 2, dev))
        st["server"] = zq.Server(0, lanes=3)
    elif kind == "host":
        n = case["n2"] // 2
        st["H"] = np.asfortranarray(gen.uniform_case(n, seed)[:, :n])
        st["D"] = np.zeros((2 * n, 2 * n), dtype=np.complex128, order="F")
        st["c"] = _weights(n, "cpu")
    else:
        ra, ca = (case["m"], case["k"]) if case["ta"] == "N" else (case["k"], case["m"])
        rb, cb = (case["k"], case["n"]) if case["tb"] == "N" else (case["n"], case["k"])
        g = torch.Generator(device=dev).manual_seed(seed)
        for name, r, c in (("A", ra, ca), ("B", rb, cb), ("C0", case["m"], case["n"])):
            st[name] = torch.randn((c, r, 4), dtype=torch.float64, device=dev, generator=g)
        st["lda"], st["ldb"] = ra, rb
        st["C"] = st["C0"].clone()
        st["ctx"] = zq.Context(0)
    return st


# ---------------------------------------------------------------- one pass

def _check(rc):
    if rc:
        raise RuntimeError(f"solve failed: {zq.error_string(rc)} ({rc})")


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "solve":
        n2, n = case["n2"], case["n2"] // 2
        D = st["D"]
        if case["jobz"] == "V":
            D[:n].copy_(st["H"])          # this step's matrix: the solve overwrites it
        rc, eig = zq.solve_torch(st["ctx"], D[:, :n2].T, case["jobz"])
        _check(rc)
        return [eig, fix_phase(D[:, :n2], st["c"])] if case["jobz"] == "V" else [eig]
    if kind == "batch":
        vec = case["jobz"] == "V"
        for H, D in zip(st["H"], st["D"]):
            D[:, : D.shape[1] // 2].copy_(H)
        st["ctx"].set_stream(torch.cuda.current_stream().cuda_stream)
        _check(st["ctx"].zquatev_batched_device(st["sizes"], st["ptr"], st["sizes"], st["eptr"], case["jobz"]))
        return [list(st["eig"]), [fix_phase(D, c) for D, c in zip(st["D"], st["c"])] if vec else []]
    if kind == "serve":
        for H, D in zip(st["H"], st["D"]):
            D[: D.shape[0] // 2].copy_(H)
        torch.cuda.current_stream().synchronize()     # the server's lanes are streams of their own
        for D, eig, n2, job in zip(st["D"], st["eig"], st["sizes"], st["jobs"]):
            st["server"].submit(n2, D.data_ptr(), n2, eig.data_ptr(), job)
        st["server"].drain()
        for rec in st["server"].poll():
            _check(rec["info"])
        return [list(st["eig"]), [fix_phase(D, c) for D, c, job in zip(st["D"], st["c"], st["jobs"]) if job == "V"]]
    if kind == "host":
        D = st["D"]
        D[:, : D.shape[1] // 2] = st["H"]
        info, eig = zq.zquatev(D)
        _check(info)
        return [eig, fix_phase(torch.from_numpy(D.T), st["c"])]
    ctx = st["ctx"]
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    st["C"].copy_(st["C0"])
    _check(ctx.qgemm_device(case["ta"], case["tb"], case["m"], case["n"], case["k"], -1.0, st["A"].data_ptr(),
                            st["lda"], st["B"].data_ptr(), st["ldb"], 1.0, st["C"].data_ptr(), case["m"],
                            case["lower"]))
    return [st["C"]]


# ---------------------------------------------------------------- accounting

def _solve_work(n2, jobz):
    """Reads the lower triangles of A and B; writes the eigenvalues, and the
    2n x 2n eigenvectors; flops of the reduction (64/3) n^3 and of the
    back-transform 32 n^3."""
    n = n2 // 2
    b = 16.0 * n * (n + 1) + 8.0 * n
    f = 64.0 / 3.0 * float(n) ** 3
    if jobz == "V":
        b += 64.0 * n * n
        f += 32.0 * float(n) ** 3
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "qgemm":
        m, n, k = case["m"], case["n"], case["k"]
        outs = m * (m + 1) / 2 if case["lower"] else m * n
        return {"bytes": 32.0 * (m * k + k * n + 2 * outs), "flops": 32.0 * outs * k}
    if kind in ("solve", "host"):
        parts = [_solve_work(case["n2"], case.get("jobz", "V"))]
    elif kind == "batch":
        parts = [_solve_work(n2, case["jobz"]) for n2 in _sizes(case)]
    else:
        parts = [_solve_work(n2, j) for n2, j in zip(_sizes(case), _jobs(case))]
    return {"bytes": float(sum(b for b, _ in parts)), "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    """Measured between panel widths 16, 24 and 32 (the same path with its sums
    in another order) and against ``exact``; stated: about four times the most seen.
    Eigenvectors differ between two correct FP64 solvers by about eps ||H||
    over the distance to the next eigenvalue: up to 2.4e-13 over 2n = 64 ..
    8192 and both distributions (twice that again for closer pairs than the
    measured ones).  Eigenvalues alone: up to 2e-15.  Products: 2.5e-15."""
    if case["kind"] == "qgemm" or case.get("jobz") == "N":
        return {"rel": 1e-14}
    return {"rel": 2e-12}


def _eigh(H, n):
    """Eigenvalues (one per pair) and phase-fixed eigenvectors of the full
    Hermitian matrix, laid out as run() gives them (rows are columns)."""
    w, Y = torch.linalg.eigh(H)
    eig = w.view(n, 2).mean(1)
    # the pair's vectors span a quaternion column x up to a unit quaternion:
    # take the combination with sum_r c_r (U_r, V_r) = (positive, 0)
    c = _weights(n, Y.device)
    P = Y.T.reshape(n, 2, 2, n) @ c                      # (pair, vector, upper or lower): the functional
    B = P / torch.linalg.vector_norm(P[:, :, 0:1], dim=1, keepdim=True)
    left = torch.einsum("pv,pvr->pr", B[:, :, 0].conj(), Y.T.reshape(n, 2, 2 * n))
    right = torch.cat([-left[:, n:].conj(), left[:, :n].conj()], 1)
    return eig, torch.cat([left, right], 0)


def _exact_solve(n2, matrix, seed, jobz):
    n = n2 // 2
    cols = torch.zeros((n, n2), dtype=torch.complex128, device="cuda")
    _fill(cols, matrix, seed)
    H = gen.full_hermitian_t(cols.cpu(), n)
    if jobz == "N":
        return torch.linalg.eigvalsh(H).view(n, 2).mean(1), None
    return _eigh(H, n)


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        if case["n2"] > (2048 if case["jobz"] == "V" else 3000):
            return None
        eig, X = _exact_solve(case["n2"], case["matrix"], seed, case["jobz"])
        return [eig, X] if case["jobz"] == "V" else [eig]
    if kind == "batch":
        sizes = sorted(_sizes(case), reverse=True)
        if sum(v ** 3 for v in sizes) > 8e9:
            return None
        every = [_exact_solve(n2, "fock", seed + 7919 * i, case["jobz"]) for i, n2 in enumerate(sizes)]
        eigs, vecs, at = [], [], 0
        for n2 in sorted(set(sizes), reverse=True):
            k = sizes.count(n2)
            eigs.append(torch.stack([e for e, _ in every[at:at + k]]))
            if case["jobz"] == "V":
                vecs.append(torch.stack([X for _, X in every[at:at + k]]))
            at += k
        return [eigs, vecs]
    if kind == "serve":
        sizes, jobs = _sizes(case), _jobs(case)
        if sum(v ** 3 for v in sizes) > 2e10:
            return None
        every = [_exact_solve(n2, "fock", seed + 7919 * i, j) for i, (n2, j) in enumerate(zip(sizes, jobs))]
        return [[e for e, _ in every], [X for _, X in every if X is not None]]
    if kind == "host":
        n = case["n2"] // 2
        D = gen.uniform_case(n, seed)
        eig, X = _eigh(torch.from_numpy(gen.full_hermitian(D, n)), n)
        return [eig, X]
    # quaternion product through the 2 x 2 complex blocks: [[Aa, -conj Ab], [Ab, conj Aa]] [Ba; Bb]
    st = prepare(case, seed)

    def parts(Q, trans):
        z = torch.view_as_complex(Q.view(Q.shape[0], Q.shape[1], 2, 2))
        a, b = z[..., 0].T, z[..., 1].T
        return (a.mH, -b.mT) if trans == "C" else (a, b)

    Aa, Ab = parts(st["A"], case["ta"])
    Ba, Bb = parts(st["B"], case["tb"])
    left = torch.cat([torch.cat([Aa, -Ab.conj()], 1), torch.cat([Ab, Aa.conj()], 1)], 0)
    prod = left.resolve_conj() @ torch.cat([Ba, Bb], 0).resolve_conj()
    m = case["m"]
    P = torch.view_as_real(torch.stack([prod[:m].T, prod[m:].T], 2)).reshape(case["n"], m, 4)
    if case["lower"]:
        P = P * torch.ones((m, m), dtype=torch.float64, device=P.device).triu()[..., None]
    return [st["C0"] - P]
