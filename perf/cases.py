"""Performance cases of pyci_amd: what a user's configuration-interaction program has it do.

    fullci_solve   the full CI space, its operator and its lowest states (the headline workload)
    csr_product    a product with the stored (CSR) operator of the full space, for a user's own iteration
    doci_solve     the same program over a seniority-zero (DOCI) space
    rdms           one- and two-particle density matrices of a state
    selection      one step of selected CI: operator, ground state, heat-bath additions
    enpt2          the Epstein-Nesbet correction of a selected state
    train          training of the learned selector on a selected state
    batch          many uneven full CI problems in one call

Integrals, determinant sets and vectors are synthetic and made from the seed alone: the integral
recipe is the benchmark's (diagonal ladder, random Cholesky vectors, decaying ones for the larger
orbital bases); selected sets hold the reference determinant, its singles and doubles and a
sample of higher excitations near the Fermi level, with a dominant reference coefficient.
"""
import math
from itertools import combinations

import numpy as np
import torch

import pyci_amd as pyci


def listed():
    return [
        # smallest calls: a minimal-basis molecule, where launches and latency are everything
        {"name": "fullci_tiny", "kind": "fullci_solve", "nbasis": 4, "nup": 2, "ndn": 2, "nroot": 1, "precision": "f64"},
        # the headline workload: full CI ground state of 853,776 determinants at the default tolerance
        {"name": "fullci_12", "kind": "fullci_solve", "nbasis": 12, "nup": 6, "ndn": 6, "nroot": 1, "precision": "f64"},
        # several states of an odd-electron system in mixed precision (no alpha-beta symmetry to use)
        {"name": "fullci_block", "kind": "fullci_solve", "nbasis": 11, "nup": 5, "ndn": 4, "nroot": 4, "precision": "mixed"},
        # density matrices of the headline state
        {"name": "fullci_rdms", "kind": "rdms", "wfn": "fullci_all", "nbasis": 12, "nup": 6, "ndn": 6, "ndet": 853776, "flips": False},
        # one product with the headline operator as a user's own iteration calls it, from and to host vectors
        {"name": "csr_product", "kind": "csr_product", "nbasis": 12, "nup": 6, "ndn": 6},
        # an ordinary small program: DOCI of five pairs in nineteen orbitals
        {"name": "doci", "kind": "doci_solve", "nbasis": 19, "npair": 5},
        # selected CI over spin orbitals, grown from the singles and doubles of all spin changes
        {"name": "genci_step", "kind": "selection", "wfn": "genci", "nbasis": 24, "nup": 6, "ndn": 6, "ndet": 60000, "flips": True, "eps": 5e-4},
        # selected CI over alpha and beta strings, a small molecule in a double-zeta basis
        {"name": "fullci_step", "kind": "selection", "wfn": "fullci", "nbasis": 24, "nup": 5, "ndn": 5, "ndet": 17317, "flips": False, "eps": 2e-4},
        # density matrices of a selected state
        {"name": "genci_rdms", "kind": "rdms", "wfn": "genci", "nbasis": 20, "nup": 5, "ndn": 5, "ndet": 30011, "flips": False},
        # perturbative correction of a selected state
        {"name": "enpt2", "kind": "enpt2", "wfn": "fullci", "nbasis": 24, "nup": 5, "ndn": 5, "ndet": 12345, "flips": False, "eps": 1e-5},
        # the learned selector, retrained between two selection steps
        {"name": "train", "kind": "train", "wfn": "genci", "nbasis": 24, "nup": 6, "ndn": 6, "ndet": 60000, "flips": True, "steps": 300, "batch": 8192},
        # a scan of uneven problems, two states each
        {"name": "batch", "kind": "batch", "nprob": 16, "nbasis_max": 10, "nocc_max": 5},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fullci_solve", "fullci_solve", "csr_product", "doci_solve", "rdms_all", "rdms", "selection",
                       "selection", "enpt2", "train", "batch"])
    if kind in ("fullci_solve", "csr_product", "rdms_all"):
        nbasis = rng.randint(4, 12)
        nup = rng.randint(2, min(6, nbasis - 1))
        ndn = nup - (rng.random() < 0.3)
        dim = math.comb(nbasis, nup) * math.comb(nbasis, ndn)
        if kind == "csr_product":
            return {"kind": kind, "nbasis": nbasis, "nup": nup, "ndn": ndn}
        if kind == "rdms_all":
            return {"kind": "rdms", "wfn": "fullci_all", "nbasis": nbasis, "nup": nup, "ndn": ndn, "ndet": dim, "flips": False}
        nroot = rng.choice([1, 1, 2, 3, 4]) if 400 <= dim <= 200000 else 1
        return {"kind": kind, "nbasis": nbasis, "nup": nup, "ndn": ndn, "nroot": nroot, "precision": rng.choice(["f64", "f64", "mixed"])}
    if kind == "doci_solve":
        return {"kind": kind, "nbasis": rng.randint(6, 24), "npair": rng.randint(2, 5)}
    if kind == "train":
        return {"kind": kind, "wfn": rng.choice(["genci", "fullci"]), "nbasis": rng.randint(12, 24), "nup": 5, "ndn": 5,
                "ndet": _log_uniform(rng, 2000, 60000), "flips": rng.random() < 0.5, "steps": rng.choice([100, 200, 300]),
                "batch": rng.choice([1024, 2048, 4096, 8192])}
    if kind == "batch":
        return {"kind": kind, "nprob": rng.randint(4, 16), "nbasis_max": rng.randint(7, 10), "nocc_max": rng.randint(3, 5)}
    # a selected set; the smallest bases hold at least the asked number of determinants
    nbasis = rng.randint(12, 24)
    nup = rng.randint(3, 6)
    ndn = nup - (rng.random() < 0.3)
    case = {"kind": kind, "wfn": rng.choice(["genci", "fullci"]), "nbasis": nbasis, "nup": nup, "ndn": ndn,
            "ndet": _log_uniform(rng, 500, 50000), "flips": rng.random() < 0.5}
    if kind == "selection":
        case["eps"] = rng.choice([1e-3, 5e-4, 2e-4])
    if kind == "enpt2":
        case["ndet"] = _log_uniform(rng, 500, 20000)
        case["eps"] = rng.choice([1e-4, 3e-5, 1e-5])
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _integrals(rng, n, large):
    """One- and two-electron integrals (physicists' order); `large`: the decaying recipe of the larger bases."""
    h = np.triu(rng.normal(0.0, 0.05, (n, n)), 1)
    h += h.T
    h[np.diag_indices(n)] = (-3.0 + 0.2 * np.arange(n)) if large else (-2.0 + 0.25 * np.arange(n))
    L = np.triu(rng.normal(0.0, 0.1, (64 if large else 32, n, n)))
    L += np.triu(L, 1).transpose(0, 2, 1)
    if large:
        L *= np.exp(-np.abs(np.arange(n)[:, None] - np.arange(n)) / 6.0)
    L = L.reshape(len(L), n * n)
    return h, np.ascontiguousarray((L.T @ L).reshape(n, n, n, n).transpose(0, 2, 1, 3))


def _spin_orbital(h, g):
    n = len(h)
    H, G = np.zeros((2 * n, 2 * n)), np.zeros((2 * n,) * 4)
    for a in (0, n):
        H[a:a + n, a:a + n] = h
        for b in (0, n):
            G[a:a + n, b:b + n, a:a + n, b:b + n] = g
    return H, G


def _reference_energy(h, g, nup, ndn):
    a, b = np.arange(nup), np.arange(ndn)
    coulomb, exchange = np.einsum("ijij->ij", g), np.einsum("ijji->ij", g)
    same = sum((coulomb - exchange)[np.ix_(o, o)].sum() / 2 for o in (a, b))
    return float(h[a, a].sum() + h[b, b].sum() + same + coulomb[np.ix_(a, b)].sum())


def _pick(rng, count, weights, k):
    """`count` samples of k[i] <= len(weights) distinct positions each, as bit masks."""
    order = np.argsort(-(np.log(weights) + rng.gumbel(size=(count, len(weights)))), axis=1)
    return np.where(np.arange(len(weights)) < k[:, None], np.uint64(1) << order.astype(np.uint64), np.uint64(0)).sum(axis=1, dtype=np.uint64)


def _excite(rng, n, nocc, k):
    """Strings k[i] excitations away from the lowest one: holes and particles near the Fermi level."""
    holes = _pick(rng, len(k), np.exp((np.arange(nocc) - nocc) / 3.0), k)
    particles = _pick(rng, len(k), np.exp(-np.arange(n - nocc) / 6.0), k) << np.uint64(nocc)
    return np.uint64((1 << nocc) - 1) ^ holes ^ particles


def _selected(rng, case):
    """The determinants (alpha, beta) of a selected set, or spin-orbital strings where it holds spin flips."""
    n, nu, nd, want = case["nbasis"], case["nup"], case["ndn"], case["ndet"]
    top = min(nu + nd, 4)
    found, parts, shift = None, [np.zeros((1, 2), np.uint64)], np.uint64(n)
    parts[0][0] = (1 << nu) - 1, (1 << nd) - 1
    while True:
        m = want
        level = rng.choice(np.arange(1, top + 1), size=m, p=np.array([0.1, 0.5, 0.25, 0.15])[:top] / sum([0.1, 0.5, 0.25, 0.15][:top]))
        ka = np.minimum(rng.binomial(level, 0.5), min(nu, n - nu))
        kb = np.minimum(level - ka, min(nd, n - nd))
        new = np.stack([_excite(rng, n, nu, ka), _excite(rng, n, nd, kb)], axis=1)
        if case["flips"] and case["wfn"] == "genci":  # one electron in four changes its spin, to any free orbital
            i = np.flatnonzero(rng.random(m) < 0.25)
            a, b = new[i, 0], new[i, 1]
            low = a & (~a + np.uint64(1))
            free = ~b & np.uint64((1 << n) - 1)
            to = free & (~free + np.uint64(1))
            new[i, 0], new[i, 1] = a ^ low, b ^ to
        parts.append(new)
        both = np.concatenate(parts)
        _, first = np.unique(both[:, 0] | (both[:, 1] << shift), return_index=True)
        both = both[np.sort(first)]
        if len(both) >= want or len(parts) > 20:
            found = both[:want]
            break
        parts = [both]
    return found


def _amplitudes(rng, ndet):
    """A normalised CI vector: a dominant first coefficient and a tail over five decades."""
    c = rng.normal(size=ndet) * 10.0 ** rng.uniform(-5.0, -1.5, size=ndet)
    c[0] = 1.0
    return c / np.linalg.norm(c)


def _wavefunction(case, dets):
    n = case["nbasis"]
    if case["wfn"] == "fullci":
        return pyci.fullci_wfn(n, case["nup"], case["ndn"], dets.reshape(-1, 2, 1))
    strings = dets[:, 0] | (dets[:, 1] << np.uint64(n))
    return pyci.genci_wfn(2 * n, case["nup"] + case["ndn"], 0, strings.reshape(-1, 1))


def _sizes(case, rng):
    """nbasis and electrons of each spin of a batch's problems."""
    lo, hi, top = 6, case["nbasis_max"], case["nocc_max"]
    return [(int(n), int(k)) for n, k in zip(rng.integers(lo, hi + 1, case["nprob"]), rng.integers(3, top + 1, case["nprob"]))]


def prepare(case, seed):
    rng, kind = np.random.default_rng(seed), case["kind"]
    s = {"case": case}
    if kind == "batch":
        s["raw"] = []
        for n, k in _sizes(case, np.random.default_rng(case["nprob"] * 100 + case["nbasis_max"])):
            s["raw"].append((*_integrals(rng, n, False), min(k, n - 1)))
        s["problems"] = [(pyci.hamiltonian(0.0, h, g), k, k) for h, g, k in s["raw"]]
        return s
    n = case["nbasis"]
    h, g = _integrals(rng, n, n > 12)
    s["integrals"] = h, g
    if kind in ("fullci_solve", "doci_solve"):
        s["ham"] = pyci.hamiltonian(0.0, h, g)
    elif kind == "csr_product" or case.get("wfn") == "fullci_all":
        s["ham"] = pyci.hamiltonian(0.0, h, g)
        s["wfn"] = pyci.fullci_wfn(n, case["nup"], case["ndn"])
        s["wfn"].add_all_dets()
        s["c"] = _amplitudes(rng, len(s["wfn"]))
        if kind == "csr_product":
            s["op"] = pyci.sparse_op(s["ham"], s["wfn"], storage="csr")
    else:
        dets = s["dets"] = _selected(rng, case)
        s["c"] = _amplitudes(rng, len(dets))
        if kind in ("selection", "enpt2"):
            s["ham"] = pyci.hamiltonian(0.0, *(_spin_orbital(h, g) if case["wfn"] == "genci" else (h, g)))
        if kind in ("rdms", "enpt2", "train"):
            s["wfn"] = _wavefunction(case, dets)
        if kind == "enpt2":  # the energy that the state's solve returned
            s["energy"] = _reference_energy(h, g, case["nup"], case["ndn"]) - 0.2
        if kind == "selection":
            s["start"] = np.zeros(len(dets))
            s["start"][0] = 1.0
            s["grown"], s["held"] = np.zeros((1 << 21, 2 if case["wfn"] == "fullci" else 1), np.int64), 0
        if kind == "train":
            s["net"] = pyci.mlp_selector(2 * n, seed)
            s["weights"] = s["net"].params
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "fullci_solve":
        wfn = pyci.fullci_wfn(case["nbasis"], case["nup"], case["ndn"])
        wfn.add_all_dets()
        es, cs = pyci.sparse_op(s["ham"], wfn).solve(n=case["nroot"], precision=case["precision"])
        return {"es": es, "cs": cs}
    if kind == "doci_solve":
        wfn = pyci.doci_wfn(case["nbasis"], case["npair"], case["npair"])
        wfn.add_all_dets()
        es, cs = pyci.sparse_op(s["ham"], wfn).solve()
        return {"es": es, "cs": cs}
    if kind == "csr_product":
        return s["op"](s["c"])
    if kind == "rdms":
        d1, d2 = pyci.compute_rdms(s["wfn"], s["c"])
        return {"d1": d1, "d2": d2}
    if kind == "selection":
        wfn = _wavefunction(case, s["dets"])
        es, cs = pyci.sparse_op(s["ham"], wfn).solve(c0=s["start"])
        pyci.add_hci(s["ham"], wfn, cs[0], eps=case["eps"])
        dets = wfn.to_det_array().view(np.int64).reshape(len(wfn), -1)
        s["grown"][:len(dets)] = dets  # into the program's own array, which holds more than one step adds
        s["grown"][len(dets):s["held"]] = 0
        s["held"] = len(dets)
        return {"es": es, "cs": cs, "dets": s["grown"], "count": len(dets)}
    if kind == "enpt2":
        return pyci.compute_enpt2(s["ham"], s["wfn"], s["c"], s["energy"], eps=case["eps"])
    if kind == "train":
        net = s["net"]
        net.params = s["weights"]
        loss = net.train(s["wfn"], s["c"], steps=case["steps"], batch=case["batch"])
        return {"loss": np.float32(loss), "params": net.params}
    es, _ = pyci.batch_solve(s["problems"])
    return es


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _connected(n, nu, nd):
    """Determinants that one Hamiltonian row of the full space couples."""
    su, sd = nu * (n - nu), nd * (n - nd)
    du, dd = (math.comb(o, 2) * math.comb(n - o, 2) for o in (nu, nd))
    return 1 + su + sd + su * sd + du + dd


def work(case):
    """Inputs read and outputs written once. The eigensolvers are counted with 16 products a state, a product with two
    operations for each coupled pair of determinants; those of a selected set are estimated."""
    kind = case["kind"]
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for n, k in _sizes(case, np.random.default_rng(case["nprob"] * 100 + case["nbasis_max"])):
            w = work({"kind": "fullci_solve", "nbasis": n, "nup": min(k, n - 1), "ndn": min(k, n - 1), "nroot": 2})
            total = {q: total[q] + w[q] for q in total}
        return total
    n = case["nbasis"]
    ints = 8.0 * (n ** 4 + n * n)
    if kind == "doci_solve":
        dim, row = math.comb(n, case["npair"]), 1 + case["npair"] * (n - case["npair"])
        return {"bytes": ints + 12.0 * dim * row + 16.0 * dim, "flops": 16.0 * 2 * dim * row}
    nu, nd = case["nup"], case["ndn"]
    if kind == "fullci_solve":
        dim = math.comb(n, nu) * math.comb(n, nd)
        return {"bytes": ints + (16.0 + 8 * case["nroot"]) * dim, "flops": 16.0 * case["nroot"] * 2 * dim * _connected(n, nu, nd)}
    if kind == "csr_product":
        dim, row = math.comb(n, nu) * math.comb(n, nd), _connected(n, nu, nd)
        return {"bytes": 12.0 * dim * row + 16.0 * dim, "flops": 2.0 * dim * row}
    dim = case["ndet"]
    if kind == "train":
        return {"bytes": 24.0 * dim, "flops": 6.0 * case["steps"] * case["batch"] * (64 * 256 + 256 * 256 + 256)}
    row = min(dim, _connected(n, nu, nd) if case["wfn"] == "fullci_all" else 400)
    if kind == "rdms":
        out = 8.0 * (2 * n * n + 3 * n ** 4 if case["wfn"] != "genci" else 4 * n * n + 16 * n ** 4)
        return {"bytes": out + 24.0 * dim, "flops": 2.0 * dim * row}
    if kind == "enpt2":
        return {"bytes": ints + 24.0 * dim, "flops": 10.0 * dim * 1000}
    return {"bytes": ints + 12.0 * dim * row + 40.0 * dim, "flops": 16.0 * 2 * dim * row}


# ---------------------------------------------------------------------------
# 64-bit values, by annihilating every pair of electrons: with A[pq, K] the amplitude of the
# (N-2)-electron string K in a_q a_p |c>, the Hamiltonian is A^T G A with pair integrals G that hold
# the one-electron part, and the two-particle density matrix is A A^T.
# ---------------------------------------------------------------------------
class _PairSpace:
    def __init__(self, strings, nso):
        """strings: determinants as spin-orbital bit strings (alpha orbitals first)."""
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        d = torch.from_numpy(np.ascontiguousarray(strings).view(np.int64)).to(dev)
        self.ndet, self.nso, self.dev = len(d), nso, dev
        self.pairs = list(combinations(range(nso), 2))
        below = [torch.zeros_like(d, dtype=torch.int8)]
        for p in range(nso):
            below.append(below[-1] + ((d >> p) & 1).to(torch.int8))
        det, key, sign, pair = [], [], [], []
        for t, (p, q) in enumerate(self.pairs):
            i = torch.nonzero((d >> p) & (d >> q) & 1).flatten()
            det.append(i)
            key.append(d[i] ^ (1 << p) ^ (1 << q))
            sign.append(1 - 2 * ((below[p][i] + below[q][i]) & 1))
            pair.append(torch.full_like(i, t))
        keys, where = torch.unique(torch.cat(key), return_inverse=True)
        self.det, self.sign = torch.cat(det), torch.cat(sign).double()
        self.nk = len(keys)
        self.at = torch.cat(pair) * self.nk + where

    def annihilated(self, c):
        a = torch.zeros(len(self.pairs) * self.nk, dtype=torch.float64, device=self.dev)
        a[self.at] = self.sign * c[self.det]
        return a.view(len(self.pairs), self.nk)

    def pair_integrals(self, h, g, nelec):
        p = torch.tensor(self.pairs, device=self.dev)
        i, j = p[:, 0], p[:, 1]
        h, g, one = (torch.from_numpy(np.ascontiguousarray(x)).to(self.dev) for x in (h, g, np.eye(len(h))))
        r, c = (lambda x: x[:, None]), (lambda x: x[None, :])
        G = g[r(i), r(j), c(i), c(j)] - g[r(i), r(j), c(j), c(i)]
        return G + (h[r(i), c(i)] * one[r(j), c(j)] + h[r(j), c(j)] * one[r(i), c(i)]
                    - h[r(i), c(j)] * one[r(j), c(i)] - h[r(j), c(i)] * one[r(i), c(j)]) / (nelec - 1)

    def product(self, G, c):
        w = (G @ self.annihilated(c)).view(-1)
        return torch.zeros_like(c).index_add_(0, self.det, self.sign * w[self.at])

    def diagonal(self, G):
        pair = torch.div(self.at, self.nk, rounding_mode="floor")
        return torch.zeros(self.ndet, dtype=torch.float64, device=self.dev).index_add_(0, self.det, torch.diagonal(G)[pair])

    def lowest(self, G, n):
        """The n lowest eigenvalues, by block Davidson."""
        diag = self.diagonal(G)
        k = min(n + 2, self.ndet)
        gen = torch.Generator(device=self.dev).manual_seed(1)
        V = torch.randn(self.ndet, k, dtype=torch.float64, device=self.dev, generator=gen) * 1e-2 / math.sqrt(self.ndet)
        V[torch.argsort(diag)[:k], torch.arange(k, device=self.dev)] += 1.0
        V = torch.linalg.qr(V)[0]
        W = torch.stack([self.product(G, V[:, j]) for j in range(k)], dim=1)
        for _ in range(400):
            e, u = torch.linalg.eigh(V.T @ W)
            X, HX = V @ u[:, :k], W @ u[:, :k]
            R = HX - X * e[:k]
            if float(R[:, :n].norm(dim=0).max()) < 1e-10 * max(1.0, float(e[:n].abs().max())) or V.shape[1] >= self.ndet:
                break
            if V.shape[1] + k > min(12 * k, self.ndet):
                V, W = X, HX
                V, t = torch.linalg.qr(V)
                W = torch.linalg.solve_triangular(t, W, upper=True, left=False)
            shift = e[:k] - diag[:, None]
            T = R / torch.where(shift.abs() < 1e-3, torch.full_like(shift, 1e-3), shift)
            for _ in range(2):
                T = T - V @ (V.T @ T)
                T = torch.linalg.qr(T)[0]
            V = torch.cat([V, T], dim=1)
            W = torch.cat([W] + [self.product(G, T[:, j])[:, None] for j in range(T.shape[1])], dim=1)
        return torch.flip(e[:n], (0,)) if n > 1 else e[:n]

    def density(self, c, nelec):
        """<a+_p a_r> and <a+_p a+_q a_s a_r> over spin orbitals."""
        a = self.annihilated(c)
        m, n = a @ a.T, self.nso
        p = torch.tensor(self.pairs, device=self.dev)
        i, j = p[:, 0], p[:, 1]
        d2 = torch.zeros(n, n, n, n, dtype=torch.float64, device=self.dev)
        for x, y, s in ((i, j, 1.0), (j, i, -1.0)):
            for z, w, t in ((i, j, 1.0), (j, i, -1.0)):
                d2[x[:, None], y[:, None], z[None], w[None]] = s * t * m
        return torch.einsum("pqrq->pr", d2) / (nelec - 1), d2


def _all_strings(n, k):
    """All k-electron strings over n orbitals in colexicographic order."""
    return np.array(sorted(sum(1 << p for p in c) for c in combinations(range(n), k)), dtype=np.uint64)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("enpt2", "train"):
        return None  # a sum over screened couplings; a trajectory that rounding in 16 bits decides
    s = prepare(case, seed)
    if kind == "batch":
        es = []
        for h, g, k in s["raw"]:
            a = _all_strings(len(h), k)
            space = _PairSpace((a[:, None] | (a[None, :] << np.uint64(len(h)))).ravel(), 2 * len(h))
            es.append(space.lowest(space.pair_integrals(*_spin_orbital(h, g), 2 * k), 2))
        return torch.stack(es)
    h, g = _spin_orbital(*s["integrals"])
    n = case["nbasis"]
    if kind == "doci_solve":
        nelec, a = 2 * case["npair"], _all_strings(n, case["npair"])
        strings = a | (a << np.uint64(n))
    else:
        nelec = case["nup"] + case["ndn"]
        if kind in ("fullci_solve", "csr_product") or case["wfn"] == "fullci_all":
            strings = (_all_strings(n, case["nup"])[:, None] | (_all_strings(n, case["ndn"])[None, :] << np.uint64(n))).ravel()
        else:
            strings = s["dets"][:, 0] | (s["dets"][:, 1] << np.uint64(n))
    space = _PairSpace(strings, 2 * n)
    if kind == "rdms":
        d1, d2 = space.density(torch.from_numpy(s["c"]).to(space.dev), nelec)
        if case["wfn"] != "genci":
            a, b = slice(0, n), slice(n, 2 * n)
            d1, d2 = torch.stack([d1[a, a], d1[b, b]]), torch.stack([d2[a, a, a, a], d2[b, b, b, b], d2[a, b, a, b]])
        return {"d1": d1, "d2": d2}
    G = space.pair_integrals(h, g, nelec)
    if kind == "csr_product":
        return space.product(G, torch.from_numpy(s["c"]).to(space.dev))
    found = {"es": space.lowest(G, case.get("nroot", 1)), "cs": None}
    return found if kind != "selection" else {**found, "dets": None, "count": None}
