"""What is timed: the calls that a user of this framework makes, with inputs of the sizes they meet.

Systems are the synthetic molecules of dice_amd.synth (orbital counts 8 to 40, one- and two-word determinants) and its
periodic Hubbard lattices.  A seed moves every integral of the named molecule a little, as a step of a geometry scan does.
Determinant spaces come from heat-bath selection, as in a run: from the reference determinant, then from what it
selected, with eps1 lowered until the wanted number of determinants is there.
"""
import ctypes

import numpy as np
import torch

from dice_amd import shci, synth

# orbitals: (alpha electrons, beta electrons, Cholesky vectors, random stream); half filled, as the benchmark's systems
MOLECULES = {8: (4, 4, 32, 8), 16: (8, 8, 64, 0), 24: (12, 12, 96, 1), 32: (16, 16, 128, 2), 40: (20, 20, 160, 3)}


def listed():
    return [
        # a whole variational step of a small molecule (an H8 chain's size): launches and host control, no throughput
        {"name": "step_8orb", "kind": "step", "norb": 8, "eps1": 2e-3, "iters": 4, "roots": 1, "fp32": False,
         "n": 2500, "pairs": 400000, "products": 86},
        # the benchmark's molecule, its first two iterations and the final Davidson: screening, merge, build, Davidson
        {"name": "step_24orb", "kind": "step", "norb": 24, "eps1": 7e-3, "iters": 3, "roots": 1, "fp32": False,
         "n": 400000, "pairs": 140000000, "products": 240},
        # one product with host vectors on a small space (an interactive user, an outer solver in Python)
        {"name": "sigma_small", "kind": "sigma", "norb": 16, "n": 2471, "k": 1, "fp32": False, "host": True,
         "pairs": 257270},
        # the benchmark's final space, the product that its Davidson repeats
        {"name": "sigma_24orb", "kind": "sigma", "norb": 24, "n": 1000003, "k": 1, "fp32": False, "host": False,
         "pairs": 466000000},
        # FP32 values and the two vectors of a two-root calculation, two-word determinants
        {"name": "sigma_fp32_k2", "kind": "sigma", "norb": 40, "n": 300007, "k": 2, "fp32": True, "host": False,
         "pairs": 340000000},
        # a Hamiltonian from scratch over given determinants and its first product
        {"name": "hamiltonian_24orb", "kind": "hamiltonian", "norb": 24, "n": 400009, "fp32": False, "pairs": 138500000},
        # selection: the new determinants of one iteration
        {"name": "screen_24orb", "kind": "screen", "norb": 24, "n": 200003, "new": 500000},
        # diagonalisation, two roots, the reference's Davidson
        {"name": "davidson_40orb", "kind": "davidson", "norb": 40, "n": 57963, "roots": 2, "fp32": False, "block": False,
         "pairs": 23350000, "products": 184},
        # the batching form: four roots of the 6x6 Hubbard lattice, block Davidson with graphs
        {"name": "step_hubbard", "kind": "step", "norb": 36, "eps1": 2e-4, "iters": 3, "roots": 4, "fp32": False,
         "block": True, "n": 400000, "pairs": 140000000, "products": 100},
        # perturbation step after a variational run
        {"name": "pt_24orb", "kind": "pt", "norb": 24, "n": 27685, "eps2": 3e-4, "external": 33000000},
        # the reference's default perturbation step: a deterministic part and sampled iterations, two-word determinants
        {"name": "pt_stochastic_40orb", "kind": "pt_stochastic", "norb": 40, "n": 57963, "eps2": 3e-4, "large": 2e-2,
         "sample": 200, "iters": 10},
        # density matrices of the final state
        {"name": "rdm_24orb", "kind": "rdm", "norb": 24, "n": 200003, "pairs": 57440000},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step", "sigma", "sigma", "hamiltonian", "screen", "davidson", "davidson", "pt",
                       "pt_stochastic", "rdm"])
    norb = rng.choice([16, 24, 24, 32, 40])
    if kind == "step":
        norb = rng.choice([8, 16, 24])
        eps1 = {8: (1e-3, 1e-2), 16: (4e-3, 2e-2), 24: (7e-3, 3e-2)}[norb]
        roots = rng.choice([1, 1, 2])
        return {"kind": kind, "norb": norb, "eps1": round(eps1[0] * (eps1[1] / eps1[0]) ** rng.random(), 6),
                "iters": 1 if norb == 24 and roots == 2 else rng.choice([1, 2]), "roots": roots,
                "fp32": rng.random() < 0.3}
    if kind == "sigma":
        host = rng.random() < 0.25
        return {"kind": kind, "norb": norb, "n": _spread(rng, 500, 20000 if norb == 16 or host else 700000),
                "k": rng.choice([1, 1, 2, 3, 4]), "fp32": rng.random() < 0.4, "host": host}
    if kind == "hamiltonian":
        return {"kind": kind, "norb": norb, "n": _spread(rng, 500, 20000 if norb == 16 else 300000),
                "fp32": rng.random() < 0.4}
    if kind == "screen":
        n = _spread(rng, 100, 10000 if norb == 16 else 200000)
        return {"kind": kind, "norb": norb, "n": n, "new": int(n * rng.uniform(0.5, 2.5)) + 50}
    if kind == "davidson":
        block = rng.random() < 0.4
        norb = rng.choice([16, 24, 36, 40])
        return {"kind": kind, "norb": norb, "n": _spread(rng, 500, 20000 if norb == 16 else 80000),
                "roots": rng.choice([1, 2, 3, 4]) if block else rng.choice([1, 1, 2]), "fp32": rng.random() < 0.3,
                "block": block}
    if kind == "pt":
        return {"kind": kind, "norb": norb, "n": _spread(rng, 300, 20000),
                "eps2": round(4e-4 * 10 ** rng.random(), 7)}
    if kind == "pt_stochastic":
        return {"kind": kind, "norb": norb, "n": _spread(rng, 300, 20000), "eps2": round(3e-4 * 10 ** rng.random(), 7),
                "large": round(1e-2 * 4 ** rng.random(), 6), "sample": rng.choice([100, 200]),
                "iters": rng.randint(6, 10)}
    return {"kind": kind, "norb": norb, "n": _spread(rng, 500, 20000 if norb == 16 else 200000)}


# ---- inputs -----------------------------------------------------------------------------

def _integrals(norb, seed):
    """(h, eri over orbital pairs, alpha, beta electrons) of the named system, moved a little by the seed."""
    rng = np.random.default_rng(int(seed))
    iu = np.tril_indices(norb)
    if norb == 36:  # 6x6 Hubbard lattice, t = 1, U = 4, with site energies that tell its degenerate roots apart
        h, u = synth.hubbard_integrals(6, 6, 1.0, 4.0 * (1 + 0.02 * rng.uniform(-1, 1)))
        pair = np.zeros(norb * (norb + 1) // 2)
        eri = np.zeros((len(pair), len(pair)))
        d = np.arange(norb)
        eri[d * (d + 3) // 2, d * (d + 3) // 2] = u
        return h + np.diag(rng.normal(0.0, 1.0, norb)), eri, 18, 18
    na, nb, nchol, stream = MOLECULES[norb]
    h, L = synth.molecular_integrals(stream, norb, nchol)
    w = rng.normal(0.0, 0.01, h.shape)
    h = h + (w + w.T) * np.abs(h)
    v = L[:, iu[0], iu[1]] * (1 + rng.normal(0.0, 0.01, (nchol, len(iu[0]))))
    return h, v.T @ v, na, nb


def _system(norb, seed):
    h, eri, na, nb = _integrals(norb, seed)
    s = shci.System.from_integrals(h, eri[np.tril_indices(len(eri))], na + nb)
    occ = synth.neel_occupation(6, 6) if norb == 36 else synth.hf_occupation(na, nb)
    ref = np.zeros((1, s.words), dtype=np.uint64)
    for o in occ:
        ref[0, o // 64] |= np.uint64(1) << np.uint64(o % 64)
    return s, ref.view(np.int64)


def _select(s, cmax, want):
    """New determinants of a heat-bath selection with eps1 lowered until about `want` are selected."""
    n = ctypes.c_int64()

    def count(eps):
        s._check(s._lib.shci_screen(s._h, _doubles(cmax), float(eps), ctypes.byref(n)))
        return n.value

    hi, lo = 0.5, 0.25
    got = count(lo)
    while got < want and lo > 1e-7:
        hi, lo = lo, lo * 0.6
        got = count(lo)
    for _ in range(16):
        if got <= want * 1.01:
            break
        mid = (hi * lo) ** 0.5
        at = count(mid)
        if at < want:
            hi = mid
        else:
            lo, got = mid, at
    return s.get_determinants_variational(cmax, lo), lo


def _space(s, ref, want, seed):
    """`want` determinants and coefficients: the reference, what it selects, what that selects, ..."""
    rng = np.random.default_rng(int(seed) + 1)
    dets, c = ref, np.ones(1)
    e0 = s.energy(ref)[0]
    while len(dets) < want:
        s.set_dets(dets)
        # the first block whole, the others as far as wanted
        new = s.get_determinants_variational(np.abs(c), 5e-3) if len(dets) == 1 else \
            _select(s, np.abs(c), want - len(dets))[0]
        if len(new) == 0:
            break
        if len(dets) + len(new) > want:
            keep = np.sort(rng.permutation(len(new))[:want - len(dets)])
            new = new[keep]
        gap = s.energy(new) - e0
        cn = rng.normal(0.0, 0.1, len(new)) / (np.abs(gap) + 0.5)
        dets, c = np.concatenate([dets, new]), np.concatenate([c, cn])
    s.set_dets(dets)
    return dets, c / np.linalg.norm(c), e0


def prepare(case, seed):
    s, ref = _system(case["norb"], seed)
    st = {"case": case, "s": s, "ref": ref}
    kind = case["kind"]
    rng = np.random.default_rng(int(seed) + 2)
    if case.get("fp32") or case.get("block"):
        s.set_options(precision=shci.PREC_FP32 if case.get("fp32") else shci.PREC_FP64,
                      davidson_block=bool(case.get("block")), hip_graphs=bool(case.get("block")))
    if kind == "step":  # the caller's buffers, large enough for any schedule here
        room = 4900 if case["norb"] == 8 else 2000000
        st["dets"], st["ci"] = np.zeros((room, s.words), dtype=np.int64), np.zeros(room * case["roots"])
        return st
    st["dets"], st["c"], e0 = _space(s, ref, case["n"], seed)
    n = len(st["dets"])
    if kind == "screen":
        st["cmax"] = np.abs(st["c"])
        st["eps1"] = _select(s, st["cmax"], case["new"])[1]
        st["new"] = np.zeros((case["new"] * 3 // 2, s.words), dtype=np.int64)
    elif kind in ("pt", "pt_stochastic"):
        # the variational energy, to the digits that every solver agrees on
        s.make_hamiltonian()
        st["e0"] = np.floor(100 * s.davidson(st["c"])[0][0]) / 100
    elif kind == "rdm":
        s.make_hamiltonian()
    elif kind == "davidson":
        s.make_hamiltonian()
        x0 = np.zeros((n, case["roots"]), order="F")
        x0[:, 0] = st["c"]
        low = np.argsort(s.energy(st["dets"][1:]), kind="stable") + 1
        for r in range(1, case["roots"]):  # the lowest determinants beside the reference, with some of each other
            x0[low[r - 1], r] = 1.0
            x0[:, r] += 0.1 * rng.normal(size=n) / np.sqrt(n)
        st["x0"] = x0
    else:
        k = case.get("k", 1)
        x = rng.normal(size=(k, n)) / (1 + np.arange(n)) ** 0.3
        x /= np.linalg.norm(x, axis=1)[:, None]
        st["k"], st["n"] = k, n
        if case.get("host"):
            st["x"] = x[0] if k == 1 else np.asfortranarray(x.T)
        else:  # k vectors of n values, one after the other
            st["x"] = torch.from_numpy(x).cuda()
            st["y"] = torch.empty_like(st["x"])
        if kind == "sigma":
            s.make_hamiltonian()
    return st


# ---- one pass ---------------------------------------------------------------------------

def _doubles(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _ints(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))


def _product(st):
    s = st["s"]
    s._check(s._lib.shci_sigma_device(s._h, st["x"].data_ptr(), st["y"].data_ptr(), st["k"], st["n"]))
    return st["y"]


def run(st):
    case, s = st["case"], st["s"]
    kind = case["kind"]
    if kind == "step":
        e = s.variational(st["ref"], [case["eps1"]] * case["iters"], nroots=case["roots"])
        s._check(s._lib.shci_get_dets(s._h, _ints(st["dets"]), len(st["dets"])))
        s._check(s._lib.shci_run_ci(s._h, _doubles(st["ci"]), len(st["ci"])))
        return {"energies": e, "number": s.num_dets(), "dets": st["dets"], "ci": st["ci"]}
    if kind == "sigma":
        return s.hmult(st["x"]) if case["host"] else _product(st)
    if kind == "hamiltonian":
        s.set_dets(st["dets"])
        elements = s.make_hamiltonian()
        return {"elements": elements, "y": _product(st)}
    if kind == "screen":
        new = ctypes.c_int64()
        s._check(s._lib.shci_screen(s._h, _doubles(st["cmax"]), st["eps1"], ctypes.byref(new)))
        s._check(s._lib.shci_get_new_dets(s._h, _ints(st["new"]), len(st["new"])))
        return {"number": new.value, "dets": st["new"]}
    if kind == "davidson":
        e, x, _ = s.davidson(st["x0"].copy(order="F"), tol=5e-5)
        return {"energies": e, "vectors": x}
    if kind == "pt":
        e, psi, external = s.pt_deterministic(st["c"], st["e0"], case["eps2"])
        return {"energy": e, "norm": psi, "external": external}
    if kind == "pt_stochastic":
        e, per, _, error = s.pt_semistochastic(st["c"], st["e0"], case["eps2"], case["large"], case["sample"],
                                               case["iters"], 1e-12, 1)
        return {"energy": e, "estimates": per, "error": error}
    g1, g2 = s.rdm(st["c"])
    return {"one": g1, "two": g2}


# ---- what a pass cannot do without --------------------------------------------------------

def _pairs(case):
    """Stored connections (J < I) of the case's space: counted once for the listed ones, else an estimate."""
    n = case.get("n", 30000)
    return case.get("pairs") or n * 4.0 * n ** 0.35 * case["norb"] / 24


def work(case):
    kind, n, words = case["kind"], case.get("n", 30000), 1 if case["norb"] < 32 else 2
    pairs, k = _pairs(case), case.get("k", 1)
    entry = 8 if case.get("fp32") else 12  # a value and a column
    product = {"bytes": pairs * entry + n * (8 + 8) + k * n * 16, "flops": k * (4.0 * pairs + 2.0 * n)}
    build = {"bytes": pairs * entry + n * (8 * words + 16), "flops": 0.0}
    if kind == "sigma":
        return product
    if kind == "hamiltonian":
        return {m: product[m] + build[m] for m in product}
    if kind in ("davidson", "step"):  # every product, and for a step the builds; the determinants in and out
        products = case.get("products") or 40 * case["roots"]
        built = build["bytes"] if kind == "step" else 16.0 * n * case["roots"]
        return {"bytes": products * product["bytes"] + built, "flops": products * product["flops"]}
    if kind == "screen":
        return {"bytes": n * (8.0 * words + 8) + case["new"] * 8.0 * words, "flops": 0.0}
    if kind in ("pt", "pt_stochastic"):  # every external determinant and its numerator written and read once
        external = case.get("external") or 1e7
        return {"bytes": external * 2 * (8.0 * words + 8) + n * (8.0 * words + 8),
                "flops": external * (4.0 * case["norb"]) ** 2 / 8}
    return {"bytes": pairs * 4 + n * (8.0 * words + 16) + 8.0 * case["norb"] ** 4, "flops": 4.0 * pairs}


# ---- the same in plain numpy ----------------------------------------------------------------

EXACT_MOST = 20000  # determinants: the pairs of larger spaces take too long here


def _occupations(dets, nso):
    words = np.ascontiguousarray(dets).view(np.uint64)
    return ((words[:, np.arange(nso) // 64] >> (np.arange(nso) % 64).astype(np.uint64)) & np.uint64(1)).astype(bool)


def _connections(occ):
    """For blocks of rows: (I, J, holes and particles) of the pairs J < I one and two excitations apart, as
    (single: I, J, p, r, sign) and (double: I, J, p, q, r, s, sign) with p < q only in I and r < s only in J."""
    n, nso = occ.shape
    f, below = occ.astype(np.float32), np.cumsum(occ, axis=1) - occ
    nelec = int(occ[0].sum())
    for b in range(0, n, 1000):
        e = min(n, b + 1000)
        apart = nelec - (f[b:e] @ f[:e].T).astype(np.int32)
        apart[np.arange(b, e)[:, None] <= np.arange(e)[None, :]] = 9
        I, J = np.nonzero(apart == 1)
        I = I + b
        p, r = np.argmax(occ[I] & ~occ[J], axis=1), np.argmax(occ[J] & ~occ[I], axis=1)
        single = (I, J, p, r, 1.0 - 2.0 * ((below[I, p] + below[J, r]) % 2))
        I, J = np.nonzero(apart == 2)
        I = I + b
        a, c = occ[I] & ~occ[J], occ[J] & ~occ[I]
        p, q = np.argmax(a, axis=1), nso - 1 - np.argmax(a[:, ::-1], axis=1)
        r, s = np.argmax(c, axis=1), nso - 1 - np.argmax(c[:, ::-1], axis=1)
        yield single, (I, J, p, q, r, s, 1.0 - 2.0 * ((below[I, p] + below[I, q] + below[J, r] + below[J, s]) % 2))


def _slater_condon(h, eri, occ):
    """Diagonal, and the (I, J, value) blocks below it."""
    norb = len(h)
    P, Q = np.meshgrid(np.arange(norb), np.arange(norb), indexing="ij")
    pair = np.maximum(P, Q) * (np.maximum(P, Q) + 1) // 2 + np.minimum(P, Q)
    two = lambda p, q, r, s: eri[pair[p, q], pair[r, s]]  # noqa: E731
    a, b = occ[:, 0::2].astype(float), occ[:, 1::2].astype(float)
    coulomb, exchange = two(P, P, Q, Q), two(P, Q, P, Q)
    t = a + b
    diag = t @ np.diag(h) + 0.5 * (((t @ coulomb) * t).sum(1) - ((a @ exchange) * a).sum(1) - ((b @ exchange) * b).sum(1))
    k = np.arange(norb)
    c3, x3 = two(P[:, :, None], Q[:, :, None], k, k), two(P[:, :, None], k, Q[:, :, None], k)

    def blocks():
        for (I, J, p, r, sign), (I2, J2, p2, q2, r2, s2, sign2) in _connections(occ):
            same = p % 2 == r % 2
            I, J, p, r, sign = I[same], J[same], p[same], r[same], sign[same]
            common = (occ[I] & occ[J])
            ca, cb = common[:, 0::2].astype(float), common[:, 1::2].astype(float)
            mine = np.where((p % 2 == 0)[:, None], ca, cb)
            v = h[p // 2, r // 2] + ((ca + cb) * c3[p // 2, r // 2]).sum(1) - (mine * x3[p // 2, r // 2]).sum(1)
            yield I, J, sign * v
            v = np.where((p2 % 2 == r2 % 2) & (q2 % 2 == s2 % 2), two(p2 // 2, r2 // 2, q2 // 2, s2 // 2), 0.0) - \
                np.where((p2 % 2 == s2 % 2) & (q2 % 2 == r2 % 2), two(p2 // 2, s2 // 2, q2 // 2, r2 // 2), 0.0)
            yield I2, J2, sign2 * v

    return diag, blocks()


def _density(occ, c):
    """Spatial one- and two-body density matrices of the real state c."""
    n, nso = occ.shape
    norb = nso // 2
    g1, g2 = np.zeros((norb, norb)), np.zeros(norb ** 4)

    def add(p, q, r, s, w):  # <a+_p a+_q a_s a_r> of spin-orbitals, kept where the spins of (p, r) and (q, s) agree
        ok = (p % 2 == r % 2) & (q % 2 == s % 2)
        at = ((p // 2 * norb + q // 2) * norb + r // 2) * norb + s // 2
        g2[:] += np.bincount(at[ok], w[ok], norb ** 4)

    w = c * c
    f = occ.astype(float)
    both = (f * w[:, None]).T @ f
    g1 += np.diag((w @ f).reshape(norb, 2).sum(1))
    p, q = np.nonzero(~np.eye(nso, dtype=bool))
    add(p, q, p, q, both[p, q])
    add(p, q, q, p, -both[p, q])
    for (I, J, p, r, sign), (I2, J2, p2, q2, r2, s2, sign2) in _connections(occ):
        same = p % 2 == r % 2
        I, J, p, r, w = I[same], J[same], p[same], r[same], (sign * c[I] * c[J])[same]
        np.add.at(g1, (p // 2, r // 2), w)
        np.add.at(g1, (r // 2, p // 2), w)
        row, k = np.nonzero(occ[I] & occ[J])
        for x, y in ((p[row], r[row]), (r[row], p[row])):
            add(x, k, y, k, w[row])
            add(k, x, k, y, w[row])
            add(x, k, k, y, -w[row])
            add(k, x, y, k, -w[row])
        w = sign2 * c[I2] * c[J2]
        for a, b, d, e in ((p2, q2, r2, s2), (r2, s2, p2, q2)):
            add(a, b, d, e, w)
            add(b, a, e, d, w)
            add(a, b, e, d, -w)
            add(b, a, d, e, -w)
    return g1, g2.reshape((norb,) * 4)


def exact(case, seed):
    if case["kind"] not in ("sigma", "hamiltonian", "davidson", "rdm") or case["n"] > EXACT_MOST:
        return None
    if case["kind"] == "davidson" and case["n"] > 4000:
        return None
    st = prepare(case, seed)
    h, eri, _, _ = _integrals(case["norb"], seed)
    occ = _occupations(st["dets"], 2 * case["norb"])
    if case["kind"] == "rdm":
        one, two = _density(occ, st["c"])
        return {"one": one, "two": two}
    diag, blocks = _slater_condon(h, eri, occ)
    if case["kind"] == "davidson":  # (a root's sign, and vectors within a degenerate pair, are free)
        H = np.diag(diag)
        for I, J, v in blocks:
            H[I, J] = v
        return {"energies": np.linalg.eigvalsh(H)[:case["roots"]], "vectors": None}
    x = st["x"].cpu().numpy() if torch.is_tensor(st["x"]) else np.asarray(st["x"])
    cols = x.T if torch.is_tensor(st["x"]) else x.reshape(len(diag), -1)
    y, elements = diag[:, None] * cols, len(diag)
    for I, J, v in blocks:
        elements += len(I)
        for k in range(cols.shape[1]):
            y[:, k] += np.bincount(I, v * cols[J, k], len(diag)) + np.bincount(J, v * cols[I, k], len(diag))
    y = y.T if torch.is_tensor(st["x"]) else y.reshape(x.shape)
    return y if case["kind"] == "sigma" else {"elements": elements, "y": y}
