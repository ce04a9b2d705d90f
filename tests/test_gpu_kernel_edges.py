"""Kernels at the sizes where their work split changes (partial tiles, few or
many work units, remainders), against the oracle."""
import numpy as np
import pytest

import helpers
from oracle_bind import OracleSystem

pytestmark = pytest.mark.gpu


def _space(path, occ, n, W):
    o = OracleSystem(path)
    dets = helpers.occ_to_det(occ, W)[None, :]
    eps = 1e-2
    while len(dets) < n:
        new = o.screen(dets, np.ones(len(dets)), eps)
        if len(new):
            dets = np.concatenate([dets, new])
        eps *= 0.5
    return dets[:n]


def _system(case, tmp_path):
    from dice_amd import synth
    path = str(tmp_path / "FCIDUMP")
    if case == "w1":
        synth.write_molecular_fcidump(path, 0, 16, 8, 8, 64)
        return path, synth.hf_occupation(8, 8), 1
    synth.write_molecular_fcidump(path, 5, 34, 6, 6, 12)
    return path, synth.hf_occupation(6, 6), 2


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("case,n", [("w1", 1), ("w1", 2), ("w1", 255), ("w1", 257), ("w1", 6001), ("w2", 1025)])
def test_sigma_work_units(case, n, prec, tmp_path):
    """Blocks without entries, of less than one unit and of many units.  Bar:
    1e-12 of the largest element in FP64 (sums of about a thousand terms), 3e-6
    with FP32 values and vectors (two roundings of 2^-24 a term)."""
    from dice_amd import shci
    path, occ, W = _system(case, tmp_path)
    dets = _space(path, occ, n, W)
    s = shci.System.from_fcidump(path)
    s.set_options(precision=prec)
    s.set_dets(dets)
    s.make_hamiltonian()
    o = OracleSystem(path)
    o.csr_append(dets)
    x = np.random.default_rng(n).normal(size=n)
    yo = o.sigma(x)
    assert np.max(np.abs(s.hmult(x) - yo)) <= (3e-6 if prec else 1e-12) * np.max(np.abs(yo))


@pytest.mark.parametrize("eps2", [0.0, 1e-4, 3e-2])
@pytest.mark.parametrize("case,n", [("w1", 1), ("w1", 65), ("w2", 130)])
def test_pt_candidates_of_few_sources(case, n, eps2, tmp_path):
    """Few sources (cut by electron pairs), lists walked (large eps2) and open
    orbitals enumerated (small), sums against the oracle's to 1e-11 (thousands
    of terms of one sign in another order)."""
    from dice_amd import shci
    path, occ, W = _system(case, tmp_path)
    dets = _space(path, occ, n, W)
    s = shci.System.from_fcidump(path)
    s.set_dets(dets)
    c = np.random.default_rng(n).normal(size=n)
    c /= np.linalg.norm(c)
    e0 = s.energy(dets).min() - 2.0
    o = OracleSystem(path)
    got, ref = s.pt_deterministic(c, e0, eps2), o.pt_deterministic(dets, c, e0, eps2)
    assert got[2] == ref[2]
    np.testing.assert_allclose(got[:2], ref[:2], rtol=1e-11, atol=0)


@pytest.mark.parametrize("case,n", [("w1", 65), ("w2", 130)])
def test_pt_candidates_of_zero_coefficients(case, n, tmp_path):
    """eps2 0 and coefficients that are 0: their threshold |0 / 0| cuts no
    double excitation off, so its external determinants are counted (with
    numerators 0), from the lists and from the open orbitals alike."""
    from dice_amd import shci
    path, occ, W = _system(case, tmp_path)
    dets = _space(path, occ, n, W)
    s = shci.System.from_fcidump(path)
    s.set_dets(dets)
    c = np.random.default_rng(n).normal(size=n)
    c[1:] = 0.0
    e0 = s.energy(dets).min() - 2.0
    got, ref = s.pt_deterministic(c, e0, 0.0), OracleSystem(path).pt_deterministic(dets, c, e0, 0.0)
    assert got[2] == ref[2]
    np.testing.assert_allclose(got[:2], ref[:2], rtol=1e-11, atol=0)


@pytest.mark.parametrize("eps", [1e-5, 3e-3, 10.0])
@pytest.mark.parametrize("case,n", [("w1", 1), ("w1", 3), ("w1", 1200), ("w2", 1), ("w2", 65)])
def test_screening_of_few_sources(case, n, eps, tmp_path):
    """Sources cut into parts and whole, candidates by the queue's 64s and its
    rest, none at all: the same new determinants as the oracle's, each once."""
    from dice_amd import shci
    path, occ, W = _system(case, tmp_path)
    dets = _space(path, occ, n, W)
    ci = np.linspace(1.0, 0.1, n)
    s = shci.System.from_fcidump(path)
    s.set_dets(dets)
    got = s.get_determinants_variational(ci, eps)
    want = OracleSystem(path).screen(dets, ci, eps)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n,roots", [(n, r) for n in (3, 8, 257, 1500) for r in (1, 2, 9) if r <= n])
def test_davidson_subspaces(n, roots, tmp_path):
    """Subspaces that grow to 4, 5 and 12 columns or to the whole space, and
    vectors shorter than a workgroup: from random vectors, orthonormal
    eigenvectors of the GPU's own rows (residuals of the tolerance 1e-5; a root
    found twice would overlap by 1) with eigenvalues of the dense matrix to 1e-8
    (the square of the residual over the gaps); from the lowest eigenvectors with
    noise, the lowest eigenvalues, each once (to 4e-8: residuals up to 2e-5, gaps
    from 0.0128 on)."""
    from dice_amd import shci
    path, occ, W = _system("w1", tmp_path)
    dets = _space(path, occ, n, W)
    s = shci.System.from_fcidump(path)
    s.set_dets(dets)
    rp, cols, vals = s.hamiltonian_rows()
    H = np.zeros((n, n))
    for i in range(n):
        H[i, cols[rp[i]:rp[i + 1]]] = vals[rp[i]:rp[i + 1]]
    H = np.tril(H) + np.tril(H, -1).T
    ev, U = np.linalg.eigh(H)
    rng = np.random.default_rng(n)
    x0 = rng.normal(size=(n, roots))
    x0[:roots] += 5.0 * np.eye(roots)
    noise = rng.normal(size=(n, roots)) * 0.02 / np.sqrt(n)
    for start, low in ((x0, False), (U[:, :roots] + noise, True)):
        e, x, _ = s.davidson(start, max_copies=max(roots + 3, 4), tol=1e-5)
        assert np.max(np.linalg.norm(H @ x - x * e, axis=0)) < 2e-5
        assert np.max(np.abs(x.T @ x - np.eye(roots))) < 1e-6
        if low:
            np.testing.assert_allclose(e, ev[:roots], rtol=0, atol=4e-8)
        elif n <= 8:
            np.testing.assert_allclose(e, ev[:roots], rtol=0, atol=1e-8)
        else:
            assert all(np.min(np.abs(ev - v)) < 1e-8 for v in e)


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("size", [63, 511, 512, 700])
def test_rows_of_groups_with_and_without_bitmap(size, half, tmp_path, monkeypatch):
    """Three alpha strings times `size` beta strings, below and above the
    group size from which beta singles are looked up in a bitmap, in random
    order: rows equal the oracle's."""
    import itertools
    from dice_amd import shci, synth
    path = str(tmp_path / "FCIDUMP")
    synth.write_molecular_fcidump(path, 7, 16, 1, 4, 24)
    rng = np.random.default_rng(size)
    beta = list(itertools.combinations(range(16), 4))
    beta = [beta[i] for i in rng.permutation(len(beta))[:size]]
    dets = np.array([(1 << (2 * a)) | sum(1 << (2 * x + 1) for x in b) for a in range(3) for b in beta],
                    dtype=np.int64).reshape(-1, 1)
    dets = dets[rng.permutation(len(dets))]
    monkeypatch.setenv("SHCI_STORAGE", "half" if half else "full")
    s, o = shci.System.from_fcidump(path), OracleSystem(path)
    s.set_dets(dets)
    rp, cols, vals = s.hamiltonian_rows()
    o.csr_append(dets)
    orp, ocols, ovals = o.csr()
    np.testing.assert_array_equal(rp, orp)
    for i in range(len(dets)):
        a, b = rp[i], rp[i + 1]
        order = np.argsort(ocols[a + 1:b], kind="stable")
        np.testing.assert_array_equal(cols[a + 1:b], ocols[a + 1:b][order])
        np.testing.assert_array_equal(vals[a + 1:b], ovals[a + 1:b][order])
