"""Reductions at the sizes where their launch shapes change: outcome tables
with qubits below and above the 64-term runs, in any order, of one to many
waves, on statevectors and density matrices, and Pauli sums of more groups
than one launch takes.  Sums are compensated FP64, so tables agree with numpy's
(pairwise) sums to a few ulps of the total: 1e-14 is allowed."""

import ctypes as C

import numpy as np
import pytest

from quest_amd import circuits as qc

pytestmark = pytest.mark.gpu


def table_of(p, qubits):
    key = np.zeros(p.size, dtype=np.int64)
    idx = np.arange(p.size)
    for i, q in enumerate(qubits):
        key |= ((idx >> q) & 1) << i
    return np.bincount(key, weights=p, minlength=1 << len(qubits))


TABLES = [(1, [0]), (2, [1, 0]), (3, [2]), (5, [4, 0, 2]), (6, [5, 3]), (7, [6]), (7, [0, 6, 3]), (9, [8, 7, 6]),
          (12, [11, 0, 5, 6]), (14, list(range(14))[::-1]), (16, [3]), (16, [9, 2, 15, 7, 0]), (18, [17]),
          (18, list(range(6))), (18, list(range(6, 18))), (20, [0, 19, 10]), (20, list(range(5, 20))),
          (21, [20, 1, 13, 6, 2, 9, 18])]


@pytest.mark.parametrize("prec", [2, 1])
@pytest.mark.parametrize("n,qubits", TABLES)
def test_outcome_tables(api, n, qubits, prec):
    print(f"[gpu] outcome table n={n} qubits={qubits} prec={prec}", flush=True)
    amps = qc.random_state(n, 11 * n + len(qubits))
    q = api.createCustomPrecisionQureg(n, 0, prec)
    try:
        api.set_amps(q, amps)
        a = api.get_amps(q)
        want = table_of(a.real ** 2 + a.imag ** 2, qubits)
        assert np.max(np.abs(api.probs_of_all_outcomes(q, qubits) - want)) <= 1e-14
    finally:
        api.destroyQureg(q)


@pytest.mark.parametrize("n,qubits", [(1, [0]), (3, [2, 0]), (7, [6, 1]), (9, [0, 8, 4, 7])])
def test_outcome_tables_of_density_matrices(api, n, qubits):
    print(f"[gpu] density outcome table n={n} qubits={qubits}", flush=True)
    rho = qc.random_state(n, 5 * n, True)
    q = api.createDensityQureg(n)
    try:
        api.set_amps(q, rho)
        p = rho.reshape(1 << n, 1 << n).diagonal().real
        assert np.max(np.abs(api.probs_of_all_outcomes(q, qubits) - table_of(p, qubits))) <= 1e-14
    finally:
        api.destroyQureg(q)


@pytest.mark.parametrize("n", [1, 2, 9, 11, 13])
def test_pauli_sums_of_many_groups(api, n):
    """60 strings with (almost all) different X/Y masks, Z strings and the
    identity among them: several launches of groups, one workgroup each below
    11 qubits and more above."""
    print(f"[gpu] pauli sum of many groups n={n}", flush=True)
    rng = np.random.default_rng(n)
    amps = qc.random_state(n, 3 * n)
    words = ["".join(rng.choice(list("IXYZ"), size=n)) for _ in range(58)] + ["Z" * n, "I" * n]
    weights = rng.uniform(-1, 1, size=len(words))
    idx = np.arange(1 << n)
    want = 0.0
    for word, w in zip(words, weights):
        x = sum(1 << i for i, c in enumerate(word) if c in "XY")
        z = sum(1 << i for i, c in enumerate(word) if c in "YZ")
        sign = 1 - 2 * (np.array([bin(i & z).count("1") for i in idx]) & 1)
        # P|j> = i^#Y (-1)^(j & z) |j ^ x>
        want += w * ((1j ** word.count("Y")) * np.vdot(amps[idx ^ x], sign * amps)).real
    strs = (api.PauliStr * len(words))(*[api.pauli_str(s, range(n)) for s in words])
    coeffs = (api.qcomp * len(words))(*[api.qcomp(w, 0.0) for w in weights])
    s = api.createPauliStrSum(strs, coeffs, len(words))
    q = api.createQureg(n)
    try:
        api.set_amps(q, amps)
        assert abs(api.calcExpecPauliStrSum(q, s) - want) <= 1e-13
        for word, w in zip(words[-3:], weights[-3:]):
            assert np.isfinite(api.calcExpecPauliStr(q, api.pauli_str(word, range(n))))
    finally:
        api.destroyPauliStrSum(s)
        api.destroyQureg(q)


@pytest.mark.parametrize("n,prec", [(21, 2), (22, 1), (22, 2), (23, 2)])
def test_pauli_sums_sharing_reads(api, n, prec):
    """Groups that share a read of the state (from 22 qubits): masks that are
    XORs of others, masks of low qubits only, one to eight strings a group,
    one to four groups left over."""
    print(f"[gpu] pauli sum sharing reads n={n} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    amps = qc.random_state(n, 3 * n)
    q = api.createCustomPrecisionQureg(n, 0, prec)
    idx = np.arange(1 << n)
    masks = [0b1, 0b11, 0b10, 1 << (n - 1), (1 << (n - 1)) | 0b101, 1 << 7, (1 << 7) | 0b11, 0b110000, 0]
    masks += [int(m) for m in rng.integers(1, 1 << n, size=2 + n % 3)]
    terms = []
    for i, m in enumerate(masks):
        for _ in range(1 + (3 * i) % 8):
            y = m & int(rng.integers(0, 1 << n))
            terms.append((m & ~y, y, int(rng.integers(0, 1 << n)) & ~m))
    weights = rng.uniform(-1, 1, size=len(terms))
    nt = len(terms)
    col = [(C.c_uint64 * nt)(*[t[i] for t in terms]) for i in range(3)]
    coeffs = (C.c_double * (2 * nt))(*[v for w in weights for v in (w, 0.0)])
    vals, out = (C.c_double * (2 * nt))(), (C.c_double * 2)()
    try:
        api.set_amps(q, amps)
        a = api.get_amps(q)
        assert api.gpu().qa_statevec_calcExpecPauliStrSum(C.c_void_p(q.gpuAmps), prec, n, C.c_int64(nt), *col, coeffs,
                                                          vals, out) == 0
    finally:
        api.destroyQureg(q)
    for t, (x, y, z) in enumerate(terms):
        par = idx & (y | z)
        for sh in (16, 8, 4, 2, 1):
            par = par ^ (par >> sh)
        want = (1j ** bin(y).count("1")) * np.vdot(a[idx ^ (x | y)], (1 - 2 * (par & 1)) * a)
        assert abs(complex(vals[2 * t], vals[2 * t + 1]) - want) <= 1e-14, (t, bin(x | y))


@pytest.mark.parametrize("n,prec", [(1, 2), (5, 1), (8, 2), (9, 2), (9, 1), (33, 1)])
def test_every_qubit_probabilities_ten_at_a_time(api, n, prec):
    """Below 10 qubits and above 32 (33: 64 GiB) a read serves up to ten
    qubits; a product state has each qubit's probabilities in closed form.
    The tolerance is the states' own: a gate rounds by a few units."""
    print(f"[gpu] every-qubit probabilities ten at a time n={n} prec={prec}", flush=True)
    angles = [0.2 + 0.08 * t for t in range(n)]
    q = api.createCustomPrecisionQureg(n, 0, prec)
    out = np.zeros(2 * n)
    try:
        api.initZeroState(q)
        for t, x in enumerate(angles):
            api.applyRotateY(q, t, x)
        assert api.gpu().qa_statevec_calcProbsOfEveryQubit(C.c_void_p(q.gpuAmps), prec, n, out.ctypes.data_as(C.c_void_p)) == 0
    finally:
        api.destroyQureg(q)
    tol = 4 * n * (2.0 ** -53 if prec == 2 else 2.0 ** -24)
    assert np.max(np.abs(out[1::2] - np.sin(np.array(angles) / 2) ** 2)) <= tol
    assert np.max(np.abs(out[0::2] - np.cos(np.array(angles) / 2) ** 2)) <= tol
