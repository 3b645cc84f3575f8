"""Damping, Pauli, two-qubit dephasing and two-qubit depolarising channels
inside fused passes, against the CPU oracle (1e-12 relative L2) and, at a size
the oracle is slow for, against the channels' own kernels."""

import numpy as np
import pytest

from quest_amd import circuits as qc

pytestmark = pytest.mark.gpu


def noisy(n: int, depth: int, seed: int, extremes: bool = False) -> qc.Circuit:
    rng = qc.SplitMix64(seed)
    c = qc.Circuit(n, True, [], ("random", seed), f"channels_n{n}")
    for _ in range(depth):
        for q in range(n):
            c.ops.append(("U1", q, qc.haar_unitary(rng, 2)))
            kind = rng.randint(4)
            if kind == 0:
                c.ops.append(("DAMP", q, 1.0 if extremes and rng.randint(4) == 0 else 0.1 * rng.uniform()))
            elif kind == 1:
                c.ops.append(("PAULIS", q, 0.1 * rng.uniform(), 0.1 * rng.uniform(), 0.1 * rng.uniform()))
        perm = rng.permutation(n)
        for k in range(n // 2):
            a, b = perm[2 * k], perm[2 * k + 1]
            c.ops.append(("CZ", a, b))
            kind = rng.randint(3)
            if kind == 0:
                c.ops.append(("DEPOL2", a, b, 15 / 16 if extremes and rng.randint(4) == 0 else 0.1 * rng.uniform()))
            elif kind == 1:
                c.ops.append(("DEPH2", a, b, 0.75 if extremes and rng.randint(4) == 0 else 0.1 * rng.uniform()))
    return c


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,tile,low", [(2, 12, 4), (3, 12, 4), (4, 5, 1), (5, 8, 3), (6, 13, 3), (7, 12, 4)])
@pytest.mark.parametrize("jit", [0, 2])
def test_channels_in_passes_match_oracle(api, n, tile, low, jit):
    from oracle import qoracle as O
    print(f"[gpu] channel fusion n={n} tile={tile} low={low} jit={jit}", flush=True)
    before = api.get_fusion()
    c = noisy(n, 3, 40 + n, extremes=True)
    want, _ = O.run(c)
    api.set_fusion(True, tile, low, 512)
    api.set_fusion_jit(jit, 1)
    try:
        q, _ = qc.run(c)
        got = api.get_amps(q)
        api.destroyQureg(q)
        assert rel(got, want) <= 1e-12
        # complex64: a gate rounds the state by at most a few 2^-24, gates add up
        q = api.createCustomPrecisionQureg(n, 1, 1)
        q, _ = qc.run(c, q)
        got = api.get_amps(q)
        api.destroyQureg(q)
        assert rel(got, want) <= 4 * 2.0 ** -24 * len(c.ops)
    finally:
        api.set_fusion_jit(1, 2)
        api.set_fusion(bool(before[0]), *before[1:])


def test_channels_in_passes_match_their_own_kernels(api):
    n = 10
    print(f"[gpu] channel fusion n={n} against unfused and exact", flush=True)
    before = api.get_fusion()
    c = noisy(n, 2, 77)
    amps = []
    try:
        for enabled, exact in ((True, False), (False, False), (True, True)):
            api.set_fusion(enabled, 12, 4, 512)
            api.set_fusion_exact(exact)
            q, _ = qc.run(c)
            amps.append(api.get_amps(q))
            api.destroyQureg(q)
    finally:
        api.set_fusion_exact(False)
        api.set_fusion(bool(before[0]), *before[1:])
    assert rel(amps[0], amps[1]) <= 1e-13
    assert np.array_equal(amps[1], amps[2])  # exact fusion keeps the channels' own kernels


@pytest.mark.parametrize("min_gates", [1, 2])
def test_channels_in_mfma_blocks(api, min_gates):
    """complex64 passes whose runs on 5 index bits are multiplied into one
    32x32 matrix hold the channels too, strong ones so that a lost one shows;
    3-target matrices end a run.  A gate rounds the state by at most a few
    2^-24, and a block's elements are rounded once."""
    from oracle import qoracle as O
    print(f"[gpu] channels in MFMA blocks, from {min_gates} gates", flush=True)
    before = api.get_fusion()
    n = 6
    rng = qc.SplitMix64(61)
    c = qc.Circuit(n, True, [], ("random", 62), "channels_blocks")
    for i in range(24):
        a, b = rng.sample(n, 2)
        c.ops.append([("DEPOL2", a, b, 0.5), ("DEPH2", a, b, 0.4), ("DAMP", a, 0.3), ("PAULIS", b, 0.1, 0.2, 0.05)][i % 4])
        if i % 3 == 0:
            c.ops.append(("U1", a, qc.haar_unitary(rng, 2)))
        if i % 8 == 5:
            c.ops.append(("UN", rng.sample(n, 3), qc.haar_unitary(rng, 8)))
    want, _ = O.run(c)
    api.set_fusion(True, 10, 3, 512)
    assert api.gpu().qa_setFusionBlocks(min_gates) == 0
    try:
        q = api.createCustomPrecisionQureg(n, 1, 1)
        q, _ = qc.run(c, q)
        got = api.get_amps(q)
        api.destroyQureg(q)
    finally:
        api.gpu().qa_setFusionBlocks(0)
        api.set_fusion(bool(before[0]), *before[1:])
    assert rel(got, want) <= 8 * 2.0 ** -24 * len(c.ops)


@pytest.mark.parametrize("prec", [2, 1])
@pytest.mark.parametrize("jit", [0, 2])
def test_two_qubit_dephasing_rounds_once(api, prec, jit):
    """In a pass, on qubits in and outside the registers and the tile, the
    channel multiplies each amplitude once and by the factor of its own kernel:
    the results are equal, bit for bit."""
    print(f"[gpu] two-qubit dephasing in passes prec={prec} jit={jit}", flush=True)
    before = api.get_fusion()
    n = 7
    c = qc.Circuit(n, True, [], ("random", 93), "dephasing")
    for a, b, p in [(0, 1, 0.3), (0, 6, 0.11), (5, 6, 0.75), (2, 4, 0.05), (3, 6, 0.4), (1, 5, 0.2)]:
        c.ops.append(("DEPH2", a, b, p))
    got = []
    try:
        for enabled in (False, True):
            api.set_fusion(enabled, 8, 3, 512)
            api.set_fusion_jit(jit, 1)
            q = api.createCustomPrecisionQureg(n, 1, prec)
            q, _ = qc.run(c, q)
            got.append(api.get_amps(q))
            api.destroyQureg(q)
    finally:
        api.set_fusion_jit(1, 2)
        api.set_fusion(bool(before[0]), *before[1:])
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("kind", ["DAMP", "PAULIS", "DEPH2"])
def test_channels_keep_infinite_amplitudes(api, kind):
    """One infinite amplitude: a channel in a pass touches what its own kernel
    touches, where a matrix would make NaN of the whole group."""
    print(f"[gpu] infinite amplitudes under {kind}", flush=True)
    before = api.get_fusion()
    n = 5
    rho = qc.random_state(n, 91, True)
    rho[0b00111_10110] = np.inf
    c = qc.Circuit(n, True, [], ("given",), "infinite")
    for q in (1, 0, 1, 3, 1):
        c.ops.append((kind, q, *{"DAMP": [0.2], "PAULIS": [0.1, 0.2, 0.05], "DEPH2": [4, 0.2]}[kind]))
    got = []
    try:
        for enabled in (False, True):
            api.set_fusion(enabled, 8, 3, 512)
            q = api.createDensityQureg(n)
            api.set_amps(q, rho)
            q, _ = qc.run(c, q)
            got.append(api.get_amps(q))
            api.destroyQureg(q)
    finally:
        api.set_fusion(bool(before[0]), *before[1:])
    assert np.count_nonzero(np.isnan(got[0].real)) == 0
    assert np.allclose(got[1].real, got[0].real, rtol=1e-13, atol=1e-15)
    assert np.array_equal(np.isfinite(got[1]), np.isfinite(got[0]))
