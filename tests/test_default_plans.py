"""The plans the library makes by itself (searched passes, special-unitary gates
with their global phase, shapes by size, complex64 forwards in gate order),
emulated on the CPU against the oracle."""
import math
import time

import numpy as np
import pytest

import oracle
from damavand_amd import _native as N
from damavand_amd import workloads as wl
from tests.libhelpers import NativeCircuit
from tests.test_tile_emulation import random_gates, zero_state
from tests.tile_emulator import TileEmulator, plan_json


@pytest.mark.parametrize("dtype,elem", [(N.C128, 16), (N.C64, 8)])
@pytest.mark.parametrize("n,count,seed", [(9, 60, 1), (10, 200, 2), (12, 250, 3), (13, 250, 4), (16, 300, 5), (18, 150, 6),
                                          (19, 120, 7), (20, 120, 8)])
def test_default_forward_plan(n, count, seed, dtype, elem):
    """Amplitudes, not only probabilities: the phases taken out of the gates come back."""
    if dtype == N.C64 and n <= 13:
        pytest.skip("a whole-state kernel's size")
    gates = random_gates(np.random.default_rng(seed), n, count)
    nc = NativeCircuit(n, gates)
    plan = plan_json(nc.h, dtype=dtype)
    got = TileEmulator(plan, elem=elem).forward(zero_state(n))
    np.testing.assert_allclose(got, oracle.run_gates(n, gates).amp, atol=1e-12)


@pytest.mark.parametrize("kind,params", [(wl.GATE_H, ()), (wl.GATE_Y, ()), (wl.GATE_U3, (0.3, 2.1, 5.0)),
                                         (wl.GATE_U3, (math.pi, 0.0, 0.0)), (wl.GATE_T, ()), (wl.GATE_RX, (0.0,))])
def test_global_phase_of_one_gate(kind, params):
    """One gate of determinant other than 1 on each qubit, so that the phase has to be kept by another gate's op, or by its own."""
    n = 13
    for last in (0, n - 1):
        gates = [(kind, -1, q, params) for q in range(n)] + [(wl.GATE_RY, -1, last, (0.4,))]
        nc = NativeCircuit(n, gates)
        got = TileEmulator(plan_json(nc.h)).forward(zero_state(n))
        np.testing.assert_allclose(got, oracle.run_gates(n, gates).amp, atol=1e-13)


def test_complex64_forward_keeps_gate_order():
    """The general matrices, in the order of the gates: what a program samples depends on a state's last bits."""
    n = 17
    gates = random_gates(np.random.default_rng(11), n, 200)
    nc = NativeCircuit(n, gates)
    auto = plan_json(nc.h, dtype=N.C64)
    m = np.array([op["m"] for P in auto["passes"] for ph in P["phases"] for op in ph["ops"] if op["kind"] == 0])
    m = m[:, ::2] + 1j * m[:, 1::2]
    assert (np.abs(m[:, 0] * m[:, 3] - m[:, 1] * m[:, 2] - 1.0) > 0.1).sum() > len(m) // 4  # determinants are kept
    given = [plan_json(nc.h, dtype=N.C64, tile_qubits=auto["k"], tlog=auto["tlog"], max_gen=g) for g in (8, 12)]
    assert auto["passes"] in [g["passes"] for g in given]


@pytest.mark.parametrize("n,layers", [(9, 1), (11, 1), (12, 1), (13, 1), (15, 1)])
def test_default_reverse_plan(n, layers):
    """The reverse sweep by itself: psi back to |0>, gradients against parameter shift."""
    gates, a, b = wl.ansatz_circuit(n, layers, 900 + n)
    gates = [(wl.GATE_H, -1, 0, ()), (wl.GATE_U3, -1, n - 1, (0.2, 0.7, 1.9))] + gates + [(wl.GATE_T, -1, n // 2, ())]
    pairs = wl.chain_pairs(n)
    nc = NativeCircuit(n, gates)
    st = oracle.run_gates(n, gates)
    idx = np.arange(1 << n)
    h = sum(c * (1.0 - 2.0 * ((idx >> q) & 1)) for q, c in enumerate(a))
    h = h + sum(c * (1.0 - 2.0 * (((idx >> i) ^ (idx >> j)) & 1)) for (i, j), c in zip(pairs, b))
    psi0, _, grads = TileEmulator(plan_json(nc.h, adjoint=True)).reverse(st.amp, h * st.amp)
    # up to a global phase, which no gradient sees
    assert abs(abs(psi0[0]) - 1.0) <= 1e-12 and np.abs(psi0[1:]).max() <= 1e-12
    ref = []
    for gi in [i for i, g in enumerate(gates) if g[0] in wl.PARAMETRIC]:
        vals = []
        for s in (0.5 * math.pi, -0.5 * math.pi):
            kk, c, t, p = gates[gi]
            vals.append(oracle.run_gates(n, gates[:gi] + [(kk, c, t, (p[0] + s,))] + gates[gi + 1:]).expect_zz(a, pairs, b))
        ref.append(0.5 * (vals[0] - vals[1]))
    np.testing.assert_allclose(grads, ref, atol=1e-10)


@pytest.mark.parametrize("kib,most", [(1, 8), (2, 16), (8, 64)])
def test_reverse_plan_within_its_partials(kib, most):
    """Passes of a bounded number of gradient entries (128 bytes of partials each at 13 qubits), in order all the
    same: the gradients of the unbounded plan."""
    n = 13
    gates, a, b = wl.ansatz_circuit(n, 4, 31)
    gates = [(k, -1, q, (0.3 * q + j,)) for q in range(n) for j, k in enumerate((wl.GATE_RX, wl.GATE_RY, wl.GATE_RX))] + gates
    nc = NativeCircuit(n, gates)
    psi = oracle.run_gates(n, gates).amp
    idx = np.arange(1 << n)
    lam = psi * sum(c * (1.0 - 2.0 * ((idx >> q) & 1)) for q, c in enumerate(a))
    free = plan_json(nc.h, adjoint=True)
    N.tune_set("adjoint_partial_kib", kib)
    try:
        plan = plan_json(nc.h, adjoint=True)
    finally:
        N.tune_set("adjoint_partial_kib", -1)
    per_pass = [[op["slot"] for ph in p["phases"] for op in ph["ops"] if op["slot"] >= 0] for p in plan["passes"]]
    assert max(len(s) for s in per_pass) <= most
    assert sorted(s for p in per_pass for s in p) == list(range(sum(g[0] in wl.PARAMETRIC for g in gates)))
    want = TileEmulator(free).reverse(psi, lam)[2]
    np.testing.assert_allclose(TileEmulator(plan).reverse(psi, lam)[2], want, atol=1e-11)


def exact_amplitudes(n, ops):
    """State after (matrix, control mask, target) ops, in 80 bits."""
    v = np.zeros(1 << n, dtype=np.clongdouble)
    v[0] = 1
    idx = np.arange(1 << n)
    for m, ctrl, target in ops:
        m = np.asarray(m, dtype=np.clongdouble)
        w = v.reshape(-1, 2, 1 << target)
        x, y = w[:, 0], w[:, 1]
        out = np.stack([m[0, 0] * x + m[0, 1] * y, m[1, 0] * x + m[1, 1] * y], axis=1).reshape(-1)
        v = np.where((idx & ctrl) == ctrl, out, v) if ctrl else out
    return v


def exact_u3(th, ph, la):
    def e(x):
        return np.cos(np.longdouble(x)) + 1j * np.sin(np.longdouble(x))

    c, s = np.cos(np.longdouble(th) / 2), np.sin(np.longdouble(th) / 2)
    return [[c, -e(la) * s], [e(ph) * s, e(np.longdouble(ph) + np.longdouble(la)) * c]]


def test_special_unitary_matrices_lose_nothing():
    """U3 gates (any determinant) and CNOTs.  The matrices of complex128 plans, phases taken out and put back, against
    the merged gates as they are (the ops of complex64 plans): they are no further from the exact state, on the
    geometric mean of eight circuits."""
    ratios = []
    for seed in range(8):
        n, rng = 9 + seed % 3, np.random.default_rng(40 + seed)
        gates = []
        for _ in range(3 + 2 * seed):
            gates += [(wl.GATE_U3, -1, q, tuple(rng.uniform(0, 2 * math.pi, 3))) for q in range(n)]
            gates += [(wl.GATE_CNOT, q, q + 1, ()) for q in range(0, n - 1, 2)]
        want = exact_amplitudes(n, [([[0, 1], [1, 0]], 1 << c, t) if k == wl.GATE_CNOT else (exact_u3(*p), 0, t)
                                    for k, c, t, p in gates])
        nc = NativeCircuit(n, gates)
        error = []
        for dtype in (N.C128, N.C64):
            _, target, ctrl, m, _ = nc.plan_ops(dtype=dtype)
            got = exact_amplitudes(n, [(x, int(c), int(t)) for x, c, t in zip(m, ctrl, target)])
            error.append(np.sqrt((np.abs(got - want) ** 2).sum()))
        ratios.append(float(error[0] / error[1]))
    assert np.exp(np.log(ratios).mean()) <= 1.0, ratios


def test_planning_time_grows_with_the_gates():
    """A state of one tile is one pass, however long the circuit: ten times the gates take about ten times as long to plan."""
    n, best = 12, []
    for layers in (150, 1500):
        nc = NativeCircuit(n, wl.ansatz_circuit(n, layers, 3)[0])
        times = []
        for _ in range(3):
            t = time.perf_counter()
            assert nc.plan_stats()[0] == 1
            times.append(time.perf_counter() - t)
        best.append(min(times))
    assert best[1] < 40 * best[0], best


@pytest.mark.parametrize("n,dtype,whole", [(9, N.C128, True), (10, N.C128, False), (13, N.C64, True), (14, N.C64, False)])
def test_small_forwards_need_no_plan(n, dtype, whole):
    """Up to 9 qubits (complex64 13) a forward is one launch that takes the ops in order."""
    passes, phases, _, _ = NativeCircuit(n, wl.layered_circuit(n, 4, 1)).plan_stats(dtype=dtype)
    assert ((passes, phases) == (1, 1)) == whole


def test_default_forward_plan_of_a_large_state():
    """21 qubits: 16 amplitudes a thread, passes searched with and without a bit to split their transposes by."""
    n = 21
    gates = random_gates(np.random.default_rng(21), n, 90)
    nc = NativeCircuit(n, gates)
    plan = plan_json(nc.h)
    assert (plan["k"], plan["tlog"]) == (12, 8)
    got = TileEmulator(plan).forward(zero_state(n))
    np.testing.assert_allclose(got, oracle.run_gates(n, gates).amp, atol=1e-12)
