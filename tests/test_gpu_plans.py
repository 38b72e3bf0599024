"""Plans kept across angles, sizes on both sides of the shape rules, and the
batch's tiles and groups, against the oracle or a fresh handle."""
import math
import threading

import numpy as np
import pytest

import oracle
from damavand_amd import batch_forward_adjoint
from damavand_amd import workloads as wl
from tests.test_gpu_parity import build_circuit, random_gates

pytestmark = pytest.mark.gpu

# |amplitude| <= 1 and a gate rounds each a few times: gates * 8 units in the last place
EPS = {"complex128": 2.0 ** -53, "complex64": 2.0 ** -24}


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [8, 9, 10, 12, 13, 14, 19, 20])
def test_forward_at_shape_edges(native, n, dtype):
    print(f"case forward n={n} {dtype}", flush=True)
    gates = random_gates(np.random.default_rng(60 + n), n, 150)
    c = build_circuit(n, gates, dtype)
    c.forward()
    err = np.abs(c.retrieve_amplitudes_on_host() - oracle.run_gates(n, gates).amp).max()
    print(f"  {err:.2e}", flush=True)
    assert err <= 150 * 8 * EPS[dtype]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [8, 9, 11, 12, 13])
def test_gradient_at_shape_edges(native, n, dtype):
    """A layer's gradients against parameter shift on the oracle."""
    print(f"case gradient n={n} {dtype}", flush=True)
    gates, a, b = wl.ansatz_circuit(n, 1, 70 + n)
    pairs = wl.chain_pairs(n)
    e, g = build_circuit(n, gates, dtype).gradient(a, pairs, b)
    ref = []
    for gi in [i for i, x in enumerate(gates) if x[0] in wl.PARAMETRIC]:
        k, c, t, p = gates[gi]
        v = [oracle.run_gates(n, gates[:gi] + [(k, c, t, (p[0] + s,))] + gates[gi + 1:]).expect_zz(a, pairs, b)
             for s in (0.5 * math.pi, -0.5 * math.pi)]
        ref.append(0.5 * (v[0] - v[1]))
    # gates * 8 roundings of two states, weighed by the observable's norm
    tol = 2 * len(gates) * 8 * EPS[dtype] * (np.abs(a).sum() + np.abs(b).sum())
    assert abs(e - oracle.run_gates(n, gates).expect_zz(a, pairs, b)) <= tol
    assert np.abs(g - np.array(ref)).max() <= tol


@pytest.mark.parametrize("n,dtype", [(7, "complex128"), (11, "complex128"), (16, "complex128"), (16, "complex64")])
def test_new_angles_on_a_kept_plan(native, n, dtype):
    """New angles, angles whose gates vanish or become diagonal, a gate more: the results of a fresh circuit each time, to the bit."""
    print(f"case angles n={n} {dtype}", flush=True)
    gates, a, b = wl.ansatz_circuit(n, 2, 80 + n)
    pairs = wl.chain_pairs(n)
    rng = np.random.default_rng(n)
    c = build_circuit(n, gates, dtype)
    for step in range(5):
        if step == 4:
            gates = gates + [(wl.GATE_U3, -1, 1, (0.4, 0.2, 1.0))]
            c.add_gate(*gates[-1])
        theta = rng.uniform(0, 2 * math.pi, c.num_parameters)
        if step == 2:
            theta[::3] = 0.0
        if step == 3:
            theta[::2] = math.pi
        c.set_parameters(theta)
        e, g = c.gradient(a, pairs, b)
        c.reset_amplitudes()
        c.forward()
        it = iter(theta)
        fresh = build_circuit(n, [(k, q, t, (float(next(it)),)) if k in wl.PARAMETRIC else (k, q, t, p) for k, q, t, p in gates],
                              dtype)
        e2, g2 = fresh.gradient(a, pairs, b)
        fresh.forward()
        assert e == e2 and np.array_equal(g, g2)
        assert np.array_equal(c.retrieve_amplitudes_on_host(), fresh.retrieve_amplitudes_on_host())


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_batch_of_many_structures(native, dtype):
    """Circuits below, at and above the tile's size, equal structures at other angles, a circuit without parameters
    and one without gates."""
    print(f"case batch {dtype}", flush=True)
    rng = np.random.default_rng(90)
    circuits = wl.batch_workload(10, 91, n_range=(2, 13), layer_range=(1, 3))
    for n, layers in ((4, 2), (11, 2), (12, 1), (10, 3)):
        gates, a, b = wl.ansatz_circuit(n, layers, 92 + n)
        for _ in range(3):
            circuits.append((n, [(k, c, t, (rng.uniform(0, 6.0),)) if k in wl.PARAMETRIC else (k, c, t, p)
                                 for k, c, t, p in gates], a, b))
    circuits.append((12, [(wl.GATE_H, -1, 3, ()), (wl.GATE_CNOT, 3, 11, ())], rng.standard_normal(12), rng.standard_normal(11)))
    circuits.append((5, [], rng.standard_normal(5), rng.standard_normal(4)))
    for order in (range(len(circuits)), rng.permutation(len(circuits))):
        some = [circuits[i] for i in order]
        energy, grads = batch_forward_adjoint(some, dtype=dtype)
        for (n, gates, a, b), e, g in zip(some, energy, grads):
            ref = build_circuit(n, gates)
            e1, g1 = ref.gradient(a, wl.chain_pairs(n), b)
            tol = 2 * (len(gates) + 8) * 8 * EPS[dtype] * (np.abs(a).sum() + np.abs(b).sum())
            assert abs(e - e1) <= tol and (g.size == 0 or np.abs(g - g1).max() <= tol)


def test_threads_share_plans(native):
    """Threads with circuits of the same structure and of different ones, and batches beside them."""
    print("case threads", flush=True)
    n = 13
    gates, a, b = wl.ansatz_circuit(n, 2, 95)
    pairs = wl.chain_pairs(n)
    batch = wl.batch_workload(6, 96, n_range=(6, 12), layer_range=(1, 2))
    want = build_circuit(n, gates).gradient(a, pairs, b)
    want_batch = batch_forward_adjoint(batch)
    bad = []

    def work(i):
        try:
            for r in range(6):
                extra = [(wl.GATE_H, -1, (i + r) % n, ())] * 2  # H H: another structure, the same circuit
                c = build_circuit(n, gates + (extra if r % 2 else []))
                e, g = c.gradient(a, pairs, b)
                if abs(e - want[0]) > 1e-12 or np.abs(g - want[1]).max() > 1e-12:
                    bad.append(("circuit", i, r))
                eb, gb = batch_forward_adjoint(batch)
                if not np.array_equal(eb, want_batch[0]) or any(not np.array_equal(x, y) for x, y in zip(gb, want_batch[1])):
                    bad.append(("batch", i, r))
        except Exception as e:  # reported by the main thread
            bad.append(repr(e))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in ts) and not bad, bad


@pytest.mark.parametrize("mib", [1, 2, 6])
def test_batch_in_groups(native, mib):
    """Groups of one circuit, of a few and of all of them: the same results to the bit."""
    print(f"case batch groups {mib} MiB", flush=True)
    circuits = wl.batch_workload(24, 97, n_range=(9, 14), layer_range=(1, 3))
    want = batch_forward_adjoint(circuits)
    native.tune_set("batch_pool_mib", mib)
    try:
        got = batch_forward_adjoint(circuits)
    finally:
        native.tune_set("batch_pool_mib", -1)
    assert np.array_equal(got[0], want[0])
    assert all(np.array_equal(x, y) for x, y in zip(got[1], want[1]))
