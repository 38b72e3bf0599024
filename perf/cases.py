"""The workloads whose speed this library is held to, and their exact results.

Every case is a plain dict.  ``kind`` names the work, through the public entry points that a program calls:

* ``circuit``: a circuit is run from |0...0> and read out as the reference's example programs do: amplitudes stay
  on the device, probabilities, samples and <Z> of every qubit come to the host (``Circuit``).
* ``forward``: a circuit too large for its probabilities to be wanted one by one: run from |0...0>, <Z> of every
  qubit read, the new state left on the device for what follows (``Circuit``, ``StateVector``).
* ``gradient``: one step of a variational program in complex128: new angles in, the energy of a Z/ZZ chain and its
  gradient by every angle out (``Circuit.set_parameters``, ``Circuit.gradient``).
* ``torch``: the same through ``autograd.expectation`` and ``backward()``, in the angles' precision.
* ``batch``: many circuits of uneven size, energies and gradients of all of them in one call
  (``batch_forward_adjoint_packed``).
* ``readout``: observables, a fidelity and samples of a large state that is already there (``StateVector``).

Circuits: ``layered`` (per layer H, RX, RY, RZ on every qubit, then a CNOT ladder), ``ansatz`` (RY, RZ on every
qubit, then a CNOT ring) and ``random`` (U3 on every qubit, then CNOT or CZ on random pairs), the three shapes of the
framework's benchmark.  Single-precision programs (complex64) keep their results in 32 bits.
"""
import ctypes
import math

import numpy as np
import torch

from damavand_amd import Circuit, batch_forward_adjoint_packed, pack_circuits
from damavand_amd import _native as N
from damavand_amd import autograd

H, RX, RY, RZ, CNOT, U3, CZ = N.GATE_H, N.GATE_RX, N.GATE_RY, N.GATE_RZ, N.GATE_CNOT, N.GATE_U3, N.GATE_CZ
AMP_BYTES = {"complex128": 16, "complex64": 8}


# ------------------------------------------------------------------------------------------------------- the cases --
def listed():
    return [
        # a small variational model inside a torch training loop: one step is latency and launches
        dict(name="torch_10q", kind="torch", circuit="ansatz", n=10, layers=4, dtype="complex128"),
        # a teaching-sized circuit read out in full; the whole state fits one workgroup
        dict(name="circuit_12q", kind="circuit", circuit="layered", n=12, layers=6, dtype="complex128"),
        # the reference's CPU benchmark: 990 gates, probabilities, 1000 samples, <Z>
        dict(name="circuit_20q", kind="circuit", circuit="layered", n=20, layers=10, dtype="complex128"),
        # a variational step at the size that such programs mostly have
        dict(name="gradient_16q", kind="gradient", circuit="ansatz", n=16, layers=8, dtype="complex128"),
        # a shallow one in single precision from torch, odd size
        dict(name="torch_21q_c64", kind="torch", circuit="ansatz", n=21, layers=4, dtype="complex64"),
        # the benchmark's gradient: 960 angles at 24 qubits
        dict(name="gradient_24q", kind="gradient", circuit="ansatz", n=24, layers=20, dtype="complex128"),
        # random-circuit sampling in single precision, high-index pairs
        dict(name="random_27q_c64", kind="forward", circuit="random", n=27, layers=6, dtype="complex64"),
        # the headline: 745 gates over 16 GiB
        dict(name="layered_30q", kind="forward", circuit="layered", n=30, layers=5, dtype="complex128"),
        # a minibatch of small models of uneven size, in one call
        dict(name="batch_32", kind="batch", count=32, n_min=8, n_max=14, layers_min=2, layers_max=8,
             dtype="complex128"),
        # the benchmark's batch at a quarter of its count, in both precisions
        dict(name="batch_1024", kind="batch", count=1024, n_min=12, n_max=18, layers_min=4, layers_max=12,
             dtype="complex128"),
        dict(name="batch_1024_c64", kind="batch", count=1024, n_min=12, n_max=18, layers_min=4, layers_max=12,
             dtype="complex64"),
        # every observable of one large state
        dict(name="readout_28q", kind="readout", circuit="layered", n=28, layers=1, dtype="complex128",
             samples=100000),
    ]


def draw(rng):
    kind = rng.choice(["torch", "circuit", "gradient", "forward", "batch", "readout"])
    dtype = rng.choice(["complex128", "complex128", "complex64"])
    if kind == "batch":
        lo = rng.randint(3, 14)
        return dict(kind=kind, count=int(round(2 ** rng.uniform(1, 8))), n_min=lo, n_max=rng.randint(lo, min(18, lo + 6)),
                    layers_min=2, layers_max=rng.randint(2, 12), dtype=dtype)
    if kind == "readout":
        return dict(kind=kind, circuit="layered", n=rng.randint(12, 28), layers=1, dtype=dtype,
                    samples=int(round(10 ** rng.uniform(2, 5))))
    if kind in ("gradient", "torch"):
        n = rng.randint(4, 23)
        if kind == "gradient":
            dtype = "complex128"
        layers = rng.randint(2, 4 if dtype == "complex64" else 10)  # deep ones have energies that 32 bits do not hold
        return dict(kind=kind, circuit=rng.choice(["ansatz", "layered"]), n=n, layers=layers, dtype=dtype)
    n = rng.randint(4, 20) if kind == "circuit" else rng.randint(13, 28)
    return dict(kind=kind, circuit=rng.choice(["layered", "ansatz", "random"]), n=n, layers=rng.randint(2, 10),
                dtype=dtype)


# ------------------------------------------------------------------------------------------------------ the inputs --
def gates_of(circuit, n, layers, rng):
    """[(kind, control, target, angles)], angles uniform in [0, 2 pi); those of a single-precision program are
    32-bit values."""
    out = []
    for _ in range(layers):
        if circuit == "layered":
            out += [(H, -1, q, ()) for q in range(n)]
            for kind in (RX, RY, RZ):
                out += [(kind, -1, q, (float(t),)) for q, t in enumerate(rng.uniform(0, 2 * math.pi, n))]
            out += [(CNOT, q, q + 1, ()) for q in range(n - 1)]
        elif circuit == "ansatz":
            for kind in (RY, RZ):
                t = rng.uniform(0, 2 * math.pi, n).astype(np.float32)
                out += [(kind, -1, q, (float(x),)) for q, x in enumerate(t)]
            out += [(CNOT, q, (q + 1) % n, ()) for q in range(n)]
        else:
            for q, t in enumerate(rng.uniform(0, 2 * math.pi, (n, 3))):
                out.append((U3, -1, q, tuple(float(x) for x in t)))
            for _ in range(n // 2):
                c, t = rng.choice(n, 2, replace=False)
                out.append((CNOT if rng.integers(2) else CZ, int(c), int(t), ()))
    return out


def chain(n, rng):
    """Coefficients of H = sum a_q Z_q + sum b_q Z_q Z_{q+1}."""
    return rng.standard_normal(n), rng.standard_normal(n - 1)


def single(case, seed):
    """Gates, chain coefficients and sampling seed of a one-circuit case."""
    rng = np.random.default_rng([int(seed), 1])
    gates = gates_of(case["circuit"], case["n"], case["layers"], rng)
    if case["kind"] == "torch" and case["dtype"] == "complex64":
        gates = [(k, c, t, tuple(float(np.float32(x)) for x in p)) for k, c, t, p in gates]
    a, b = chain(case["n"], rng)
    return gates, a, b, int(rng.integers(1 << 62))


def batch_of(case, seed):
    """[(n, gates, a, b)]: ansatz circuits of uneven qubit and layer counts.  The counts are spread evenly over their
    range whatever the seed, so that every seed is the same amount of work."""
    rng = np.random.default_rng([int(seed), 2])
    k = np.arange(case["count"])
    n = case["n_min"] + k % (case["n_max"] - case["n_min"] + 1)
    layers = case["layers_min"] + (k * 7) % (case["layers_max"] - case["layers_min"] + 1)
    out = []
    for i in rng.permutation(case["count"]):
        gates = gates_of("ansatz", int(n[i]), int(layers[i]), rng)
        out.append((int(n[i]), gates) + chain(int(n[i]), rng))
    return out


TABLE_WIRES = 8


def readout_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 3])
    wires = [int(q) for q in rng.choice(case["n"], TABLE_WIRES, replace=False)]
    return wires, rng.standard_normal(1 << TABLE_WIRES), int(rng.integers(1 << 62))


def near(gates, seed):
    """The same circuit at angles nearby: the state that a fidelity is taken with."""
    rng = np.random.default_rng([int(seed), 4])
    return [(k, c, t, tuple(x + 0.05 * rng.standard_normal() for x in p)) for k, c, t, p in gates]


def build(n, gates, dtype):
    c = Circuit(n, apply_method="gpu", dtype=dtype)
    for g in gates:
        c.add_gate(*g)
    return c


class Buffer:
    """A state's device buffer as torch sees it (2^n interleaved amplitudes in the state's own element order)."""

    def __init__(self, state, dtype):
        p, size = ctypes.c_void_p(), ctypes.c_uint64(0)
        N.call("dmv_state_device_ptr", state.handle, ctypes.byref(p), ctypes.byref(size))
        self.state = state  # keeps the buffer alive
        amp = AMP_BYTES[dtype]
        self.__cuda_array_interface__ = {"shape": (size.value // amp,), "typestr": "<c%d" % amp,
                                         "data": (p.value, False), "version": 3}


def view(state, dtype):
    return torch.as_tensor(Buffer(state, dtype), device="cuda")


def prepare(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "batch":
        return dict(kind=kind, dtype=dtype, batch=pack_circuits(batch_of(case, seed)))
    n = case["n"]
    gates, a, b, sampling = single(case, seed)
    c = build(n, gates, dtype)
    s = dict(kind=kind, dtype=dtype, circuit=c, a=a, b=b, pairs=[(q, q + 1) for q in range(n - 1)], seed=sampling)
    if kind == "gradient":
        s["theta"] = np.array([g[3][0] for g in gates if g[0] in (RX, RY, RZ)])
    elif kind == "torch":
        s["theta"] = torch.tensor([g[3][0] for g in gates if g[0] in (RX, RY, RZ)],
                                  dtype=torch.float32 if dtype == "complex64" else torch.float64, requires_grad=True)
    elif kind == "forward":
        s["view"] = view(c.state, dtype)
    elif kind == "readout":
        c.forward()
        other = build(n, near(gates, seed), dtype)
        other.forward()
        s["other"] = other.state
        s["wires"], s["table"], s["seed"] = readout_inputs(case, seed)
        s["samples"] = case["samples"]
    return s


# -------------------------------------------------------------------------------------------------------- the work --
def kept(dtype, x):
    """A double-precision result as the program keeps it."""
    return np.asarray(x, dtype=np.float32 if dtype == "complex64" else np.float64)


def run(s):
    kind, dtype = s["kind"], s["dtype"]
    if kind == "batch":
        energy, grad = batch_forward_adjoint_packed(s["batch"], dtype)
        return {"energy": kept(dtype, energy), "grad": kept(dtype, grad)}
    c = s["circuit"]
    if kind == "gradient":
        c.set_parameters(s["theta"])
        e, g = c.gradient(s["a"], s["pairs"], s["b"])
        return {"energy": kept(dtype, e), "grad": g}
    if kind == "torch":
        theta = s["theta"]
        theta.grad = None
        e = autograd.expectation(c, theta, s["a"], s["pairs"], s["b"])
        e.backward()
        return {"energy": e.detach(), "grad": theta.grad}
    if kind == "readout":
        v = c.state
        overlap = v.inner(s["other"])
        return {"z": kept(dtype, v.expect_z()), "energy": kept(dtype, v.expect_zz(s["a"], s["pairs"], s["b"])),
                "diag": kept(dtype, v.expect_diag(s["wires"], s["table"])), "norm": kept(dtype, v.norm_sqr()),
                "inner": kept(dtype, np.array([overlap.real, overlap.imag])),
                "samples": v.sample(s["samples"], s["seed"])}
    c.reset_amplitudes()
    c.forward()
    if kind == "forward":
        return {"z": kept(dtype, c.expectation_z()), "state": s["view"]}
    return {"probabilities": kept(dtype, c.measure()), "samples": c.sample(1000, seed=s["seed"]),
            "z": kept(dtype, c.expectation_z())}


def merged_one_qubit(gates):
    """One-qubit matrices and two-qubit gates that a circuit cannot do without: [uncontrolled, controlled]."""
    open_, ones, twos = set(), 0, 0
    for kind, control, target, _ in gates:
        if control < 0:
            ones += target not in open_
            open_.add(target)
        else:
            twos += 1
            open_ -= {control, target}
    return ones, twos


def forward_flops(gates, n):
    """28 operations a pair for every merged one-qubit matrix; X and CNOT move values only."""
    return merged_one_qubit(gates)[0] * 28 * 2.0 ** (n - 1)


def gradient_flops(gates, n):
    """The forward, the same on two states backwards, and 8 operations an amplitude for each angle's sum."""
    angles = sum(g[0] in (RX, RY, RZ) for g in gates)
    return 3 * forward_flops(gates, n) + angles * 8 * 2.0 ** n


def work(case):
    """The state is written once (and read once where it is read out); gates' operations, no passes between."""
    kind = case["kind"]
    if kind == "batch":
        bytes_ = flops = 0.0
        for n, gates, a, b in batch_of(case, 1):
            angles = sum(g[0] in (RX, RY, RZ) for g in gates)
            bytes_ += 16 * angles + 8 * (2 * n)
            flops += gradient_flops(gates, n)
        return {"bytes": bytes_, "flops": flops}
    n, amp = case["n"], AMP_BYTES[case["dtype"]]
    gates = single(case, 1)[0]
    angles = sum(g[0] in (RX, RY, RZ) for g in gates)
    if kind in ("gradient", "torch"):
        return {"bytes": 16.0 * angles + 16 * n, "flops": gradient_flops(gates, n)}
    if kind == "readout":
        return {"bytes": 2.0 * amp * 2 ** n + 8 * case["samples"], "flops": 16.0 * 2 ** n}
    if kind == "forward":
        return {"bytes": float(amp * 2 ** n + 8 * n), "flops": forward_flops(gates, n)}
    return {"bytes": 8.0 * 2 ** n + 8 * 1000 + 8 * n, "flops": forward_flops(gates, n) + 3.0 * 2 ** n}


# ---------------------------------------------------------------------------------------------- exact, in 64 bits --
# States are (circuits, 2^n) complex128 tensors, so that the circuits of a batch that have one size go together.
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def matrix(kind, p):
    """2x2 of a gate, per circuit: p is an array (circuits, angles)."""
    m = np.zeros((len(p), 2, 2), dtype=np.complex128)
    if kind == H:
        m[:] = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
        return m
    c, s = np.cos(p[:, 0] / 2), np.sin(p[:, 0] / 2)
    if kind == RX:
        m[:, 0, 0], m[:, 0, 1], m[:, 1, 0], m[:, 1, 1] = c, -1j * s, -1j * s, c
    elif kind == RY:
        m[:, 0, 0], m[:, 0, 1], m[:, 1, 0], m[:, 1, 1] = c, -s, s, c
    elif kind == RZ:
        m[:, 0, 0], m[:, 1, 1] = np.exp(-0.5j * p[:, 0]), np.exp(0.5j * p[:, 0])
    elif kind == U3:
        m[:, 0, 0], m[:, 0, 1] = c, -np.exp(1j * p[:, 2]) * s
        m[:, 1, 0], m[:, 1, 1] = np.exp(1j * p[:, 1]) * s, np.exp(1j * (p[:, 1] + p[:, 2])) * c
    return m


def apply_one(v, m, q):
    """m (circuits, 2, 2) on qubit q, in place."""
    w = v.view(v.shape[0], -1, 2, 1 << q)
    m = torch.from_numpy(m).to(v.device).view(-1, 2, 2, 1, 1)
    a, b = w[:, :, 0], w[:, :, 1]
    t = m[:, 0, 0] * a
    t.addcmul_(m[:, 0, 1].expand_as(b), b)
    b.mul_(m[:, 1, 1])
    b.addcmul_(m[:, 1, 0].expand_as(a), a)
    a.copy_(t)


def apply_two(v, kind, c, t):
    """CNOT or CZ, in place."""
    hi, lo = max(c, t), min(c, t)
    w = v.view(v.shape[0], -1, 2, 1 << (hi - lo - 1), 2, 1 << lo)
    if kind == CZ:
        w[:, :, 1, :, 1].neg_()
        return
    x, y = (w[:, :, 1, :, 0], w[:, :, 1, :, 1]) if c == hi else (w[:, :, 0, :, 1], w[:, :, 1, :, 1])
    z = x.clone()
    x.copy_(y)
    y.copy_(z)


def steps(gates):
    """(kind, control, target, angles) with runs of one-qubit gates on a qubit as one matrix: what forward needs."""
    out, last = [], {}
    for kind, control, target, p in gates:
        if control >= 0:
            last.pop(control, None)
            last.pop(target, None)
            out.append([kind, control, target, None])
            continue
        m = matrix(kind, p)
        if target in last:
            out[last[target]][3] = m @ out[last[target]][3]
        else:
            last[target] = len(out)
            out.append([None, -1, target, m])
    return out


def zero_state(count, n):
    v = torch.zeros(count, 1 << n, dtype=torch.complex128, device=DEVICE)
    v[:, 0] = 1
    return v


def simulate(gates, count, n):
    v = zero_state(count, n)
    for kind, c, t, m in steps(gates):
        if c < 0:
            apply_one(v, m, t)
        else:
            apply_two(v, kind, c, t)
    return v


def stacked(gates):
    """Gates of one circuit with their angles as (1, angles) arrays."""
    return [(k, c, t, np.array([p])) for k, c, t, p in gates]


def bit_signs(n, q, device):
    z = torch.ones(1 << n, dtype=torch.float64, device=device)
    z.view(-1, 2, 1 << q)[:, 1] = -1
    return z


def chain_energy(n, a, b):
    """h(x), per circuit: (circuits, 2^n)."""
    a, b = torch.from_numpy(np.atleast_2d(a)).to(DEVICE), torch.from_numpy(np.atleast_2d(b)).to(DEVICE)
    h = torch.zeros(a.shape[0], 1 << n, dtype=torch.float64, device=DEVICE)
    before = None
    for q in range(n):
        z = bit_signs(n, q, DEVICE)
        h += a[:, q:q + 1] * z
        if before is not None:
            h += b[:, q - 1:q] * (before * z)
        before = z
    return h


def energy_and_gradient(gates, n, a, b):
    """Of circuits of one shape: gates with (circuits, angles) arrays; (circuits,), (circuits, angles)."""
    count = len(np.atleast_2d(a))
    v = simulate(gates, count, n)
    h = chain_energy(n, a, b)
    energy = (h * (v.real ** 2 + v.imag ** 2)).sum(1)
    w = h * v
    both = torch.cat([v, w])
    v, w = both[:count], both[count:]
    del h
    grads = []
    for kind, c, t, p in reversed(gates):
        if c >= 0:
            apply_two(both, kind, c, t)
            continue
        if kind in (RX, RY, RZ):
            x, y = v.view(count, -1, 2, 1 << t), w.view(count, -1, 2, 1 << t)
            dot = lambda i, j: (y[:, :, i].conj() * x[:, :, j]).sum((1, 2))  # noqa: E731
            g = dot(0, 1) + dot(1, 0) if kind == RX else 1j * (dot(1, 0) - dot(0, 1)) if kind == RY else \
                dot(0, 0) - dot(1, 1)
            grads.append(g.imag)
        m = matrix(kind, p).conj().transpose(0, 2, 1).copy()
        apply_one(both, np.concatenate([m, m]), t)
    return energy, torch.stack(grads[::-1], 1)


def exact_batch(case, seed):
    circuits = batch_of(case, seed)
    energy, grads = [None] * len(circuits), [None] * len(circuits)
    groups = {}
    for i, (n, gates, a, b) in enumerate(circuits):
        groups.setdefault((n, len(gates)), []).append(i)
    for (n, count), which in groups.items():
        most = max(1, (1 << 27) >> n)
        for at in range(0, len(which), most):
            part = which[at:at + most]
            first = circuits[part[0]][1]
            gates = [(k, c, t, np.array([circuits[i][1][j][3] for i in part])) for j, (k, c, t, _) in enumerate(first)]
            e, g = energy_and_gradient(gates, n, np.array([circuits[i][2] for i in part]),
                                       np.array([circuits[i][3] for i in part]))
            for row, i in enumerate(part):
                energy[i], grads[i] = e[row], g[row]
    return {"energy": torch.stack(energy), "grad": torch.cat(grads)}


def element_order(v, n, dtype):
    """The amplitudes in the element order of a state's buffer (include/damavand_gpu.h, dmv_state_layout): in spans of
    2 MiB, element = amplitude ^ (P(span) << block)."""
    shift, block = (18, 7) if dtype == "complex64" else (17, 6)
    if n <= shift:
        return v
    out = torch.empty_like(v)
    low = torch.arange(1 << (shift - block), device=v.device)
    for s in range(1 << (n - shift)):
        p = 0
        for j in range(n - shift):
            p ^= ((s >> j) & 1) << ((7 * j) % 11)
        out[s << shift:(s + 1) << shift].view(-1, 1 << block)[low ^ p] = \
            v[s << shift:(s + 1) << shift].view(-1, 1 << block)
    return out


def all_z(prob, n):
    out = torch.empty(n, dtype=torch.float64, device=prob.device)
    for q in range(n):
        w = prob.view(-1, 2, 1 << q)
        out[q] = w[:, 0].sum() - w[:, 1].sum()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return exact_batch(case, seed)
    n = case["n"]
    gates, a, b, _ = single(case, seed)
    if kind in ("gradient", "torch"):
        e, g = energy_and_gradient(stacked(gates), n, a, b)
        return {"energy": e[0], "grad": g[0]}
    v = simulate(stacked(gates), 1, n)[0]
    if kind == "forward":
        z = all_z(v.real ** 2 + v.imag ** 2, n)
        return {"z": z, "state": element_order(v, n, case["dtype"])}
    prob = v.real ** 2 + v.imag ** 2
    if kind == "circuit":
        return {"probabilities": prob, "samples": None, "z": all_z(prob, n)}
    wires, table, _ = readout_inputs(case, seed)
    inner = torch.vdot(v, simulate(stacked(near(gates, seed)), 1, n)[0])
    del v
    h = torch.zeros_like(prob)
    index = torch.zeros(1 << n, dtype=torch.int32, device=prob.device)
    for j, q in enumerate(wires):
        index.view(-1, 2, 1 << q)[:, 1] += 1 << j
    h = torch.from_numpy(table).to(prob.device)[index.long()]
    diag = (h * prob).sum()
    del h, index
    energy = (chain_energy(n, a, b)[0] * prob).sum()
    return {"z": all_z(prob, n), "energy": energy, "diag": diag, "norm": prob.sum(),
            "inner": np.array([inner.real.item(), inner.imag.item()]), "samples": None}
