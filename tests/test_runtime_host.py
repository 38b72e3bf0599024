"""The library's host code against a HIP runtime without a GPU
(tests/hip_stand_in.cpp): what is left after a refused allocation, and how much
memory a call asks for.  Each test runs in a process of its own, since the
stand-in has to be loaded before the library."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes, sys
S = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
for name in ("stand_in_launches", "stand_in_bad_launches", "stand_in_peak", "stand_in_reset_peak"):
    getattr(S, name).restype = ctypes.c_int64
S.stand_in_capacity.argtypes = [ctypes.c_uint64]
import numpy as np
from damavand_amd import _native as N, workloads as wl
from damavand_amd.circuit import Circuit

def build(n, gates, dtype="complex128"):
    c = Circuit(n, dtype=dtype)
    for g in gates:
        c.add_gate(*g)
    return c
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("hip") / "stand_in.so")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", os.path.join(ROOT, "tests", "hip_stand_in.cpp"), "-o", lib],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return lib


def run(stand_in, code, *args):
    env = {k: v for k, v in os.environ.items() if not k.startswith("DMV_")}
    env["PYTHONPATH"] = ROOT
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, stand_in, *args], env=env, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("adjoint", [0, 1])
def test_refused_allocation_leaves_no_plan(stand_in, adjoint):
    """Gates are added, an allocation of the new plan is refused, and the call is made again: the passes and phases
    that it launches are the new plan's, on the device."""
    run(stand_in, r"""
adjoint = int(sys.argv[2])
refused = 0
live = S.stand_in_reset_peak()
for nth in range(1, 30):
    c = build(16, wl.layered_circuit(16, 1, 1))
    work = (lambda: c.gradient(np.ones(16))) if adjoint else c.forward
    work()
    for g in wl.layered_circuit(16, 6, 2):
        c.add_gate(*g)
    S.stand_in_fail_malloc(nth)
    try:
        work()
        done = True
    except N.OutOfDeviceMemory:
        done = False
    S.stand_in_fail_malloc(0)
    before = S.stand_in_launches()
    work()
    again = S.stand_in_launches() - before
    fresh = build(16, wl.layered_circuit(16, 1, 1) + wl.layered_circuit(16, 6, 2))
    (fresh.gradient(np.ones(16)) if adjoint else fresh.forward())
    assert S.stand_in_bad_launches() == 0, nth
    assert c.plan_stats() == fresh.plan_stats()
    refused += not done
    del c, fresh, work
    assert S.stand_in_reset_peak() == live, "device memory left behind"
    if done:
        break
assert done and refused >= 2
""", str(adjoint))


def test_refused_allocation_leaves_no_buffer_size(stand_in):
    """A workspace that could not grow is gone with its size: what needs less of it afterwards allocates it again."""
    run(stand_in, r"""
refused = 0
a, few, many = np.ones(16), [(0, 1)], [(q, q + 1) for q in range(15)]
for nth in range(1, 30):
    c = build(16, wl.layered_circuit(16, 1, 1))
    c.gradient(a, few, np.ones(1))
    c.expectation(a, few, np.ones(1))
    for g in wl.layered_circuit(16, 6, 2):
        c.add_gate(*g)
    S.stand_in_fail_malloc(nth)
    for work in (lambda: c.gradient(a, many, np.ones(15)), lambda: c.expectation(a, many, np.ones(15))):
        try:
            work()
        except N.OutOfDeviceMemory:
            refused += 1
    S.stand_in_fail_malloc(0)
    c.reset()
    for g in wl.layered_circuit(16, 1, 1):
        c.add_gate(*g)
    c.gradient(a, few, np.ones(1))
    c.expectation(a, few, np.ones(1))
    assert S.stand_in_bad_launches() == 0, nth
    if refused < nth:
        break
assert refused >= 5
""")


def test_no_pinned_memory(stand_in):
    """Copies that go through pinned memory for speed are made without it where there is none."""
    run(stand_in, r"""
S.stand_in_fail_host(1)
c = build(16, wl.layered_circuit(16, 2, 1))
c.forward()
c.expectation(np.ones(16), [(0, 1)], np.ones(1))
c.state.expect_diag([1, 3], np.ones(4))
c.gradient(np.ones(16))
c.set_parameters(np.zeros(c.num_parameters))
c.gradient(np.ones(16))
assert S.stand_in_bad_launches() == 0
""")


BRICKWORK = r"""
def brickwork(n, layers):
    rng = np.random.default_rng(n)
    gates = []
    for layer in range(layers):
        for kind in (wl.GATE_RX, wl.GATE_RY, wl.GATE_RZ):
            gates += [(kind, -1, q, (t,)) for q, t in enumerate(rng.uniform(0, 6, n))]
        gates += [(wl.GATE_CZ, q, q + 1, ()) for q in range(layer % 2, n - 1, 2)]
    return gates
"""


def test_gradient_of_the_largest_states_fits(stand_in):
    """33 qubits: two states of 128 GiB and the partials of 1980 angles on a card of 288 GiB."""
    run(stand_in, BRICKWORK + r"""
from tests.libhelpers import NativeCircuit
n = 33
c = NativeCircuit(n, brickwork(n, 20))
psi, lam, e = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_double(0)
N.call("dmv_state_create", n, N.C128, ctypes.byref(psi))
N.call("dmv_state_create", n, N.C128, ctypes.byref(lam))
a, g = np.ones(n), np.empty(3 * 20 * n)
before = S.stand_in_reset_peak()
N.call("dmv_circuit_adjoint", c.h, psi, lam, N.dptr(a), 0, None, None, None, ctypes.byref(e), N.dptr(g))
assert S.stand_in_bad_launches() == 0
assert S.stand_in_peak() - before <= (1 << n) + (1 << 20)  # the partials: a byte an amplitude
""")


@pytest.mark.parametrize("mib", [40, 16, 6])
def test_gradient_plans_for_the_memory_there_is(stand_in, mib):
    """24 qubits, where the widest pass would take 79 MiB of partials, with less than that left on the device."""
    run(stand_in, BRICKWORK + r"""
n, left = 24, int(sys.argv[2]) << 20
c = build(n, brickwork(n, 20))
c._scratch = (c.state, build(n, []).state)
c.forward()
S.stand_in_capacity(S.stand_in_reset_peak() + left)
for _ in range(2):
    c.gradient(np.ones(n))
    c.set_parameters(np.zeros(c.num_parameters))
assert S.stand_in_bad_launches() == 0
""", str(mib))


@pytest.mark.parametrize("n,layers,dtype", [(30, 5, "complex128"), (20, 4, "complex128"), (14, 4, "complex128"),
                                            (10, 2, "complex128"), (20, 3, "complex64")])
def test_autotuner_can_keep_the_default(stand_in, tmp_path, n, layers, dtype):
    """Where every launch takes as long, tuning chooses no plan with more launches than the default's, and another
    process that reads the choice from the file makes that plan."""
    run(stand_in, r"""
import os
n, layers, dtype = int(sys.argv[2]), int(sys.argv[3]), sys.argv[4]
gates = wl.layered_circuit(n, layers, 1)

def forward_launches(c):
    before = S.stand_in_launches()
    c.forward()
    return S.stand_in_launches() - before

default = forward_launches(build(n, gates, dtype))
os.environ["DMV_TUNE_CACHE"] = sys.argv[5]
N.call("dmv_tune_forget")
c = build(n, gates, dtype)
k = c.autotune()
shape = c.tile_shape()
assert k == shape["tile_qubits"] and k <= n
tuned = forward_launches(c)
assert tuned <= default, (tuned, default, shape)
N.call("dmv_tune_forget")
fresh = build(n, gates, dtype)
assert fresh.tile_shape() == shape and forward_launches(fresh) == tuned
""", str(n), str(layers), dtype, str(tmp_path / "tune.jsonl"))


@pytest.mark.parametrize("n,dtype", [(23, "complex128"), (13, "complex128"), (10, "complex128"), (12, "complex64")])
def test_adjoint_autotuner_can_keep_the_default(stand_in, n, dtype):
    run(stand_in, r"""
n, dtype = int(sys.argv[2]), sys.argv[3]
gates = wl.layered_circuit(n, 4, 1)

def launches(c):
    c.gradient(np.ones(n))
    before = S.stand_in_launches()
    c.gradient(np.ones(n))
    return S.stand_in_launches() - before

default = launches(build(n, gates, dtype))
c = build(n, gates, dtype)
k = c.autotune(adjoint=True)
assert k == c.tile_shape(adjoint=True)["tile_qubits"] and 9 <= k <= n
assert launches(c) <= default, (launches(c), default)
""", str(n), dtype)


@pytest.mark.parametrize("n", [9, 10, 11])
def test_tuning_entry_larger_than_the_state(stand_in, tmp_path, n):
    """An entry whose tile is larger than the state does not apply (it never did at these sizes)."""
    (tmp_path / "tune.jsonl").write_text("".join(
        '{"key": "gfx950/n%d/c128/%s", "tile_qubits": 12, "threads_log2": 8, "max_gen_per_pass": 8}\n' % (n, kind)
        for kind in ("forward", "adjoint")))
    run(stand_in, r"""
import os
os.environ["DMV_TUNE_CACHE"] = sys.argv[2]
n = int(sys.argv[3])
c = build(n, wl.layered_circuit(n, 2, 1))
c.forward()
c.gradient(np.ones(n))
""", str(tmp_path / "tune.jsonl"), str(n))


def test_batch_takes_the_memory_there_is(stand_in):
    """64 circuits that take 20 MiB together, with more and more left on the device."""
    run(stand_in, r"""
from damavand_amd import batch_forward_adjoint
circuits = wl.batch_workload(64, 5, n_range=(12, 14), layer_range=(2, 4))
N.synchronize()
S.stand_in_capacity(1 << 18)  # not even room for one circuit
try:
    batch_forward_adjoint(circuits)
    assert False
except N.OutOfDeviceMemory:
    pass
launches = []
for mib in (3, 8, 16, 64):
    S.stand_in_capacity(mib << 20)
    before = S.stand_in_launches()
    batch_forward_adjoint(circuits)
    launches.append(S.stand_in_launches() - before)
assert S.stand_in_bad_launches() == 0
assert launches[0] > launches[1] > launches[2] > launches[3], launches
""")


def test_batch_without_threads():
    """The host threads of a batch are a matter of speed: none can be made here, since their stacks exceed the address
    space that is left.  (No stand-in: the call ends when it finds no GPU.)"""
    code = r"""
import resource
from damavand_amd import _native as N, workloads as wl, batch_forward_adjoint
circuits = wl.batch_workload(64, 5, n_range=(3, 5), layer_range=(1, 2))
N.device_count()
size = next(int(l.split()[1]) for l in open("/proc/self/status") if l.startswith("VmSize")) << 10
resource.setrlimit(resource.RLIMIT_AS, (size + (6 << 20),) * 2)
try:
    batch_forward_adjoint(circuits)
except N.NoDeviceError:
    pass
"""
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, PYTHONPATH=ROOT, HIP_VISIBLE_DEVICES="-1"),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
