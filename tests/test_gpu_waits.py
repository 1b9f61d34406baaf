"""Waits that calls owe their callers.

Calls after which the state's memory may be read from any stream: the tiled
executor and pl_sv_device_ptr with gates queued.  The engine's stream does not
order itself against others, so the amplitudes copied on the null stream right
behind the call must be the ones the engine's own wait gives.

Calls that refuse their input with a copy of the caller's memory queued: the
next call on the handle gives the oracle's result."""
import numpy as np
import pytest

from conftest import random_state, rel_err
from lightning_unification_amd.circuits import Tape, random_layers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,n", [(np.complex128, 25), (np.complex64, 22), (np.complex64, 24)])
@pytest.mark.parametrize("how", ["tiled", "deferred"])
def test_state_is_final_when_the_call_returns(dtype, n, how):
    import ctypes
    from lightning_unification_amd import capi
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    tape = random_layers(n, 8, seed=3)
    print(f"final on return: {how} n={n} {np.dtype(dtype).name}", flush=True)
    with capi.DeviceStateVector(n, dtype) as sv, capi.DeviceStateVector(n, dtype) as copy:
        to = copy.device_ptr()
        copy.synchronize()
        at = sv.device_ptr()
        if how == "tiled":
            sv.apply_tape_tiled(tape)
        else:
            sv.set_deferred(True)
            sv.apply_tape(tape)
            at = sv.device_ptr()
        # on the null stream, which the engine's streams do not wait for
        assert hip.hipMemcpy(to, at, sv.size * np.dtype(dtype).itemsize, 3) == 0  # hipMemcpyDeviceToDevice
        assert hip.hipDeviceSynchronize() == 0
        assert copy.distance(sv) == 0
        assert abs(copy.norm2() - 1) < 1e-4


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_vjp_that_refuses_its_tape_has_finished_its_upload(oracle, dtype):
    from lightning_unification_amd import capi
    n = 15
    good, bad, wrong = Tape(), Tape(), Tape()
    for w in range(n):
        good.add("RX", [w], [0.1 + w])
    bad.add("Rot", [0], [0.1, 0.2, 0.3])  # more than one parameter
    bad.ops += good.ops
    wrong.ops = [("RY", [n], False, [0.3])] + list(good.ops)  # no such wire
    tol = 1e-12 if dtype == np.complex128 else 5e-5
    s, dy = random_state(n, 1, dtype), random_state(n, 2, dtype)
    with capi.DeviceStateVector.from_array(s) as sv:
        for tape in (bad, wrong):
            with pytest.raises(ValueError):
                sv.vjp(tape, random_state(n, 3, dtype), list(range(n + 1)))
            got = sv.vjp(good, dy, list(range(n)))
            exp = oracle.vjp(s.astype(np.complex128), good, dy.astype(np.complex128), list(range(n)))
            assert rel_err(got, exp) < tol


def test_tapes_run_ahead_of_the_device():
    """A tape's call does not wait for the tape before it: three queued behind
    each other take a fraction of their run time to submit, and many short ones,
    whose programs go round the upload ring several times, give the oracle's state."""
    import time
    from lightning_unification_amd import capi
    tape = random_layers(28, 4, seed=6)
    with capi.DeviceStateVector(28) as sv:
        sv.apply_tape(tape)
        sv.synchronize()
        t0 = time.perf_counter()
        for _ in range(3):
            sv.apply_tape(tape)
        queued = time.perf_counter() - t0
        sv.synchronize()
        assert queued < 0.5 * (time.perf_counter() - t0)


@pytest.mark.parametrize("n,layers,times", [(6, 2, 60), (12, 25, 4), (14, 120, 2)])
def test_programs_round_the_ring(oracle, n, layers, times):
    """Short programs many times round the ring, and tapes whose programs grow it."""
    from lightning_unification_amd import capi
    s = random_state(n, 3)
    exp = s.copy()
    with capi.DeviceStateVector.from_array(s) as sv:
        for i in range(times):
            tape = random_layers(n, layers, seed=i)
            sv.apply_tape(tape)
            oracle.apply_tape(exp, tape)
        assert rel_err(sv.state(), exp, floor=0.1) < 1e-12 * times


def test_a_handle_per_circuit_in_several_threads(oracle):
    """Handles that come and go take over the upload ring and the pinned area of
    earlier ones; four threads at once, tapes that grow the ring among them,
    give the oracle's states and expectation values."""
    from concurrent.futures import ThreadPoolExecutor
    from lightning_unification_amd import capi
    from lightning_unification_amd.circuits import random_hamiltonian

    def circuit(i):
        n = 4 + i % 9
        tape, ham = random_layers(n, 40 if i % 8 == 7 else 2, seed=i), random_hamiltonian(n, 6, seed=i)
        exp = np.zeros(1 << n, np.complex128)
        exp[0] = 1
        oracle.apply_tape(exp, tape)
        with capi.DeviceStateVector(n) as sv:
            sv.apply_tape(tape)
            e = sv.expval(ham)
            return rel_err(sv.state(), exp, floor=0.1), abs(e - oracle.expval(exp, ham))

    with ThreadPoolExecutor(4) as pool:
        for err, de in pool.map(circuit, range(64)):
            assert err < 1e-12 and de < 1e-12
