"""Calls after which the state's memory may be read from any stream: the tiled
executor and pl_sv_device_ptr with gates queued.  The engine's stream does not
order itself against others, so the amplitudes copied on torch's stream right
behind the call must be the ones the engine's own wait gives."""
import numpy as np
import pytest

from lightning_unification_amd.circuits import random_layers

pytestmark = pytest.mark.gpu


class _Memory:
    def __init__(self, sv, ptr):
        self.sv = sv
        self.__cuda_array_interface__ = {"shape": (sv.size,), "typestr": sv.dtype.str, "version": 3,
                                         "data": (ptr, False)}


@pytest.mark.parametrize("dtype,n", [(np.complex128, 25), (np.complex64, 22), (np.complex64, 24)])
@pytest.mark.parametrize("how", ["tiled", "deferred"])
def test_state_is_final_when_the_call_returns(dtype, n, how):
    import torch
    from lightning_unification_amd import capi
    tape = random_layers(n, 8, seed=3)
    print(f"final on return: {how} n={n} {np.dtype(dtype).name}", flush=True)
    with capi.DeviceStateVector(n, dtype) as sv:
        view = torch.as_tensor(_Memory(sv, sv.device_ptr()), device="cuda")
        view.clone()  # torch's allocation for the copy below
        torch.cuda.synchronize()
        if how == "tiled":
            sv.apply_tape_tiled(tape)
        else:
            sv.set_deferred(True)
            sv.apply_tape(tape)
            sv.device_ptr()
        got = view.clone()
        torch.cuda.synchronize()
        sv.synchronize()
        assert torch.equal(got, view)
        assert abs(float(torch.linalg.vector_norm(got.abs().double())) - 1) < 1e-4
