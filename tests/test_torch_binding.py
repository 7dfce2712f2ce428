"""The native side of the Python entry points refuses what it cannot describe before it calls the library, with the same
exceptions whichever entry point takes the tensor, and holds every tensor it read until the call is over (no GPU: nothing
gets as far as a launch)."""
import gc
import weakref

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from turboexl3_amd import api


def call(entry, x):
    t = torch.zeros(8, 8, 64, dtype=torch.int16)
    v = torch.ones(128, dtype=torch.float16)
    bank = api.Bank(*(api.Proj(t[None], v[None], v[None]) for _ in range(3)))
    inds = torch.zeros(1, 1, 2, dtype=torch.int32)
    if entry == "linear":
        return api.linear(x, t, v, v)
    if entry == "unrot":
        return api.linear_unrot_parts(x, torch.zeros(128, 128))
    return api.moe(x, bank, inds, inds.float())


@pytest.mark.parametrize("entry", ["linear", "unrot", "moe"])
@pytest.mark.parametrize("x,error,name", [
    (3.0, TypeError, None),
    (torch.zeros(1, 1, 128), ValueError, None),                          # host memory
    (torch.zeros(1, 1, 128, dtype=torch.float64), api.T3Error, "BadExl3Dtype"),
    (torch.zeros([1] * 8 + [128]), api.T3Error, "BadExl3Shape"),         # nine dimensions
])
def test_tensors_the_library_cannot_take_are_refused(entry, x, error, name):
    with pytest.raises(error) as e:
        call(entry, x)
    if name:
        assert e.value.name == name


class Looked(Exception):
    """Ends a call once its tensors have been looked at."""


@pytest.mark.parametrize("entry", ["moe", "moe_shared_expert", "moe_fused_shared", "moe_fused_shared_routed"])
@pytest.mark.filterwarnings("ignore::DeprecationWarning", "ignore::UserWarning")
def test_computed_bank_attributes_are_held_for_the_call(entry):
    """A bank whose attributes make a new tensor at every access: each must still be alive when the call goes on to read its
    `dec` (device tensors without a device: the call ends there)."""
    with FakeTensorMode():
        def fake(*shape, dtype):
            return torch.empty(shape, dtype=dtype, device="cuda")

        made = []

        class Fresh:
            def __getattr__(self, name):
                if name in ("gate", "up", "down"):
                    return Fresh()
                t = fake(4, 8, 8, 64, dtype=torch.int16) if name == "trellis" else fake(4, 128, dtype=torch.float16)
                made.append(weakref.ref(t))
                return t

        class Dec:
            window_bits = 16

            @property
            def codebook(self):
                gc.collect()
                raise Looked(sum(r() is not None for r in made))

        x, v = fake(1, 1, 128, dtype=torch.float16), fake(1, dtype=torch.float16)
        inds, scores = fake(1, 1, 2, dtype=torch.int32), fake(1, 1, 2, dtype=torch.float32)
        banks = {"moe": 1}.get(entry, 2)
        with pytest.raises(Looked) as e:
            if entry == "moe":
                api.moe(x, Fresh(), inds, scores, Dec())
            elif entry == "moe_shared_expert":
                api.moe_shared_expert(x, Fresh(), inds, scores, Dec(), 0, Fresh())
            elif entry == "moe_fused_shared":
                api.moe_fused_shared(x, Fresh(), inds, scores, Dec(), Fresh(), v, v)
            else:
                api.moe_fused_shared_routed(x, Fresh(), scores, 2, Dec(), Fresh(), v, v)
        assert len(made) == 9 * banks and e.value.args[0] == len(made)
