"""What the native binding makes of the tensors it is handed: banks whose arrays are computed or strided give the bytes that
the plain bank gives."""
import numpy as np
import pytest
import torch

from tests.gpu_util import MCG, bytes_of, make_x
from tests.test_gpu_moe import dev_bank, routing

pytestmark = pytest.mark.gpu

EXPERTS, HIDDEN, INTER, TOPK = 8, 512, 256, 4


@pytest.fixture(scope="module")
def t3():
    from turboexl3_amd import api
    return api


class Computed:
    """A bank (or a projection) whose attributes are copied to new memory at every access: the call is the only owner."""

    def __init__(self, of):
        self.of = of

    def __getattr__(self, name):
        v = getattr(self.of, name)
        return v.clone() if isinstance(v, torch.Tensor) else Computed(v)


def strided(t: torch.Tensor) -> torch.Tensor:
    """t's values as every second element of a wider array."""
    wide = torch.zeros(*t.shape, 2, dtype=t.dtype, device=t.device)
    wide[..., 0] = t
    return wide[..., 0]


@pytest.mark.parametrize("rows", [1, 3, 40])
def test_computed_and_strided_banks_give_the_plain_banks_bytes(oracle, t3, rows):
    rng = np.random.default_rng(0xB1D + rows)
    bank = dev_bank(t3, oracle.synth_bank(rng, EXPERTS, HIDDEN, INTER, 48))
    dec = t3.Decode(MCG, 16)
    x, _ = make_x(rng, rows, HIDDEN, torch.bfloat16)
    s, sc = routing(rng, rows, TOPK, EXPERTS)
    x, s, sc = (t.reshape(1, rows, -1) for t in (x, torch.from_numpy(s).cuda(), torch.from_numpy(sc).cuda()))
    want = bytes_of(t3.moe(x, bank, s, sc, dec))
    assert bytes_of(t3.moe(x, Computed(bank), s, sc, dec)) == want
    assert bytes_of(t3.moe(strided(x), t3.Bank(*(t3.Proj(*(strided(a) for a in (p.trellis, p.suh, p.svh)))
                                                for p in (bank.gate, bank.up, bank.down))), strided(s), strided(sc), dec)) == want
