"""What the entry points make of the tensors and the stream they are handed: banks whose arrays are computed or strided give
the bytes that the plain bank gives, and all of a call's work is on the stream it is given."""
import threading

import numpy as np
import pytest
import torch

from tests.gpu_util import MCG, bytes_of, dev_f16_bits, dev_u16, make_x
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


class Handle:
    """A stream by its handle alone."""

    def __init__(self, stream):
        self.cuda_stream = stream.cuda_stream


@pytest.mark.parametrize("as_handle", [False, True])
def test_a_given_stream_carries_the_copies_and_the_scratch_too(oracle, t3, as_handle):
    """The current stream is busy for some 50 ms; calls on another stream copy strided operands, allocate and (in the threads'
    first call) clear a workspace, and are read when that stream alone is done."""
    rng = np.random.default_rng(0x57E)
    in_f, out_f = 1024, 512
    trellis, suh, svh = oracle.synth_linear(rng, in_f, out_f, 64)
    w = (dev_u16(trellis), dev_f16_bits(suh), dev_f16_bits(svh))
    bank = dev_bank(t3, oracle.synth_bank(rng, EXPERTS, HIDDEN, INTER, 48))
    dec = t3.Decode(MCG, 16)
    xl, _ = make_x(rng, 40, in_f, torch.float16)
    xm, _ = make_x(rng, 3, HIDDEN, torch.bfloat16)
    xm = xm.reshape(1, 3, HIDDEN)
    s, sc = routing(rng, 3, TOPK, EXPERTS)
    s, sc = torch.from_numpy(s).cuda().reshape(1, 3, TOPK), torch.from_numpy(sc).cuda().reshape(1, 3, TOPK)

    # the strided operands are there before the streams part: only the calls' own copies of them are in question
    xl1, xl, xm, s, sc, t = (strided(v) for v in (xl[:1], xl, xm, s, sc, w[0]))

    def calls(stream):
        return [t3.linear(xl1, *w, dec, stream=stream), t3.linear(xl, *w, dec, stream=stream),
                t3.moe(xm, bank, s, sc, dec, stream=stream), t3.moe_glm(xm, bank, s, dec, stream=stream),
                t3.linear_static(xl1, *w, dec, stream=stream), t3.dequant(t, dec, stream=stream),
                t3.unrot_weight(t, w[1], w[2], dec, stream=stream)[0]]

    want = [bytes_of(y) for y in calls(None)]
    torch.cuda.synchronize()
    got = []

    def worker():
        side = torch.cuda.Stream()
        torch.cuda._sleep(100_000_000)  # clock ticks: the current stream is behind from here on
        ys = calls(Handle(side) if as_handle else side)
        late = not torch.cuda.current_stream().query()
        side.synchronize()
        got.extend([late, *(y.to("cpu") for y in ys)])

    thread = threading.Thread(target=worker)
    thread.start()
    thread.join(60)
    torch.cuda.synchronize()
    assert got and got[0], "the current stream was done before the calls were made: nothing was shown"
    for i, (g, e) in enumerate(zip(got[1:], want)):
        assert bytes_of(g) == e, f"call {i}"
