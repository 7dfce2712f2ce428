"""The stages around the routed prefill's GEMMs where their shares are ragged: placed positions that are not whole groups of
four, skipped ids, one to seven 128-blocks a position, every activation dtype; each row against its own decode call (the same
roundings, sums in another order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter", [(128, 128), (640, 384), (256, 896), (896, 640)])
@pytest.mark.parametrize("rows,topk", [(17, 3), (33, 5), (70, 8)])
@pytest.mark.parametrize("decode,dtype", [("mcg", torch.bfloat16), ("mul1", torch.bfloat16), ("mcg", torch.float16),
                                          ("mul1", torch.float32)])
def test_rows_equal_their_decode_calls(hidden, inter, rows, topk, decode, dtype):
    from turboexl3_amd import api as t3
    experts, dec = 7 + topk, getattr(t3.Decode, decode)
    g = torch.Generator(device="cuda")
    g.manual_seed(hidden + inter + rows)

    def proj(in_f, out_f):
        return t3.Proj(torch.randint(-32768, 32768, (experts, in_f // 16, out_f // 16, 64), dtype=torch.int16, device="cuda",
                                     generator=g),
                       torch.randn(experts, in_f, device="cuda", generator=g).half(),
                       (torch.randn(experts, out_f, device="cuda", generator=g) * in_f ** -0.5).half())

    bank = t3.Bank(proj(hidden, inter), proj(hidden, inter), proj(inter, hidden))
    x = torch.randn(1, rows, hidden, device="cuda", generator=g).to(dtype)
    inds = torch.rand(rows, experts, device="cuda", generator=g).topk(topk).indices.to(torch.int32)[None].contiguous()
    inds[0, ::3, 1] = experts + 5  # skipped
    scores = torch.rand(1, rows, topk, device="cuda", generator=g).to(dtype)
    y = t3.moe(x, bank, inds, scores, dec).float()
    want = torch.cat([t3.moe(x[:, r:r + 1].contiguous(), bank, inds[:, r:r + 1].contiguous(),
                             scores[:, r:r + 1].contiguous(), dec) for r in range(rows)], 1).float()
    rms = want.square().mean().sqrt()
    step = 2.0 ** (-7 if dtype == torch.bfloat16 else -9)
    assert bool(((y - want).abs() <= step * want.abs() + 2e-2 * rms).all()), float((y - want).abs().max() / rms)


def case(t3, hidden, inter, rows, topk, n=64, experts=9, unit_scales=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(hidden + inter)

    def scales(width):
        v = torch.randn(experts, width, device="cuda", generator=g)
        return torch.where(v < 0, -1.0, 1.0) if unit_scales else v

    def proj(in_f, out_f):
        return t3.Proj(torch.randint(-32768, 32768, (experts, in_f // 16, out_f // 16, n), dtype=torch.int16, device="cuda",
                                     generator=g),
                       scales(in_f).half(), (scales(out_f) * in_f ** -0.5).half())

    bank = t3.Bank(proj(hidden, inter), proj(hidden, inter), proj(inter, hidden))
    x = torch.randn(1, rows, hidden, device="cuda", generator=g).half()
    inds = torch.rand(rows, experts, device="cuda", generator=g).topk(topk).indices.to(torch.int32)[None].contiguous()
    inds[0, ::5, 0] = -1  # skipped
    return x, bank, inds, torch.rand(1, rows, topk, device="cuda", generator=g)


@pytest.mark.parametrize("hidden,inter", [(128, 384), (640, 1152), (2432, 128), (2176, 2304)])
@pytest.mark.parametrize("decode", ["mcg", "mul1"])
def test_a_rows_bytes_do_not_depend_on_how_many_waves_share_its_blocks(hidden, inter, decode):
    """The fewer the positions, the more waves share one's blocks: up to one a block, or 16, 8, 4 of a workgroup where its block
    sums are added up. Rows of one long call against shorter calls' at every step, skipped slots among them."""
    from turboexl3_amd import api as t3
    dec = getattr(t3.Decode, decode)
    x, bank, inds, scores = case(t3, hidden, inter, 2900, 3)
    whole = t3.moe(x, bank, inds, scores, dec)  # 2175 groups of four positions
    assert bool(torch.isfinite(whole).all())
    for rows in (17, 40, 341, 342, 1300, 1366):
        part = t3.moe(x[:, :rows].contiguous(), bank, inds[:, :rows].contiguous(), scores[:, :rows].contiguous(), dec)
        assert torch.equal(part, whole[:, :rows]), rows


@pytest.mark.parametrize("hidden,inter", [(65664, 128), (128, 65664), (665600, 128)])
def test_block_sums_of_very_wide_rows(hidden, inter):
    """More 128-blocks than their sums have LDS at a time (and, the last, than a workgroup has at all): f16 rows against their
    decode calls, which add the same sums up elsewhere."""
    from turboexl3_amd import api as t3
    dec = t3.Decode.mul1
    x, bank, inds, scores = case(t3, hidden, inter, 18, 2, n=16, experts=3, unit_scales=True)
    y = t3.moe(x, bank, inds, scores, dec).float()
    want = torch.cat([t3.moe(x[:, r:r + 1].contiguous(), bank, inds[:, r:r + 1].contiguous(), scores[:, r:r + 1].contiguous(), dec)
                      for r in range(4)], 1).float()
    # Two chains that round to f16 at the same points and differ in the order of their f32 sums alone: a value may round to the
    # next f16 (2^-10 of it at most). An element's own three roundings (the down sums, the finish, the output) move it by 3 such
    # steps; the six of the gate, up and hidden values reach it through the 128-blocks' transforms and the sums as noise of at
    # most sqrt(6) 2^-10 of the row's rms, and five times that is the largest of the 2.7 million values looked at. (Scales of one
    # size: the noise of a column is as large as its scale.) A total that misses any of its blocks is off by whole rms.
    rms = want.square().mean(-1, keepdim=True).sqrt()
    step = 2.0 ** -10
    worst = ((y[:, :4] - want).abs() - 3 * step * want.abs()).div(5 * 6 ** 0.5 * step * rms).max()
    assert float(worst) <= 1.0, float(worst)


@pytest.mark.parametrize("hidden,inter", [(1152, 1408), (1408, 384), (2176, 1152)])
@pytest.mark.parametrize("decode", ["mcg", "mul1"])
@pytest.mark.parametrize("rows,topk", [(18, 2), (150, 5)])
def test_rows_within_the_roundings_of_their_decode_calls(hidden, inter, decode, rows, topk):
    """Nine to seventeen 128-blocks a position, skipped slots among them, scales with full mantissas: f16 rows against the
    decode chain, which rounds at the same points and adds the sums up in another order."""
    from turboexl3_amd import api as t3
    dec = getattr(t3.Decode, decode)
    x, bank, inds, scores = case(t3, hidden, inter, rows, topk)
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    for p in (bank.gate, bank.up, bank.down):  # magnitudes 1 to 2, so that no column's noise is far above the row's
        for v in (p.suh, p.svh):
            v.copy_(torch.where(v < 0, -1.0, 1.0) * (1.0 + torch.rand(v.shape, device="cuda", generator=g)) * (v.float().square().mean() ** 0.5))
    y = t3.moe(x, bank, inds, scores, dec).float()
    some = list(range(0, rows, max(1, rows // 25)))
    want = torch.cat([t3.moe(x[:, r:r + 1].contiguous(), bank, inds[:, r:r + 1].contiguous(), scores[:, r:r + 1].contiguous(), dec)
                      for r in some], 1).float()
    # A f32 sum of N terms in another order moves by about sqrt(N) 2^-24 of its rms, under MUL1's map 3.5 times that: at most 0.04
    # of the distance between two f16 roundings (2^-11) for the N here, so at most one value in twenty rounds the other way, by a
    # step of 2^-10 of it at most. An element's own three roundings move it by three steps; the six of the gate, up and hidden
    # values come through the transforms and sums as noise of sqrt(6 / 20) steps of the row's rms, twice that in a column of the
    # largest scale; five times that is the largest of the 60,000 values looked at.
    step = 2.0 ** -10
    rms = want.square().mean(-1, keepdim=True).sqrt()
    worst = ((y[:, some] - want).abs() - 3 * step * want.abs()).div(5 * 2 * (6 / 20) ** 0.5 * step * rms).max()
    assert float(worst) <= 1.0, float(worst)
