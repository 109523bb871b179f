"""How far a NaN or infinity in one row of an input reaches in the chunkwise kernels.  By the recurrence it reaches the
positions from its own on (of H, dQ) or up to its own (of dV, dK).  The kernels multiply whole tiles, in which what the
causal mask removes is a factor of zero, and zero times NaN is NaN: a tile holds at most 64 positions of the sequence on
either side of the diagonal.  The rows outside of the tile hold the very bits that they hold without the NaN."""
import pytest
import torch

from helpers import make_qkvif

pytestmark = pytest.mark.gpu

_TILE = 64


@pytest.mark.parametrize("B,NH,DQ,DV", [(1, 2, 64, 64), (1, 2, 128, 128), (1, 3, 128, 192), (2, 64, 128, 256), (1, 4, 256, 256),
                                        (2, 64, 256, 256), (1, 2, 256, 512), (2, 40, 256, 512), (1, 2, 256, 1024), (1, 2, 512, 1024),
                                        (2, 64, 512, 64), (1, 40, 192, 320)])
@pytest.mark.parametrize("S", [256, 384, 419])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_reach(B, NH, DQ, DV, S, dtype):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    print(f"{B}x{NH} S={S} {DQ}/{DV} {dtype}", flush=True)
    q, k, v, i, f = (t.cuda() for t in make_qkvif(B, NH, S, DQ, DV, seed=S, dtype=dtype))
    dH = torch.randn(B, NH, S, DV, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    bad = float("nan") if S % 2 else float("inf")

    def run(name=None, pos=0):
        x = dict(q=q, k=k, v=v, dH=dH)
        if name is not None:
            x[name] = x[name].clone()
            x[name][:, :, pos, 3] = bad
        leaves = [t.clone().requires_grad_(True) for t in (x["q"], x["k"], x["v"], i, f)]
        H = mlstm_chunkwise__hip_xl_chunk(*leaves, any_sequence_length=True)
        return H.detach(), *torch.autograd.grad(H, leaves[:3], x["dH"])

    clean = dict(zip(("H", "dQ", "dK", "dV"), run()))
    assert all(bool(torch.isfinite(t).all()) for t in clean.values())
    for pos in (5, 64, 100, 127, 128, 200, 255, S - 1):
        first, last = pos // _TILE * _TILE, (pos // _TILE + 1) * _TILE
        for name, before, after in (("v", ("H", "dQ"), ("dK",)), ("k", ("H", "dQ"), ()), ("q", (), ("dK", "dV")), ("dH", ("dQ",), ("dK", "dV"))):
            got = dict(zip(("H", "dQ", "dK", "dV"), run(name, pos)))
            for out in before:
                assert torch.equal(got[out][:, :, :first], clean[out][:, :, :first]), f"{name} at {pos} reaches back in {out}"
            for out in after:
                assert torch.equal(got[out][:, :, last:], clean[out][:, :, last:]), f"{name} at {pos} reaches on in {out}"
        reached = dict(zip(("H", "dQ", "dK", "dV"), run("v", pos)))["H"]
        assert not bool(torch.isfinite(reached[:, :, pos]).all())   # and where it belongs it is
