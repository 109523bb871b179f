"""Last states written over the initial ones (c_last = c0, n_last = n0, m_last = m0) through the C entry points."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _forward(S, DQ, DV, *, in_place, keep=0, path=0, NH=2, sig=False, noalloc=False, seed=0):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=dev, generator=g)
    q, k, v = rn(1, NH, S, DQ).bfloat16(), rn(1, NH, S, DQ).bfloat16(), rn(1, NH, S, DV).bfloat16()
    i, f = rn(1, NH, S), 3 + rn(1, NH, S)
    first = [rn(1, NH, DQ, DV), rn(1, NH, DQ), rn(1, NH)]
    last = first if in_place else [torch.empty_like(t) for t in first]
    H = torch.empty_like(v)
    head = [ptr(t) for t in (q, k, v, i, f, *first, H)] + [None, None] + [ptr(t) for t in last]
    tail = [1, NH, S, DQ, DV, 1e-6, _lib.BF16, _lib.F32, _lib.GATE_SIG if sig else _lib.GATE_EXP, 1]
    if noalloc:
        _lib.check(lib.mlstm_hip_chunkwise_fw_noalloc(*head, *tail, current_stream_ptr(dev)), "fw_noalloc")
    else:
        n = lib.mlstm_hip_chunkwise_fw_workspace_bytes(1, NH, S, DQ, DV, keep, path, 0)
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        _lib.check(lib.mlstm_hip_chunkwise_fw(*head, ptr(ws), n, keep, *tail, path, 0, _lib.NORM_NONE, 0.0, None, None,
                                              current_stream_ptr(dev)), "fw")
    torch.cuda.synchronize()
    return H, *last


# up to 512 positions: the bits of scan + H, which a forward that keeps its workspace for a backward takes at every length
@pytest.mark.parametrize("S", [1, 128, 317, 512])
@pytest.mark.parametrize("DQ,DV", [(64, 64), (256, 512)])
@pytest.mark.parametrize("sig,noalloc", [(False, False), (False, True), (True, False)])
def test_short_sequences(S, DQ, DV, sig, noalloc):
    got = _forward(S, DQ, DV, in_place=True, sig=sig, noalloc=noalloc, seed=S)
    ref = _forward(S, DQ, DV, in_place=False, sig=sig, keep=1, seed=S)
    for name, a, b in zip(("H", "C", "n", "m"), got, ref):
        assert torch.equal(a, b), name
