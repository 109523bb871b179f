"""Last states written over the initial ones (c_last = c0, n_last = n0, m_last = m0) through the C entry points."""
import pytest
import torch

from helpers import rel_norm

pytestmark = pytest.mark.gpu


def _forward(S, DQ, DV, *, in_place, keep=0, path=0, NH=2, sig=False, normalize=1, noalloc=False, seed=0, f_offset=3.0, share="Cnm"):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=dev, generator=g)
    q, k, v = rn(1, NH, S, DQ).bfloat16(), rn(1, NH, S, DQ).bfloat16(), rn(1, NH, S, DV).bfloat16()
    i, f = rn(1, NH, S), f_offset + rn(1, NH, S)
    first = [rn(1, NH, DQ, DV), rn(1, NH, DQ), rn(1, NH)]
    last = [t if in_place and x in share else torch.empty_like(t) for t, x in zip(first, "Cnm")]
    H = torch.empty_like(v)
    head = [ptr(t) for t in (q, k, v, i, f, *first, H)] + [None, None] + [ptr(t) for t in last]
    tail = [1, NH, S, DQ, DV, 1e-6, _lib.BF16, _lib.F32, _lib.GATE_SIG if sig else _lib.GATE_EXP, normalize]
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


# m alone in place: the workgroups of the short kernel all read m0 and one writes m_last
@pytest.mark.parametrize("S", [50, 300, 512])
def test_short_sequences_stabiliser_only(S):
    got, ref = (_forward(S, 128, 128, in_place=p, seed=S, share="m") for p in (True, False))
    for name, a, b in zip(("H", "C", "n", "m"), got, ref):
        assert torch.equal(a, b), name


# the path of one kernel, whose workgroups of a head all read n0; and n that the operator leaves as it is: the same bits
@pytest.mark.parametrize("path,sig,normalize", [("fused", False, 1), ("fused", True, 0), ("auto", True, 0), ("split", False, 1)])
def test_named_paths(path, sig, normalize):
    from mlstm_kernels_amd import _lib

    got, ref = (_forward(700, 128, 256, in_place=p, path=_lib.path_code(path), sig=sig, normalize=normalize, NH=3) for p in (True, False))
    for name, a, b in zip(("H", "C", "n", "m"), got, ref):
        assert torch.equal(a, b), name


# a head's gates in several workgroups, all of which need the first m, and scan + H (with so many heads not in segments) either way:
# the same bits
@pytest.mark.parametrize("S", [2048, 2049, 4100])
@pytest.mark.parametrize("DQ,DV,NH", [(64, 64, 140), (256, 512, 20)])
def test_gates_of_several_workgroups(S, DQ, DV, NH):
    got, ref = (_forward(S, DQ, DV, in_place=p, NH=NH, seed=S, f_offset=12.0) for p in (True, False))
    for name, a, b in zip(("H", "C", "n", "m"), got, ref):
        assert torch.equal(a, b), name


# Few heads and a long sequence: the scan in segments, which all read the initial state, is not taken in place.  The states are
# those of the scan in one piece (which a named path takes), H that of separate buffers but for the order of a sum in fp32.  Gates
# near one: the initial state still weighs at the end.
@pytest.mark.parametrize("S,DQ,DV,NH", [(8192, 128, 128, 2), (8200, 256, 512, 1), (2048, 64, 64, 12), (4100, 64, 64, 12), (2049, 128, 64, 32),
                                          (8200, 256, 512, 4), (8192, 128, 128, 8), (6016, 64, 256, 12)])
@pytest.mark.parametrize("sig", [False, True])
def test_long_sequences_of_few_heads(S, DQ, DV, NH, sig):
    kw = dict(NH=NH, sig=sig, seed=S, f_offset=12.0, share="Cn")
    H, C, n, _ = _forward(S, DQ, DV, in_place=True, **kw)
    _, C1, n1, _ = _forward(S, DQ, DV, in_place=False, path=_split(), **kw)
    H2, C2, n2, _ = _forward(S, DQ, DV, in_place=False, **kw)
    assert torch.equal(C, C1) and torch.equal(n, n1)
    # sums of 64 chunks in fp32 in another order: 64 * 2^-24, and room for the chunk states' own rounding to 16 bits in H
    assert rel_norm(C, C2) <= 1e-5 and rel_norm(n, n2) <= 1e-5 and rel_norm(H, H2) <= 2 ** -9


def _split():
    from mlstm_kernels_amd import _lib

    return _lib.PATH_SPLIT


def test_backward_of_few_heads():
    """dC0 over dC_last: the bits of the scan in one piece (behind the same forward, whose row normalisers it reads)."""
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    NH, S, D = 2, 8192, 128
    g = torch.Generator(device=dev).manual_seed(5)
    rn = lambda *s: torch.randn(*s, device=dev, generator=g)
    q, k, v, dH = (rn(1, NH, S, D).bfloat16() for _ in range(4))
    i, f = rn(1, NH, S), 12 + rn(1, NH, S)
    d_last = rn(1, NH, D, D)
    out = {}
    for path in (_lib.PATH_SPLIT, _lib.PATH_AUTO):
        H = torch.empty_like(v)
        n = lib.mlstm_hip_chunkwise_fw_workspace_bytes(1, NH, S, D, D, 1, _lib.PATH_SPLIT, 0)
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        _lib.check(lib.mlstm_hip_chunkwise_fw(*[ptr(t) for t in (q, k, v, i, f)], None, None, None, ptr(H), *[None] * 5, ptr(ws), n, 1,
                                              1, NH, S, D, D, 1e-6, _lib.BF16, _lib.F32, _lib.GATE_EXP, 1, _lib.PATH_SPLIT, 0, _lib.NORM_NONE,
                                              0.0, None, None, current_stream_ptr(dev)), "fw")
        nb = lib.mlstm_hip_chunkwise_bw_workspace_bytes(1, NH, S, D, D, 0)
        bws = torch.empty(nb, dtype=torch.uint8, device=dev)
        dC = d_last.clone()
        dC0 = dC if path == _lib.PATH_AUTO else torch.empty_like(dC)
        grads = [torch.empty_like(t) for t in (q, k, v)] + [torch.empty_like(t) for t in (i, f)]
        _lib.check(lib.mlstm_hip_chunkwise_bw(*[ptr(t) for t in (q, k, v, i, f, dH, dC, *grads, dC0, ws)], n, ptr(bws), nb, 1, NH, S, D,
                                              D, 1e-6, _lib.BF16, _lib.F32, _lib.GATE_EXP, 1, path, 0, current_stream_ptr(dev)), "bw")
        torch.cuda.synchronize()
        out[path] = (dC0, *grads)
    a, b = out[_lib.PATH_AUTO], out[_lib.PATH_SPLIT]
    assert torch.equal(a[0], b[0])
    for name, x, y in zip(("dQ", "dK", "dV"), a[1:], b[1:]):
        assert rel_norm(x, y) <= 1e-2, name  # other kernels behind the scan: the bf16 tolerance of the operands
