"""Operands and outputs that begin at an odd element: contiguous views, and buffers of a C caller.  Kernels that move rows to LDS
without registers in between or store 16 bytes at a time through the caches leave such calls to the others."""
import pytest
import torch

from helpers import rel_norm

pytestmark = pytest.mark.gpu


def _moved(t):
    """The same values in memory that is aligned to one element only."""
    x = torch.cat([t.new_zeros(1), t.detach().flatten()])[1:].view(t.shape)
    assert x.is_contiguous() and x.data_ptr() % 16 == t.element_size()
    return x


@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (128, 256, 256), (256, 512, 256)])
@pytest.mark.parametrize("moved", ["q", "k", "v", "dH", "all"])
@pytest.mark.parametrize("recompute", [False, True])
def test_rows(DQ, DV, width, moved, recompute):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    S, BH = 330, torch.cuda.get_device_properties(0).multi_processor_count // (DV // width)
    print(f"{BH} x {S} {DQ}/{DV} {moved}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(DQ)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = dict(q=rn(S, DQ).bfloat16(), k=rn(S, DQ).bfloat16(), v=rn(S, DV).bfloat16(), i=rn(S), f=3 + rn(S), dH=rn(S, DV).bfloat16())
    out = []
    for which in ("", moved):
        y = {n: _moved(t) if n != "i" and n != "f" and which in (n, "all") else t.clone() for n, t in x.items()}
        leaves = [y[n].requires_grad_(True) for n in ("q", "k", "v", "i", "f")]
        _lib.profile_read()
        _lib.profile_enable(True)
        try:
            H = mlstm_chunkwise__hip_xl_chunk(*leaves, any_sequence_length=True, recompute_states_in_bw=recompute)
            out.append((H.detach(), *torch.autograd.grad(H, leaves, y["dH"])))
        finally:
            _lib.profile_enable(False)
        names = set(_lib.profile_read())
        assert ("chain_h" in names) == (which in ("", "dH")) and ("chain_dv" in names) == (which in ("", "v"))
    for name, a, b in zip(("H", "dQ", "dK", "dV", "dI", "dF"), *out):
        # two ways of rounding the same operands to 16 bits: each is within 6e-3 (8e-3 with the gates' sums) of the exact result
        assert rel_norm(b, a) <= (8e-3 if name[1:] in ("I", "F") else 6e-3) * 2 ** 0.5, name


# H and dV of a C caller in memory that is aligned to one element: the other kernels, and nothing beside the rows is written
@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (128, 256, 256), (256, 512, 256)])
@pytest.mark.parametrize("moved", ["H", "dV"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_output_rows(DQ, DV, width, moved, dtype):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    S, BH = 330, torch.cuda.get_device_properties(0).multi_processor_count // (DV // width)
    print(f"{BH} x {S} {DQ}/{DV} {moved} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(DQ)
    rn = lambda *s: torch.randn(1, BH, *s, device=dev, generator=g)
    q, k, v, dH = (rn(S, d).to(dtype) for d in (DQ, DQ, DV, DV))
    i, f = rn(S), 3 + rn(S)
    code = _lib.F16 if dtype == torch.float16 else _lib.BF16
    nf = lib.mlstm_hip_chunkwise_fw_workspace_bytes(1, BH, S, DQ, DV, 1, _lib.PATH_AUTO, 0)
    nb = lib.mlstm_hip_chunkwise_bw_workspace_bytes(1, BH, S, DQ, DV, 0)

    def output(odd):  # a buffer of ones and the rows in it
        buf = torch.ones(v.numel() + 16, dtype=dtype, device=dev)
        return buf, buf[1 if odd else 8:][:v.numel()].view(v.shape)

    out = []
    for which in ("", moved):
        (bh, H), (bv, dV) = output(which == "H"), output(which == "dV")
        assert (H.data_ptr() % 16 == 0) == (which != "H") and (dV.data_ptr() % 16 == 0) == (which != "dV")
        ws, bws = (torch.empty(n, dtype=torch.uint8, device=dev) for n in (nf, nb))
        dQ, dK, dI, dF = torch.empty_like(q), torch.empty_like(k), torch.empty_like(i), torch.empty_like(f)
        _lib.profile_read()
        _lib.profile_enable(True)
        try:
            _lib.check(lib.mlstm_hip_chunkwise_fw(*[ptr(t) for t in (q, k, v, i, f)], None, None, None, ptr(H), *[None] * 5, ptr(ws), nf, 1,
                                                  1, BH, S, DQ, DV, 1e-6, code, _lib.F32, _lib.GATE_EXP, 1, _lib.PATH_AUTO, 0, _lib.NORM_NONE,
                                                  1e-6, None, None, current_stream_ptr(dev)), "forward")
            _lib.check(lib.mlstm_hip_chunkwise_bw(*[ptr(t) for t in (q, k, v, i, f, dH)], None, *[ptr(t) for t in (dQ, dK, dV, dI, dF)], None,
                                                  ptr(ws), nf, ptr(bws), nb, 1, BH, S, DQ, DV, 1e-6, code, _lib.F32, _lib.GATE_EXP, 1,
                                                  _lib.PATH_AUTO, 0, current_stream_ptr(dev)), "backward")
            torch.cuda.synchronize()
        finally:
            _lib.profile_enable(False)
        names = set(_lib.profile_read())
        assert ("chain_h" in names) == (which != "H") and ("chain_dv" in names) == (which != "dV")
        for buf, rows in ((bh, H), (bv, dV)):
            first = (rows.data_ptr() - buf.data_ptr()) // buf.element_size()
            assert bool((buf[:first] == 1).all()) and bool((buf[first + rows.numel():] == 1).all())
        out.append((H, dV, dQ, dK))
    tol = (0.25 if dtype == torch.float16 else 1.0) * 6e-3 * 2 ** 0.5  # (as above)
    for name, a, b in zip(("H", "dV", "dQ", "dK"), *out):
        assert rel_norm(b, a) <= tol, name


# a state between 32 and 112 MiB, whose stores go through the caches where they can
@pytest.mark.parametrize("in_place", [False, True])
def test_step_state(in_place):
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_step__hip_fw

    n, DQ, DV = 400, 128, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    rn = lambda *s: torch.randn(n, 1, *s, device="cuda", generator=g)
    x = [rn(DQ).bfloat16(), rn(DQ).bfloat16(), rn(DV).bfloat16(), rn(1), 3 + rn(1)]
    st = [rn(DQ, DV), rn(DQ), rn(1)]
    h, last = mlstm_recurrent_step__hip_fw(*st, *x)
    c = _moved(st[0])
    new = dict(matC_new=c if in_place else _moved(torch.zeros_like(c)), vecN_new=torch.empty_like(st[1]), scaM_new=torch.empty_like(st[2]))
    h2, last2 = mlstm_recurrent_step__hip_fw(c if in_place else st[0], *st[1:], *x, **new)
    for a, b in zip((h, *last), (h2, *last2)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T", [5, 40])
def test_sequence_state(T):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    B, DQ, DV = 3, 128, 192
    g = torch.Generator(device=dev).manual_seed(T)
    rn = lambda *s: torch.randn(B, 1, *s, device=dev, generator=g)
    x = [rn(T, DQ).bfloat16(), rn(T, DQ).bfloat16(), rn(T, DV).bfloat16(), rn(T), 3 + rn(T), rn(DQ, DV), rn(DQ), rn(1)]
    out = []
    for c in (torch.zeros_like(x[5]), _moved(torch.zeros_like(x[5]))):
        h, n, m = torch.empty_like(x[2]), torch.empty_like(x[6]), torch.empty_like(x[7])
        _lib.check(lib.mlstm_hip_recurrent_sequence(*[ptr(t) for t in (*x, h, c, n, m)], B, 1, T, DQ, DV, 1e-6, _lib.BF16, _lib.F32, _lib.F32,
                                                    current_stream_ptr(dev)), "sequence")
        out.append((h, c, n, m))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("S", [64, 300])
def test_short_prompt_output(S):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.utils import current_stream_ptr, ptr

    lib, dev = _lib.get_lib(), torch.device("cuda")
    NH, DQ, DV = 3, 128, 128
    g = torch.Generator(device=dev).manual_seed(S)
    rn = lambda *s: torch.randn(1, NH, *s, device=dev, generator=g)
    x = [rn(S, DQ).bfloat16(), rn(S, DQ).bfloat16(), rn(S, DV).bfloat16(), rn(S), 3 + rn(S)]
    n = lib.mlstm_hip_chunkwise_fw_workspace_bytes(1, NH, S, DQ, DV, 0, _lib.PATH_AUTO, 0)
    out = []
    for H in (torch.zeros_like(x[2]), _moved(torch.zeros_like(x[2]))):
        ws, last = torch.empty(n, dtype=torch.uint8, device=dev), [torch.empty(1, NH, *s, device=dev) for s in ((DQ, DV), (DQ,), (1,))]
        _lib.check(lib.mlstm_hip_chunkwise_fw(*[ptr(t) for t in x], None, None, None, ptr(H), None, None, *[ptr(t) for t in last], ptr(ws), n, 0,
                                              1, NH, S, DQ, DV, 1e-6, _lib.BF16, _lib.F32, _lib.GATE_EXP, 1, _lib.PATH_AUTO, 0, _lib.NORM_NONE,
                                              1e-6, None, None, current_stream_ptr(dev)), "forward")
        out.append((H, *last))
    for a, b in zip(*out):
        assert torch.equal(a, b)
