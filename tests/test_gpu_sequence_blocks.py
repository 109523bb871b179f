"""The recurrence over several tokens on the matrix cores, at the token counts where its blocks of 32 begin and end and at
the head dimensions where its split changes, against the fp64 oracle.  The sums are fp32-exact, so with fp16 inputs and
fp32 states the tolerances are those of fp32 arithmetic (the outputs h are rounded once)."""
import pytest
import torch

import oracle as O
from helpers import make_qkvif, rel_norm

pytestmark = pytest.mark.gpu

_DIMS = [(64, 64), (64, 192), (128, 128), (128, 320), (256, 64), (512, 128)]


@pytest.mark.parametrize("T", [1, 2, 16, 17, 31, 32, 33, 64, 97])
@pytest.mark.parametrize("dims", _DIMS, ids=str)
@pytest.mark.parametrize("dtype,state", [(torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                         (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16)], ids=str)
def test_blocks_of_tokens(T, dims, dtype, state):
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_sequence__hip

    DQ, DV = dims
    B, NH = 2, 3
    print(f"T={T} {DQ}/{DV} {dtype} {state}", flush=True)
    q, k, v, i, f = make_qkvif(B, NH, T, DQ, DV, seed=T + DQ, dtype=dtype, f_offset=2.0)
    g = torch.Generator().manual_seed(T)
    rn = lambda *s: torch.randn(*s, generator=g).to(state)
    c, n, m = rn(B, NH, DQ, DV), rn(B, NH, DQ), rn(B, NH, 1)
    d = lambda t: t.double()
    H_ref, (C_r, n_r, m_r) = O.recurrent_sequence(d(q), d(k), d(v), d(i), d(f), d(c), d(n), d(m))
    cu = lambda t: t.cuda()
    H, (C, nn, mm) = mlstm_recurrent_sequence__hip(*map(cu, (q, k, v, i, f, c, n, m)), return_last_states=True, dtype_state=state)
    out = {torch.bfloat16: 3e-3, torch.float16: 4e-4, torch.float32: 2e-6}
    assert rel_norm(H, H_ref) < out[dtype]
    for a, b in ((C, C_r), (nn, n_r), (mm, m_r)):
        assert rel_norm(a.reshape(b.shape), b) < out[state]


@pytest.mark.parametrize("T", [7, 23, 70])
@pytest.mark.parametrize("dims", [(64, 128), (256, 64)], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_values_that_are_not_finite_reach_no_earlier_token(T, dims, dtype):
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_sequence__hip

    DQ, DV = dims
    B, NH = 1, 4
    print(f"T={T} {DQ}/{DV} {dtype}", flush=True)
    q, k, v, i, f = make_qkvif(B, NH, T, DQ, DV, seed=T + DQ, dtype=dtype, f_offset=2.0)
    v[0, 0, T // 2, 3] = float("nan")
    v[0, 1, T - 2, 5] = float("inf")
    k[0, 2, T // 3, 7] = float("nan")
    g = torch.Generator().manual_seed(T)
    c, n, m = torch.randn(B, NH, DQ, DV, generator=g), torch.randn(B, NH, DQ, generator=g), torch.randn(B, NH, 1, generator=g)
    d = lambda t: t.double()
    H_ref, (C_r, n_r, m_r) = O.recurrent_sequence(*map(d, (q, k, v, i, f, c, n, m)))
    cu = lambda t: t.cuda()
    H, (C, nn, mm) = mlstm_recurrent_sequence__hip(*map(cu, (q, k, v, i, f, c, n, m)), return_last_states=True)
    out = {torch.bfloat16: 3e-3, torch.float16: 4e-4}[dtype]
    for a, b, tol in ((H, H_ref, out), (C, C_r, 2e-6), (nn, n_r, 2e-6), (mm, m_r, 2e-6)):
        a, b = a.cpu().reshape(b.shape), b
        fin = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), fin)
        assert rel_norm(a[fin], b[fin]) < tol
    assert torch.isfinite(H_ref[0, 0, : T // 2]).all() and not torch.isfinite(H_ref[0, 0, T // 2:]).all()


def _recurrence_fp32(q, k, v, i, f, c, n, m):
    """The recurrence, token by token in fp32; the larger of two as the kernels take it (a NaN is not the larger one)."""
    q, k, v, i, f, c, n, m = (t.float().cpu() for t in (q, k, v, i, f, c, n, m))
    scale, H = q.shape[-1] ** -0.5, []
    for t in range(q.shape[2]):
        lf, it = torch.nn.functional.logsigmoid(f[:, :, t, None]), i[:, :, t, None]
        m_new = torch.fmax(lf + m, it)
        fa, ia, m = torch.exp(lf + m - m_new), torch.exp(it - m_new), m_new
        qt, kt = q[:, :, t] * scale, k[:, :, t] * ia
        c = fa[..., None] * c + kt[..., None] * v[:, :, t, None, :]
        n = fa * n + kt
        den = torch.fmax((qt * n).sum(-1, keepdim=True).abs(), torch.exp(-m)) + 1e-6
        H.append((qt[..., None] * c).sum(-2) * (1 / den))
    return torch.stack(H, 2), c, n, m


@pytest.mark.parametrize("T", [1, 6, 23, 70])
@pytest.mark.parametrize("dims", [(64, 128), (256, 64)], ids=str)
@pytest.mark.parametrize("dtype,state", [(torch.bfloat16, torch.float32), (torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16)], ids=str)
def test_infinities_stay_infinities(T, dims, dtype, state):
    """An infinity and a NaN of the recurrence are the same in the block form, and so is a finite value whose products
    overflow in one of them only: every output is held to the class (NaN, which infinity, finite) that the recurrence has."""
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_sequence__hip

    DQ, DV = dims
    B, NH = 1, 8
    print(f"T={T} {DQ}/{DV} {dtype} {state}", flush=True)
    q, k, v, i, f = make_qkvif(B, NH, T, DQ, DV, seed=T + DQ, dtype=dtype, f_offset=2.0)
    g = torch.Generator().manual_seed(T)
    rn = lambda *s: torch.randn(*s, generator=g)
    c, n, m = rn(B, NH, DQ, DV), rn(B, NH, DQ), rn(B, NH, 1)
    j = T // 2
    q, k = q.clone(), k.clone()
    q[0, :2], k[0, :2] = q[0, :2].abs() + 0.01, k[0, :2].abs() + 0.01   # sums of one sign: an infinity stays one in h
    v[0, 0, j, 3] = float("inf")
    c[0, 1, 5, 9] = float("-inf")
    c[0, 2, 7, 11] = float("nan")
    c[0, 3, 60, 2] = 3.4e38                                            # finite, infinite when rounded to 16 bits
    k[0, 4, j, 13] = float("inf")
    q[0, 5, j, 17] = float("-inf")
    if dtype == torch.bfloat16:                                        # a score that overflows, products with v that do not
        q[0, 6, 0, 4], k[0, 6, T - 1, 4] = 2.0 ** 70, 2.0 ** 70
        v[0, 6] *= 2.0 ** -40
    n[0, 7, 3] = float("inf")
    c, n, m = (t.to(state) for t in (c, n, m))
    ref = _recurrence_fp32(q, k, v, i, f, c, n, m)
    H, st = mlstm_recurrent_sequence__hip(*(t.cuda() for t in (q, k, v, i, f, c, n, m)), return_last_states=True, dtype_state=state)
    assert torch.isinf(ref[0][0, 0, j, 3]) and torch.isinf(ref[0][0, 1, :, 9]).all() and torch.isinf(ref[1][0, 1, 5, 9])
    tol = {torch.bfloat16: 3e-3, torch.float16: 4e-4, torch.float32: 2e-5}   # the rounding of the type; fp32 sums of either side
    for name, a, b, kind in (("H", H, ref[0], dtype), ("C", st[0], ref[1], state), ("n", st[1], ref[2], state), ("m", st[2], ref[3], state)):
        a, b = a.float().cpu().reshape(b.shape), b.to(kind).float()
        assert torch.equal(torch.isnan(a), torch.isnan(b)), name
        assert torch.equal(torch.where(torch.isinf(a), a, 0), torch.where(torch.isinf(b), b, 0)), name
        for head in range(NH):
            x, y = a[:, head], b[:, head]
            fin = torch.isfinite(y)
            if fin.any() and y[fin].abs().max() > 0:
                assert rel_norm(x[fin], y[fin]) < tol[kind], (name, head)


@pytest.mark.parametrize("dtype,state", [("bfloat16", "float32"), ("float16", "bfloat16"), ("float32", "float32")])
@pytest.mark.parametrize("form", ["dense", "strided", "mixed", "other state type"])
def test_one_token_through_the_backend(dtype, state, form):
    """One token from given states (in native code where nothing has to be converted) against the step function, and the shapes
    that the backend refuses."""
    from mlstm_kernels_amd.torch.backend_module import mLSTMBackend, mLSTMBackendConfig
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_step__hip

    B, NH, DQ, DV = 2, 3, 64, 128
    dt, sdt = getattr(torch, dtype), getattr(torch, state)
    g = torch.Generator().manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g).cuda()
    q, k, v = rn(B, NH, 1, DQ).to(dt), rn(B, NH, 1, DQ).to(dt), rn(B, NH, 1, DV).to(dt)
    i, f = rn(B, NH, 1).to(dt), rn(B, NH, 1).to(dt)
    st = [rn(B, NH, DQ, DV).to(sdt), rn(B, NH, DQ).to(sdt), rn(B, NH, 1).to(sdt)]
    if form == "strided":
        q = rn(B, NH, 1, 2 * DQ).to(dt)[..., ::2]
    elif form == "mixed":
        f = f.double().to(torch.float32 if dt != torch.float32 else torch.bfloat16)
    elif form == "other state type":
        st = [t.half() for t in st]
    backend = mLSTMBackend(mLSTMBackendConfig(mode="inference", autocast_kernel_dtype=dtype, inference_state_dtype=state))
    h, new = backend(q, k, v, i, f, *st)
    h_ref, new_ref = mlstm_recurrent_step__hip(q.squeeze(2), k.squeeze(2), v.squeeze(2), i, f, *st, dtype_state=sdt)
    assert h.shape == v.shape and torch.equal(h[:, :, 0], h_ref)
    for a, b in zip(new, new_ref):
        assert a.dtype == sdt and torch.equal(a, b)
    with pytest.raises(ValueError):
        backend(q.squeeze(2), k.squeeze(2), v.squeeze(2), i, f, *st)
