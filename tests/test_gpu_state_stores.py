"""The recurrent kernels' ways of reading and storing the state, chosen by its size: a head's results are the same bits whatever it is
batched with, but for the order of the sum in h beyond 320 MiB, where the rows are dealt to other groups.  Heads of rows and columns
that leave row groups, lanes and the first batch of rows unfilled."""
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
_F32, _BF16 = torch.float32, torch.bfloat16


def _inputs(n, T, DQ, DV, sdt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(n, *s, device="cuda", generator=g)
    tok = () if T is None else (T,)
    x = [rn(1, *tok, DQ).bfloat16(), rn(1, *tok, DQ).bfloat16(), rn(1, *tok, DV).bfloat16(), rn(1, *(tok or (1,))), 3 + rn(1, *(tok or (1,)))]
    return x, [rn(1, DQ, DV).to(sdt), rn(1, DQ).to(sdt), rn(1, 1).to(sdt)]


# (rows, columns, state type, MiB of state: on either side of 12, 20, 32, 112 and 320)
@pytest.mark.parametrize("DQ,DV,sdt,mib", [(64, 128, _F32, 11), (64, 128, _F32, 20), (64, 128, _F32, 120), (48, 132, _F32, 20), (65, 64, _F32, 40),
                                           (127, 256, _F32, 40), (128, 256, _F32, 40), (129, 260, _F32, 40), (255, 64, _BF16, 40),
                                           (256, 512, _BF16, 40), (256, 512, _F32, 40), (100, 72, _BF16, 20), (128, 256, _F32, 330),
                                           (64, 64, _F32, 5), (64, 64, _F32, 20), (64, 64, _F32, 24), (33, 40, _BF16, 20), (127, 64, _F32, 24),
                                           (512, 64, _BF16, 40)])
@pytest.mark.parametrize("in_place", [False, True])
def test_step(DQ, DV, sdt, mib, in_place):
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_step__hip_fw

    n = (mib << 20) // (DQ * DV * (4 if sdt == _F32 else 2))
    print(n, DQ, DV, sdt, in_place, flush=True)
    x, (c, nn, m) = _inputs(n, None, DQ, DV, sdt, DQ)
    some = [0, 1, n - 2, n - 1]
    h1, (c1, n1, m1) = mlstm_recurrent_step__hip_fw(c[some], nn[some], m[some], *(t[some] for t in x), dtype_state=sdt)
    d = lambda t: t[some].double()
    ref = O.recurrent_step(*(d(t) for t in x), d(c), d(nn), d(m))  # (in front of the call, which may write over c)
    kw = dict(matC_new=c, vecN_new=torch.empty_like(nn), scaM_new=torch.empty_like(m)) if in_place else {}
    h, (c2, n2, m2) = mlstm_recurrent_step__hip_fw(c, nn, m, *x, dtype_state=sdt, **kw)
    for a, b in ((c2, c1), (n2, n1), (m2, m1)):
        assert torch.equal(a[some], b)
    if mib <= 320:
        assert torch.equal(h[some], h1)
    else:  # a sum in another order may be rounded to the other bfloat16 neighbour
        assert bool(((h[some].double() - h1.double()).abs() <= 2 ** -7 * h1.double().abs() + 1e-5 * float(h1.double().abs().max())).all())
    # the recurrence in 64 bits.  h is rounded to bfloat16, a 16-bit state to 16 bits: half a unit in the last place of each value
    ref_h, ref_states = ref
    assert float((h[some].double() - ref_h).norm() / ref_h.norm()) <= 2 ** -8
    for a, b in zip((c2, n2, m2), ref_states):
        assert float((a[some].double() - b).norm() / b.norm()) <= (1e-6 if sdt == _F32 else 2 ** -8)


# (on either side of 96 MiB of state)
@pytest.mark.parametrize("T", [2, 16, 17, 33])
@pytest.mark.parametrize("DQ,DV,sdt", [(64, 64, _F32), (128, 192, _F32), (256, 512, _F32), (512, 64, _BF16)])
def test_sequence(T, DQ, DV, sdt):
    from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_sequence__hip

    n = (100 << 20) // (DQ * DV * (4 if sdt == _F32 else 2))
    print(n, T, DQ, DV, sdt, flush=True)
    x, st = _inputs(n, T, DQ, DV, sdt, DQ + T)
    some = [0, 1, n - 2, n - 1]
    h, last = mlstm_recurrent_sequence__hip(*x, *st, return_last_states=True, dtype_state=sdt)
    h1, last1 = mlstm_recurrent_sequence__hip(*(t[some] for t in (*x, *st)), return_last_states=True, dtype_state=sdt)
    for a, b in ((h, h1), *zip(last, last1)):
        assert torch.equal(a[some], b)
