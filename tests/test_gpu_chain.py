"""The chain kernels (state recurrence and H / dV in one launch) where they can go wrong: lengths around steps of 64 positions,
chunks of 128 and windows of 256 and long ones, each width of a workgroup and head dimension, every option of the operators, one and
several rounds of workgroups, against the fp64 oracle on the first and the last (batch, head) pair.  Tolerances are norm-relative as for the other kernels of these outputs: H
6e-3, gradients 8e-3 (float16: a quarter), gate gradients 5e-2 of their scale, states 1e-3."""
import ctypes

import pytest
import torch

import oracle as O
from helpers import rel_norm

pytestmark = pytest.mark.gpu


def _names():
    from mlstm_kernels_amd import _lib

    lib, out, i = _lib.get_lib(), set(), 0
    while True:
        name, ms, n = ctypes.create_string_buffer(64), ctypes.c_float(), ctypes.c_int()
        if i >= lib.mlstm_hip_profile_read(i, name, 64, ctypes.byref(ms), ctypes.byref(n)):
            return out
        out.add(name.value.decode())
        i += 1


def _heads(DV, width):
    """Heads for one workgroup of `width` value columns on (almost) every CU."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return cus // (DV // width)


def _run(BH, S, DQ, DV, *, sig=False, normalize=True, init=False, last=False, dtype=torch.bfloat16, stride=2, f_offset=3.0, seed=0,
         recompute=False):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    print(f"{BH} x {S} {DQ}/{DV} sig={sig} normalize={normalize} init={init} last={last} {dtype} stride={stride}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    q, k, v, dH = (rn(1, BH, S, x).to(dtype) for x in (DQ, DQ, DV, DV))
    i, f = rn(1, BH, S), f_offset + rn(1, BH, S)
    c0 = n0 = m0 = dC = None
    if init:
        c0, n0, m0 = 0.1 * rn(1, BH, DQ, DV), 0.1 * rn(1, BH, DQ), 0.3 * rn(1, BH, 1)
    if last:
        dC = 0.1 * rn(1, BH, DQ, DV)
    leaves = [t.requires_grad_(True) for t in (q, k, v, i, f)] + ([c0.requires_grad_(True)] if init else [])
    kw = dict(c_initial=c0, n_initial=n0, return_last_states=last, any_sequence_length=True, chunk_size_intra=128 * stride,
              recompute_states_in_bw=recompute)
    lib = _lib.get_lib()
    _names()
    lib.mlstm_hip_profile_enable(1)
    try:
        if sig:
            out = mlstm_siging_chunkwise__hip_xl_chunk(*leaves[:5], normalize=normalize, **kw)
        else:
            out = mlstm_chunkwise__hip_xl_chunk(*leaves[:5], m_initial=m0, **kw)
        H, states = (out[0], out[1]) if last else (out, ())
        grads = torch.autograd.grad([H] + ([states[0]] if last else []), leaves, [dH] + ([dC] if last else []))
        torch.cuda.synchronize()
    finally:
        lib.mlstm_hip_profile_enable(0)
    assert {"chain_h", "chain_dv"} <= _names()   # the kernels that this is about
    tol = 0.25 if dtype == torch.float16 else 1.0
    L = next(x for x in (64, 32, 16, 8, 4, 2, 1) if S % x == 0)
    for h in (0, BH - 1):
        d = lambda t: None if t is None else t.detach()[:, h:h + 1].double().cpu()
        args = (d(q), d(k), d(v), d(i), d(f))
        m0d = None if sig else d(m0)
        o = dict(chunk_size=L, siging=sig, normalize=normalize)
        fw = O.chunkwise_fw(*args, d(c0), d(n0), m0d, **o)
        bw = O.chunkwise_bw(*args, d(dH), d(c0), d(n0), m0d, d(dC), **o)
        assert rel_norm(d(H), fw["H"]) <= 6e-3 * tol
        for name, x, ref in zip(("dQ", "dK", "dV", "dI", "dF", "dC0"), grads, bw):
            if name in ("dI", "dF"):
                assert float((d(x) - ref).abs().max()) <= 5e-2 * float(ref.abs().max()), name
            else:
                assert rel_norm(d(x), ref) <= 8e-3 * tol, name
        if last:
            assert rel_norm(d(states[0]), fw["C_last"]) <= 1e-3
            if normalize:
                assert rel_norm(d(states[1]), fw["n_last"]) <= 1e-3


@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (64, 256, 256), (128, 128, 128), (128, 256, 256), (256, 256, 256), (256, 512, 256),
                                         (256, 128, 128), (128, 384, 128)])
@pytest.mark.parametrize("S", [257, 320, 321, 383, 450])
def test_lengths(DQ, DV, width, S):
    _run(_heads(DV, width), S, DQ, DV, seed=S)


@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (64, 256, 256), (128, 128, 128), (128, 256, 256), (256, 128, 128), (256, 256, 256)])
@pytest.mark.parametrize("S", [384, 449])
@pytest.mark.parametrize("opt", [dict(init=True, last=True), dict(sig=True, init=True, last=True), dict(sig=True, normalize=False, init=True, last=True),
                                 dict(dtype=torch.float16, init=True, last=True), dict(stride=1, last=True), dict(stride=3, init=True),
                                 dict(f_offset=-4.0, last=True), dict(f_offset=9.0, init=True, last=True), dict(f_offset=9.0, dtype=torch.float16),
                                 dict(recompute=True, init=True)],
                         ids=["states", "sig", "sig-raw", "fp16", "stride1", "stride3", "forget", "keep", "fp16-keep", "recompute"])
def test_options(DQ, DV, width, S, opt):
    _run(_heads(DV, width), S, DQ, DV, seed=S + 1, **opt)


# many steps: decays that add up, sums over a long walk; forget gates that forget, that mostly keep and that keep nearly all
@pytest.mark.parametrize("DQ,DV,width,S", [(64, 128, 128, 2048), (64, 256, 256, 2111), (128, 128, 128, 4100), (128, 256, 256, 2017), (256, 128, 128, 2050),
                                           (256, 512, 256, 2200), (256, 256, 128, 1600)])
@pytest.mark.parametrize("opt", [dict(f_offset=0.0, last=True), dict(f_offset=3.0, init=True, last=True), dict(f_offset=9.0, last=True),
                                 dict(f_offset=3.0, dtype=torch.float16, last=True), dict(f_offset=9.0, dtype=torch.float16), dict(sig=True, last=True)],
                         ids=str)
def test_long(DQ, DV, width, S, opt):
    _run(_heads(DV, width), S, DQ, DV, seed=S, **opt)


@pytest.mark.parametrize("S", [257, 321, 1000, 1024, 1700])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_halves_of_wide_heads(S, dtype):
    """Half of the heads that fill the chip with 256 columns a workgroup: the scan and the streaming kernel, whether states are kept or not."""
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    BH, DQ, DV = _heads(512, 128), 256, 512
    print(f"{BH} x {S} {DQ}/{DV} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), 3 + rn(S)]
    st = [0.1 * rn(DQ, DV), 0.1 * rn(DQ), 0.3 * rn(1)]
    _names()
    _lib.profile_enable(True)
    try:
        H, last = mlstm_chunkwise__hip_xl_chunk(*x, c_initial=st[0], n_initial=st[1], m_initial=st[2], return_last_states=True, any_sequence_length=True)
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    assert "chain_h" not in _names()
    L = next(y for y in (64, 32, 16, 8, 4, 2, 1) if S % y == 0)
    for h in (0, BH - 1):
        d = lambda t: t[:, h:h + 1].double().cpu()
        fw = O.chunkwise_fw(*map(d, x), *map(d, st), chunk_size=L)
        assert rel_norm(d(H), fw["H"]) <= 6e-3 * (0.25 if dtype == torch.float16 else 1.0)
        assert rel_norm(d(last[0]), fw["C_last"]) <= 1e-5 and rel_norm(d(last[1]), fw["n_last"]) <= 1e-5


# Few heads and a long prompt, whose heads leave the chain kernel most of the chip: it is not taken, whether states are kept or not.  The last
# states are held to the 1e-5 of a scan that carries the remainder of the value operand in the chunks that weigh 2^-8 or more: what the others lose
# is up to 2^-9 of them, 2^-17 = 7.6e-6 of the state (gates around 6: it is a part of the chunks of every segment).
@pytest.mark.parametrize("BH,S,DQ,DV", [(4, 16384, 128, 256), (4, 8300, 256, 512), (8, 5000, 256, 512), (8, 10000, 256, 512), (40, 8060, 256, 512),
                                        (100, 3968, 128, 256), (4, 4428, 128, 256), (24, 3528, 128, 128), (5, 16384, 64, 128), (12, 6016, 64, 256),
                                        (7, 10185, 256, 256), (9, 6003, 128, 384)])
@pytest.mark.parametrize("opt", [dict(), dict(f_offset=6.0, init=True), dict(f_offset=9.0, init=True), dict(f_offset=0.0, last=False), dict(sig=True, init=True),
                                 dict(sig=True, normalize=False, init=True), dict(dtype=torch.float16, f_offset=9.0)],
                         ids=["", "half", "keep", "forget", "sig", "sig-raw", "fp16-keep"])
def test_long_prompts_of_few_heads(BH, S, DQ, DV, opt):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    o = dict(dict(f_offset=3.0, init=False, last=True, sig=False, normalize=True, dtype=torch.bfloat16), **opt)
    print(f"{BH} x {S} {DQ}/{DV} {opt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(o["dtype"]), rn(S, DQ).to(o["dtype"]), rn(S, DV).to(o["dtype"]), rn(S), o["f_offset"] + rn(S)]
    c0, n0, m0 = (0.1 * rn(DQ, DV), 0.1 * rn(DQ), None if o["sig"] else 0.3 * rn(1)) if o["init"] else (None, None, None)
    kw = dict(c_initial=c0, n_initial=n0, return_last_states=o["last"], any_sequence_length=True)
    _names()
    _lib.profile_enable(True)
    try:
        with torch.no_grad():
            if o["sig"]:
                out = mlstm_siging_chunkwise__hip_xl_chunk(*x, normalize=o["normalize"], **kw)
            else:
                out = mlstm_chunkwise__hip_xl_chunk(*x, m_initial=m0, **kw)
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    assert "chain_h" not in _names()
    H, last = out if o["last"] else (out, None)
    L = max(y for y in range(1, 257) if S % y == 0)  # (the oracle's chunks)
    for h in {0, BH - 1}:
        d = lambda t: None if t is None else t[:, h:h + 1].double().cpu()
        fw = O.chunkwise_fw(*map(d, x), d(c0), d(n0), d(m0), chunk_size=L, siging=o["sig"], normalize=o["normalize"])
        assert rel_norm(d(H), fw["H"]) <= 6e-3 * (0.25 if o["dtype"] == torch.float16 else 1.0)
        if last is not None:
            assert rel_norm(d(last[0]), fw["C_last"]) <= 1e-5
            if o["normalize"]:
                assert rel_norm(d(last[1]), fw["n_last"]) <= 1e-5


# two rounds of workgroups (the last head is in the second one), and a first round that is all there is, not quite full
@pytest.mark.parametrize("DQ,DV,width,share", [(128, 256, 256, 2.0), (256, 512, 256, 1.95), (64, 128, 128, 2.0), (128, 256, 256, 0.9)])
def test_rounds(DQ, DV, width, share):
    _run(int(_heads(DV, width) * share), 330, DQ, DV, seed=7, last=True)


@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (64, 256, 256), (128, 128, 128), (128, 256, 256), (256, 128, 128), (256, 512, 256)])
@pytest.mark.parametrize("S", [513, 1100, 2048])
@pytest.mark.parametrize("dtype,init", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, False)], ids=str)
def test_without_kept_states(DQ, DV, width, S, dtype, init):
    """A forward without a backward keeps no states; H and the last states are the bits of one that does."""
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    BH = _heads(DV, width)
    print(f"{BH} x {S} {DQ}/{DV} {dtype} init={init}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), 3 + rn(S)]
    st = (0.1 * rn(DQ, DV), 0.1 * rn(DQ), 0.3 * rn(1)) if init else (None,) * 3
    out = []
    for grad in (False, True):
        leaves = [t.clone().requires_grad_(grad) for t in x]
        _names()
        _lib.profile_enable(True)
        try:
            H, last = mlstm_chunkwise__hip_xl_chunk(*leaves, *st, return_last_states=True, any_sequence_length=True)
        finally:
            _lib.profile_enable(False)
        assert "chain_h" in _names()
        out.append([t.detach() for t in (H, *last)])
    for a, b in zip(*out):
        assert torch.equal(a, b)
    L = next(y for y in (64, 32, 16, 8, 4, 2, 1) if S % y == 0)
    for h in (0, BH - 1):
        d = lambda t: None if t is None else t.detach()[:, h:h + 1].double().cpu()
        fw = O.chunkwise_fw(*(d(t) for t in x), *(d(t) for t in st), chunk_size=L)
        assert rel_norm(d(out[0][0]), fw["H"]) <= 6e-3 * (0.25 if dtype == torch.float16 else 1.0)
        assert rel_norm(d(out[0][1]), fw["C_last"]) <= 1e-3 and rel_norm(d(out[0][2]), fw["n_last"]) <= 1e-3


def test_closed_gates():
    """A forget gate that forgets everything (decay zero) and an input gate that stays shut for several steps."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    BH, S, DQ, DV = _heads(256, 256), 400, 128, 256
    g = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    q, k, v = (rn(1, BH, S, x).bfloat16() for x in (DQ, DQ, DV))
    i, f = rn(1, BH, S), 3 + rn(1, BH, S)
    f[:, :, 130] = -200.0
    i[:, :, 200:330] = -float("inf")
    from mlstm_kernels_amd import _lib

    _names()
    _lib.profile_enable(True)
    try:
        H, (C, n, m) = mlstm_chunkwise__hip_xl_chunk(q, k, v, i, f, return_last_states=True, any_sequence_length=True)
    finally:
        _lib.profile_enable(False)
    assert "chain_h" in _names()
    for h in (0, BH - 1):
        d = lambda t: t[:, h:h + 1].double().cpu()
        # (the recurrence itself: an infinite gate is a weight of zero there)
        ref, (Cr, nr, mr) = O.recurrent_sequence(d(q), d(k), d(v), d(i), d(f), torch.zeros(1, 1, DQ, DV, dtype=torch.float64),
                                                 torch.zeros(1, 1, DQ, dtype=torch.float64), torch.zeros(1, 1, 1, dtype=torch.float64))
        assert rel_norm(d(H), ref) <= 6e-3 and rel_norm(d(C), Cr) <= 1e-3 and rel_norm(d(n), nr) <= 1e-3


@pytest.mark.parametrize("DQ,DV,width,S", [(64, 128, 128, 700), (64, 256, 256, 300), (128, 128, 128, 1025), (128, 256, 256, 641), (256, 128, 128, 512),
                                           (256, 512, 256, 600)])
@pytest.mark.parametrize("opt", [dict(), dict(stride=1, f_offset=9.0), dict(stride=3, init=True, last=True), dict(dtype=torch.float16, f_offset=9.0),
                                 dict(sig=True, normalize=False, init=True), dict(norm="layer")], ids=str)
def test_recomputed_states_are_the_kept_ones(DQ, DV, width, S, opt):
    """recompute_states_in_bw: the gradients are bit for bit those of the kept states, whichever kernel made them (a head norm keeps
    the forward from this one)."""
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    BH, dtype, init, norm = _heads(DV, width), opt.get("dtype", torch.bfloat16), opt.get("init", False), opt.get("norm", "none")
    print(f"{BH} x {S} {DQ}/{DV} {opt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), opt.get("f_offset", 3.0) + rn(S)]
    dH, state = rn(S, DV).to(dtype), (rn(DQ, DV), rn(DQ), rn(1)) if init else (None, None, None)
    grads, names = [], []
    for recompute in (False, True):
        leaves = [t.clone().requires_grad_(True) for t in x]
        kw = dict(c_initial=state[0], n_initial=state[1], return_last_states=opt.get("last", False), any_sequence_length=True,
                  chunk_size_intra=128 * opt.get("stride", 2), recompute_states_in_bw=recompute, head_norm=norm)
        _lib.profile_read()
        _lib.profile_enable(True)
        try:
            if opt.get("sig"):
                out = mlstm_siging_chunkwise__hip_xl_chunk(*leaves, normalize=opt.get("normalize", True), **kw)
            else:
                out = mlstm_chunkwise__hip_xl_chunk(*leaves, m_initial=state[2], **kw)
            H = out[0] if opt.get("last") else out
            grads.append((H.detach(), *torch.autograd.grad(H, leaves, dH)))
        finally:
            _lib.profile_enable(False)
        names.append(set(_lib.profile_read()))
    assert ("chain_h" in names[0]) == (norm == "none") and "scan_fw_recompute" in names[1]
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize("DQ,DV,width,S", [(64, 128, 128, 700), (64, 256, 256, 1500), (128, 128, 128, 1500), (128, 256, 256, 700), (256, 128, 128, 700),
                                           (256, 512, 256, 1500)])
@pytest.mark.parametrize("name,power", [("v", 104), ("dH", 104), ("v", -80), ("dH", -80)])
def test_range_of_values(DQ, DV, width, S, name, power):
    """What is linear in v or dH scales with a power of two exactly, also where the state is within a few powers of two of the largest
    float32 value: nothing that the kernels hold is larger than the state."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    BH = _heads(DV, width)
    print(f"{BH} x {S} {DQ}/{DV} {name} {power}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).bfloat16(), rn(S, DQ).bfloat16(), rn(S, DV).bfloat16(), rn(S), 3 + rn(S)]
    dH, state = rn(S, DV).bfloat16(), (rn(DQ, DV), rn(DQ), rn(1))
    scale = 2.0 ** power
    out = []
    for factor in (1.0, scale):
        y = [t * factor if j == 2 and name == "v" else t for j, t in enumerate(x)]
        c0 = state[0] * factor if name == "v" else state[0]
        leaves = [t.clone().requires_grad_(True) for t in y]
        H, (C, n, m) = mlstm_chunkwise__hip_xl_chunk(*leaves, c0, *state[1:], return_last_states=True, any_sequence_length=True)
        out.append((H.detach(), C.detach(), *torch.autograd.grad(H, leaves, dH * factor if name == "dH" else dH)))
    linear = (True, True, True, True, False, True, True) if name == "v" else (False, False) + (True,) * 5
    for what, a, b, lin in zip(("H", "C", "dQ", "dK", "dV", "dI", "dF"), *out, linear):
        assert bool(torch.isfinite(b).all()), what
        assert torch.equal(a * scale if lin else a, b), what


@pytest.mark.parametrize("DQ,DV,width", [(64, 128, 128), (64, 256, 256), (128, 128, 128), (128, 256, 256), (256, 128, 128), (256, 512, 256)])
@pytest.mark.parametrize("opt", [dict(S=512), dict(S=1024), dict(S=768, stride=1, init=True), dict(S=512, sig=True, init=True),
                                 dict(S=512, sig=True, normalize=False), dict(S=768, stride=3, dtype=torch.float16)], ids=str)
def test_every_element_within_tolerance_of_the_rounding_emulation(DQ, DV, width, opt):
    """H, dQ, dK, dV against the fp64 emulation that rounds what the kernels round, in steps of 64 positions (tests/rounding_emulation.py): every
    element inside |x - ref| <= 2e-2 + 2e-2 |ref|.  The row normalisers are held to fp32 summation accuracy first and then handed to it."""
    import rounding_emulation as R
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import hip_xl_chunk as X
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    BH, S, stride, dtype = _heads(DV, width), opt["S"], opt.get("stride", 2), opt.get("dtype", torch.bfloat16)
    sig, normalize, init = opt.get("sig", False), opt.get("normalize", True), opt.get("init", False)
    print(f"{BH} x {S} {DQ}/{DV} {opt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S + DQ)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), opt.get("f_offset", 3.0) + rn(S)]
    dH, st = rn(S, DV).to(dtype), (0.1 * rn(DQ, DV), 0.1 * rn(DQ), torch.zeros(1, BH, 1, device="cuda")) if init else (None,) * 3
    leaves = [t.clone().requires_grad_(True) for t in x]
    kw = dict(c_initial=st[0], n_initial=st[1], chunk_size_intra=128 * stride)
    _names()
    _lib.profile_enable(True)
    try:
        H = mlstm_siging_chunkwise__hip_xl_chunk(*leaves, normalize=normalize, **kw) if sig else mlstm_chunkwise__hip_xl_chunk(*leaves, m_initial=st[2], **kw)
        got = (H, *torch.autograd.grad(H, leaves[:3], dH))
    finally:
        _lib.profile_enable(False)
    assert {"chain_h", "chain_dv"} <= _names()
    track_n = not (sig and not normalize)
    _, qb, kb, vb, ib, fb, c0f, n0f, m0f = X._prep_inputs(*x, *st, sig)
    n_kernel = torch.empty(1, BH, S, device="cuda")
    X._fw_launch(qb, kb, vb, ib, fb, c0f, n0f, m0f, 1e-6, sig, normalize, False, False, _lib.PATH_AUTO, stride, n_out=n_kernel)
    for h in (0, BH - 1):
        d = lambda t: None if t is None else t.detach()[:, h:h + 1].double().cpu()
        args, first = [d(t) for t in x], [d(t) for t in st]
        ekw = dict(stride=stride, siging=sig, normalize=normalize, rnd=R.rounder(dtype), chain=True)
        own = R.chunkwise_fw_rounded(*args, *first, **ekw)
        nk = d(n_kernel) if track_n else None
        if track_n:  # a sum of up to 64 + DHQK fp32 terms, and the state's own of up to S
            assert float(((nk - own["nmax_own"]).abs() - (2e-6 * own["den_abs"] + 1e-6 * own["nmax_own"])).max()) <= 0
        ref = (R.chunkwise_fw_rounded(*args, *first, nmax_given=nk, **ekw)["H"],
               *R.chunkwise_bw_rounded(*args, d(dH), *first, nmax_given=nk, **ekw))
        for name, a, b in zip(("H", "dQ", "dK", "dV"), got, ref):
            worst = float(((d(a) - b).abs() / (2e-2 + 2e-2 * b.abs())).max())
            print(f"  {name} head {h}: {worst:.2f} x the bound", flush=True)
            assert worst <= 1, (name, h, worst)


@pytest.mark.parametrize("DQ,DV,width,S", [(64, 128, 128, 1000), (128, 256, 256, 1024), (256, 512, 256, 1024)])
@pytest.mark.parametrize("opt", [dict(f_offset=0.0), dict(), dict(f_offset=9.0), dict(sig=True), dict(f_offset=9.0, dtype=torch.float16)], ids=str)
def test_as_exact_as_scan_and_h(DQ, DV, width, S, opt):
    """Distance from 64 bits by norm, over eight heads, against that of the scan and the kernels over chunks ("split")."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    BH, dtype, sig = _heads(DV, width), opt.get("dtype", torch.bfloat16), opt.get("sig", False)
    print(f"{BH} x {S} {DQ}/{DV} {opt}", flush=True)
    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    g = torch.Generator(device="cuda").manual_seed(S + DQ)
    rn = lambda *s: torch.randn(1, BH, *s, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), opt.get("f_offset", 3.0) + rn(S)]
    dH, heads = rn(S, DV).to(dtype), list(range(0, BH, BH // 8))
    d = lambda t: t.detach()[:, heads].double().cpu()
    L = next(y for y in (64, 32, 16, 8) if S % y == 0)
    fw = O.chunkwise_fw(*(d(t) for t in x), chunk_size=L, siging=sig)
    bw = O.chunkwise_bw(*(d(t) for t in x), d(dH), chunk_size=L, siging=sig)
    err = []
    for path in ("auto", "split"):
        leaves = [t.clone().requires_grad_(True) for t in x]
        H, last = op(*leaves, return_last_states=True, any_sequence_length=True, kernel_path=path)
        grads = torch.autograd.grad(H, leaves[:3], dH)
        err.append([rel_norm(d(a), b) for a, b in zip((H, *grads, *last[:2]), (fw["H"], *bw[:3], fw["C_last"], fw["n_last"]))])
    print(err, flush=True)
    for a, b in zip(err[0][:4], err[1][:4]):
        assert a <= 1.02 * b
    for a, b in zip(err[0][4:], err[1][4:]):
        assert a <= max(1.05 * b, 2 ** -20)  # (fp32 sums of up to S terms, in another order)
