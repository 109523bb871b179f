"""The streaming kernels at the lengths where they can go wrong (one position, either side of a chunk and of a window of
two chunks, several windows with a ragged last one), forward and backward, against the fp64 oracle; and the padding
adapter, which hands such a length over as it is, against explicit padding.  Tolerances are norm-relative as in the
randomised sweep: H 6e-3, gradients 8e-3, gate gradients 5e-2 of their scale."""
import pytest
import torch

import oracle as O
from helpers import make_qkvif, rel_norm

pytestmark = pytest.mark.gpu


def _run(S, DQ, DV, *, B=1, NH=2, sig=False, norm="none", init=False, seed=0, dtype=torch.bfloat16, path="auto",
         f_offset=3.0):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    q, k, v, i, f = make_qkvif(B, NH, S, DQ, DV, seed=seed, dtype=dtype, f_offset=f_offset)
    g = torch.Generator().manual_seed(seed + 1)
    dH = torch.randn(B, NH, S, DV, generator=g).to(dtype)
    st = (None, None, None)
    if init:
        st = (0.1 * torch.randn(B, NH, DQ, DV, generator=g), 0.1 * torch.randn(B, NH, DQ, generator=g), 0.3 * torch.randn(B, NH, 1, generator=g))
    d = lambda t: None if t is None else t.double()
    L = next(x for x in (64, 32, 16, 8, 4, 2, 1) if S % x == 0)
    m0 = None if sig else d(st[2])
    fw = O.chunkwise_fw(d(q), d(k), d(v), d(i), d(f), d(st[0]), d(st[1]), m0, chunk_size=L, siging=sig)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v, i, f)]
    cu = lambda t: None if t is None else t.cuda()
    print(f"S={S} {DQ}/{DV} sig={sig} norm={norm} init={init} {dtype} {path}", flush=True)
    H, last = op(*leaves, c_initial=cu(st[0]), n_initial=cu(st[1]), m_initial=cu(st[2]), return_last_states=True, chunk_size=128,
                 any_sequence_length=True, kernel_path=path, head_norm=norm)
    H.backward(dH.cuda())
    if norm == "none":
        H_ref, dH_ref = fw["H"], d(dH)
    else:
        raw = fw["H"].detach().requires_grad_(True)
        x = raw - raw.mean(-1, keepdim=True) if norm == "layer" else raw
        H_ref = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
        (dH_ref,) = torch.autograd.grad(H_ref, raw, d(dH))
    bw = O.chunkwise_bw(d(q), d(k), d(v), d(i), d(f), dH_ref, d(st[0]), d(st[1]), m0, None, chunk_size=L, siging=sig)
    tol = 4.0 if norm != "none" else 1.0   # the norm removes the scale of a row: what is left of dQ and dK cancels in part
    assert rel_norm(H, H_ref) <= 6e-3 * tol
    # (the norm of the only row of a sequence removes its scale, which is all q and k change: their gradients vanish)
    grads = list(zip(("dQ", "dK", "dV"), leaves, bw[:3]))[2 if norm != "none" and S == 1 else 0:]
    for name, leaf, ref in grads:
        assert rel_norm(leaf.grad, ref) <= 8e-3 * tol, name
    for name, leaf, ref in zip(("dI", "dF"), leaves[3:], bw[3:5]) if len(grads) == 3 else ():
        # (a sequence of one has dF = 0: the oracle's own rounding is no scale)
        scale = max(float(ref.abs().max()), 1e-3 * float(bw[3].abs().max()))
        assert float((leaf.grad.double().cpu() - ref).abs().max()) <= 5e-2 * tol * scale, name
    assert rel_norm(last[0], fw["C_last"]) <= 1e-3


@pytest.mark.parametrize("S", [1, 63, 127, 129, 255, 257, 384, 385, 1001])
@pytest.mark.parametrize("opt", [dict(), dict(sig=True, init=True), dict(norm="layer"), dict(dtype=torch.float16, init=True)],
                         ids=["exp", "sig-init", "norm", "fp16-init"])
def test_ragged_lengths(S, opt):
    _run(S, 256, 512, seed=S, **opt)


@pytest.mark.parametrize("DQ,DV", [(64, 64), (64, 128), (128, 128), (128, 256), (256, 256), (512, 1024), (192, 320), (256, 192),
                                   (128, 384), (64, 512), (512, 64)])
@pytest.mark.parametrize("S", [40, 256, 390])
@pytest.mark.parametrize("opt", [dict(), dict(sig=True, init=True), dict(norm="rms"), dict(dtype=torch.float16)],
                         ids=["exp", "sig-init", "norm", "fp16"])
def test_head_dimensions(DQ, DV, S, opt):
    if "norm" in opt and DV not in (64, 128, 256, 512):
        pytest.skip("the fused head norm needs DHHV = 64, 128, 256 or 512")
    _run(S, DQ, DV, seed=S + DQ + DV, **opt)


@pytest.mark.parametrize("B,NH,S,DQ,DV,opt", [
    (1, 2, 8 * 128, 256, 512, dict()),                 # one segment per chunk group: the shortest that is cut
    (1, 2, 65 * 128 - 5, 128, 128, dict(init=True)),   # eight segments, the last one shorter and ragged
    (1, 1, 67 * 128 + 3, 64, 64, dict(sig=True, init=True)),
    (1, 4, 4100, 256, 512, dict(dtype=torch.float16)),
])
@pytest.mark.parametrize("f_offset", [3.0, 9.0])       # only the last chunks / all chunks weigh in the last state
def test_segmented_scan(B, NH, S, DQ, DV, opt, f_offset):
    _run(S, DQ, DV, B=B, NH=NH, seed=S, f_offset=f_offset, **opt)


# segments of two to six chunks, up to sixteen of them, the last one shorter than the others
@pytest.mark.parametrize("NH,S,DQ,DV,opt", [(4, 20 * 128 - 3, 64, 64, dict()), (1, 32 * 128 + 1, 64, 128, dict(init=True)), (2, 33 * 128, 128, 128, dict(sig=True)),
                                            (1, 41 * 128 + 5, 128, 64, dict(init=True, dtype=torch.float16)), (3, 24 * 128, 64, 192, dict(init=True, sig=True))])
@pytest.mark.parametrize("f_offset", [3.0, 9.0])
def test_short_segments(NH, S, DQ, DV, opt, f_offset):
    _run(S, DQ, DV, NH=NH, seed=S, f_offset=f_offset, **opt)


@pytest.mark.parametrize("NH,S,DQ,DV", [(1, 8200, 128, 128), (2, 8192, 256, 512), (8, 4100, 256, 512)])
@pytest.mark.parametrize("path", ["auto", "split"])
def test_segmented_scan_is_recomputed_in_segments(NH, S, DQ, DV, path):
    """recompute_states_in_bw: the gradients are bit for bit those of the kept states where no last state is returned, also
    where the forward's scan ran in segments."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    q, k, v, i, f = (t.cuda() for t in make_qkvif(1, NH, S, DQ, DV, seed=S, f_offset=9.0))   # (states that remember)
    dH = torch.randn(1, NH, S, DV, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    grads = []
    for recompute in (False, True):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v, i, f)]
        H = mlstm_chunkwise__hip_xl_chunk(*leaves, any_sequence_length=True, kernel_path=path, recompute_states_in_bw=recompute)
        grads.append((H.detach(), *torch.autograd.grad(H, leaves, dH)))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize("S", [2047, 2048, 2049])      # a head's gates in one workgroup up to 2048 positions
@pytest.mark.parametrize("opt", [dict(), dict(init=True), dict(sig=True, init=True)], ids=["exp", "init", "sig-init"])
def test_gates_in_one_or_two_launches(S, opt):
    _run(S, 64, 64, seed=S, **opt)


# the most heads with half tiles (scan: 16, 42, 64), half items or one column group a workgroup (the others, at one length)
@pytest.mark.parametrize("DQ,DV,BH", [(256, 512, 16), (192, 128, 42), (128, 256, 64), (256, 512, 14), (256, 512, 64), (256, 1024, 32),
                                      (512, 1024, 32)])
@pytest.mark.parametrize("S", [129, 1024, 1100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_width_of_the_tiles(DQ, DV, BH, S, dtype):
    """The tiles of the scans and the items of the H / dV kernels split the value columns: their width changes no bit of the
    results.  (Window or tiled kernel, and segments of the scan, are chosen by the number of heads too, and do change some:
    the shapes here are those at which only the widths differ between the two batches.)"""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    print(f"S={S} {DQ}/{DV} {BH}", flush=True)
    q, k, v, i, f = (t.cuda() for t in make_qkvif(BH + 1, 1, S, DQ, DV, seed=S, dtype=dtype))
    dH = torch.randn(BH + 1, 1, S, DV, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    out = []
    for n in (BH, BH + 1):
        leaves = [t[:n].clone().requires_grad_(True) for t in (q, k, v, i, f)]
        H, last = mlstm_chunkwise__hip_xl_chunk(*leaves, return_last_states=True, any_sequence_length=True)
        grads = torch.autograd.grad(H, leaves, dH[:n])
        out.append([t.detach()[:BH] for t in (H, *last, *grads)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("path,S,DQ,DV", [("split", 8192, 128, 128), ("stream", 8192, 256, 512), ("split", 8200, 64, 64), ("stream", 256, 256, 512),
                                          ("split", 1024, 64, 128), ("split", 1100, 192, 256)])
def test_named_paths_do_not_depend_on_the_batch(path, S, DQ, DV):
    """With the path named a sequence gets the same bits alone (where the scan of "auto" runs in segments and fewer windows
    change the kernels it takes) and in a batch."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    n = 100 if DQ < 256 else 40
    q, k, v, i, f = (t.cuda() for t in make_qkvif(n + 1, 1, S, DQ, DV, seed=S, f_offset=9.0))
    dH = torch.randn(n + 1, 1, S, DV, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    out = []
    for rows in (slice(n, n + 1), slice(0, n + 1)):
        leaves = [t[rows].clone().requires_grad_(True) for t in (q, k, v, i, f)]
        H, last = mlstm_chunkwise__hip_xl_chunk(*leaves, return_last_states=True, any_sequence_length=True, kernel_path=path)
        grads = torch.autograd.grad(H, leaves, dH[rows])
        out.append([t.detach()[-1] for t in (H, *last, *grads)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


# State tiles on persistent workgroups: fewer, as many and many more than the CUs hold (the last: more than 32 for each); the
# chunks behind the last kept state are not run, with and without a last state, with strides that divide the chunks and not.
# With the path named a head's bits do not depend on how the tiles fall to the workgroups.
@pytest.mark.parametrize("DQ,DV,BH,S", [(256, 512, 33, 129), (256, 512, 80, 640), (64, 64, 514, 385), (128, 64, 300, 257), (64, 128, 300, 640),
                                        (64, 64, 16500, 130),
                                        # tiles smaller than 128 x 128 around the line below which each has a workgroup of its own
                                        (256, 320, 26, 385), (256, 320, 35, 640), (256, 320, 36, 257), (192, 192, 57, 257), (192, 192, 80, 640),
                                        (64, 384, 119, 129), (64, 384, 120, 385)])
@pytest.mark.parametrize("last,stride,init", [(False, 1, False), (False, 2, True), (False, 3, False), (True, 2, False), (True, 3, True)])
def test_state_tiles_on_persistent_workgroups(DQ, DV, BH, S, last, stride, init):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    if BH > 1000 and (stride, init) != (2, False) and stride != 1:
        pytest.skip("the most workgroups: two options only")
    q, k, v, i, f = (t.cuda() for t in make_qkvif(BH, 1, S, DQ, DV, seed=S, f_offset=3.0))
    dH = torch.randn(BH, 1, S, DV, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    g = torch.Generator().manual_seed(2)
    c0 = [torch.randn(BH, 1, *d, generator=g).cuda() for d in ((DQ, DV), (DQ,))] + [torch.zeros(BH, 1, 1).cuda()] if init else [None] * 3
    out = []
    pick = [0, BH // 3, BH - 1]
    for rows in (pick, slice(0, BH)):
        leaves = [t[rows].clone().requires_grad_(True) for t in (q, k, v, i, f)]
        H = mlstm_chunkwise__hip_xl_chunk(*leaves, *(None if t is None else t[rows] for t in c0), return_last_states=last,
                                          any_sequence_length=True, kernel_path="split", chunk_size_intra=128 * stride)
        H, state = H if last else (H, ())
        grads = torch.autograd.grad(H, leaves, dH[rows])
        out.append([t.detach() if rows is pick else t.detach()[pick] for t in (H, *state, *grads)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


# The forward of short prompts (H and the last state in one launch) at either side of its blocks of 32, of its slabs of 64, of a
# chunk and of its longest sequence; every head dimension it is built for and two it leaves to the other kernels.  H as above (the
# gated scores and the products are rounded once each); the last state carries 16 bits of every value and 24 of every weight:
# 2^-16 of the terms, whose sums are a few times smaller than their terms.
@pytest.mark.parametrize("S", [1, 31, 33, 63, 64, 65, 127, 128, 129, 257, 320, 321, 449, 512, 513])
@pytest.mark.parametrize("DQ,DV", [(64, 64), (64, 128), (128, 192), (128, 256), (256, 64), (256, 512), (512, 64), (512, 128), (192, 128)])
@pytest.mark.parametrize("opt", [dict(), dict(init=True), dict(sig=True, dtype=torch.float16), dict(sig=True, init=True, normalize=False)], ids=str)
def test_short_prompts(S, DQ, DV, opt):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    sig, init, dtype, normalize = opt.get("sig", False), opt.get("init", False), opt.get("dtype", torch.bfloat16), opt.get("normalize", True)
    NH = 3
    q, k, v, i, f = make_qkvif(1, NH, S, DQ, DV, seed=S + DQ, dtype=dtype, f_offset=3.0)
    g = torch.Generator().manual_seed(S)
    st = [None] * 3
    if init:
        st = [torch.randn(1, NH, DQ, DV, generator=g), torch.randn(1, NH, DQ, generator=g), None if sig else torch.randn(1, NH, 1, generator=g)]
    d = lambda t: None if t is None else t.double()
    L = next(x for x in (64, 32, 16, 8, 4, 2, 1) if S % x == 0)
    okw = dict(normalize=normalize) if sig else {}
    ref = O.chunkwise_fw(d(q), d(k), d(v), d(i), d(f), *(d(t) for t in st), chunk_size=L, siging=sig, **okw)
    cu = lambda t: None if t is None else t.cuda()
    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    for last in (True, False):
        with torch.no_grad():
            out = op(*(t.cuda() for t in (q, k, v, i, f)), *(cu(t) for t in st), return_last_states=last, any_sequence_length=True, **okw)
        H = out[0] if last else out
        assert rel_norm(H, ref["H"]) <= 6e-3
        if last:
            assert rel_norm(out[1][0], ref["C_last"]) <= 5e-5
            if normalize:
                assert rel_norm(out[1][1], ref["n_last"]) <= 5e-6
            if not sig:
                assert float((out[1][2].double().cpu() - ref["m_last"].reshape(out[1][2].shape)).abs().max()) <= 1e-5


@pytest.mark.parametrize("S,pos", [(40, 0), (200, 63), (317, 130), (512, 511)])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_short_prompts_values_not_finite(S, pos, which, bad):
    """A NaN or infinity at one position reaches no row more than 31 positions in front of it (its own block of 32 keys)."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    x = dict(zip("qkvif", (t.cuda() for t in make_qkvif(1, 2, S, 128, 128, seed=S, f_offset=3.0))))
    x[which][0, 0, pos, 5] = bad
    with torch.no_grad():
        H, _ = mlstm_chunkwise__hip_xl_chunk(*x.values(), return_last_states=True, any_sequence_length=True)
    assert bool(torch.isfinite(H[0, 1]).all()) and bool(torch.isfinite(H[0, 0, :pos // 32 * 32]).all())
    if which == "q":
        assert bool(torch.isfinite(H[0, 0, pos + 1:]).all())


@pytest.mark.parametrize("S", [1, 33, 65, 129, 257, 321, 496, 497])
@pytest.mark.parametrize("DQ,DV", [(64, 64), (128, 192), (256, 512), (512, 128)])
def test_short_prompts_in_used_memory(S, DQ, DV):
    """What the launches before left in the memory of the compute units does not matter: the same bits after launches full of NaN
    as after launches full of zeros, also where the last tile of 16 keys is the first of its block of 32."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    x = [t.cuda() for t in make_qkvif(1, 3, S, DQ, DV, seed=S + DQ, f_offset=3.0)]
    out = []
    for value in (0.0, float("nan")):
        fill = [torch.full((1, 128, 512, d), value, device="cuda", dtype=torch.bfloat16) for d in (DQ, DQ, DV)]
        gates = [torch.zeros(1, 128, 512, device="cuda")] * 2
        with torch.no_grad():
            mlstm_chunkwise__hip_xl_chunk(*fill, *gates, return_last_states=True, any_sequence_length=True)
            H, state = mlstm_chunkwise__hip_xl_chunk(*x, return_last_states=True, any_sequence_length=True)
        out.append((H, *state))
    for a, b in zip(*out):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.parametrize("S,DQ,DV", [(256, 64, 64), (317, 256, 512), (512, 128, 192)])
def test_short_prompts_from_a_large_state(S, DQ, DV):
    """float16 from a state beyond its range: finite, and as exact as from a small one, in the chunks where it has decayed."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    q, k, v, i, f = make_qkvif(1, 2, S, DQ, DV, seed=S, dtype=torch.float16, f_offset=3.0)
    g = torch.Generator().manual_seed(S)
    st = [1e5 * torch.randn(1, 2, DQ, DV, generator=g), 1e5 * torch.randn(1, 2, DQ, generator=g), torch.zeros(1, 2, 1)]
    with torch.no_grad():
        H, last = mlstm_chunkwise__hip_xl_chunk(*(t.cuda() for t in (q, k, v, i, f, *st)), return_last_states=True,
                                                any_sequence_length=True)
    ref = O.chunkwise_fw(*(t.double() for t in (q, k, v, i, f)), *(t.double() for t in st), chunk_size=S)
    assert rel_norm(H[:, :, 128:], ref["H"][:, :, 128:]) <= 1.5e-3  # an eighth of bf16's 6e-3 (three bits more), doubled
    assert rel_norm(last[0], ref["C_last"]) <= 5e-5 and rel_norm(last[1], ref["n_last"]) <= 5e-6


# One launch or scan + H (what a forward that keeps its workspace for a backward runs, here by its name): they round the same
# values once each, in another order of the sums, and so are equally far from 64 bits.  5 %: what a sample of this size scatters
# (2^15 values or more whose errors are independent between the rows: 1 / sqrt(S) at most).
@pytest.mark.parametrize("S,DQ,DV", [(129, 256, 512), (317, 256, 512), (512, 128, 256), (400, 64, 64), (300, 512, 128)])
@pytest.mark.parametrize("init,dtype", [(False, torch.bfloat16), (True, torch.bfloat16), (True, torch.float16)], ids=str)
def test_short_prompts_are_as_exact_as_scan_and_h(S, DQ, DV, init, dtype):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    NH = 4
    x = make_qkvif(1, NH, S, DQ, DV, seed=S, dtype=dtype, f_offset=3.0)
    g = torch.Generator().manual_seed(S)
    st = [torch.randn(1, NH, *d, generator=g) for d in ((DQ, DV), (DQ,), (1,))] if init else []
    ref = O.chunkwise_fw(*(t.double() for t in x), *(t.double() for t in st), chunk_size=S)
    err = []
    for path in ("auto", "split"):
        with torch.no_grad():
            H, last = mlstm_chunkwise__hip_xl_chunk(*(t.cuda() for t in (*x, *st)), return_last_states=True, any_sequence_length=True,
                                                    kernel_path=path)
        err.append([rel_norm(H, ref["H"]), rel_norm(last[0], ref["C_last"]), rel_norm(last[1], ref["n_last"])])
    print(err)
    assert err[0][0] <= 1.05 * err[1][0]
    for a, b in zip(err[0][1:], err[1][1:]):
        assert a <= max(1.05 * b, 2 ** -22)  # (states: below it, what the last rounding to 32 bits leaves)


# Without a gradient "auto" takes H of a short sequence from another kernel: each is within 2.5e-3 of 64 bits (above), so they are
# within the sum of it of each other; with the path named the bits are the same.
@pytest.mark.parametrize("S,DQ,DV", [(65, 64, 64), (317, 256, 512), (512, 128, 256)])
@pytest.mark.parametrize("path", ["auto", "split"])
@pytest.mark.parametrize("last", [False, True])
def test_forward_with_and_without_a_gradient(S, DQ, DV, path, last):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    x = [t.cuda().requires_grad_(True) for t in make_qkvif(1, 4, S, DQ, DV, seed=S, f_offset=3.0)]
    out = []
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            r = mlstm_chunkwise__hip_xl_chunk(*x, return_last_states=last, any_sequence_length=True, kernel_path=path)
        out.append([t.detach() for t in ((r[0], *r[1]) if last else (r,))])
    for a, b, tol in zip(*out, (5e-3, 1e-5, 1e-6, 0.0)):
        assert torch.equal(a, b) if path == "split" else rel_norm(a, b) <= tol


# Beyond 512 positions "auto" takes the same kernels with a gradient and without one: the same bits.
@pytest.mark.parametrize("NH,S,DQ,DV", [(4, 8300, 256, 512), (8, 8192, 128, 128), (12, 6016, 64, 256), (4, 4428, 128, 256), (1, 8200, 256, 512), (128, 700, 256, 512),
                                          (64, 513, 256, 512), (64, 700, 256, 512), (64, 1300, 256, 512), (64, 1700, 256, 512)])
@pytest.mark.parametrize("f_offset", [3.0, 9.0])
@pytest.mark.parametrize("last", [False, True])
def test_long_forward_with_and_without_a_gradient(NH, S, DQ, DV, f_offset, last):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    print(f"{NH} x {S} {DQ}/{DV} {f_offset} {last}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *s: torch.randn(1, NH, *s, device="cuda", generator=g)
    x = [t.requires_grad_(True) for t in (rn(S, DQ).bfloat16(), rn(S, DQ).bfloat16(), rn(S, DV).bfloat16(), rn(S), f_offset + rn(S))]
    out = []
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            r = mlstm_chunkwise__hip_xl_chunk(*x, return_last_states=last, any_sequence_length=True)
        out.append([t.detach() for t in ((r[0], *r[1]) if last else (r,))])
    for a, b in zip(*out):
        assert torch.equal(a, b)


# The short kernel scans the gates itself: 16-bit gates are the same numbers as those of 32 bits, so every bit is the same.  Gates in
# memory that is aligned to one element only.
@pytest.mark.parametrize("S", [1, 127, 128, 129, 257, 385, 512])
@pytest.mark.parametrize("gates", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sig", [False, True])
def test_short_prompts_gate_types(S, gates, sig):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    q, k, v, i, f = (t.cuda() for t in make_qkvif(1, 3, S, 64, 128, seed=S, f_offset=3.0))
    i, f = i.to(gates), f.to(gates)
    moved = [torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for t in (i, f)]
    out = []
    for x in ((i.float(), f.float()), (i, f), moved):
        with torch.no_grad():
            H, state = op(q, k, v, *x, return_last_states=True, any_sequence_length=True)
        out.append((H, *state[:2], *([] if sig else state[2:])))
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert torch.equal(a, b)


# Few workgroups scan the gates themselves, many take them from the pre-pass: the same numbers, so that a head's bits do not depend on
# how many there are (the rule is at three workgroups a CU: more than 768 for all heads here, fewer for two of them).
@pytest.mark.parametrize("S,DQ,DV,NH", [(17, 64, 128, 512), (64, 128, 192, 300), (65, 64, 64, 300), (128, 256, 64, 260), (129, 64, 64, 400),
                                        (200, 128, 256, 128), (320, 64, 64, 160)])
@pytest.mark.parametrize("opt", [dict(), dict(init=True), dict(sig=True, init=True), dict(dtype=torch.float16)], ids=str)
def test_short_prompts_gates_of_the_pre_pass(S, DQ, DV, NH, opt):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    init, sig, dtype = opt.get("init", False), opt.get("sig", False), opt.get("dtype", torch.bfloat16)
    if init:
        if S == 320:
            pytest.skip("from a state so many heads do not take the short kernel")
        NH = {200: 80, 129: 272}.get(S, NH)  # (as many as take one launch from a state)
    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    g = torch.Generator(device="cuda").manual_seed(S)
    rn = lambda *d: torch.randn(1, NH, *d, device="cuda", generator=g)
    x = [rn(S, DQ).to(dtype), rn(S, DQ).to(dtype), rn(S, DV).to(dtype), rn(S), 3 + rn(S)]
    state = [rn(DQ, DV), rn(DQ), None if sig else rn(1)] if init else [None] * 3
    _lib.profile_read()
    _lib.profile_enable(True)
    try:
        with torch.no_grad():
            H, last = op(*x, *state, return_last_states=True, any_sequence_length=True)
    finally:
        _lib.profile_enable(False)
    assert {"gates", "short_fw"} <= set(_lib.profile_read())
    cut = lambda t: None if t is None else t[:, NH - 2:].contiguous()
    with torch.no_grad():
        H2, last2 = op(*(cut(t) for t in x), *(cut(t) for t in state), return_last_states=True, any_sequence_length=True)
    for a, b in zip((H, *last), (H2, *last2)):
        assert torch.equal(cut(a), b)


# Up to 128 positions many heads take scan + H as well: the most heads that the short kernel takes, and one more.
@pytest.mark.parametrize("S,DQ,DV,init,most", [(128, 256, 512, False, 112), (65, 256, 512, True, 56), (64, 256, 512, True, 384),
                                               (100, 128, 256, False, 768), (128, 64, 192, True, 1024)])
@pytest.mark.parametrize("more", [0, 1])
def test_short_prompts_of_many_heads(S, DQ, DV, init, most, more):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    NH = most + more
    x = [torch.randn(1, NH, *d, device="cuda").bfloat16() for d in ((S, DQ), (S, DQ), (S, DV))]
    gates = [torch.randn(1, NH, S, device="cuda"), 3 + torch.randn(1, NH, S, device="cuda")]
    state = [torch.randn(1, NH, *d, device="cuda") for d in ((DQ, DV), (DQ,), (1,))] if init else [None] * 3
    _lib.profile_read()
    _lib.profile_enable(True)
    try:
        with torch.no_grad():
            mlstm_chunkwise__hip_xl_chunk(*x, *gates, *state, return_last_states=True, any_sequence_length=True)
    finally:
        _lib.profile_enable(False)
    assert ("short_fw" in _lib.profile_read()) == (more == 0)


def _fill_free_memory_with_nan(sizes):
    """What the allocator hands out next is full of NaN: blocks of up to 1 MiB, which have a pool of their own, and larger ones.
    Checked for blocks of `sizes` bytes."""
    torch.cuda.empty_cache()
    nan = lambda n_bytes: torch.full((n_bytes // 4,), float("nan"), device="cuda")
    full = [nan(1 << 30)] + [nan(1 << 20) for _ in range(64)]
    # and the gaps between blocks in use
    full += [nan(b["size"]) for seg in torch.cuda.memory_snapshot() for b in seg["blocks"] if b["state"] == "inactive"]
    del full
    probes = [torch.empty(n // 4, device="cuda") for n in sizes]
    for t in probes:
        assert bool(t.isnan().all())


# States that are known to be zero are neither written nor multiplied: the same bits as with zeros handed over, whatever the
# workspace holds (it is taken from memory full of NaN), for one window, several, and a ragged last one of either length.
@pytest.mark.parametrize("DQ,DV,path", [(256, 512, "auto"), (256, 512, "stream"), (256, 512, "split"), (64, 64, "auto"), (128, 256, "auto"),
                                        (512, 512, "auto"), (128, 128, "split")])
@pytest.mark.parametrize("NH,S", [(1, 64), (2, 256), (3, 384), (2, 600), (96, 700), (40, 1300)])
@pytest.mark.parametrize("stride,sig,dtype", [(2, False, torch.bfloat16), (2, True, torch.float16), (3, False, torch.bfloat16)], ids=str)
def test_zero_states_that_are_left_out(DQ, DV, path, NH, S, stride, sig, dtype):
    from mlstm_kernels_amd import _lib
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    if path == "stream":
        S = (S + 127) // 128 * 128
    lib, code = _lib.get_lib(), _lib.path_code(path)
    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    q, k, v, i, f = (t.cuda() for t in make_qkvif(1, NH, S, DQ, DV, seed=S, dtype=dtype, f_offset=3.0))
    dH = torch.randn(1, NH, S, DV, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    zeros = [torch.zeros(1, NH, *d, device="cuda") for d in ((DQ, DV), (DQ,), (1,))]
    out = []
    for init, d_last in ((None, False), (zeros, True)):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v, i, f)]
        st = dict(zip(("c_initial", "n_initial", "m_initial"), init)) if init else {}
        _fill_free_memory_with_nan([lib.mlstm_hip_chunkwise_fw_workspace_bytes(1, NH, S, DQ, DV, 1, code, stride),
                                    lib.mlstm_hip_chunkwise_bw_workspace_bytes(1, NH, S, DQ, DV, stride)])
        H, last = op(*leaves, **st, return_last_states=True, any_sequence_length=True, kernel_path=path, chunk_size_intra=128 * stride)
        if d_last:
            grads = torch.autograd.grad((H, last[0]), leaves, (dH, torch.zeros_like(last[0])))
        else:
            grads = torch.autograd.grad(H, leaves, dH)
        out.append([H.detach(), *(t.detach() for t in last), *grads])
    for name, a, b in zip(("H", "C", "n", "m", "dQ", "dK", "dV", "dI", "dF"), *out):
        assert torch.equal(a, b), name
        assert bool(torch.isfinite(a).all()), name


@pytest.mark.parametrize("S,DQ,DV,NH", [(1100, 64, 64, 4), (1100, 128, 128, 2), (300, 256, 512, 5), (700, 256, 512, 26)])
def test_items_that_are_no_multiple_of_eight(S, DQ, DV, NH):
    _run(S, DQ, DV, NH=NH, seed=S + NH)


# the tiled kernel with a workgroup for every column group of the most heads that fit the CUs, the window kernel with one more
@pytest.mark.parametrize("DQ,DV,S,NH", [(128, 384, 200, 21), (64, 320, 390, 6), (64, 448, 129, 9)])
@pytest.mark.parametrize("more", [0, 1])
def test_several_column_groups(DQ, DV, S, NH, more):
    _run(S, DQ, DV, NH=NH + more, seed=S + NH)


@pytest.mark.parametrize("S", [64, 200])
def test_stream_path_takes_whole_chunks(S):
    with pytest.raises(RuntimeError, match="S % 128 == 0"):
        _run(S, 256, 512, path="stream")


@pytest.mark.parametrize("S,chunk", [(1, 64), (65, 64), (200, 128), (1000, 64)])
def test_padding_adapter_without_padding(S, chunk):
    from mlstm_kernels_amd.torch.backend_module import mLSTMBackend, mLSTMBackendConfig

    backend = mLSTMBackend(mLSTMBackendConfig(mode="train_with_padding", chunk_size=chunk, return_last_states=False))
    q, k, v, i, f = make_qkvif(2, 2, S, 256, 512, seed=S)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v, i, f)]
    dH = torch.randn(2, 2, S, 512, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    grads = torch.autograd.grad(backend(*leaves), leaves, dH)
    S_pad = -(-S // chunk) * chunk
    padded = [torch.cat([t.cuda(), t.new_zeros(*t.shape[:2], S_pad - S, *t.shape[3:]).cuda()], dim=2).requires_grad_(True)
              for t in (q, k, v, i, f)]
    ref = torch.autograd.grad(mLSTMBackend(mLSTMBackendConfig(mode="train", chunk_size=chunk, return_last_states=False))(*padded)[:, :, :S],
                              padded, dH)
    for name, x, y in zip(("dQ", "dK", "dV", "dI", "dF"), grads, ref):
        assert rel_norm(x, y[:, :, :S]) <= 2e-3, name


@pytest.mark.parametrize("S", [1, 127, 2049])
@pytest.mark.parametrize("gates", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sig", [False, True])
def test_gradients_of_16_bit_gates(S, gates, sig):
    """dI and dF leave the kernel in the gates' type: those of the same gates in 32 bits, rounded once."""
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk, mlstm_siging_chunkwise__hip_xl_chunk

    op = mlstm_siging_chunkwise__hip_xl_chunk if sig else mlstm_chunkwise__hip_xl_chunk
    q, k, v, i, f = (t.cuda() for t in make_qkvif(1, 2, S, 64, 64, seed=S, f_offset=3.0))
    dH = torch.randn(v.shape, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    grads = []
    for gi, gf in ((torch.float32, torch.float32), (gates, gates), (gates, torch.float32)):
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v, i.to(gates).to(gi), f.to(gates).to(gf))]
        grads.append(torch.autograd.grad(op(*leaves, any_sequence_length=True), leaves, dH))
        assert grads[-1][3].dtype == gi and grads[-1][4].dtype == gf
    for other in grads[1:]:
        for a, b in zip(grads[0], other):
            assert torch.equal(a.to(b.dtype), b)
