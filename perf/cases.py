"""The calls whose speed this package is judged by, through its public entry points.

A case is a dict of plain values.  `listed()` names the ones that are always measured, `draw(rng)` gives more of the same
ranges, `prepare` makes what a program has in hand before the call, `run` makes one call, `work` states the bytes and
operations that the call cannot do without and `tolerance` how far another correct implementation may be off.

Kinds:
  decode   one token for every (batch, head): `mLSTMBackend` in inference mode with S = 1
  inplace  the same with the state matrix updated where it lies: `mlstm_recurrent_step__hip_fw(..., matC_new=matC_old)`
  tokens   T tokens for every (batch, head) in one call: `mlstm_recurrent_sequence__hip`
  prefill  a prompt of any length, last states returned: `mLSTMBackend` in inference mode
  train    forward and backward: `mLSTMBackend` in train or train_with_padding mode, or the chunkwise operator itself
           where the backend has no field for an option (head norm, recomputed states)
"""
import math

import torch

from mlstm_kernels_amd.torch.backend_module import mLSTMBackend, mLSTMBackendConfig
from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk
from mlstm_kernels_amd.torch.recurrent import mlstm_recurrent_sequence__hip, mlstm_recurrent_step__hip_fw

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
# (DHQK, DHHV, NH): the head shapes of this repository's benchmark and tests; the first one is the layer that the
# benchmark is about, and the one that is used most
_HEADS = [(256, 512, 8), (256, 512, 8), (256, 512, 8), (128, 256, 16), (128, 256, 16), (128, 128, 8), (64, 128, 8), (64, 64, 4),
          (256, 256, 8), (512, 1024, 4)]
_DEFAULT_HEADS = {"NH": 8, "dqk": 256, "dhv": 512}


def listed():
    h = dict(_DEFAULT_HEADS)
    return [
        # one user's chat: a token at a time, nothing else on the card
        {"name": "decode_1", "kind": "decode", "B": 1, **h, "dtype": "bf16", "gates": "bf16", "state": "fp32"},
        # a small serving batch
        {"name": "decode_16", "kind": "decode", "B": 16, **h, "dtype": "bf16", "gates": "bf16", "state": "fp32"},
        # a full serving batch whose state outgrows every cache, updated in place
        {"name": "decode_256_inplace", "kind": "inplace", "B": 256, **h, "dtype": "bf16", "gates": "fp32", "state": "fp32"},
        # several tokens at once: a draft that is verified, the short remainder of a prompt
        {"name": "tokens_16x16", "kind": "tokens", "B": 16, "T": 16, **h, "dtype": "bf16", "gates": "bf16", "state": "fp32"},
        # one prompt of ordinary, ragged length
        {"name": "prefill_prompt", "kind": "prefill", "B": 1, "S": 317, **h, "dtype": "bf16", "gates": "bf16", "chunk": 64, "init": False},
        # one long document
        {"name": "prefill_document", "kind": "prefill", "B": 1, "S": 10000, **h, "dtype": "bf16", "gates": "bf16", "chunk": 64, "init": False},
        # prompts of a batch that then decodes together
        {"name": "prefill_batch", "kind": "prefill", "B": 16, "S": 2048, **h, "dtype": "bf16", "gates": "fp32", "chunk": 128, "init": False},
        # the smallest training call: a toy model, a unit test, a quick experiment
        {"name": "train_small", "kind": "train", "B": 1, "S": 256, "NH": 4, "dqk": 64, "dhv": 64, "dtype": "bf16", "gates": "fp32", "chunk": 64,
         "sig": False, "normalize": True, "norm": "none", "pad": False, "last": True, "init": False, "recompute": False},
        # a layer of a language model on one device's share of the batch, the multi-head norm that follows the cell fused in
        {"name": "train_layer_norm", "kind": "train", "B": 16, "S": 1024, **h, "dtype": "bf16", "gates": "fp32", "chunk": 128,
         "sig": False, "normalize": True, "norm": "layer", "pad": False, "last": False, "init": False, "recompute": False},
        # narrower heads, sigmoid input gate
        {"name": "train_sig_narrow", "kind": "train", "B": 8, "S": 2048, "NH": 16, "dqk": 128, "dhv": 256, "dtype": "bf16", "gates": "fp32",
         "chunk": 128, "sig": True, "normalize": False, "norm": "none", "pad": False, "last": False, "init": False, "recompute": False},
        # ragged sequences, padded by the backend
        {"name": "train_padded", "kind": "train", "B": 8, "S": 1000, **h, "dtype": "bf16", "gates": "fp32", "chunk": 64,
         "sig": False, "normalize": True, "norm": "none", "pad": True, "last": False, "init": False, "recompute": False},
        # the benchmark's own layer at long context
        {"name": "train_long", "kind": "train", "B": 4, "S": 16384, **h, "dtype": "bf16", "gates": "fp32", "chunk": 128,
         "sig": False, "normalize": True, "norm": "none", "pad": False, "last": False, "init": False, "recompute": False},
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


# What a drawn chunkwise case may cost: half of the largest listed one's values in and out (batch * heads * positions *
# head dimensions), since small head dimensions take more time for each.
_MOST_VALUES = 65536 * 8 * (256 + 512) // 2


def draw(rng):
    dqk, dhv, nh = rng.choice(_HEADS)
    heads = {"NH": nh, "dqk": dqk, "dhv": dhv}
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    gates = rng.choice([dtype, "fp32"])
    kind = rng.choice(["decode", "inplace", "tokens", "prefill", "prefill", "train", "train", "train"])
    if kind in ("decode", "inplace"):
        most = min(512, 256 * 8 * 256 * 512 // (nh * dqk * dhv))
        return {"kind": kind, "B": _log_int(rng, 1, most), **heads, "dtype": dtype, "gates": gates,
                "state": rng.choice(["fp32", "fp32", "bf16"])}
    if kind == "tokens":
        T = _log_int(rng, 2, 128)
        most = min(256, 64 * 8 * 256 * 512 // (nh * dqk * dhv))
        return {"kind": kind, "B": _log_int(rng, 1, most), "T": T, **heads, "dtype": dtype, "gates": gates, "state": "fp32"}
    if kind == "prefill":
        S = _log_int(rng, 17, 16384)
        most = max(1, min(64, _MOST_VALUES // (nh * S * (dqk + dhv))))
        return {"kind": kind, "B": _log_int(rng, 1, most), "S": S, **heads, "dtype": dtype, "gates": gates,
                "chunk": rng.choice([64, 128]), "init": rng.random() < 0.3}
    pad = rng.random() < 0.25
    chunk = rng.choice([64, 128])
    S = _log_int(rng, 129, 16384)
    if not pad:
        S = max(chunk, S // chunk * chunk)
    most = max(1, min(64, _MOST_VALUES // (nh * S * (dqk + dhv))))
    case = {"kind": "train", "B": _log_int(rng, 1, most), "S": S, **heads, "dtype": dtype, "gates": gates, "chunk": chunk,
            "sig": False, "normalize": True, "norm": "none", "pad": pad, "last": False, "init": False, "recompute": False}
    if not pad:
        option = rng.choice(["plain", "plain", "sig", "norm", "last", "init", "recompute"])
        if option == "sig":
            case.update(sig=True, normalize=rng.random() < 0.5)
        elif option == "norm" and dhv <= 512:
            case.update(norm=rng.choice(["layer", "rms"]))
        elif option == "last":
            case.update(last=True)
        elif option == "init":
            case.update(init=True, last=True)
        elif option == "recompute":
            case.update(recompute=True)
    return case


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=dev, generator=gen)
    B, NH, dqk, dhv = case["B"], case["NH"], case["dqk"], case["dhv"]
    dt, gdt = _DTYPES[case["dtype"]], _DTYPES[case["gates"]]
    kind = case["kind"]
    steps = {"decode": 1, "inplace": 1, "tokens": case.get("T")}.get(kind) or case["S"]
    tok = (B, NH) if kind == "inplace" else (B, NH, steps)
    s = {"kind": kind, "case": case}
    # projections of normalised activations, an input gate around zero and a forget gate that mostly keeps
    s["q"], s["k"], s["v"] = rn(*tok, dqk).to(dt), rn(*tok, dqk).to(dt), rn(*tok, dhv).to(dt)
    gate = (B, NH, 1) if kind == "inplace" else tok
    s["i"], s["f"] = rn(*gate).to(gdt), (3 + rn(*gate)).to(gdt)
    if kind in ("decode", "inplace", "tokens"):
        sdt = _DTYPES[case["state"]]
        s["c"], s["n"], s["m"] = rn(B, NH, dqk, dhv).to(sdt), rn(B, NH, dqk).to(sdt), rn(B, NH, 1).to(sdt)
        s["sdt"] = sdt
        if kind == "inplace":
            s["n_next"], s["m_next"] = torch.empty_like(s["n"]), torch.empty_like(s["m"])
    elif case["init"]:
        s["c"], s["n"], s["m"] = 0.1 * rn(B, NH, dqk, dhv), 0.1 * rn(B, NH, dqk), torch.zeros(B, NH, 1, device=dev)
    else:
        s["c"] = s["n"] = s["m"] = None
    names = {"bf16": "bfloat16", "fp16": "float16", "fp32": "float32"}
    if kind in ("decode", "prefill"):
        s["backend"] = mLSTMBackend(mLSTMBackendConfig(
            mode="inference", chunk_size=case.get("chunk", 64), autocast_kernel_dtype=names[case["dtype"]],
            inference_state_dtype=names[case.get("state", "fp32")]))
    if kind == "train":
        s["dh"] = rn(B, NH, steps, dhv).to(dt)
        s["leaves"] = [s[x].requires_grad_(True) for x in ("q", "k", "v", "i", "f")]
        s["backend"] = mLSTMBackend(mLSTMBackendConfig(
            chunkwise_kernel="chunkwise--hip_xl_chunk" + ("_siging" if case["sig"] else ""), chunk_size=case["chunk"],
            mode="train_with_padding" if case["pad"] else "train", return_last_states=case["last"],
            autocast_kernel_dtype=names[case["dtype"]], normalize_siging=case["normalize"]))
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "inplace":
        h, (s["c"], n, m) = mlstm_recurrent_step__hip_fw(
            s["c"], s["n"], s["m"], s["q"], s["k"], s["v"], s["i"], s["f"],
            matC_new=s["c"], vecN_new=s["n_next"], scaM_new=s["m_next"], dtype_state=s["sdt"])
        s["n"], s["n_next"], s["m"], s["m_next"] = n, s["n"], m, s["m"]
        return h, s["c"], n, m
    if kind == "tokens":
        return mlstm_recurrent_sequence__hip(s["q"], s["k"], s["v"], s["i"], s["f"], s["c"], s["n"], s["m"],
                                             return_last_states=True, dtype_state=s["sdt"])
    if kind in ("decode", "prefill"):
        with torch.no_grad():
            return s["backend"](s["q"], s["k"], s["v"], s["i"], s["f"], s["c"], s["n"], s["m"])
    q, k, v, i, f = s["leaves"]
    if case["norm"] != "none" or case["recompute"]:
        out = mlstm_chunkwise__hip_xl_chunk(
            q, k, v, i, f, s["c"], s["n"], s["m"], return_last_states=case["last"], chunk_size=case["chunk"],
            autocast_kernel_dtype=_DTYPES[case["dtype"]], head_norm=case["norm"], recompute_states_in_bw=case["recompute"])
    else:
        out = s["backend"](q, k, v, i, f, s["c"], s["n"], s["m"])
    h = out[0] if case["last"] else out
    grads = torch.autograd.grad(h, s["leaves"], s["dh"])
    return out, grads


def work(case):
    bh, dqk, dhv = case["B"] * case["NH"], case["dqk"], case["dhv"]
    e, g = _BYTES[case["dtype"]], _BYTES[case["gates"]]
    kind = case["kind"]
    token = (2 * dqk + 2 * dhv) * e + 2 * g   # q, k, v and the gates in, h out
    state = dqk * dhv + dqk + 1
    if kind in ("decode", "inplace", "tokens"):
        T = case.get("T", 1)
        # each state value is decayed, gets its outer product added and enters the read-out
        return {"bytes": bh * (2 * state * _BYTES[case["state"]] + T * token), "flops": bh * T * 5 * dqk * dhv}
    S = case["S"]
    L = min(S, 128)
    fw = 4 * dqk * dhv + L * (dqk + dhv)      # per position: state update, read-out, the causal half inside a chunk
    nbytes = bh * S * token
    last = True if kind == "prefill" else case["last"]
    nbytes += bh * state * 4 * (int(last) + int(case["init"]))
    flops = bh * S * fw
    if kind == "train":
        nbytes += bh * S * ((2 * dqk + 2 * dhv) * e + 2 * g)   # dh in; dq, dk, dv and the gates' gradients out
        flops += bh * S * (8 * dqk * dhv + L * (3 * dqk + 2 * dhv))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] in ("decode", "inplace", "tokens"):
        # 32-bit arithmetic; outputs (and a 16-bit state) are rounded once, and a sum that ends near the middle of two
        # 16-bit values may be rounded the other way
        return {"rel": 2e-3, "max": 2e-2} if case["dtype"] == "bf16" or case["state"] == "bf16" else {"rel": 3e-4, "max": 3e-3}
    # 16-bit operands on the matrix units, 32-bit sums; rows whose normaliser nearly cancels are off by more than the rest
    fine = 0.25 if case["dtype"] == "fp16" else 1.0
    if case["kind"] == "prefill":
        return {"rel": 5e-3 * fine, "max": 0.3 * fine}
    # the forget gates' gradient is a sum over all later positions of differences of such products: its error grows with
    # the square root of the length
    rel = 1e-2 * fine * math.sqrt(1 + case["S"] / 2048)
    return {"rel": rel, "max": 30 * rel}
