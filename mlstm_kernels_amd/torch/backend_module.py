"""``mLSTMBackend``: the operator-level entry point, with the configuration fields, defaults, validation
and mode logic of mlstm_kernels/torch/backend_module.py:43-218 in the reference.  Only the kernel-name
defaults differ: this package ships the HIP kernels, so they are the defaults."""
from __future__ import annotations

from dataclasses import dataclass
from functools import partial
from typing import Literal

import torch
from torch import nn

from .. import _lib
from . import get_mlstm_kernel, get_mlstm_sequence_kernel, get_mlstm_step_kernel
from .recurrent.hip_step import _STATE_CODES, mlstm_recurrent_step__hip
from .kernel_wrappers import wrap_chunkwise__arbitrary_sequence_length, wrap_chunkwise__pad_zeros

ChunkwiseKernelType = Literal["chunkwise--hip_xl_chunk", "chunkwise--hip_xl_chunk_siging"]
SequenceKernelType = Literal["native_sequence__hip"]
StepKernelType = Literal["hip"]
DtypeType = Literal["float32", "bfloat16", "float16"]
BackendModeType = Literal["train", "train_with_padding", "inference"]


@dataclass
class mLSTMBackendConfig:
    chunkwise_kernel: ChunkwiseKernelType = "chunkwise--hip_xl_chunk"
    """Kernel for chunkwise-parallel processing (training, prefill)."""
    sequence_kernel: SequenceKernelType = "native_sequence__hip"
    """Token-loop kernel for the short remainder of a prefill in inference mode."""
    step_kernel: StepKernelType = "hip"
    """Single-step kernel for generation in inference mode."""
    mode: BackendModeType = "train"
    """'train', 'train_with_padding' (inputs zero-padded to a multiple of chunk_size) or 'inference'."""
    chunk_size: int = 64
    return_last_states: bool = True
    """Return the last (C, n, m) in training mode; inference mode always returns them."""
    autocast_kernel_dtype: DtypeType = "bfloat16"
    """Under autocast all inputs are cast to this dtype before the kernel is called."""
    eps: float = 1e-6
    inference_state_dtype: DtypeType = "float32"
    normalize_siging: bool = True
    """Normalise H in the sigmoid-input-gate kernels (ignored by mLSTMexp kernels)."""

    def __post_init__(self):
        if self.return_last_states and "parallel" in self.chunkwise_kernel:
            raise ValueError("return_last_states=True is not supported with parallel kernels.")
        if self.return_last_states and self.mode == "train_with_padding":
            raise ValueError("return_last_states=True is not supported with train_with_padding mode.")


class mLSTMBackend(nn.Module):
    """Wraps the mLSTM kernels behind one ``forward(q, k, v, i, f, ...)`` for training and inference."""

    config_class = mLSTMBackendConfig
    _native_step = None  # (here as well: modules pickled before there was one have none of their own)

    def __init__(self, config: mLSTMBackendConfig):
        super().__init__()
        self.config = config
        self.chunkwise_kernel_fn = get_mlstm_kernel(config.chunkwise_kernel)
        self.sequence_kernel_fn = get_mlstm_sequence_kernel(config.sequence_kernel)
        self.step_kernel_fn = get_mlstm_step_kernel(config.step_kernel)
        state_dtype = getattr(torch, config.inference_state_dtype)
        kernel_dtype = getattr(torch, config.autocast_kernel_dtype)
        self._inference_fn = partial(
            wrap_chunkwise__arbitrary_sequence_length,
            mlstm_chunkwise_kernel=self.chunkwise_kernel_fn,
            mlstm_sequence_kernel=partial(self.sequence_kernel_fn, dtype_state=state_dtype),
            mlstm_step_kernel=partial(self.step_kernel_fn, dtype_state=state_dtype),
            chunk_size=config.chunk_size,
            eps=config.eps,
            autocast_kernel_dtype=kernel_dtype,
            return_last_states=True,
            dtype_state=state_dtype,
        )
        # One token from given states goes to the native step without the layers in between (sequence adapter, partials, step
        # function): a call of one sequence, whose kernel takes 6.6 us, 10.9 -> 9.4 us.  None: another step kernel or state type
        if self.step_kernel_fn is mlstm_recurrent_step__hip and state_dtype in _STATE_CODES:
            self._native_step = (None, None, None, config.eps, _STATE_CODES[state_dtype])
        train_fn = partial(
            self.chunkwise_kernel_fn,
            autocast_kernel_dtype=kernel_dtype,
            eps=config.eps,
            chunk_size=config.chunk_size,
        )
        if "with_padding" in config.mode:
            train_fn = partial(wrap_chunkwise__pad_zeros, mlstm_chunkwise_kernel=train_fn)
        self._train_fn = train_fn

    def forward(
        self,
        q: torch.Tensor,  # (B, NH, S, DHQK)
        k: torch.Tensor,  # (B, NH, S, DHQK)
        v: torch.Tensor,  # (B, NH, S, DHHV)
        i: torch.Tensor,  # (B, NH, S)
        f: torch.Tensor,  # (B, NH, S)
        c_initial: torch.Tensor = None,  # (B, NH, DHQK, DHHV)
        n_initial: torch.Tensor = None,  # (B, NH, DHQK)
        m_initial: torch.Tensor = None,  # (B, NH, 1)
        return_last_states: bool = None,
        mode: Literal["train", "inference"] = None,
    ):
        """Returns H (B,NH,S,DHHV), or (H, (C, n, m)) when last states are requested / in inference mode."""
        if mode is None:
            mode = self.config.mode
        if "train" in mode:
            if return_last_states is None:
                return_last_states = self.config.return_last_states
            if self.config.mode == "train_with_padding":
                assert not return_last_states, "return_last_states=True is not supported with train_with_padding mode."
            kwargs = dict(q=q, k=k, v=v, i=i, f=f, c_initial=c_initial, n_initial=n_initial,
                          m_initial=m_initial, return_last_states=return_last_states)
            if "siging" in self.config.chunkwise_kernel:
                kwargs["normalize"] = self.config.normalize_siging
            return self._train_fn(**kwargs)
        elif "inference" in mode:
            if c_initial is not None and self._native_step is not None and q.dim() == 4:
                # (None back: more than one token, or an argument to be made, converted or refused)
                out = _lib.get_host().step(c_initial, n_initial, m_initial, q, k, v, i, f, *self._native_step)
                if out is not None:
                    return out
            return self._inference_fn(q=q, k=k, v=v, i=i, f=f, c_initial=c_initial, n_initial=n_initial,
                                      m_initial=m_initial)
        else:
            raise ValueError(f"Unknown mode: {self.config.mode}")

    def extra_repr(self) -> str:
        return f"{self.config}"
