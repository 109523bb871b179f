"""The chunkwise operator has no forward-mode derivative: tangents are refused, with and without reverse mode, and not dropped."""
import pytest
import torch

from helpers import make_qkvif

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("which", range(5))
def test_tangents_are_refused(which, reverse):
    from mlstm_kernels_amd.torch.chunkwise import mlstm_chunkwise__hip_xl_chunk

    args = [t.cuda() for t in make_qkvif(1, 1, 128, 64, 64, seed=0)]
    if reverse:
        args[0].requires_grad_(True)
    mlstm_chunkwise__hip_xl_chunk(*args)
    with torch.autograd.forward_ad.dual_level():
        args[which] = torch.autograd.forward_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(RuntimeError, match="jvp"):
            mlstm_chunkwise__hip_xl_chunk(*args)
