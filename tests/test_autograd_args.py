"""The autograd function's micro-kernel argument: any form of the number, as the other entries take it."""
import numpy as np
import pytest
import torch

import stkfmm_amd as S
from stkfmm_amd.autograd import P2PFunction

FORMS = [int, np.int64, np.array, torch.tensor, str, S.UKER]


@pytest.mark.parametrize("form", FORMS, ids=["int", "int64", "0-d array", "0-d tensor", "text", "enum"])
def test_micro_kernel_in_any_form(form):
    x = torch.zeros((3, 3), dtype=torch.float64)
    with pytest.raises(Exception) as e:  # host tensors: refused, but not for want of an adjoint kernel
        P2PFunction.apply(form(int(S.UKER.STOKES_VEL)), 0, x, x, x)
    assert "adjoint kernel" not in str(e.value) and not isinstance(e.value, TypeError)
    with pytest.raises(ValueError, match="no adjoint kernel for LAPLACE_PGRADGRAD"):
        P2PFunction.apply(form(int(S.UKER.LAPLACE_PGRADGRAD)), 0, x, x[:, :1], x)
