"""q/k/v of a matrix whose rows are not as long as those of x: refused before anything is launched, at every number of rows."""
import pytest
import torch

from servelab_amd.kernels import HipOps, KernelError
from servelab_amd.kernels.tuning import Tuning
from servelab_amd.kernels.values import LinearWeight


class Recorded(HipOps):
    """The table's host side without a device: what it would launch is written down."""

    def __init__(self):
        Tuning().apply(self)
        self.act_dtype, self.device, self._num_cus = torch.bfloat16, torch.device("cpu"), 256
        self.use_block_products = self.fuse_rope = self.fuse_norms = self.tile_few_rows = True
        self._tuning, self._tuned, self._untiled = False, set(), None
        self.launched = []

    def _check(self, *a, **k):
        pass

    def _call(self, stem, name, *a):
        self.launched.append(name)


@pytest.mark.parametrize("M", [1, 16, 17, 64, 100, 300, 600])
@pytest.mark.parametrize("K_of_x", [512, 2048])
def test_rows_of_another_length_are_refused(M, K_of_x):
    ops, (nh, nkv, D) = Recorded(), (8, 2, 64)
    N, K = (nh + 2 * nkv) * D, 1024
    weight = LinearWeight(torch.zeros(N, K, dtype=torch.bfloat16), torch.zeros(N * K, dtype=torch.bfloat16))
    x = torch.zeros(M, K_of_x, dtype=torch.bfloat16)
    with pytest.raises(KernelError):
        ops.qkv_rope_store(x, weight, None, nh, nkv, D, None, None, None, None, None, 16)
    assert ops.launched == []
