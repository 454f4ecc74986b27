"""LogicLayer kernels on rows of any number of samples: four samples per lane, the last lane of a row steps back.  Against the float64 kernels
on the same wiring, at row lengths around a lane's four samples, a row of 16 / 32 / 64 lanes and a second pass."""
import pytest
import torch

import convlogic_amd as C
from convlogic_amd.hip import difflogic_hip as D
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 5, 15, 16, 17, 18, 63, 65, 66, 67, 127, 130, 255, 257, 259, 513])
def test_rows_of_any_length(batch):
    torch.manual_seed(batch)
    i, o = 50, 83
    layer = C.LogicLayer(i, o, implementation="cuda").to(DEV)
    a, b, w = layer.indices_0, layer.indices_1, layer.weights.detach()
    which = torch.argsort(torch.cat([a, b]) * (2 * o) + torch.arange(o, device=DEV).repeat(2), stable=True)
    flat = torch.arange(o, device=DEV).repeat(2)[which].contiguous()
    start = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.bincount(torch.cat([a, b]), minlength=i).cumsum(0)]).contiguous()
    # rows behind a value that is not finite: it must not reach a neighbour
    x, gy = torch.rand(i, batch, device=DEV), torch.randn(o, batch, device=DEV)
    x[3, batch // 2] = float("inf")
    y, probs, folded = D.forward_logits(x, a, b, w)
    y64, probs64, folded64 = D.forward_logits(x.double(), a, b, w.double())
    gx, gx64 = (D.backward_x_folded(v, a, b, f, g, start, flat) for v, f, g in ((x, folded, gy), (x.double(), folded64, gy.double())))
    gw, gw64 = (D.backward_logits(v, a, b, p, g) for v, p, g in ((x, probs, gy), (x.double(), probs64, gy.double())))
    for got, want, bound in ((y, y64, 1e-6), (D.forward_folded(x, a, b, folded), y64, 1e-6), (gx, gx64, 1e-6 * o), (gw, gw64, 1e-6 * (batch + 16))):
        ok = want.isfinite()
        assert torch.equal(got.isfinite(), ok)
        # coefficients and values of magnitude <= 2 in sums of at most `o` consumers or `batch` samples of |grad_y| < 6: 2^-24 per step
        assert (got.double() - want)[ok].abs().max().item() <= bound * 6
