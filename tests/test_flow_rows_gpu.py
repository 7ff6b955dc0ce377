"""mt_flow_euler_assemble where the embedder's rows pass through LDS (latent 64, hidden up to 1024) and
just past it, against the two launches it stands for, bit for bit."""
import pytest
import torch

import mingtts as mt
from _gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden", [8, 129, 1000, 1024, 1032])
def test_rows_of_64_equal_the_two_launches(gpu, hidden, dt):
    g = torch.Generator(device=gpu)
    g.manual_seed(hidden)
    r = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
    y0, pred, hist, cemb, temb = r(64), r(6, 64), r(64), r(hidden), r(hidden)
    xw, xb, null = r(hidden, 64).to(dt), r(hidden).to(dt), r(hidden).to(dt)
    say(f"flow rows hidden={hidden} {dt}")
    y1, x1 = y0.clone(), torch.zeros(6, hidden, device=gpu)
    mt.flow_euler_assemble(y1, pred, 2, 5, 2.0, 0.0625, hist, cemb, null, temb, xw, xb, x1)
    y2, x2 = y0.clone(), torch.zeros(6, hidden, device=gpu)
    mt.flow_euler(y2, pred, 2, 5, 2.0, 0.0625)
    mt.flow_assemble(y2, hist, cemb, null, temb, xw, xb, x2)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2) and torch.equal(x1, x2)
