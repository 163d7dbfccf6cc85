"""Line gradients on both sides of the line count from which a line has one lane
instead of eight: a batch of copies of one scene against that scene alone."""
import math

import numpy as np
import pytest
import torch

from tileink_amd import diff

pytestmark = pytest.mark.gpu

LANES_MAX = 1 << 20  # TK_LINE_LANES_MAX


def test_copies_of_a_scene_have_its_line_gradients(ctx):
    scene = diff.random_scene(3, 96, 80, fills=1500, radius_mu=math.log(9.0))
    verts, counts = scene.polygons()
    weight = np.random.default_rng(1).normal(size=(80 * 96, 4))

    def gradients(n):
        plan = diff.Plan(ctx, [scene] * n, [verts] * n, [counts] * n)
        colors = plan.full_paint(torch.cat([scene.paint_records()] * n)).to("cuda", torch.float32)
        image = plan.forward(colors)
        assert image.shape[0] == plan.pixels
        grad = torch.zeros((plan.pixels, 4), dtype=torch.float32, device="cuda")
        for at in plan.offsets:
            grad[at:at + 80 * 96] = torch.as_tensor(weight, dtype=torch.float32, device="cuda")
        lines, _ = plan.backward(grad)
        return lines.cpu().double().numpy()

    one = gradients(1)
    below = (LANES_MAX - 1) // len(one)
    assert 1 < below < 200
    for copies in (below, below + 1):
        got = gradients(copies)
        assert (len(got) >= LANES_MAX) == (copies > below)
        # The same FP32 terms, some 10 to 100 a line, summed in another order.
        assert np.abs(got.reshape(copies, *one.shape) - one).max() <= 1e-5 * np.abs(one).max()
