"""What a context chooses when it is created: every product is timed as it then runs."""

import pytest
import torch

from pi05_infer import _ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [1, 10])
def test_projector_is_timed_as_it_runs(depth):
    """The weights of 10 layers (307 MB) do not stay in the 256 MB cache behind the L2s, those of one do; the
    projector's follow them, so its tile is timed with W from HBM where the layers' products are."""
    print(f"case vision choices: depth {depth}, 1 image", flush=True)
    d = _ext.vision_default_dims()
    d.depth, d.n_images = depth, 1
    ctx = _ext.VisionContext(d, torch.device("cuda"))
    got = ctx.products()
    ctx.close()
    print(got, flush=True)
    assert {n: p["cold"] for n, p in got.items()} == dict.fromkeys(got, depth == 10)
