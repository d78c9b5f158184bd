"""Priming and the vision tower's embedding and attention at the sizes where their splits can go wrong.

Tolerances are those of the parity tests (bf16 on the GPU against the oracle's bf16 rounding points);
what must not depend on a layout or an alignment is compared bit for bit."""

from dataclasses import replace

import pytest
import torch

from oracle import denoise_oracle as O
from oracle import siglip_oracle as SO
from pi05_infer import synthetic as S
from pi05_infer.engine import Observation, OpenPi0InferConfig, OpenPi0Inference
from test_gpu_vision import G, _close, _context, _pixels

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def expert2():
    g = replace(S.ExpertGeometry(), depth=2)
    return g, S.make_weights(g)


@pytest.fixture(scope="module")
def tower2():
    return SO.random_weights(G, 2, seed=21, std=0.03)


@pytest.mark.parametrize("schedule", ["persistent", "graph"])
@pytest.mark.parametrize("plen", [1, 31, 32, 33, 77])
def test_priming_block_edges_strides_and_masks(expert2, plen, schedule):
    """One key, a block less one, a block, one more: against the oracle; K/V rows of 264 values and a uint8
    mask give the same bits as contiguous rows and a bool mask."""
    g, w = expert2
    print(f"case priming: B=2, P={plen}, {schedule}", flush=True)
    k, v = S.make_prefix_kv(g, plen, 2)
    pad = S.full_prefix_pad(plen, 2)
    pad[1, plen // 2:] = plen == 1
    x1 = S.make_noise(g, 2)
    model = OpenPi0Inference(OpenPi0InferConfig(num_steps=2), g)
    model.load_state_dict(w)
    model.to("cuda")
    model.set_schedule(schedule)
    act = model.sample_actions(Observation(k.cuda(), v.cuda(), pad.cuda()), x1.cuda())["actions"].clone()
    wide = [torch.full((*t.shape[:3], 264), float("nan"), dtype=t.dtype, device="cuda") for t in (k, v)]
    for t, src in zip(wide, (k, v)):
        t[..., :256] = src.cuda()
    obs = Observation(wide[0][..., :256], wide[1][..., :256], pad.cuda().to(torch.uint8))
    strided = model.sample_actions(obs, x1.cuda())["actions"]
    torch.cuda.synchronize()
    assert torch.equal(act, strided)
    ref, _ = O.sample_actions(w, O.geometry_from(g), k, v, pad, x1, 2)
    _close(ref, act.float(), f"P={plen} {schedule} actions")
    model.close()


@pytest.mark.parametrize("n_images", [1, 2, 5])
def test_vision_patch_rows_and_pixel_alignment(tower2, n_images):
    """16, 32 and 80 patch rows over a workgroup's stride (the last one uneven); pixels that are only 4-byte
    aligned give the same bits."""
    print(f"case vision: depth 2, {n_images} images", flush=True)
    layers, heads = tower2
    px = _pixels(n_images, 5)
    ctx, _keep = _context(layers, heads, n_images)
    got = ctx.forward(px.cuda()).clone()
    flat = torch.empty(px.numel() + 1, device="cuda")
    shifted = flat[1:].view(px.shape)
    shifted.copy_(px)
    assert shifted.data_ptr() % 16 == 4
    again = ctx.forward(shifted)
    torch.cuda.synchronize()
    assert torch.equal(got, again)
    ref = SO.image_features(px, layers, heads, G)
    for i in range(n_images):
        _close(ref[i], got[i].float(), f"image {i} of {n_images}")
    ctx.close()
