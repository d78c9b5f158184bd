"""The matrix products of the prefill and the vision tower (csrc/pi05_mm.h), every tile and epilogue at the
sizes where a tile can go wrong: one row, a row past a tile's edge, a column remainder, one k-tile, fewer
k-tiles than a tile keeps in flight, uneven K splits, rows longer than the product.

Reference: the product of the same bf16 values in float64 on the CPU.  A sum of K fp32 terms in any order is
off by at most K 2^-24 times the sum of the terms' magnitudes, and a bf16 rounding by 2^-8 of the value (2^-9, and
the sum's error may move it over a rounding boundary)."""

import pytest
import torch

from pi05_infer import _ext

pytestmark = pytest.mark.gpu

BF16, GELU, F32, GEGLU = range(4)
TILES = ["256x256", "256x192", "192x256", "128x128", "128x96", "128x64", "64x96", "64x64"]
SIZES = [(1, 32, 64, 1), (63, 160, 128, 1), (65, 272, 832, 3), (257, 288, 192, 2), (200, 544, 1152, 5)]


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("epi", [BF16, GELU, F32, GEGLU], ids=["bf16", "gelu", "f32", "geglu"])
@pytest.mark.parametrize("cfg", range(8), ids=TILES)
def test_product(cfg, epi, size):
    m, n, k, split = size
    split = split if epi == F32 else 1
    n_out, n_w = (n // 32 * 16, n // 32 * 32) if epi == GEGLU else (n, n)
    lda, ldw, ldc = k + 64, k + 8, n_out + 12
    gen = torch.Generator().manual_seed(7)
    a = torch.randn(m, lda, generator=gen).to(torch.bfloat16)
    w = torch.randn(n_w, ldw, generator=gen).to(torch.bfloat16)
    bias = torch.randn(n_w, generator=gen) if epi in (BF16, GELU) else None
    mark = -77.0
    out = torch.full((split * m + 1, ldc), mark, dtype=torch.float32 if epi == F32 else torch.bfloat16, device="cuda")
    ag, wg, bg = a.cuda(), w.cuda(), bias.cuda() if bias is not None else None
    print(f"tile {TILES[cfg]} epi {epi} M={m} N={n_w} K={k} split={split}", flush=True)
    rc = _ext.load_prefix_library().pi05_debug_product(
        cfg, epi, ag.data_ptr(), wg.data_ptr(), out.data_ptr(), bg.data_ptr() if bg is not None else None, m, n_w, k, lda, ldw, ldc, split, None)
    if epi == GEGLU and TILES[cfg] in ("256x192", "128x96", "64x96"):
        assert rc == -1  # gate and up columns do not pair up in these tiles
        return
    assert rc == 0
    torch.cuda.synchronize()
    got = out.cpu().double()
    assert (got[split * m:] == mark).all() and (got[:, n_out:] == mark).all(), "written outside the product"
    a64, w64 = a[:, :k].double(), w[:, :k].double()
    ref, bound = a64 @ w64.T, k * 2.0**-24 * (a64.abs() @ w64.abs().T)
    got = got[: split * m, :n_out]
    if epi == F32:
        got = got.view(split, m, n_out).sum(0)
    elif epi == GEGLU:
        g, u = (x.reshape(m, n_out) for x in ref.view(m, -1, 2, 16).unbind(2))
        eg, eu = (x.reshape(m, n_out) + 2.0**-8 * y.abs() for x, y in zip(bound.view(m, -1, 2, 16).unbind(2), (g, u)))
        ref = _gelu(g) * u
        # |gelu'| <= 1.13; the error of each factor times the other one (with its own error), one rounding
        bound = 1.13 * eg * (u.abs() + eu) + _gelu(g).abs() * eu + 2.0**-8 * ref.abs() + 1e-6 * u.abs()
    else:
        ref, bound = ref + bias.double(), bound + 2.0**-24 * (ref.abs() + bias.double().abs())
        bound = bound + 2.0**-8 * ref.abs()
        if epi == GELU:
            ref, bound = _gelu(ref), 1.13 * bound + 2.0**-8 * _gelu(ref).abs() + 1e-6
    over = (got - ref).abs() - bound
    assert torch.isfinite(got).all() and over.max() <= 0, f"error {(got - ref).abs().max():.3e}, over its bound by {over.max():.3e}"


def test_products_that_do_not_fit_are_refused():
    lib = _ext.load_prefix_library()
    a, w, c = (torch.zeros(256 * 256, dtype=torch.bfloat16, device="cuda") for _ in range(3))

    def rc(cfg=7, epi=BF16, pa=a.data_ptr(), pw=w.data_ptr(), m=16, n=64, k=64, lda=64, ldw=64, ldc=64, split=1):
        return lib.pi05_debug_product(cfg, epi, pa, pw, c.data_ptr(), None, m, n, k, lda, ldw, ldc, split, None)

    assert rc() == 0
    torch.cuda.synchronize()
    for bad in (dict(cfg=8), dict(cfg=-1), dict(epi=4), dict(pa=None), dict(pa=a.data_ptr() + 2), dict(pw=w.data_ptr() + 8), dict(m=0), dict(n=24),
                dict(k=96, lda=96, ldw=96), dict(lda=32), dict(ldw=68), dict(ldc=32), dict(split=2), dict(split=2, epi=F32), dict(epi=GEGLU, n=48)):
        assert rc(**bad) == -1, bad


# 1800 rows: 8 to 29 m-tiles, the last band shorter than the others.  256 x 256 tiles: 272 and 536 on at most 256
# workgroups, so these take up to 3 tiles each; the splits' 288 tiles cross from split to split in one workgroup.
MANY = [(1800, 8512, 64, 1), (1800, 17056, 320, 1), (1800, 2080, 576, 4)]
CACHED = 256  # PI05_DEBUG_PRODUCT_CACHED
UNPAIRED = ("256x192", "128x96", "64x96")  # gate and up columns do not pair up in these tiles
MANY_CASES = [(c, e, s) for c in range(8) for e in (BF16, GELU, F32, GEGLU) for s in MANY
              if (s[3] > 1) == (e == F32) and not (e == GEGLU and TILES[c] in UNPAIRED)]


@pytest.mark.parametrize("cached", [0, CACHED], ids=["hbm", "cached"])
@pytest.mark.parametrize("cfg, epi, size", MANY_CASES, ids=[f"{TILES[c]}-epi{e}-{'x'.join(map(str, s))}" for c, e, s in MANY_CASES])
def test_product_over_many_tiles(cfg, epi, size, cached):
    """More tiles than workgroups and more m-tiles than a band.  Reference and bounds as above, in float64 on the GPU; a
    row or column that a tile leaves out, takes twice or swaps is off by whole values."""
    m, n, k, split = size
    n_out = n // 2 if epi == GEGLU else n
    gen = torch.Generator(device="cuda").manual_seed(9)
    a = torch.randn(m, k, generator=gen, device="cuda").to(torch.bfloat16)
    w = torch.randn(n, k, generator=gen, device="cuda").to(torch.bfloat16)
    bias = torch.randn(n, generator=gen, device="cuda") if epi in (BF16, GELU) else None
    mark = -77.0
    out = torch.full((split * m + 1, n_out), mark, dtype=torch.float32 if epi == F32 else torch.bfloat16, device="cuda")
    print(f"tile {TILES[cfg]} epi {epi} M={m} N={n} K={k} split={split} cached={cached}", flush=True)
    rc = _ext.load_prefix_library().pi05_debug_product(
        cfg, epi + cached, a.data_ptr(), w.data_ptr(), out.data_ptr(), bias.data_ptr() if bias is not None else None, m, n, k, k, k, n_out, split,
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert (out[split * m:] == mark).all(), "written outside the product"
    a64, w64 = a.double(), w.double().T.contiguous()
    ref, bound = a64 @ w64, k * 2.0**-24 * (a64.abs() @ w64.abs())
    got = out[: split * m].double()
    if epi == F32:
        got = got.view(split, m, n_out).sum(0)
    elif epi == GEGLU:
        g, u = (x.reshape(m, n_out) for x in ref.view(m, -1, 2, 16).unbind(2))
        eg, eu = (x.reshape(m, n_out) + 2.0**-8 * y.abs() for x, y in zip(bound.view(m, -1, 2, 16).unbind(2), (g, u)))
        ref = _gelu(g) * u
        bound = 1.13 * eg * (u.abs() + eu) + _gelu(g).abs() * eu + 2.0**-8 * ref.abs() + 1e-6 * u.abs()
    else:
        ref, bound = ref + bias.double(), bound + 2.0**-24 * (ref.abs() + bias.double().abs())
        bound = bound + 2.0**-8 * ref.abs()
        if epi == GELU:
            ref, bound = _gelu(ref), 1.13 * bound + 2.0**-8 * _gelu(ref).abs() + 1e-6
    over = (got - ref).abs() - bound
    assert torch.isfinite(got).all() and over.max() <= 0, f"error {(got - ref).abs().max():.3e}, over its bound by {over.max():.3e}"
