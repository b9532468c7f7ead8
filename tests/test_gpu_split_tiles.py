"""Tiled product on the bf16 pipe for 64 output columns on either side of the number of rows where its
tiles change, last tiles of one row and of all, rows sent elsewhere."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 1535 * 128, 1535 * 128 + 1, 1536 * 128, 1536 * 128 + 129])
@pytest.mark.parametrize("scattered", [False, True])
def test_tiles_of_64_columns(n, scattered):
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cint, i64, ptr, stream
    r, f = 64, 64
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, r, device="cuda", generator=gen)
    wt = torch.randn(f, r, device="cuda", generator=gen)
    rows = torch.randperm(n, device="cuda", generator=gen).int() if scattered else None
    out = torch.full((n, f), float("nan"), device="cuda")
    _lib.call("final_product_wt", stream(), i64(n), cint(r), ptr(x), cint(f), ptr(wt),
              None if rows is None else ptr(rows), ptr(out))
    got = out if rows is None else out[rows.long()]
    expect = x.double() @ wt.double().t()
    mag = x.double().abs() @ wt.double().abs().t()
    # parts left out below 2^-24 of a product, 6 r float32 additions
    assert bool(((got.double() - expect).abs() <= (6 * r + 1) * 2.0 ** -24 * mag).all())
