"""Operand preparation of the layers through the C ABI: padded row gathers and the forms of a
layer's weights, compared with the same arrangement made of tensor operations (copies: exact)."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def abi():
    from tensorflow_graphics_point_clouds_amd import _lib
    _lib.lib()
    return _lib


@pytest.mark.parametrize("n,stride,first,cols,out_cols,permuted", [
    (1, 1, 0, 1, 16, True), (1000, 6, 0, 6, 16, True), (513, 48, 16, 32, 64, True),
    (77, 64, 4, 12, 16, False), (300, 50, 3, 7, 16, True), (64, 128, 0, 128, 128, True)])
def test_gather_rows_padded(abi, n, stride, first, cols, out_cols, permuted):
    gen = torch.Generator(device="cuda").manual_seed(n)
    src = torch.randn((n, stride), device="cuda", generator=gen)
    rows = torch.randperm(n, device="cuda", generator=gen).int() if permuted else None
    out = torch.full((n, out_cols), float("nan"), device="cuda")
    abi.call("gather_rows_padded", abi.stream(), abi.i64(n), abi.ptr(rows), abi.ptr(src),
             abi.i64(stride), abi.cint(first), abi.cint(cols), abi.cint(out_cols), abi.ptr(out))
    expect = torch.zeros_like(out)
    picked = src[:, first:first + cols]
    expect[:, :cols] = picked if rows is None else picked[rows.long()]
    assert torch.equal(out, expect)


# (C, H, G, mlps of the layer, first, per, C', H', G')
@pytest.mark.parametrize("c,h,g,mlps,first,per,cp,hp,gp", [
    (1, 8, 16, 1, 0, 1, 16, 16, 16), (6, 8, 8, 4, 2, 2, 16, 8, 8), (64, 16, 64, 1, 0, 1, 64, 16, 64),
    (48, 15, 45, 1, 0, 1, 64, 16, 64), (5, 3, 7, 4, 0, 4, 16, 4, 8)])
def test_pack_and_unpack_layer_weights(abi, c, h, g, mlps, first, per, cp, hp, gp):
    dims = 3
    gen = torch.Generator(device="cuda").manual_seed(c + h)
    final = torch.randn((mlps, c * h, g), device="cuda", generator=gen)
    kw = torch.randn((mlps, dims, h), device="cuda", generator=gen)
    kb = torch.randn((mlps, h), device="cuda", generator=gen)
    k, f = per * hp, per * gp
    dense = torch.zeros((cp, per, hp, per, gp), device="cuda")
    blocks = final.reshape(mlps, c, h, g)
    for m in range(per):
        dense[:c, m, :h, m, :g] = blocks[first + m]
    dense = dense.reshape(cp, k, f)
    new = lambda *s: torch.full(s, float("nan"), device="cuda")
    w, wt, w2, w2t = new(cp * k, f), new(f, cp * k), new(f * k, cp), new(cp, f * k)
    kwp, kbp = new(per, dims, hp), new(per * hp)
    shape = [abi.cint(v) for v in (dims, c, h, g, first, per, cp, hp, gp)]
    abi.call("pack_layer_weights", abi.stream(), *shape, *[abi.ptr(t) for t in (
        final, kw, kb, w, wt, w2, w2t, kwp, kbp)])
    assert torch.equal(w, dense.reshape(cp * k, f)) and torch.equal(wt, w.t())
    assert torch.equal(w2t.reshape(cp, f, k), dense.permute(0, 2, 1))
    assert torch.equal(w2, w2t.t())
    pad = torch.nn.functional.pad
    assert torch.equal(kwp, pad(kw[first:first + per], (0, hp - h)))
    assert torch.equal(kbp.reshape(per, hp), pad(kb[first:first + per], (0, hp - h)))

    ddense = torch.randn((cp, f * k), device="cuda", generator=gen)
    dfinal, dkw, dkb = new(mlps, c * h, g), new(mlps, dims, h), new(mlps, h)
    abi.call("unpack_layer_grads", abi.stream(), *shape, *[abi.ptr(t) for t in (
        ddense, kwp, kbp, dfinal, dkw, dkb)])
    d = ddense.reshape(cp, per, gp, per, hp)
    for m in range(per):
        got = dfinal[first + m].reshape(c, h, g)
        assert torch.equal(got, d[:c, m, :g, m, :h].permute(0, 2, 1))
    assert torch.equal(dkw[first:first + per], kwp[:, :, :h])
    assert torch.equal(dkb[first:first + per], kbp.reshape(per, hp)[:, :h])


@pytest.mark.parametrize("n,r,cols,padded", [(1, 256, 48, 64), (3000, 256, 48, 64), (700, 1024, 96, 128),
                                             (5000, 1024, 160, 192), (33, 2048, 80, 128)])
def test_padded_columns_leave_the_bits_alone(n, r, cols, padded):
    """The product with zero columns behind the weights equals the one without, bit for bit."""
    from ctypes import c_int64
    from tensorflow_graphics_point_clouds_amd import _lib
    from tensorflow_graphics_point_clouds_amd._lib import cint, ptr, stream
    gen = torch.Generator(device="cuda").manual_seed(n + r)
    x = torch.randn(n, r, device="cuda", generator=gen)
    w = torch.randn(r, cols, device="cuda", generator=gen)
    wide = torch.nn.functional.pad(w, (0, padded - cols)).contiguous()
    expect, got = torch.empty(n, cols, device="cuda"), torch.empty(n, padded, device="cuda")
    _lib.call("final_product", stream(), c_int64(n), cint(r), ptr(x), cint(cols), ptr(w),
              ptr(None), ptr(expect))
    _lib.call("final_product_padded", stream(), c_int64(n), cint(r), ptr(x), cint(padded),
              cint(cols), ptr(wide), ptr(None), ptr(got))
    assert torch.equal(got[:, :cols], expect)
