"""Pair tables regrouped for another order of their centres: fewer centres than a wavefront takes,
last wavefronts that are not full, empty and long segments, both numbers of slots per wavefront."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,most", [(1, 5), (3, 300), (5, 0), (17, 40), (257, 9), (4099, 70),
                                    (131071, 6), (131072, 6), (131089, 40)])
@pytest.mark.parametrize("empty", [False, True])
def test_regrouped_segments(n, most, empty):
    from tensorflow_graphics_point_clouds_amd import _lib
    host = _lib.host()
    gen = torch.Generator(device="cuda").manual_seed(n)
    counts = torch.randint(0, most + 1, (n,), device="cuda", generator=gen)
    if empty:                                        # runs of empty segments, one long one
        counts[: n // 2] = 0
        counts[n // 2] = 700
    ranges = torch.cumsum(counts, 0)
    seg = torch.repeat_interleave(torch.arange(n, device="cuda"), counts)
    ids = torch.randint(0, n, (seg.shape[0],), device="cuda", generator=gen)
    pairs = torch.stack([ids, seg], dim=1).int().contiguous()
    order = torch.randperm(n, device="cuda", generator=gen)
    point_map = torch.randperm(n, device="cuda", generator=gen)
    pdf = torch.rand(n, device="cuda", generator=gen)
    out = host.reorder_ranges(ranges.int(), order.int())
    assert torch.equal(out.long(), torch.cumsum(counts[order], 0))
    new_seg = torch.repeat_interleave(torch.arange(n, device="cuda"), counts[order])
    start = torch.cat([out.new_zeros(1), out[:-1]]).long()
    first = (ranges - counts)[order]
    new_ids = ids[first[new_seg] + torch.arange(seg.shape[0], device="cuda") - start[new_seg]]
    got = host.reorder_pairs(ranges.int(), pairs, order.int(), out, None)
    assert torch.equal(got.long(), torch.stack([new_ids, new_seg], dim=1))
    got = host.reorder_pairs(ranges.int(), pairs, order.int(), out, point_map.int())
    assert torch.equal(got.long(), torch.stack([point_map[new_ids], new_seg], dim=1))
    assert torch.equal(host.reorder_pdf(ranges.int(), pairs, order.int(), out, pdf), pdf[new_ids])
