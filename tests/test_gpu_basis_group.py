"""Gradients of the basis projection by groups of centres, on tables made to hit the edges of the
kernels: lists of 0, 1, 16, 17, 64, 65 and several hundred pairs, a point listed twice by a
centre, and groups with more distinct points than the LDS table has rows."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 16, 17, 64, 65, 31, 33, 700, 5]


@pytest.mark.parametrize("c,k,points,centres", [
    (3, 8, 40, 1), (7, 64, 900, 37), (16, 16, 64, 10), (24, 32, 4000, 83), (64, 8, 300, 21),
    (64, 64, 5000, 64), (96, 16, 500, 129), (104, 32, 2000, 50), (128, 64, 1000, 33),
    (128, 32, 3000, 260), (128, 32, 40, 1), (128, 16, 40, 1), (64, 32, 700, 130)])
def test_grouped_gradients(c, k, points, centres):
    from tensorflow_graphics_point_clouds_amd import _lib
    host = _lib.host()
    rng = np.random.default_rng(c * 100 + k)
    lengths = np.resize(LENGTHS, centres)
    ranges = np.cumsum(lengths).astype(np.int32)
    owner = np.repeat(np.arange(centres), lengths)
    ids = np.concatenate([np.sort(rng.choice(points, n, replace=n > points))
                          for n in lengths] + [np.zeros(0, np.int64)])
    if len(ids) > 2:
        ids[2] = ids[1]                                  # listed twice by its centre
    pairs = np.stack([ids, owner], axis=1).astype(np.int32)
    basis = rng.standard_normal((len(ids), k)).astype(np.float32)
    feat = rng.standard_normal((points, c)).astype(np.float32)
    up = rng.standard_normal((centres, c, k)).astype(np.float32)
    args = [torch.from_numpy(x).cuda() for x in (basis, feat, pairs, ranges, up)]
    order = host.neighbourhood_order(args[2], args[3])
    assert np.array_equal(np.sort(order.cpu().numpy()), np.arange(centres))
    dbasis, dfeat = (x.cpu().numpy() for x in host.basis_proj_grads_grouped(*args, order))

    def reference(basis, feat, up):
        db = np.einsum("mck,mc->mk", up[owner], feat[ids])
        df = np.zeros_like(feat)
        np.add.at(df, ids, np.einsum("mck,mk->mc", up[owner], basis))
        return db, df
    # A sum of n float32 products in any order is off by less than (n + 1) 2^-24 times the sum of
    # their absolute values: n = c for dbasis, k times the pairs of a point for dfeat.
    wide = [x.astype(np.float64) for x in (basis, feat, up)]
    db, df = reference(*wide)
    db_mag, df_mag = reference(*map(np.abs, wide))
    terms = k * np.bincount(ids, minlength=points)[:, None]
    assert np.all(np.abs(dbasis - db) <= (c + 1) * 2.0 ** -24 * db_mag)
    assert np.all(np.abs(dfeat - df) <= (terms + 1) * 2.0 ** -24 * df_mag)


@pytest.mark.parametrize("c,k,spare", [(24, 8, 1), (96, 16, 700), (64, 64, 65), (128, 32, 70)])
def test_rows_behind_the_last_list_have_zero_gradients(c, k, spare):
    """A table of more rows than its lists hold (a search into a given capacity): the kernels per
    pair and channel leave zeros there, the grouped ones write them."""
    from tensorflow_graphics_point_clouds_amd import _lib
    host, stream, ptr, i64, cint = _lib.host(), _lib.stream, _lib.ptr, _lib.i64, _lib.cint
    gen = torch.Generator(device="cuda").manual_seed(c)
    centres, points, per = 300, 200, 20
    used, rows = centres * per, centres * per + spare
    pairs = torch.zeros(rows, 2, dtype=torch.int32, device="cuda")
    pairs[:used, 0] = torch.randint(points, (used,), device="cuda", generator=gen)
    pairs[:used, 1] = torch.arange(centres, device="cuda").repeat_interleave(per)
    ranges = torch.arange(per, used + 1, per, device="cuda", dtype=torch.int32)
    basis, feat, up = (torch.randn(*s, device="cuda", generator=gen)
                       for s in ((rows, k), (points, c), (centres, c, k)))
    order = host.neighbourhood_order(pairs, ranges)
    size = _lib.lib().mccnn_basis_proj_grads_grouped_workspace_bytes
    size.restype = _lib.csize
    ws = _lib.workspace(size(i64(centres), i64(rows)), "cuda")
    dbasis, dfeat = torch.full_like(basis, float("nan")), torch.empty_like(feat)
    _lib.call("basis_proj_grads_grouped", stream(), i64(points), cint(k), ptr(basis), cint(c),
              ptr(feat), i64(rows), ptr(pairs), i64(centres), ptr(ranges), ptr(order), ptr(up),
              ptr(ws), _lib.csize(ws.numel()), ptr(dbasis), ptr(dfeat))
    assert torch.equal(dbasis[used:], torch.zeros_like(dbasis[used:]))
    terms = up[pairs[:used, 1].long()].double() * feat[pairs[:used, 0].long()].double()[:, :, None]
    expect, size = terms.sum(1), terms.abs().sum(1)
    assert torch.all((dbasis[:used] - expect).abs() <= (c + 1) * 2.0 ** -24 * size)


@pytest.mark.parametrize("c,k,longest,window", [(64, 32, 40, 60), (128, 32, 66, 80), (128, 32, 130, 2000)])
def test_gradients_of_more_groups_than_blocks(c, k, longest, window):
    """More groups than the device takes blocks at once, with centres without pairs (which the order of
    the table's own has last), lists that share their points and groups whose points overflow the
    table.  A kernel for either gradient; larger tables, of which one forms both, are below."""
    from tensorflow_graphics_point_clouds_amd import _lib
    host = _lib.host()
    gen = torch.Generator(device="cuda").manual_seed(c + k)
    rand = lambda high, n: torch.randint(high, (n,), device="cuda", generator=gen)
    centres = 10 * 400 * 256 // longest
    points = centres
    lengths = rand(longest + 1, centres)
    lengths[5000:5400] = 0
    lengths[-1] = 0
    ranges = torch.cumsum(lengths, 0).int()
    owner = torch.repeat_interleave(torch.arange(centres, device="cuda"), lengths)
    ids = (owner + rand(window, len(owner))) % points        # (a point twice in a list among them)
    pairs = torch.stack([ids, owner], 1).int().contiguous()
    basis, feat, up = (torch.randn(*s, device="cuda", generator=gen)
                       for s in ((len(ids), k), (points, c), (centres, c, k)))
    dbasis, dfeat = host.basis_proj_grads_grouped(basis, feat, pairs, ranges, up,
                                                  host.neighbourhood_order(pairs, ranges))
    df, df_mag = (torch.zeros(points, c, device="cuda", dtype=torch.float64) for _ in range(2))
    for part in torch.arange(len(ids), device="cuda").split(16384):
        g, b, i = up[owner[part]].double(), basis[part].double(), ids[part]
        terms = g * feat[i].double()[:, :, None]
        assert torch.all((dbasis[part] - terms.sum(1)).abs() <=
                         (c + 1) * 2.0 ** -24 * terms.abs().sum(1))
        terms = g * b[:, None, :]
        df.index_add_(0, i, terms.sum(2))
        df_mag.index_add_(0, i, terms.abs().sum(2))
    terms = k * torch.bincount(ids, minlength=points)[:, None]
    assert torch.all((dfeat - df).abs() <= (terms + 1) * 2.0 ** -24 * df_mag)


def _check(dbasis, dfeat, basis, feat, ids, owner, up):
    """Against the sums in 64 bits; the bounds are those of test_grouped_gradients."""
    c, k = up.shape[1:]
    df, df_mag = (torch.zeros(feat.shape, device="cuda", dtype=torch.float64) for _ in range(2))
    for part in torch.arange(len(ids), device="cuda").split(16384):
        g, b, i = up[owner[part]].double(), basis[part].double(), ids[part]
        terms = g * feat[i].double()[:, :, None]
        assert torch.all((dbasis[part] - terms.sum(1)).abs() <=
                         (c + 1) * 2.0 ** -24 * terms.abs().sum(1))
        terms = g * b[:, None, :]
        df.index_add_(0, i, terms.sum(2))
        df_mag.index_add_(0, i, terms.abs().sum(2))
    terms = k * torch.bincount(ids, minlength=len(feat))[:, None]
    assert torch.all((dfeat - df).abs() <= (terms + 1) * 2.0 ** -24 * df_mag)


@pytest.mark.parametrize("order", ["index", "random"])
@pytest.mark.parametrize("c,k,longest,of_group", [(128, 32, 130, 350), (64, 16, 146, 400)])
def test_groups_without_pairs_between_others(order, c, k, longest, of_group):
    """Orders of the caller's own, by which a block that forms both gradients comes to one, two and three
    groups without pairs in a row between two others (the order of the table's own has them last);
    and a shape of a kernel for either."""
    from tensorflow_graphics_point_clouds_amd import _lib
    host = _lib.host()
    group, window = 8, 60
    gen = torch.Generator().manual_seed(3)
    rand = lambda high, n: torch.randint(high, (n,), generator=gen)
    blocks = torch.cuda.get_device_properties(0).multi_processor_count // 8 * 8
    rounds = (30 * 256 + blocks - 1) // blocks
    centres = rounds * blocks * group - 5
    slot = torch.arange(centres) // group                    # group of the centre by its place in the order
    empty = torch.tensor([[0, 0, 0, 0, 0, 0, 0, 0, 0], [0, 1, 0, 1, 0, 1, 0, 0, 0],
                          [0, 1, 1, 0, 1, 1, 0, 0, 1], [1, 0, 1, 1, 1, 0, 1, 0, 0]], dtype=torch.bool)
    lengths = torch.where(empty[slot % blocks % 4, slot // blocks % 9], 0, rand(longest + 1, centres))
    # what the library makes of these sizes
    assert lengths.sum() >= 9 << 18 and int(of_group / (int(lengths.sum()) / centres)) == group
    by_order = torch.arange(centres) if order == "index" else torch.randperm(centres, generator=gen)
    lengths = torch.empty_like(lengths).scatter_(0, by_order, lengths)
    owner = torch.repeat_interleave(torch.arange(centres), lengths)
    place = torch.empty_like(by_order).scatter_(0, by_order, torch.arange(centres))
    ids = (place[owner] + rand(window, len(owner))) % centres      # (centres of a group share points)
    pairs = torch.stack([ids, owner], 1).int().cuda()
    ranges = torch.cumsum(lengths, 0).int().cuda()
    gen = torch.Generator(device="cuda").manual_seed(4)
    basis, feat, up = (torch.randn(*s, device="cuda", generator=gen)
                       for s in ((len(ids), k), (centres, c), (centres, c, k)))
    dbasis, dfeat = host.basis_proj_grads_grouped(basis, feat, pairs, ranges, up, by_order.int().cuda())
    _check(dbasis, dfeat, basis, feat, ids.cuda(), owner.cuda(), up)


@pytest.mark.parametrize("rows,spare,longest,window", [
    ((9 << 18) - 1, 0, 40, 60), (9 << 18, 0, 40, 60), (9 << 18, 70, 66, 80), ((9 << 18) + 1, 1, 130, 2000),
    ((9 << 18) + 77, 700, 700, 900)])
def test_tables_on_either_side_of_both_gradients_at_once(rows, spare, longest, window):
    """Lists of 0, 1, .. `longest` pairs with points listed twice among them, groups that overflow
    their table, rows behind the last list; and one pair fewer than are worked on by one kernel."""
    from tensorflow_graphics_point_clouds_amd import _lib
    host = _lib.host()
    c, k, used = 128, 32, rows - spare
    gen = torch.Generator(device="cuda").manual_seed(longest)
    rand = lambda high, n: torch.randint(high, (n,), device="cuda", generator=gen)
    lengths = rand(longest + 1, 3 * used // longest)
    lengths[1000:1400] = 0
    centres = int((torch.cumsum(lengths, 0) < used).sum()) + 1
    ranges = torch.cumsum(lengths[:centres], 0).clamp(max=used).int()
    owner = torch.searchsorted(ranges, torch.arange(used, device="cuda", dtype=torch.int32), right=True)
    ids = (owner + rand(window, used)) % centres
    pairs = torch.zeros(rows, 2, dtype=torch.int32, device="cuda")
    pairs[:used] = torch.stack([ids, owner], 1).int()
    basis, feat, up = (torch.randn(*s, device="cuda", generator=gen)
                       for s in ((rows, k), (centres, c), (centres, c, k)))
    dbasis, dfeat = host.basis_proj_grads_grouped(basis, feat, pairs, ranges, up,
                                                  host.neighbourhood_order(pairs, ranges))
    assert not dbasis[used:].any()
    _check(dbasis, dfeat, basis, feat, ids, owner, up)
