"""The C-ABI library loads without a GPU, exports every symbol the header
declares, and rejects invalid arguments before touching the device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "mccnn_hip.h")
LIB = os.path.join(ROOT, "tensorflow_graphics_point_clouds_amd", "libmccnn_hip.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        pytest.fail("libmccnn_hip.so is not built; run __graft_entry__.build()")
    handle = ctypes.CDLL(LIB)
    handle.mccnn_last_error.restype = ctypes.c_char_p
    return handle


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mccnn_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported(lib):
    names = declared_symbols()
    assert len(names) >= 20
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_abi_version(lib):
    assert lib.mccnn_abi_version() == 1


def test_invalid_arguments_return_status_not_abort(lib):
    i64 = ctypes.c_int64
    rc = lib.mccnn_compute_keys(None, i64(10), 7, None, i64(10), None, i64(1), 7, None, 7, None,
                                7, None, None)
    assert rc == 1 and b"dimension" in lib.mccnn_last_error()
    rc = lib.mccnn_compute_keys(None, i64(10), 3, None, i64(9), None, i64(1), 3, None, 3, None,
                                3, None, None)
    assert rc == 1 and b"batch ids" in lib.mccnn_last_error()
    # K must be 8/16/32/64, C < 8 or a multiple of 8, pairs need two columns
    args = lambda k, c, cols: (None, i64(5), k, None, i64(4), c, None, i64(5), 2, cols, None,
                               i64(3), None, None)
    assert lib.mccnn_basis_proj(*args(12, 8, 2)) == 1
    assert lib.mccnn_basis_proj(*args(8, 12, 2)) == 1
    assert lib.mccnn_basis_proj(*args(8, 8, 3)) == 1
    # sampling and pdf modes
    total = i64(0)
    rc = lib.mccnn_sampling_count(None, 2, i64(4), 3, None, i64(4), None, i64(4), None, 3, None,
                                  i64(4), 2, 2, None, i64(4), None, None, ctypes.c_size_t(0),
                                  ctypes.byref(total))
    assert rc == 1 and b"mode" in lib.mccnn_last_error()
    rc = lib.mccnn_compute_pdf(None, i64(4), 3, None, i64(4), 2, 2, None, i64(5), None, 3, None,
                               3, None, 0, None)
    assert rc == 1 and b"same points as samples" in lib.mccnn_last_error()
    host = (ctypes.c_int32 * 3)(1, 1, 1)
    rc = lib.mccnn_build_grid_ds(None, i64(4), None, 3, None, 3, host, 0, None)
    assert rc == 1 and b"batch size" in lib.mccnn_last_error()


def test_grid_in_one_call_wants_both_host_outputs_or_neither(lib):
    """The shape without the key width was written through a null pointer; neither is enough only
    where the grid is one launch (more clouds than a block keeps the extents of are not)."""
    i64, sz, vp = ctypes.c_int64, ctypes.c_size_t, ctypes.c_void_p
    cells, bits = (ctypes.c_int32 * 3)(), ctypes.c_int(0)
    lib.mccnn_build_grid_single_launch_max.restype = i64
    most = lib.mccnn_build_grid_single_launch_max()

    def status(points, batch, shape, width):
        rc = lib.mccnn_build_grid_pinned(None, i64(points), 3, None, None, batch, *[None] * 12,
                                         sz(1 << 40), shape, width)
        assert rc == 1
        return lib.mccnn_last_error()
    for points in (4, most, most + 1):
        assert b"or neither" in status(points, 2, cells, None)
        assert b"or neither" in status(points, 2, None, ctypes.byref(bits))
    single = lib.mccnn_build_grid_is_single_launch
    for points, batch, expect in ((1, 1, 1), (most, 170, 1), (most, 171, 0), (most + 1, 1, 0),
                                  (0, 1, 0), (5, 0, 0), (5, 1 << 30, 0)):
        assert single(i64(points), 3, batch) == expect, (points, batch)
        message = status(points, batch, None, None)
        assert (b"null tensor" if expect else b"needs host outputs") in message


def test_pointconv_density_entry_points_validate_before_the_device(lib):
    i64, sz = ctypes.c_int64, ctypes.c_size_t
    rc = lib.mccnn_pointconv_density(None, i64(5), None, 2, None, None, None, None, None, None, None)
    assert rc == 1 and b"point_column" in lib.mccnn_last_error()
    assert lib.mccnn_pointconv_density(None, i64(0), None, 0, None, None, None, None, None, None,
                                       None) == 0
    rc = lib.mccnn_pointconv_density_grads(None, i64(5), None, 0, None, None, None, None, None, None,
                                           None, 5, None, None, sz(0), None)
    assert rc == 1 and b"slabs" in lib.mccnn_last_error()
    lib.mccnn_pointconv_density_grads_workspace_bytes.restype = sz
    assert lib.mccnn_pointconv_density_grads_workspace_bytes(i64(10 ** 6)) >= 49 * 4


def test_layer_entry_points_reject_uncovered_shapes(lib):
    i64, sz = ctypes.c_int64, ctypes.c_size_t
    assert lib.mccnn_mc_conv_supported(3, 64, 16) == 1 and lib.mccnn_mc_conv_supported(3, 24, 16) == 0
    assert lib.mccnn_mc_conv_layer_supported(3, 64, 16, 64) == 1
    assert lib.mccnn_mc_conv_layer_supported(4, 64, 16, 64) == 0
    assert lib.mccnn_weight_grad_product_supported(64, 1024) == 1
    assert lib.mccnn_weight_grad_product_supported(48, 1024) == 0
    assert lib.mccnn_projection_grad_product_supported(64, 1024) == 1
    assert lib.mccnn_projection_grad_product_supported(128, 1024) == 1
    assert lib.mccnn_projection_grad_product_supported(96, 1024) == 0
    assert lib.mccnn_final_product_supported(2048, 128) == 1
    assert lib.mccnn_final_product_supported(1000, 128) == 0
    # K = 8 is not covered by the fused projection
    rc = lib.mccnn_mc_conv_project(None, 3, i64(10), None, 64, None, i64(10), None, i64(20), None,
                                   None, None, 8, 1, 0, None, None, None, None, None)
    assert rc == 1 and b"K in {16,32,64}" in lib.mccnn_last_error()
    assert lib.mccnn_mc_conv_project_supported(3, 48, 32) == 1
    assert lib.mccnn_mc_conv_weight_grads_supported(3, 64, 64) == 1
    assert lib.mccnn_mc_conv_supported(3, 64, 32) == 0          # no feature-gradient half there
    rc = lib.mccnn_kp_conv_project(None, 3, i64(10), None, 64, None, i64(10), None, i64(20), None,
                                   None, None, 33, None, 0, ctypes.c_float(1.0), None, None)
    assert rc == 1 and b"kernel points" in lib.mccnn_last_error()
    rc = lib.mccnn_weight_grad_product(None, i64(10), 48, None, 1024, None, None, sz(0), None)
    assert rc == 1 and b"output rows" in lib.mccnn_last_error()
    rc = lib.mccnn_projection_grad_product(None, i64(10), 96, None, 1024, None, None)
    assert rc == 1 and b"input columns" in lib.mccnn_last_error()
    # a feature table too large for 32-bit byte offsets is refused, not truncated
    rc = lib.mccnn_mc_conv_project(None, 3, i64(1 << 25), None, 64, None, i64(10), None, i64(20),
                                   None, None, None, 16, 1, 0, None, None, None, None, None)
    assert rc == 1 and b"2^30" in lib.mccnn_last_error()
    fn = lib.mccnn_mc_conv_project_grads_workspace_bytes
    fn.restype = sz
    assert fn(3, 16, i64(1000)) >= 32 * 64 * 4


def test_workspace_queries(lib):
    for name in ("mccnn_sort_keys_workspace_bytes", "mccnn_sampling_workspace_bytes"):
        fn = getattr(lib, name)
        fn.restype = ctypes.c_size_t
        assert fn(ctypes.c_int64(1000)) > 1000 * 4
    fn = lib.mccnn_find_neighbors_workspace_bytes
    fn.restype = ctypes.c_size_t
    assert fn(3, ctypes.c_int64(1000)) >= 1000 * 9 * 8
    assert fn(9, ctypes.c_int64(1000)) == 0


def test_product_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "tensorflow_graphics_point_clouds_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                text = open(os.path.join(base, f)).read()
                assert "mccnn_oracle" not in text and "from oracle" not in text, f


def test_grouped_basis_gradients_stop_short_of_the_last_pair_indices(lib):
    """The grouped kernels look up to 128 pairs past a centre's last one in 32 bits: tables within
    that of 2^31 pairs are left to the other kernels and refused."""
    i64, sz = ctypes.c_int64, ctypes.c_size_t
    most = 2 ** 31 - 1024
    pays = lambda m: lib.mccnn_basis_proj_grads_grouped_pays(24, 8, i64(10 ** 7), i64(m))
    assert pays(most) == 1 and pays(most + 1) == 0 and pays(2 ** 31 - 1) == 0
    for pairs in (most + 1, 2 ** 31 - 1):
        rc = lib.mccnn_neighbourhood_order(None, i64(5), i64(pairs), None, None, None, sz(0), None)
        assert rc == 1 and b"2^31 - 1024" in lib.mccnn_last_error()
        rc = lib.mccnn_basis_proj_grads_grouped(None, i64(0), 8, None, 24, None, i64(pairs), None,
                                                i64(5), None, None, None, None, sz(0), None, None)
        assert rc == 1 and b"2^31 - 1024" in lib.mccnn_last_error()


@pytest.mark.parametrize("c,k,centres,pairs,grouped", [
    # short lists: the kernels per pair and channel take 0.4 to 0.8 of the time
    (64, 8, 3413, 23249, 0), (96, 8, 9102, 62418, 0), (24, 16, 9102, 62418, 0),
    (16, 8, 13653, 94583, 0), (96, 16, 2275, 14775, 0), (128, 8, 4551, 43397, 0),
    # the grouped ones take 0.1 to 0.9 of it: more pairs, longer lists, more columns
    (24, 8, 36408, 256794, 1), (16, 32, 27306, 191624, 1), (96, 8, 5461, 106117, 1),
    (64, 64, 3413, 23249, 1), (128, 64, 1706, 11124, 1), (3, 64, 174762, 3739442, 1),
    # under 2^20 pairs x channels
    (3, 64, 3000, 150000, 0)])
def test_small_tables_of_short_lists_keep_the_ungrouped_basis_gradients(lib, c, k, centres, pairs,
                                                                        grouped):
    i64 = ctypes.c_int64
    assert lib.mccnn_basis_proj_grads_grouped_pays(c, k, i64(centres), i64(pairs)) == grouped
