"""The C-ABI library: every symbol declared in include/tk3d.h is exported, and the
argument checks reject bad calls before anything is launched (so they can be
exercised without a GPU)."""
import ctypes
import os
import re

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(REPO, "include", "tk3d.h")


@pytest.fixture(scope="module")
def lib():
    from torkit3d_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        from torkit3d_amd import build

        build.build()
    return _lib.lib()


DEBUG_HEADER = os.path.join(REPO, "torkit3d_amd", "csrc", "tk3d_debug.h")


def declared_symbols(header=HEADER):
    text = open(header).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tk3d_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_families():
    names = declared_symbols()
    for family in ("chamfer_distance_forward", "chamfer_distance_backward", "knn_distance",
                   "ball_query", "sample_farthest_points", "group_points_forward",
                   "group_points_backward", "interpolate_forward", "interpolate_backward"):
        assert "tk3d_%s_f32" % family in names
        assert "tk3d_%s_f64" % family in names
    assert "tk3d_version" in names and "tk3d_error_string" in names


def test_every_declared_symbol_is_exported(lib):
    for name in declared_symbols():
        assert hasattr(lib, name), "%s declared in tk3d.h but not exported" % name


def test_test_only_entry_points_are_exported_and_outside_the_boundary(lib):
    # what the tests and the benchmark call besides the boundary: declared in a header of its
    # own, none of it in include/tk3d.h
    debug = declared_symbols(DEBUG_HEADER)
    assert debug and all(name.startswith("tk3d_debug_") for name in debug)
    assert not any(name.startswith("tk3d_debug_") for name in declared_symbols())
    for name in debug:
        assert hasattr(lib, name), "%s declared in tk3d_debug.h but not exported" % name
    fn = lib.tk3d_debug_chamfer_forward_route_f32
    fn.restype = ctypes.c_int
    null = ctypes.c_void_p(0)
    # argument checks come before any launch
    assert fn(null, null, i64(-1), i64(4), i64(4), null, null, null, null, ctypes.c_int(1), null) == -2
    assert fn(null, null, i64(1), i64(4), i64(4), null, null, null, null, ctypes.c_int(1), null) == -1


def test_exchanges_through_lds_within_a_wave_are_fenced():
    # (a wave barrier orders no memory for the compiler: every one of them comes with the fence)
    csrc = os.path.dirname(DEBUG_HEADER)
    for name in sorted(os.listdir(csrc)):
        text = open(os.path.join(csrc, name)).read()
        fenced = re.findall(r'__builtin_amdgcn_fence\(__ATOMIC_ACQ_REL, "wavefront"\);\s*'
                            r"__builtin_amdgcn_wave_barrier\(\);", text)
        assert len(fenced) == text.count("__builtin_amdgcn_wave_barrier("), name


def test_version_and_error_strings(lib):
    from torkit3d_amd import _lib

    assert lib.tk3d_version() == 100
    assert _lib.error_string(0) == "success"
    assert "Invalid version" in _lib.error_string(-4)
    for code in range(-6, 0):
        assert "unknown" not in _lib.error_string(code)
    assert "unknown" in _lib.error_string(-99)


def i64(v):
    return ctypes.c_int64(v)


NULL = ctypes.c_void_p(0)
FAKE = ctypes.c_void_p(256)  # never dereferenced: the checks below fail first


def test_argument_errors_are_reported_without_launching(lib):
    for sfx in ("_f32", "_f64"):
        fwd = getattr(lib, "tk3d_chamfer_distance_forward" + sfx)
        assert fwd(FAKE, FAKE, i64(-1), i64(4), i64(4), FAKE, FAKE, FAKE, FAKE, NULL) == -2
        assert fwd(NULL, FAKE, i64(1), i64(4), i64(4), FAKE, FAKE, FAKE, FAKE, NULL) == -1
        assert fwd(NULL, NULL, i64(0), i64(4), i64(4), NULL, NULL, NULL, NULL, NULL) == 0
        knn = getattr(lib, "tk3d_knn_distance" + sfx)
        assert knn(FAKE, FAKE, i64(1), i64(8), i64(4), i64(5), 1, FAKE, FAKE, NULL) == -3  # k > N2
        assert knn(FAKE, FAKE, i64(1), i64(8), i64(4), i64(0), 1, FAKE, FAKE, NULL) == -3
        assert knn(FAKE, FAKE, i64(1), i64(8), i64(4), i64(2), 7, FAKE, FAKE, NULL) == -4
        fps = getattr(lib, "tk3d_sample_farthest_points" + sfx)
        assert fps(FAKE, i64(1), i64(10), i64(0), FAKE, NULL, ctypes.c_size_t(0), NULL) == -3
        assert fps(FAKE, i64(1), i64(10), i64(11), FAKE, NULL, ctypes.c_size_t(0), NULL) == -3
        assert fps(NULL, i64(1), i64(10), i64(5), FAKE, NULL, ctypes.c_size_t(0), NULL) == -1
        # a cloud too large for the register kernel needs a workspace
        assert fps(FAKE, i64(1), i64(100000), i64(5), FAKE, NULL, ctypes.c_size_t(0), NULL) == -5
        ball = getattr(lib, "tk3d_ball_query" + sfx)
        assert ball(FAKE, FAKE, i64(1), i64(4), i64(4), ctypes.c_float(0.1), i64(-1), FAKE, NULL) == -3
        interp = getattr(lib, "tk3d_interpolate_forward" + sfx)
        assert interp(FAKE, FAKE, FAKE, i64(1), i64(2), i64(4), i64(4), i64(9), FAKE, NULL) == -3
        group = getattr(lib, "tk3d_group_points_backward" + sfx)
        assert group(FAKE, FAKE, i64(1), i64(-2), i64(4), i64(4), i64(2), FAKE, NULL) == -2
        # entry points that fuse Python-side steps of the reference
        ball = getattr(lib, "tk3d_ball_query_bcn" + sfx)
        assert ball(FAKE, FAKE, i64(1), i64(4), i64(4), ctypes.c_float(0.1), i64(-1), FAKE, NULL) == -3
        assert ball(NULL, FAKE, i64(1), i64(4), i64(4), ctypes.c_float(0.1), i64(2), FAKE, NULL) == -1
        fps = getattr(lib, "tk3d_sample_farthest_points_gather" + sfx)
        assert fps(FAKE, 1, i64(1), i64(10), i64(11), FAKE, NULL, NULL, ctypes.c_size_t(0), NULL) == -3
        assert fps(NULL, 0, i64(1), i64(10), i64(5), FAKE, NULL, NULL, ctypes.c_size_t(0), NULL) == -1
        nn3 = getattr(lib, "tk3d_three_nn" + sfx)
        eps = ctypes.c_double(1e-10)
        assert nn3(FAKE, FAKE, 0, i64(1), i64(8), i64(2), eps, FAKE, FAKE, FAKE, NULL) == -3
        assert nn3(FAKE, FAKE, 1, i64(1), i64(8), i64(4), eps, FAKE, FAKE, NULL, NULL) == -1
        assert nn3(NULL, NULL, 1, i64(0), i64(8), i64(4), eps, NULL, NULL, NULL, NULL) == 0
        cat = getattr(lib, "tk3d_group_points_concat_forward" + sfx)
        assert cat(NULL, FAKE, FAKE, FAKE, i64(1), i64(2), i64(4), i64(4), i64(2), FAKE, NULL) == -1
        assert cat(NULL, FAKE, FAKE, FAKE, i64(1), i64(0), i64(4), i64(-4), i64(2), FAKE, NULL) == -2
        cat = getattr(lib, "tk3d_group_points_concat_backward" + sfx)
        assert cat(FAKE, FAKE, i64(1), i64(2), i64(4), i64(4), i64(2), NULL, NULL, NULL) == 0


def test_fps_workspace_size(lib):
    fn = lib.tk3d_sample_farthest_points_workspace_bytes
    fn.restype = ctypes.c_size_t
    assert fn(i64(16), i64(4096), ctypes.c_size_t(4)) == 0
    assert fn(i64(8), i64(16384), ctypes.c_size_t(4)) == 0
    need = fn(i64(2), i64(100000), ctypes.c_size_t(4))
    assert need >= 2 * 100000 * 4


def test_chamfer_workspace_size_and_argument_checks(lib):
    # the size function is host code: the dispatch rule of the sorted path, no GPU needed
    size = lib.tk3d_chamfer_distance_forward_workspace_bytes
    size.restype = ctypes.c_size_t

    def nbytes(b, n1, n2, always):
        return size(i64(b), i64(n1), i64(n2), ctypes.c_int(always))

    assert nbytes(32, 16384, 16384, 0) > 0          # the benchmark shape is served
    assert nbytes(1, 65536, 65536, 0) > 0
    assert nbytes(2, 1024, 1024, 0) == 0            # too little work to repay the sort
    assert nbytes(16, 4096, 4096, 0) == 0
    assert nbytes(4, 65536, 2048, 0) == 0           # lengths more than a factor of four apart
    assert nbytes(64, 3000, 3000, 0) == 0           # clouds under 4096 points
    for shape in ((2, 1024, 1024), (16, 4096, 4096), (4, 65536, 2048), (1, 1, 1)):
        assert nbytes(*shape, 1) > 0                # ... but can be, on request
    assert nbytes(1, 65537, 4096, 1) == 0 and nbytes(0, 4096, 4096, 1) == 0
    # 16 + 32 bytes per padded point, a box per 32 points, headers, flags and far-key lists
    b, n = 3, 5000
    pad = (n + 127) // 128 * 128
    low = 2 * b * pad * 48
    assert low < nbytes(b, n, n, 1) < low + 2 * b * (pad // 2 + 1024) + 4096
    # null or short workspace: the call is the plain entry point, with its argument checks
    fn = lib.tk3d_chamfer_distance_forward_ws_f32
    args = (FAKE, FAKE, i64(1), i64(8), i64(8), FAKE, FAKE, FAKE)
    assert fn(*args, NULL, NULL, ctypes.c_size_t(0), NULL) == -1          # idx2 missing
    assert fn(FAKE, FAKE, i64(-1), i64(8), i64(8), FAKE, FAKE, FAKE, FAKE, NULL,
              ctypes.c_size_t(0), NULL) == -2
    assert fn(NULL, NULL, i64(0), i64(8), i64(8), NULL, NULL, NULL, NULL, NULL,
              ctypes.c_size_t(0), NULL) == 0


# Calls that lost to the copy (or took it for nothing), then calls that win by it, as timed.
@pytest.mark.parametrize("b,n1,n2,channels_first,copied", [
    (1, 1025, 1025, 0, False),    # the only batch element starts on 16 bytes as it is
    (2, 1025, 1025, 0, False),    # few workgroups: the vector pre-filter
    (128, 1000, 999, 0, False),
    (4, 2049, 400, 0, False),     # few workgroups, a short cloud: the exact sweep
    (32, 489, 1130, 0, False),    # the matrix kernel, but the last 128 keys are nearly full
    (4, 5001, 300, 1, False), (1, 2049, 400, 1, False), (8, 126, 1144, 1, False),
    (16, 1024, 2048, 0, False), (16, 1024, 2048, 1, False),
    (16, 1025, 1025, 0, True), (8, 4099, 4097, 0, True), (4, 7569, 1552, 0, True),
    (24, 1550, 8803, 0, True),
    (1, 1025, 1025, 1, True), (8, 2500, 3001, 1, True), (8, 5001, 300, 1, True),
    (8, 1000, 1000, 1, True), (1, 257, 300, 1, True),
])
def test_chamfer_clouds_are_copied_where_it_pays(lib, b, n1, n2, channels_first, copied):
    fn = lib.tk3d_chamfer_distance_forward_rows_bytes
    fn.restype = ctypes.c_size_t
    for sizes in ((n1, n2), (n2, n1)):
        padded = sum((n + 3) // 4 * 4 for n in sizes)
        want = b * padded * 12 if copied else 0
        assert fn(i64(b), i64(sizes[0]), i64(sizes[1]), ctypes.c_int(channels_first)) == want


# Lengths that are no multiple of four: up to which estimate the small launches' sweep reads the clouds in place.
@pytest.mark.parametrize("b,n1,n2,taken", [
    (8, 2500, 3001, True), (16, 3001, 770, True), (2, 5891, 3001, True), (4, 4099, 770, True), (64, 1026, 1026, True),
    (8, 4099, 515, False), (4, 5891, 770, False), (4, 4099, 4099, False), (32, 1537, 1537, False)])
@pytest.mark.parametrize("channels_first", [0, 1])
def test_chamfer_clouds_are_read_in_place_where_it_pays(lib, b, n1, n2, channels_first, taken):
    for sizes in ((n1, n2), (n2, n1)):
        args = i64(b), i64(sizes[0]), i64(sizes[1]), ctypes.c_int(channels_first)
        assert bool(lib.tk3d_chamfer_distance_forward_in_place(*args)) is taken


# What the products of include/tk3d_mlp.h are called with.
pointer, i32 = ctypes.c_void_p, ctypes.c_int32
IN_RAW, IN_GRAD, OUT_PLAIN, OUT_EVAL, OUT_MASK = 0, 3, 1, 3, 6


@pytest.mark.parametrize("planes,roots,n1,n2,taken", [
    (1, 0, 8192, 8192, True), (1, 0, 8193, 5, False), (0, 1, 8192, 8192, True), (0, 1, 5, 8193, False),
    (1, 1, 8192, 4096, True), (1, 1, 4096, 8192, True), (1, 1, 4097, 4097, False), (1, 1, 8193, 1, False)])
def test_chamfer_backward_reads_planes_and_roots_where_it_pays(lib, planes, roots, n1, n2, taken):
    args = [ctypes.c_int(planes), ctypes.c_int(roots), ctypes.c_int64(n1), ctypes.c_int64(n2)]
    assert bool(lib.tk3d_chamfer_distance_backward_takes_forms(*args)) is taken


class Source(ctypes.Structure):
    _fields_ = [(n, pointer) for n in ("x", "y", "coef", "w")] + [("batch_stride", ctypes.c_int64)] + [
        (n, i32) for n in ("K", "wk", "wc")]


class Norm(ctypes.Structure):
    _fields_ = [(n, pointer) for n in ("mean", "var", "gamma", "beta")] + [("eps", ctypes.c_float)]


class Product(ctypes.Structure):
    _fields_ = [("src", Source * 2), ("in_norm", Norm), ("out_norm", Norm)] + [
        (n, pointer) for n in ("out", "out2", "yprev", "bias", "add", "partial")] + [
        (n, i32) for n in ("B", "C", "C0", "P", "group", "M")]


class Outer(ctypes.Structure):
    _fields_ = [("row", Source), ("col", Source), ("row_norm", Norm), ("col_norm", Norm),
                ("partial", pointer), ("rowsum", pointer), ("B", i32), ("P", i32)]


# The kernel's byte offsets within a batch element are 32-bit: (channels + 8) * positions up to 2^29, as in the
# products on their own. No pointer is read.
@pytest.mark.parametrize("rows,columns,positions,taken", [
    (128, 128, 3947580, True), (128, 128, 3947584, False), (16, 128, 3947584, False), (128, 64, 3947584, False),
    (16, 16, 3947584, True), (16, 16, 22369620, True), (16, 16, 22369624, False), (128, 128, 2**31 - 4, False),
    (128, 128, 2046, False), (129, 64, 64, False), (64, 129, 64, False), (128, 32, 64, False), (32, 128, 64, True)])
def test_layers_whose_two_gradients_share_a_launch(lib, rows, columns, positions, taken):
    product, outer = Product(B=1, C=columns, C0=columns, P=positions), Outer(B=1, P=positions)
    product.src[0].K = outer.row.K = rows
    outer.col.K = columns
    assert (lib.tk3d_mlp_pair_slots(ctypes.byref(product), ctypes.byref(outer)) > 0) is taken


# Wide products go through tiles in LDS (a slot per 128 positions) where their workgroups' rounds are not padding for
# the most part: rows under 128 and just over, channels just over a tile, few rounds; else wave tiles. (256 CUs)
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("rows,columns,b,positions,tiles", [
    (512, 256, 128, 128, True), (1024, 320, 16, 1024, True), (320, 1024, 4, 1024, True), (384, 384, 64, 1024, True),
    (256, 512, 64, 1024, True), (256, 256, 4096, 16, False), (200, 300, 73, 224, False), (256, 512, 256, 64, False),
    (130, 70, 292, 224, False), (256, 256, 2, 1024, False), (64, 256, 128, 128, False), (512, 512, 31, 132, True)])
def test_products_that_take_tiles_in_lds(lib, rows, columns, b, positions, tiles, masked):
    product = Product(B=b, C=columns, C0=columns, P=positions, group=1, M=positions)
    product.src[0].K, product.src[0].wk, product.src[0].wc = rows, columns, 1
    slots = lib.tk3d_mlp_product_slots(IN_GRAD, OUT_MASK if masked else OUT_PLAIN, ctypes.byref(product))
    assert (slots == b * -(-positions // 128)) is tiles


# Products of more tiles than SIMDs whose weights lie apart (rows of W that are no multiple of eight, in
# evaluation) share tiles among waves (a slot a tile) where the last round of wave tiles is half empty, others
# up to four tiles per SIMD. (256 CUs)
@pytest.mark.parametrize("rows,columns,b,positions,evaluation,gradient", [
    (323, 1024, 64, 33, False, True), (131, 256, 512, 31, False, True), (131, 512, 1, 2050, True, True),
    (515, 128, 1, 9001, True, True), (131, 256, 32, 256, False, True), (128, 1024, 64, 33, True, True),
    (512, 256, 9, 1777, True, True), (131, 67, 1, 9001, True, True), (120, 256, 9, 1777, False, False),
    (512, 256, 10, 1777, False, False)])
def test_products_whose_waves_share_tiles(lib, rows, columns, b, positions, evaluation, gradient):
    product = Product(B=b, C=columns, C0=columns, P=positions, group=1, M=positions)
    product.src[0].K = rows
    for way, out, wk, wc, taken in ((IN_RAW, OUT_EVAL, 1, rows, evaluation), (IN_GRAD, OUT_MASK, columns, 1, gradient),
                                    (IN_GRAD, OUT_PLAIN, columns, 1, gradient)):
        product.src[0].wk, product.src[0].wc = wk, wc
        slots = lib.tk3d_mlp_product_slots(way, out, ctypes.byref(product))
        assert (slots == b * -(-positions // 32)) is taken


class GroupedPool(ctypes.Structure):  # tk3d_mlp_grouped_pool
    _fields_ = [("pointers", pointer * 7), ("norms", pointer * 15), ("out", pointer), ("sizes", i32 * 8)]


# Three layers behind a grouping go in one launch unless that is slower: chains of products that are long for the tiles
# there are, layers that leave most waves of a CU's only workgroup idle. (256 CUs, b x m groups of s)
@pytest.mark.parametrize("widths,b,m,s,taken", [
    ((64, 64, 128), 1, 1, 64, True), ((96, 96, 96), 1, 32, 64, True), ((128, 128, 256), 1, 32, 64, True),
    ((192, 64, 64), 1, 32, 64, False), ((256, 32, 64), 1, 32, 64, False), ((256, 32, 64), 1, 32, 32, True),
    ((32, 480, 64), 1, 32, 32, False), ((480, 32, 64), 1, 32, 32, False), ((256, 256, 512), 1, 32, 32, False),
    ((128, 256, 512), 1, 32, 32, True), ((256, 256, 512), 1, 64, 64, False),
    ((256, 256, 512), 2, 64, 64, True), ((32, 480, 64), 2, 64, 64, True),
    ((224, 32, 64), 2, 64, 64, False), ((448, 64, 64), 2, 64, 64, False), ((480, 32, 64), 2, 64, 64, False),
    ((480, 32, 64), 32, 128, 64, False), ((224, 32, 64), 32, 128, 64, True), ((256, 64, 128), 16, 32, 32, True),
    ((256, 64, 128), 32, 128, 64, False), ((32, 480, 64), 32, 128, 64, False), ((96, 256, 32), 32, 128, 64, False),
    ((96, 256, 32), 16, 32, 32, True), ((128, 192, 32), 32, 128, 64, True), ((256, 256, 512), 32, 128, 64, True)])
def test_grouped_layers_that_share_a_launch(lib, widths, b, m, s, taken):
    sizes = GroupedPool(sizes=(67, b, 4 * m, m, s, *widths))
    assert bool(lib.tk3d_mlp_grouped_pool_supported(ctypes.byref(sizes))) is taken


def test_edge_backward_workspace_has_the_selected_values_only_where_they_may_be_gathered(lib):
    size = lib.tk3d_mlp_edge_backward_bytes
    size.restype = ctypes.c_int64
    b, o, c = 1, 64, 3

    def bytes_of(n):
        return size(*[ctypes.c_int(v) for v in (b, n, o, c)])

    selected = 8 * b * o * 6144
    assert bytes_of(6145) - bytes_of(6144) >= selected
    # rows that are added in LDS: both halves of the gradient, the points as rows and their sums, and partial sums, which
    # do not grow with the points beyond their parts
    assert bytes_of(6144) - bytes_of(2048) < 4 * b * 4096 * (2 * o + 3 * c) + selected // 2
