"""CPU-side checks: the C-ABI library loads and exports every symbol the header declares,
and the host-side mirror keeps the reference's module structure, names and init."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from pyramidconvblock_amd import _lib

    header = open(os.path.join(ROOT, "include", "pdw.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(pdw_\w+)\s*\(", header))
    assert len(declared) >= 13
    L = _lib.lib()  # loads libpdw.so (built in-tree); no compute call is made here
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(raw, name), f"libpdw.so does not export {name}"
    assert declared == set(_lib.EXPORTS), declared ^ set(_lib.EXPORTS)
    assert L.pdw_version() >= 1
    assert L.pdw_conv_out_size(56, 13, 1, 6, 1) == 56
    assert L.pdw_conv_out_size(5, 9, 1, 0, 1) == 0
    assert L.pdw_conv_out_size(32, 7, 2, 3, 1) == 16


def test_argument_validation_without_gpu():
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    # invalid arguments are rejected before any HIP call
    assert L.pdw_dwconv_fwd(None, None, None, 1, 4, 4, 8, 3, 3, 1, 1, 1, 1, 1, 1, 7, None) != 0
    assert b"dtype" in L.pdw_last_error()
    assert L.pdw_dwconv_fwd(None, None, None, 1, 4, 4, 8, 3, 3, 0, 1, 1, 1, 1, 1, 0, None) != 0
    assert b"stride" in L.pdw_last_error()
    assert L.pdw_gate_fwd(None, None, 4, 7, 0, 0, None) != 0
    assert L.pdw_dwconv_wgrad_workspace_bytes(2, 8, 8, 16, 3, 3, 1, 1, 1, 1, 1, 1, 0) > 0
    assert L.pdw_dwconv_wgrad(1, 1, 1, None, 0, 2, 8, 8, 16, 3, 3, 1, 1, 1, 1, 1, 1, 0, None) != 0
    assert b"workspace" in L.pdw_last_error()


def test_single_call_block_host_logic_without_gpu():
    """pdw_convblock_*: which shapes are covered, workspace sizes, and rejection before any HIP call."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    BF16, F16, F32 = 2, 1, 0
    assert L.pdw_convblock_supported(32, 56, 56, 128, 64, 13, BF16) == 1
    assert L.pdw_convblock_supported(1, 4, 8, 128, 64, 3, F16) == 1
    assert L.pdw_convblock_supported(2, 32, 32, 64, 32, 7, BF16) == 1
    assert L.pdw_convblock_supported(8, 112, 112, 96, 48, 17, F16) == 1
    for bad in ((32, 56, 56, 128, 64, 13, F32),    # 16-bit types only
                (32, 57, 56, 128, 64, 13, BF16),   # odd extent: the pooled scale is not an exact half
                (32, 56, 56, 128, 64, 12, BF16),   # even filter
                (32, 56, 56, 160, 80, 13, BF16),   # widths beyond the dense kernels (128)
                (0, 56, 56, 128, 64, 13, BF16),
                (2, 6, 6, 128, 64, 3, BF16)):      # 36 rows per image: not whole row tiles
        assert L.pdw_convblock_supported(*bad) == 0, bad
        assert L.pdw_convblock_fwd_workspace_bytes(*bad) == 0 and L.pdw_convblock_bwd_workspace_bytes(*bad) == 0
    shape = (32, 56, 56, 128, 64, 13, BF16)
    fwd, bwd = L.pdw_convblock_fwd_workspace_bytes(*shape), L.pdw_convblock_bwd_workspace_bytes(*shape)
    n = 32 * 56 * 56
    assert fwd >= n // L.pdw_dense_colsum_rows() * 128 * 4 + 32 * 128 * 4
    assert bwd >= 3 * n * 64 * 2 + L.pdw_dense_wgrad_workspace_bytes(n, 128, 64) * 2
    assert L.pdw_convblock_fwd(*([None] * 16), 0, *shape, None) != 0 and b"null" in L.pdw_last_error()
    assert L.pdw_convblock_fwd(*([1] * 16), 16, *shape, None) != 0 and b"workspace" in L.pdw_last_error()
    assert L.pdw_convblock_bwd(*([1] * 22), 16, *shape, None) != 0 and b"workspace" in L.pdw_last_error()
    assert L.pdw_convblock_bwd(*([1] * 22), 1 << 40, 32, 57, 56, 128, 64, 13, BF16, None) != 0
    assert b"not covered" in L.pdw_last_error()


@pytest.mark.parametrize("B,H,W,D,K,dtype", [(32, 56, 56, 128, 13, 2), (3, 57, 61, 200, 9, 2), (32, 56, 56, 128, 13, 0),
                                             (4, 64, 64, 1152, 13, 1), (8, 7, 7, 512, 3, 1)])
def test_block_buffers_hold_no_scratch_beyond_its_use(B, H, W, D, K, dtype):
    """pdw_block_*: the buffer between the passes holds what the backward reads and one row per image (the sums of x lie in
    y until it is written); the backward's workspace holds two gradients at full resolution, two pooled ones and partial
    sums (the gradient of the concatenation makes room for conv_up's)."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    es, I, h, w = (4 if dtype == 0 else 2), D // 2, H // 2, W // 2
    Il = I if I % 8 == 0 or dtype == 0 else 2 * ((I // 2 + 7) // 8 * 8)
    up = lambda b: (b + 255) // 256 * 256
    full, half = up(B * H * W * Il * es), up(B * h * w * Il * es)
    packed = 0 if Il == I else 2 * up(Il * D * es) + 2 * up(K * K * Il * es)
    shape = (B, H, W, h, w, D, I, K, dtype)
    assert L.pdw_block_supported(*shape)
    assert L.pdw_block_saved_bytes(*shape) == 3 * full + 2 * half + up(B * D * es) + packed + up(B * D * 4)
    wgrads = sum(up(L.pdw_dwconv_wgrad_workspace_bytes(B, *hw, Il, K, K, 1, 1, K // 2, K // 2, 1, 1, dtype)) for hw in ((H, W), (h, w)))
    n = B * H * W
    wgrads += up(L.pdw_dense_wgrad_workspace_bytes(n, D, Il)) + up(L.pdw_dense_wgrad_workspace_bytes(n, Il, D))
    sums = up((n + 31) // 32 * D * 4) + up(2 * D * es) + up(B * D * 4)
    mean = max(B * 33 * D * 4 + 512, up(L.pdw_pool_branch_workspace_bytes(B, H * W, D)))   # (at most 32 partial sums an image)
    assert L.pdw_block_bwd_workspace_bytes(*shape) <= 2 * full + 2 * half + wgrads + sums + mean
    # y is written early: it must not be x
    for y in (1 << 20, (1 << 20) + B * H * W * D * es - 16):
        assert L.pdw_block_fwd(1 << 20, *([1 << 40] * 7), y, 1 << 40, 1 << 60, *shape, None) == 1
        assert b"overlaps" in L.pdw_last_error()


@pytest.mark.parametrize("N,M,NO", [(458752, 4096, 2048), (458752, 2048, 4096), (1 << 20, 2040, 1020), (1 << 17, 16376, 64),
                                    (8490, 63592, 168), (136435, 32464, 64)])   # (fewer ranges would save the launch of both products a round)
def test_wide_weight_gradient_ranges_fit_32_bit_offsets(N, M, NO):
    """pdw_dense_wgrad of wide layers cuts the rows into ranges whose operands 32-bit offsets reach, also where the layer's
    tiles alone fill the chip: the workspace holds a partial result for each."""
    from pyramidconvblock_amd import _lib

    parts = _lib.lib().pdw_dense_wgrad_workspace_bytes(N, M, NO) // (M * NO * 4)
    reach = (2**31 - 1) // (max(M, NO) * 4) // 64 * 64   # (the larger of the types; the workspace is for either)
    assert parts * reach >= N


def test_block_extents_beyond_the_pools_bins():
    """pdw_block_supported: extents whose products do not fit the pool's 32-bit bins, of rows and of columns, are not taken
    (the single calls refuse them), unless the fused launches do, which have no bins."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    for dtype in (0, 1, 2):
        for H, W in ((2, 70001), (70001, 2), (2, 70000), (70000, 2)):
            assert L.pdw_block_supported(1, H, W, H // 2, W // 2, 8, 4, 3, dtype) == 0
            assert L.pdw_avgpool_fwd(1 << 20, 1 << 21, 1, H, W, 4, H // 2, W // 2, dtype, None) == 1
            assert b"too large" in L.pdw_last_error()
        assert L.pdw_block_supported(1, 2, 65535, 1, 32767, 8, 4, 3, dtype) == 1
    assert L.pdw_block_supported(1, 4, 70000, 2, 35000, 64, 32, 3, 2) == 1


@pytest.mark.parametrize("shape", [(128, 2, 64, 64, 3), (128, 4, 64, 64, 3), (128, 6, 64, 64, 13), (96, 2, 34, 16, 5),
                                   (512, 6, 40, 128, 17), (32, 56, 56, 64, 13), (8, 56, 56, 64, 13), (1, 8, 36, 16, 9),
                                   (8, 112, 112, 48, 17), (128, 56, 56, 64, 13)])
def test_bwd3_planner_strip_shaped_inputs(shape):
    """The planner of the backward's three-problem launch (host code, no device touched): images of fewer than four
    rows at the half scale, with batch x channels large enough that only whole-image bands are tried, must still get
    a plan with at least one band per problem (a plan of zero bands is a division by zero in the launcher)."""
    from pyramidconvblock_amd import _lib

    L = _lib.lib()
    bands = (ctypes.c_int * 3)(-1, -1, -1)
    rc = L.pdw_dwconv_bwd3_plan(*shape, _lib.dtype_code(torch.bfloat16), ctypes.addressof(bands))
    assert rc == 0, L.pdw_last_error()
    B, H, W, C, K = shape
    assert 1 <= bands[0] <= H and 1 <= bands[1] <= H and 1 <= bands[2] <= max(1, H // 2), list(bands)
    # not covered: fp32, odd extents, narrow images
    assert L.pdw_dwconv_bwd3_plan(*shape, _lib.dtype_code(torch.float32), ctypes.addressof(bands)) == 3
    assert L.pdw_dwconv_bwd3_plan(B, H, 16, C, K, 2, ctypes.addressof(bands)) == 3
    assert L.pdw_dwconv_bwd3_plan(B, H + 1, W, C, K, 2, ctypes.addressof(bands)) == 1
    assert L.pdw_dwconv_bwd3_plan(B, H, W, C, K, 2, None) == 1


@pytest.mark.parametrize("shape", [(64, 8192, 34, 16, 5), (2, 65536, 34, 16, 13), (3, 40000, 36, 32, 7), (256, 4096, 34, 16, 3)])
def test_bwd3_planner_tall_images(shape):
    """Batches of tall images, whose rows one below the other are more than the kernel's quotients by an image's rows are exact
    for, are walked image by image (host code, no device touched)."""
    from pyramidconvblock_amd import _lib

    bands = (ctypes.c_int * 3)(-1, -1, -1)
    rc = _lib.lib().pdw_dwconv_bwd3_plan(*shape, _lib.dtype_code(torch.bfloat16), ctypes.addressof(bands))
    assert rc == 0, _lib.lib().pdw_last_error()
    B, H, _, C, _ = shape
    assert all(1 <= n <= H for n in bands) and B * bands[0] * C // 16 >= 48, list(bands)   # (a useful share of the chip)


def test_module_structure_and_seeded_init_match_reference_recipe():
    import pyramid_dwconv
    from oracle import torch_path

    torch.manual_seed(0)
    m = pyramid_dwconv.ConvBlock(dim=64, kernel_size=7)
    torch.manual_seed(0)
    P = torch_path.default_params(64, 7)
    sd = m.state_dict()
    assert list(sd.keys()) == list(P.keys())
    for k in P:
        assert sd[k].dtype == P[k].dtype and torch.equal(sd[k], P[k]), k
    assert tuple(sd["gates.1.conv_spatial.weight"].shape) == (7, 7, 32)
    assert sd["gates.0.conv_spatial.weight"].dtype == torch.float16
    assert m.gates[1].scale_factor == 0.5 and abs(m.gates[0].scale - 16 ** -0.5) < 1e-12
    mb = m.to(torch.bfloat16)
    assert all(v.dtype == torch.bfloat16 for v in mb.state_dict().values())


def test_no_cpu_path():
    import pyramidconvblock_amd as P

    conv = P.OptimizedDepthwiseConv2d(8, 3, padding=1, dtype=torch.float32)
    assert conv.weight.dtype == torch.float16  # dtype argument ignored, as in the reference
    with pytest.raises(RuntimeError, match="HIP device"):
        conv(torch.zeros(1, 4, 4, 8, dtype=torch.float16))
    with pytest.raises(AssertionError):
        conv(torch.zeros(1, 4, 4, 9))
    with pytest.raises(RuntimeError, match="HIP device"):
        P.ConvBlock(8, kernel_size=3)(torch.zeros(1, 4, 4, 8))
    from pyramidconvblock_amd.conv_block import convblock_infer

    m = P.ConvBlock(128, kernel_size=3).bfloat16()
    args = [m.conv_up.weight, m.conv_out.weight, m.conv_out.bias, m.conv_pool.weight, m.conv_pool.bias]
    for x, a in ((torch.zeros(1, 4, 8, 128).bfloat16(), args), (None, args), (torch.zeros(1, 4, 8, 128).bfloat16(), [None] * 5)):
        with pytest.raises(RuntimeError, match="HIP device"):
            convblock_infer(x, *a, [g.conv_spatial.weight for g in m.gates])


def test_the_library_builds_without_torch(tmp_path):
    """build.py as a script in an interpreter without torch (the compiler stands in by a script that writes its output):
    libpdw.so is linked, the host extension is left out, and nothing raises."""
    hipcc = tmp_path / "hipcc"
    hipcc.write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\necho built > "$2"\n')
    hipcc.chmod(0o755)
    code = ("import sys, importlib.util as u; sys.modules['torch'] = None\n"
            f"spec = u.spec_from_file_location('b', {os.path.join(ROOT, 'pyramidconvblock_amd', 'build.py')!r})\n"
            "b = u.module_from_spec(spec); spec.loader.exec_module(b)\n"
            f"b.HERE = {str(tmp_path)!r}; b.OBJ = b.HERE + '/obj'; b.LIB = b.HERE + '/libpdw.so'; b._headers = lambda: []\n"
            "b.build()")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env={**os.environ, "HIPCC": str(hipcc)})
    assert r.returncode == 0, r.stderr
    assert (tmp_path / "libpdw.so").read_text() == "built\n" and not list(tmp_path.glob("_pdw_torch*"))


def test_the_host_extension_is_bound_to_its_torch(monkeypatch):
    """Another torch than the one the extension was compiled against: that file is not loaded, one is built."""
    from pyramidconvblock_amd import _lib, build

    assert _lib.ext() and os.path.exists(build.ext_path(torch.__version__))
    asked = []

    def build_ext():
        asked.append(torch.__version__)
        raise RuntimeError("no compiler")

    monkeypatch.setattr(_lib, "_ext", None)
    monkeypatch.setattr(build, "build_ext", build_ext)
    monkeypatch.setattr(torch, "__version__", "99.1.0+rocm9")
    with pytest.raises(RuntimeError, match="no compiler"):
        _lib.ext()
    assert asked == ["99.1.0+rocm9"]
    names = {build.ext_path(v) for v in ("2.10.0+rocm7.0", "2.10.0", "2.11.0+rocm7.0")}
    assert len(names) == 3 and all(os.path.dirname(n) == build.HERE for n in names)


def test_quotients_of_quads():
    """x / w as the high half of x * ceil(2^32 / w) (QuadRows of csrc/dense_wide.hip): exact for every x < w + 32 and w up to 32768."""
    import numpy as np

    for w in [*range(2, 700), *range(701, 32768, 97), 32767, 32768]:
        x = np.arange(w + 32, dtype=np.uint64)
        magic = np.uint64((2 ** 32 + w - 1) // w)
        assert ((x * magic) >> np.uint64(32) == x // np.uint64(w)).all(), w


@pytest.mark.parametrize("shape,k,stores", [
    # us, two launches and in the store: 16.7 and 14.3, 73.9 and 54.7, 20.0 and 17.1; 93.7 and 110, 76.6 and 90.6, 31.1 and 33.6
    ((3, 57, 61, 104), 9, True), ((70, 57, 57, 64), 7, True), ((2, 83, 82, 112), 15, True),
    ((107, 13, 14, 320), 17, False), ((3, 103, 103, 304), 17, False), ((54, 11, 8, 336), 9, False),
])
def test_where_a_pooled_gradient_is_added(shape, k, stores):
    """The plan of a block's convolution gradients says whether their launch adds the gradient of a pool of odd extents (bwd3_any_pays of
    csrc/dwconv_bwd3.h)."""
    from pyramidconvblock_amd import _lib

    class Mean(ctypes.Structure):   # MeanJob of csrc/mean_any.h: sums of one range, twice the channels
        _fields_ = [("part", ctypes.c_void_p), ("n", ctypes.c_int), ("B", ctypes.c_int), ("D", ctypes.c_int), ("inv_p", ctypes.c_float),
                    ("pointers", ctypes.c_void_p * 7), ("shared", ctypes.c_bool)]

    launch = _lib.lib()["_ZN3pdw18dwconv_bwd3_launchEPKvS1_S1_PvS1_S2_S2_S1_S1_S2_S2_iiiiiiiiP12ihipStream_tPiPKNS_7MeanJobE"]
    B, H, W, C = shape
    none, at, cuts, mean = ctypes.c_void_p(0), ctypes.c_void_p(256), (ctypes.c_int * 3)(), Mean(n=1, B=B, D=2 * C)
    for add, want in ((None, 0), (at, 0 if stores else -1)):
        assert launch(none, none, add, *[none] * 8, B, H, W, H // 2, W // 2, C, k, _lib.dtype_code(torch.bfloat16), none, cuts,
                      ctypes.byref(mean)) == want
    assert min(cuts) >= 1


@pytest.mark.parametrize("dtype,N,D,I", [(torch.bfloat16, 800, 256, 64), (torch.float16, 2000, 512, 64), (torch.float32, 848, 780, 448)])
def test_plans_of_sums_that_do_not_ride(dtype, N, D, I):
    """Where no launch takes both gradients of a layer, the column sums that would have ridden there keep the plan for where they run instead."""
    from pyramidconvblock_amd import _lib

    class Sums(ctypes.Structure):   # ColsumJob of csrc/mean_any.h
        _fields_ = [("x", ctypes.c_void_p), ("part", ctypes.c_void_p)] + [(n, ctypes.c_int) for n in ("B", "P", "C", "n", "len", "lanes_log", "slices")] \
            + [("pairs", ctypes.c_bool)]

    both = _lib.lib()["_ZN3pdw26dense_bwd_both_sums_launchEPKvS1_S1_PvS2_S2_mPKfixiiiP12ihipStream_tPNS_9ColsumJobE"]
    at, none = ctypes.c_void_p(4096), ctypes.c_void_p(0)
    given = (4096, 4096, 1, N, D, 32, -(-N // 32), 5, -(-D // 128), False)
    sums = Sums(*given)
    r = both(at, at, at, at, at, at, ctypes.c_size_t(1 << 40), none, 1, ctypes.c_longlong(N), D, I, _lib.dtype_code(dtype), none, ctypes.byref(sums))
    assert r == -1 and tuple(getattr(sums, n) for n, _ in Sums._fields_) == given


class _Sums(ctypes.Structure):   # ColsumJob of csrc/mean_any.h
    _fields_ = [("x", ctypes.c_void_p), ("part", ctypes.c_void_p)] + [(n, ctypes.c_int) for n in ("B", "P", "C", "n", "len", "lanes_log", "slices")] \
        + [("pairs", ctypes.c_bool)]


@pytest.mark.parametrize("dtype,shape,inter,rides", [
    # small; one round of products and more, of 8 to 16 MB; larger; fp32 by its size alone; many images
    (torch.bfloat16, (2, 40, 40, 640), 320, False), (torch.bfloat16, (71, 13, 12, 552), 288, False), (torch.float16, (105, 7, 7, 848), 432, False),
    (torch.bfloat16, (8, 58, 59, 168), 96, True), (torch.float16, (4, 64, 64, 1152), 576, True), (torch.float32, (32, 56, 56, 128), 64, True),
    (torch.float32, (2, 40, 40, 512), 256, False), (torch.float16, (65, 33, 44, 280), 144, True), (torch.bfloat16, (96, 33, 33, 296), 160, True),
    (torch.float32, (34, 38, 38, 280), 140, True),
])
def test_where_column_sums_ride(dtype, shape, inter, rides):
    """csrc/dense_wide.hip: the sums of an output gradient in its layer's launch, or (not) in that of the gates."""
    from pyramidconvblock_amd import _lib

    f = _lib.lib()["_ZN3pdw20dense_wide_sums_rideERKNS_9ColsumJobEii"]
    f.restype = ctypes.c_bool
    B, H, W, C = shape
    vecs = C // (4 if dtype == torch.float32 else 8)
    assert vecs > 16   # 32 vectors of a row to a workgroup
    assert f(ctypes.byref(_Sums(0, 0, B, H * W, C, 4, -(-H * W // 4), 5, -(-vecs // 32), False)), inter, _lib.dtype_code(dtype)) == rides
