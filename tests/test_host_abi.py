"""CPU-only checks of the host side: the C-ABI libraries load and export every
symbol include/*.h declares, the launch-shape table, the statistics, the runner
utilities and the stdout+abort error convention (no GPU compute calls here)."""
import ctypes as C
import itertools
import os
import re
import subprocess
import sys
import threading

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INCLUDE = os.path.join(REPO, "include")


def declared_functions(header):
    text = open(os.path.join(INCLUDE, header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"\b([A-Za-z_][A-Za-z0-9_]*)\s*\(", text)
    return sorted({n for n in names if n.startswith(("gpu", "mgpu", "imexHip", "_mlir_ciface_", "printMemref"))})


def test_runtime_exports_every_declared_symbol(host):
    rt = host.runtime()
    names = declared_functions("imex_hip_runtime.h")
    assert {"gpuCreateStream", "gpuStreamDestroy", "gpuMemAlloc", "gpuMemFree", "gpuMemCopy", "gpuModuleLoad",
            "gpuKernelGet", "gpuLaunchKernel", "gpuWait"} <= set(names)
    for n in names:
        assert getattr(rt, n) is not None, n
    assert set(names) == set(host._RUNTIME_SYMBOLS), "python mirror and header disagree"


def test_kernel_library_exports_and_catalogue(host):
    k = host.kernels()
    for n in declared_functions("imex_hip_kernels.h"):
        assert getattr(k, n) is not None, n
    names = host.kernel_names()
    assert len(names) == len(set(names)) >= 20
    header = open(os.path.join(INCLUDE, "imex_hip_kernels.h")).read()
    for n in names:
        size = C.c_size_t(0)
        blob = k.imexHipKernelModule(n.encode(), C.byref(size))
        assert blob and size.value > 1000
        magic = C.string_at(blob, 24)
        assert magic[:4] == b"\x7fELF" or magic.startswith(b"__CLANG_OFFLOAD_BUNDLE__")
        # the kernel's name is in its code object's symbol table
        assert n.encode() in C.string_at(blob, size.value)
        stem = re.sub(r"_(f32|f16|bf16|b16|b32|acc)$", "", n)
        assert stem in header, "kernel %s is not documented in imex_hip_kernels.h" % n
    assert k.imexHipKernelModule(b"no_such_kernel", None) is None


def test_ops_library_exports_every_declared_symbol(host):
    ops = host.ops()
    names = declared_functions("imex_hip_ops.h")
    assert "imexHipGemmBiasSiluBf16SplitKNoAlloc" in names and len(names) == 5
    for n in names:
        assert getattr(ops, n) is not None, n
    assert set(names) == set(host._OPS_SYMBOLS)
    # no compute without a GPU: only what needs none
    assert ops.imexHipOpsFixedWorkspaceBytes() == host.kernels().imexHipStreamKWorkspaceBytes(256)
    assert ops.imexHipOpsLastError() == b""


def test_runner_utils_exports(host):
    ru = host.runner_utils()
    for n in declared_functions("imex_runner_utils.h"):
        assert getattr(ru, n) is not None, n


def test_launch_shapes(host):
    ls = host.launch_shape
    assert ls("imex_relu_f32", [4096 * 4096]) == ((4096, 1, 1), (256, 1, 1), 0)
    assert ls("imex_relu_f32", [1])[0] == (1, 1, 1)
    assert ls("imex_maximum_f32", [256 * 256]) == ((16, 1, 1), (256, 1, 1), 0)
    assert ls("imex_exp_f32", [256 * 256]) == ((64, 1, 1), (256, 1, 1), 0)  # one vector per lane below 4 Mi elements
    assert ls("imex_relu_f32", [0])[0][0] == 0  # nothing to launch
    assert ls("imex_relu_bf16", [8193])[0] == (2, 1, 1)
    assert ls("imex_softmax_f16", [16384, 1024])[0] == (2048, 1, 1)  # a wavefront per slot of the chip; they walk the rows
    assert ls("imex_softmax_f16", [16383, 1024])[0] == (2048, 1, 1)
    assert ls("imex_softmax_f16", [1000, 512])[0] == (250, 1, 1)
    assert ls("imex_softmax_bf16", [16384, 1024])[0] == (2048, 1, 1)  # two rows per wavefront from 16384 rows on
    assert ls("imex_softmax_bf16", [16383, 1024])[0] == (4096, 1, 1)
    assert ls("imex_softmax_f32", [16, 2000])[0] == (16, 1, 1)
    assert ls("imex_rowsum_f32", [8192, 8192])[0] == (8192, 1, 1)
    assert ls("imex_rowsum_f32", [8, 256])[0] == (2, 1, 1)
    assert ls("imex_reduce_outer_f32", [32, 16 * 512 * 512])[0] == (512, 1, 1)     # 8192 outputs per workgroup
    assert ls("imex_reduce_outer_f32", [32, 1 << 20])[0] == (512, 1, 1)            # 2048
    assert ls("imex_reduce_outer_f32", [32, 5000])[0] == (5, 1, 1)                  # 1024
    assert ls("imex_transpose2d_b16", [8192, 8192])[0] == (32, 32, 1)   # 256 x 256 tiles from 2^24 elements
    assert ls("imex_transpose2d_b16", [2048, 2048])[0] == (16, 16, 1)   # 128 x 128 below
    # 128 x 128 tiles from 2^24 elements; whole tiles: 512 workgroups walk them, the next tile's loads in flight
    assert ls("imex_transpose2d_b32", [4096, 4096])[0] == (32, 16, 1)
    assert ls("imex_transpose2d_b32", [4096, 4100])[0] == (33, 32, 1)   # ragged: one workgroup per tile
    assert ls("imex_transpose2d_b32", [128, 131072])[0] == (512, 1, 1)
    assert ls("imex_transpose3d_b32", [256, 64, 1024])[0] == (8, 2, 32)
    assert ls("imex_transpose2d_b32", [2048, 4096])[0] == (64, 32, 1)   # 64 x 64 below
    assert ls("imex_transpose2d_b32", [10, 20])[0] == (1, 1, 1)
    assert ls("imex_transpose3d_b32", [16, 96, 96])[0] == (2, 1, 96)
    assert ls("imex_gemm_f16_f16_f32", [4096, 4096, 4096]) == ((256, 1, 1), (512, 1, 1), 0)
    assert ls("imex_gemm_bf16_bias_silu_bf16", [4096, 11008, 4096])[0] == (16 * 43, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [3, 3, 3])[0] == (1, 1, 1)
    # the MFMA path takes K in steps of 32 and B rows of whole 16-byte groups (N % 8 == 0); M and N need
    # not divide the 256 x 256 tile.  The catalogue must count tiles exactly when the kernel tiles.
    assert ls("imex_gemm_f16_f16_f32", [256, 256, 32])[0] == (1, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [512, 256, 96])[0] == (2, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [255, 256, 64])[0] == (1, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [257, 520, 64])[0] == (6, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [256, 256, 48])[0] == (1, 1, 1)     # K % 32 != 0 but K % 8 == 0: still tiled
    assert ls("imex_gemm_f16_f16_f32", [256, 256, 44])[0] == (4, 1, 1)     # K % 8 != 0: 128 x 128 vector-ALU tiles
    assert ls("imex_gemm_f16_f16_f32", [256, 252, 64])[0] == (4, 1, 1)     # N % 8 != 0
    assert ls("imex_gemm_f16_f16_f32_tb", [256, 252, 64])[0] == (1, 1, 1)  # B stored [N,K]: any N
    assert ls("imex_gemm_f16_f16_f32_ta", [252, 256, 64])[0] == (4, 1, 1)    # A stored [K,M]: M % 8 != 0
    assert ls("imex_gemm_f16_f16_f32_ta", [248, 256, 64])[0] == (1, 1, 1)
    # a strided operand of 2 GiB or more cannot be addressed with 32-bit offsets: the vector-ALU tiles
    assert ls("imex_gemm_f16_f16_f32", [256, 32768, 32768])[0] == (2 * 256, 1, 1)
    assert ls("imex_gemm_f16_f16_f32", [256, 32768, 32736])[0] == (128, 1, 1)
    assert ls("imex_gemm_f16_f16_f32_tb", [256, 32768, 32768])[0] == (128, 1, 1)
    assert ls("imex_gemm_4kx4kx4k_f16_f16_f32", []) == ((16, 16, 1), (512, 1, 1), 0)
    assert ls("imex_flash_attention_fwd_f16", [4, 4096]) == ((64, 4, 1), (512, 1, 1), 0)
    assert ls("imex_flash_attention_fwd_f16", [2, 100])[0] == (2, 2, 1)    # N_CTX need not divide the tiles
    assert ls("imex_flash_attention_fwd_f16", [40, 1000])[:2] == ((8, 40, 1), (512, 1, 1))
    assert ls("imex_flash_attention_fwd_f16", [64, 1000])[:2] == ((4, 64, 1), (1024, 1, 1))
    # 64, 128 or 256 queries per workgroup: the most that still leaves 256 workgroups
    assert ls("imex_flash_attention_fwd_f16", [8, 4096])[0] == (32, 8, 1)
    assert ls("imex_flash_attention_fwd_f16", [16, 4096])[:2] == ((16, 16, 1), (1024, 1, 1))  # 256 queries: 16 wavefronts
    assert ls("imex_flash_attention_fwd_f16", [64, 1024])[:2] == ((4, 64, 1), (1024, 1, 1))
    assert ls("imex_flash_attention_fwd_f16", [3, 256])[0] == (4, 3, 1)
    assert ls("imex_input_fusion_f32", [512, 1024])[:2] == ((256, 1, 1), (320, 1, 1))  # 4 columns per workgroup
    assert ls("imex_input_fusion_bf16", [512, 1024])[:2] == ((256, 1, 1), (320, 1, 1))
    assert ls("imex_input_fusion_f32", [512, 4096])[:2] == ((512, 1, 1), (256, 1, 1))
    assert ls("imex_input_fusion_f32", [512, 65536])[0] == (1024, 1, 1)    # 64
    # tall and wide: the streaming form, 576 lanes per 128-byte row segment
    assert ls("imex_input_fusion_f32", [8192, 8192])[:2] == ((256, 1, 1), (576, 1, 1))
    assert ls("imex_input_fusion_bf16", [8192, 8192])[:2] == ((128, 1, 1), (576, 1, 1))
    assert ls("imex_input_fusion_f16", [2048, 8200])[:2] == ((129, 1, 1), (576, 1, 1))
    assert ls("imex_input_fusion_f32", [2047, 8192])[1] == (256, 1, 1)
    assert ls("imex_input_fusion_f16", [8192, 4096])[1] == (256, 1, 1)
    assert ls("imex_gemm_4kx4kx4k_transpose_a", []) == ((16, 16, 1), (512, 1, 1), 0)
    assert ls("imex_gemm_f16_f16_f32_tb", [512, 256, 96])[0] == (2, 1, 1)
    with pytest.raises(ValueError):
        ls("imex_mfma_lds_ceiling_f16", [512])  # measurement kernels are not catalogue entries
    with pytest.raises(ValueError):
        ls("imex_relu_f32", [1, 2])
    with pytest.raises(ValueError):
        ls("imex_relu_f32", [-1])
    with pytest.raises(ValueError):
        ls("nope", [1])


def test_kernel_variants(host):
    """What imexHipKernelVariant names is in the catalogue, takes the operator's arguments, and stays the operator
    itself where that is the fastest form or the MFMA paths do not take the shape."""
    v = host.variant
    assert v("imex_gemm_f16_f16_f32", [4096, 4096, 4096]) == "imex_gemm_f16_f16_f32"
    assert v("imex_gemm_bf16_bias_silu_bf16", [4096, 11008, 4096]) == "imex_gemm_bf16_bias_silu_bf16"
    assert v("imex_gemm_f16_f16_f32_tb", [1000, 1000, 1000]) == "imex_gemm_f16_f16_f32_tb_t64"
    assert v("imex_relu_f32", [1000]) == "imex_relu_f32"
    assert host.kernels().imexHipKernelVariant(b"nope", None, 0) is None
    seen = set()
    for base in ("imex_gemm_f16_f16_f32", "imex_gemm_f16_f16_f32_acc", "imex_gemm_bf16_bf16_f32", "imex_gemm_f16_f16_f16",
                 "imex_gemm_bf16_bf16_f32_acc", "imex_gemm_bf16_bias_silu_bf16", "imex_gemm_f16_f16_f32_ta",
                 "imex_gemm_f16_f16_f32_tb"):
        for m in (1, 16, 64, 300, 1000, 2048):
            for n in (8, 64, 1000, 4096):
                for k in (8, 256, 1000, 4096):
                    name = v(base, [m, n, k])
                    assert name.startswith(base) and host.signature_types(name) == host.signature_types(base)
                    assert host.launch_shape(name, [m, n, k])[0][0] >= 1
                    seen.add(name[len(base):])
    assert {"_t128", "_t64", "_t32", "_t16"} <= seen


def test_kernel_variants_for_unaligned_rows(host):
    """Rows that are not 16-byte aligned: the operator's own loop for small products of short sums, the matrix cores
    beyond, and the operator again where a row holds no whole 16 bytes or an offset would not fit."""
    v, shape = host.variant, host.launch_shape
    for base in ("imex_gemm_f16_f16_f32", "imex_gemm_f16_f16_f32_ta", "imex_gemm_f16_f16_f32_tb",
                 "imex_gemm_bf16_bias_silu_bf16"):
        assert v(base, [129, 129, 17]) == base and v(base, [101, 101, 191]) == base
        assert v(base, [101, 101, 193]) == base + "_u16x16" and v(base, [1001, 1003, 99]) == base + "_u64"
        assert v(base, [4097, 4097, 4097]) == base + "_u128"
        assert shape(base + "_u64", [130, 65, 9])[0][0] == 6 and shape(base + "_u128", [130, 65, 9])[0][0] == 2
        assert v(base, [4097, 4097, 7]) == base and v(base, [4097, 4097, (1 << 22) + 1]) == base
    assert v("imex_gemm_f16_f16_f32", [99999, 7, 4097]) == "imex_gemm_f16_f16_f32"
    assert v("imex_gemm_f16_f16_f32_tb", [99999, 7, 4097]) != "imex_gemm_f16_f16_f32_tb"
    assert v("imex_gemm_f16_f16_f32_ta", [7, 99999, 4097]) == "imex_gemm_f16_f16_f32_ta"


def test_transposes_of_few_columns_keep_the_larger_tiles(host):
    """Tall 16-bit transposes of 5.5 .. 15 MB whose columns are no whole tiles of 64, up to 1.14 of the time with these."""
    form = lambda bits, *dims: host.variant("imex_transpose%dd_b%d" % (len(dims), bits), list(dims))[len("imex_transpose2d_b16"):]
    for rows, cols in ((16336, 200), (20568, 264), (20360, 232), (16336, 304), (25072, 248), (13752, 200), (8200, 456)):
        assert form(16, rows, cols) == "", (rows, cols)
    for rows, cols in ((16336, 256), (16336, 320), (13736, 200), (31240, 248), (5016, 600), (16336, 1400)):
        assert form(16, rows, cols) == "_any", (rows, cols)
    assert form(32, 20360, 232) == form(16, 16328, 3, 200) == "_any"


def test_narrow_tiles_for_unaligned_short_sums(host):
    """Between 129 and 191 k the narrow tiles for odd rows only where they should gain 6 %: ones that lost up to 8 %."""
    tile = lambda kind, *dims: host.variant("imex_gemm_" + kind, list(dims))[len("imex_gemm_" + kind):]
    for kind, *dims in (("f16_f16_f32_ta", 798, 549, 185), ("f16_f16_f32_tb", 1233, 137, 189), ("f16_f16_f32", 377, 897, 169),
                        ("f16_f16_f32_tb", 1167, 287, 133)):
        assert tile(kind, *dims) == "_u64", (kind, dims)
    assert tile("f16_f16_f32_acc", 815, 237, 73) == tile("f16_f16_f16", 327, 431, 111) == "_u32"
    assert tile("bf16_bias_silu_bf16", 341, 447, 183) == "_u32" and tile("f16_f16_f32_tb", 197, 1317, 193) == "_u32"


def test_param_desc_packing(host):
    descs, keep = host._pack_params([host.Ptr(0x1000), 7, 2.5])
    assert C.sizeof(host.ParamDesc) == 16
    assert [d.size for d in descs] == [8, 8, 4, 0]
    assert descs[3].data is None
    assert C.cast(descs[0].data, C.POINTER(C.c_void_p))[0] == 0x1000
    assert C.cast(descs[1].data, C.POINTER(C.c_int64))[0] == 7
    assert C.cast(descs[2].data, C.POINTER(C.c_float))[0] == 2.5


def test_launch_shapes_of_every_form_fit_a_launch(host):
    """HIP takes fewer than 2^32 lanes per dimension of a launch: every further form of an operator has a grid within
    that at any size (it strides over the rest), none of it empty, and the transposes' a multiple of the 8 XCDs."""
    forms = [n for n in host.kernel_names() if re.search(r"_(shared|l\d+|short|tall|deep|any|[tuq]\d+(x\d+)?)$", n)]
    assert len(forms) > 60
    sizes = [1, 8, 9, 4096, 65537, (1 << 24) - 1, 1 << 24, (1 << 28) + 8, (1 << 34) + 4]
    for name in forms:
        ndims = next(k for k in (1, 2, 3) if host.kernels().imexHipKernelLaunchShape(
            name.encode(), (C.c_int64 * 3)(1, 1, 1), k, (C.c_size_t * 3)(), (C.c_size_t * 3)(), None) == 0)
        for dims in itertools.product(sizes, repeat=ndims):
            grid, block, _ = host.launch_shape(name, list(dims))
            assert all(g >= 1 and g * b < 1 << 32 for g, b in zip(grid, block)), (name, dims, grid, block)
            if name.endswith("_any"):
                assert grid[0] % 8 == 0
    # many planes of one small tile; a lane per output
    assert host.launch_shape("imex_transpose3d_b16_any", [8, 1 << 24, 9])[0][0] == (1 << 24) - 8
    assert host.launch_shape("imex_reduce_outer_f32_deep", [2, (1 << 32) + 1])[0][0] == (1 << 24) - 8


def test_softmax_launch_rules(host):
    """Rows of 65 .. 128 whole pieces stay with the operator's wavefronts as far as these are the faster form; a workgroup's
    row gets whole wavefronts that hold it in at most four pieces per lane."""
    choice = lambda dt, rows, pieces: host.variant("imex_softmax_" + dt, [rows, pieces * (4 if dt == "f32" else 8)])
    for dt in ("f32", "bf16"):
        own, shared = "imex_softmax_" + dt, "imex_softmax_%s_shared" % dt
        assert [choice(dt, 8192, n) for n in (64, 65, 128, 129)] == [shared, own, own, shared]
        assert [choice(dt, rows, n) for rows, n in ((8193, 95), (8193, 96), (16384, 96), (16385, 96))] == [shared, own, own, shared]
        assert host.variant(own, [100, 65 * 8 + 1]) == shared
    assert choice("f16", 1 << 20, 128) == "imex_softmax_f16" and choice("f16", 1 << 20, 64) == "imex_softmax_f16_shared"
    for pieces in range(257, 4097):
        grid, block, _ = host.launch_shape("imex_softmax_f32_shared", [3000, 4 * pieces - 3])
        assert grid == (3000, 1, 1) and block[0] % 64 == 0 and block[0] <= 1024
        assert pieces <= 4 * block[0] and -(-pieces // block[0]) == -(-pieces // (256 if pieces <= 1024 else 512 if pieces <= 2048 else 1024))
    # a wavefront per row from 1024 rows of up to 256 pieces on
    assert host.launch_shape("imex_softmax_f32_shared", [1024, 800])[0] == (256, 1, 1)
    assert host.launch_shape("imex_softmax_f32_shared", [1023, 800])[0] == (1023, 1, 1)


def test_reduce_outer_launch_rules(host):
    """The outer sum's own form for large slices of whole vectors, from 4 MiB for up to four of them; chains for narrow and
    for tall matrices, a lane per vector (or column) for few slices of many columns."""
    choice = lambda dt, outer, inner: host.variant("imex_reduce_outer_" + dt, [outer, inner])[len("imex_reduce_outer_" + dt):]
    mib = 1 << 20
    for dt, width, least in (("f32", 4, 5), ("f16", 2, 8), ("bf16", 2, 8)):
        for outer in (1, 4):
            assert [choice(dt, outer, 4 * mib // width + d) for d in (-8, 0, 1)] == ["_deep", "", "_deep"]
        for outer in (5, 32):
            assert [choice(dt, outer, least * mib // width + d) for d in (-8, 0, 1)] == ["_deep", "", "_deep"]
        for cols in range(1, 17):
            assert choice(dt, 8192, cols) == choice(dt, 200, cols) == "_tall"
        assert choice(dt, 8192, 4096) == choice(dt, 64, 2000) == "_tall" and choice(dt, 64, 100000) == "_deep"
        assert choice(dt, 0, 16) == choice(dt, 16, 0) == ""
    assert choice("f32", 62, 32296) == "_tall" and choice("f32", 568, 197848) == "_deep"


def test_gemm_tile_rules(host):
    """Tiles by size: few rows narrow ones, ordinary products 64 x 64 and up, short sums with large results 256 x 256 (f32)
    or 128 x 64 (16-bit), short sums with small results 64 x 64."""
    tile = lambda kind, *dims: host.variant("imex_gemm_" + kind, list(dims))[len("imex_gemm_" + kind):]
    assert tile("f16_f16_f32", 4096, 4096, 4096) == tile("bf16_bias_silu_bf16", 4096, 11008, 4096) == ""
    assert tile("f16_f16_f32_ta", 2168, 4064, 312) == tile("bf16_bf16_f32", 2740, 3360, 216) == ""
    assert tile("f16_f16_f16", 3000, 1600, 48) == "_t128x64s"
    assert tile("f16_f16_f32_tb", 1000, 1000, 1000) == tile("f16_f16_f32", 771, 880, 112) == tile("bf16_bf16_f32", 314, 2160, 72) == "_t64"
    assert tile("bf16_bias_silu_bf16", 923, 992, 120) == "_t64"
    assert tile("bf16_bias_silu_bf16", 16, 11008, 4096) == "_t16"
    assert tile("f16_f16_f32", 16, 1680, 3992) == tile("f16_f16_f32", 256, 256, 256) == "_t16x16"
    assert tile("f16_f16_f32", 1001, 1003, 999) == "_u64"


def test_gemm_workgroups_that_fetch_rule(host):
    """256 workgroups where few tiles walk a long K over operands of 2 .. 32 MiB, a workgroup per tile elsewhere."""
    grid = lambda tile, *dims: host.launch_shape("imex_gemm_bf16_bias_silu_bf16" + tile, list(dims))[0][0]
    assert grid("_t16x16", 16, 1680, 3992) == grid("_t32", 128, 2048, 4096) == grid("_t128x64", 1000, 1000, 1024) == 256
    assert grid("_t16x16", 16, 1680, 760) == 105 and grid("_t16x16", 16, 640, 1024) == 40 and grid("_t64", 16, 8192, 4096) == 128
    assert grid("_t16x16", 16, 2816, 1024) == 176 and grid("_t128", 1000, 1000, 1024) == 64
    # operands that the L2s may hold: from 1024 k (16 x 16 1400) and 3.75 MiB, or 2560 k and 2 MiB
    assert [grid("_t16x32", 2, n, 1024) for n in (1912, 1920)] == [60, 256] and grid("_t16x32", 2, 2000, 1016) == 63
    assert [grid("_t16x16", 5, 1720, k) for k in (1184, 1392, 1400)] == [108, 108, 256]
    # an XCD's share of the operands: below 6 MiB, of a 4 MiB L2
    assert [grid("_t32", 1560, 168, k) for k in (7416, 7424, 9680)] == [256, 147, 147]
    assert [grid("_t16x16", 2, n, 2560) for n in (400, 424)] == [25, 256] and grid("_t16x16", 2, 424, 2552) == 27
    assert grid("_t16x16", 2, 1560, 1080) == 98 and grid("_t16x32", 391, 176, 1928) == 150
    assert grid("_t16x32", 141, 544, 2800) == 153 and grid("_t16x32", 141, 448, 2800) == 256  # 2 MiB: 128 tiles at most
    assert grid("_t128x64", 3409, 296, 3776) == 135 and grid("_t64", 1500, 296, 4096) == grid("_t128x64", 1500, 296, 4096) == 256
    assert grid("_t64", 1500, 384, 4096) == 256 and grid("_t128x64", 1700, 392, 4096) == 98


def test_gemm_workgroups_that_fetch_do_not_draw_problems_to_slower_tiles(host):
    """Problems that lost up to a fifth of their speed to tiles of 16 x 64 (or 16 x 32 with B^T) and workgroups that fetch."""
    tile = lambda kind, *dims: host.variant("imex_gemm_" + kind, list(dims))[len("imex_gemm_" + kind):]
    for m, n, k in ((151, 576, 3456), (257, 416, 2656), (219, 479, 3256), (682, 143, 2680)):
        assert tile("f16_f16_f32_tb", m, n, k) == "_t16x32", (m, n, k)
    assert tile("bf16_bf16_f32_acc", 329, 288, 2432) == tile("f16_f16_f32_acc", 551, 224, 3056) == "_t16x32"
    assert tile("f16_f16_f32_tb", 48, 1000, 2064) == "_t16x16" and tile("f16_f16_f16", 156, 400, 2152) == "_t16x16"
    for m, n, k in ((405, 144, 2920), (414, 136, 3456), (286, 144, 2784), (178, 224, 2656)):
        assert tile("f16_f16_f32", m, n, k) == "_t16x16", (m, n, k)
    assert tile("f16_f16_f32_ta", 104, 1648, 3288) == "_t32" and tile("bf16_bias_silu_bf16", 15, 2624, 2904) == "_t16x32"


def test_gemm_workgroups_that_fetch_do_not_draw_problems_beyond_an_l2(host):
    """Problems whose tiles of one XCD read more than its 4 MiB L2, where the fetched lines were gone before their use: up to
    1.3 times as long with the tiles that they were drawn to."""
    tile = lambda kind, *dims: host.variant("imex_gemm_" + kind, list(dims))[len("imex_gemm_" + kind):]
    for kind, *dims in (("f16_f16_f16", 200, 800, 12944), ("bf16_bf16_f32", 416, 320, 8480), ("f16_f16_f32_tb", 496, 360, 11656),
                        ("bf16_bf16_f32_acc", 64, 2272, 6520), ("bf16_bias_silu_bf16", 27, 4184, 3936)):
        assert tile(kind, *dims) == "_t16", (kind, dims)
    assert tile("f16_f16_f32", 640, 600, 12064) == "_t32"
    assert tile("bf16_bias_silu_bf16", 155, 912, 6552) == "_t32" and tile("bf16_bias_silu_bf16", 155, 912, 6560) == "_t16"


def test_plan_packs_arguments_as_the_kernel_declares_them(host):
    """Stream.launch's fast path: 8 bytes per argument, an f32 in the low four, with _pack_params' conversions and errors."""
    class Resolver:
        def kernel(self, name):
            return 1
    plan = host._Plan(Resolver(), "imex_rowsum_f32", [3, 5])
    p, q = host.Ptr(0x1000), host.Ptr(0x2000)
    want = np.array([0x1000, 0x2000, 3, 5], np.int64).tobytes() + np.array([2.5, 0], np.float32).tobytes()
    assert plan.pack([p, q, 3, 5, 2.5]) == want
    assert plan.pack([p, q, 3.0, np.int32(5), np.float64(2.5)]) == want
    assert plan.pack([p, q, 3, 5, 1e300])[-8:-4] == np.array([np.inf], np.float32).tobytes()
    assert list(plan.shape) == [1, 1, 1, 256, 1, 1, 0]
    for bad in ([p, 0x2000, 3, 5, 2.5], [p, q, 3.5, 5, 2.5], [p, q, 3, 5]):
        with pytest.raises(TypeError):
            plan.pack(bad)


def test_plan_refuses_a_grid_that_no_launch_takes(host):
    """A grid of 2^32 workgroups and more is an error, as it is for gpuLaunchKernel, not its low 32 bits."""
    class Resolver:
        def kernel(self, name):
            return 1
    rows = (1 << 34) + 4  # a workgroup per four rows: 2^32 + 1
    assert host.launch_shape("imex_rowsum_f32", [rows, 2000])[0][0] == (1 << 32) + 1
    with pytest.raises(ValueError, match="outside"):
        host._Plan(Resolver(), "imex_rowsum_f32", [rows, 2000])


def test_launch_takes_the_dims_that_launch_shape_takes(host):
    """Whole numbers of any integer type, and nothing else -- also where the plan of an equal number is kept."""
    launched = []

    class Runtime:
        def imexHipLaunchValues(self, *args):
            launched.append(args)
            return 7
    s = host.Stream.__new__(host.Stream)
    s.rt, s.handle, s._plans, s.kernel = Runtime(), 1, {}, lambda name: 1
    p = host.Ptr(0x1000)
    for n in (64, np.int64(64), np.uint8(64)):
        assert s.launch("imex_relu_f32", [n], [p, p, 64]) == 7
    for n in (64.0, np.float32(64), "64"):
        with pytest.raises(TypeError):
            host.launch_shape("imex_relu_f32", [n])
        with pytest.raises(TypeError):
            s.launch("imex_relu_f32", [n], [p, p, 64])
    assert len(launched) == 3 and len(s._plans) == 1


def test_launch_with_dependencies_uses_the_kept_plan(host):
    """The kernel of a size is resolved once, whether a launch waits for events of other streams or not, and both go
    to the variant the catalogue advises under its launch shape."""
    launched, resolved = [], []

    class Runtime:
        def imexHipLaunchValues(self, handle, fn, shape, values, count):
            launched.append((fn, tuple(shape)))

        def gpuLaunchKernel(self, handle, fn, *rest):
            launched.append((fn, rest[:7]))
    s = host.Stream.__new__(host.Stream)
    s.rt, s.handle, s._plans, s.kernel = Runtime(), 1, {}, lambda name: resolved.append(name) or name
    p = host.Ptr(0x1000)
    for deps in (None, [0x20], [0x20, 0x30]):
        s.launch("imex_rowsum_f32", [300, 40], [p, p, 300, 40, 0.0], deps=deps)
    name = host.variant("imex_rowsum_f32", [300, 40])
    grid, block, smem = host.launch_shape(name, [300, 40])
    assert name != "imex_rowsum_f32" and resolved == [name]
    assert launched == [(name, (*grid, *block, smem))] * 3


def test_staging_block_of_a_queue(host):
    """One block per caller at a time, one kept, grown by powers of two, freed when its user fails and with the queue."""
    live = {}

    class Runtime:
        def gpuMemAlloc(self, handle, nbytes, alignment, shared):
            assert shared == 1
            buf = C.create_string_buffer(nbytes)
            live[C.addressof(buf)] = buf
            return C.addressof(buf)

        def gpuMemFree(self, handle, ptr):
            del live[ptr]

        def gpuStreamDestroy(self, handle):
            assert not live
    s = host.Stream.__new__(host.Stream)
    s.rt, s.handle, s._staging = Runtime(), 1, []
    with s.staging(100) as (p, block):
        assert len(block) == 1 << 18 and p in live
        with s.staging(100) as (q, _):  # a second thread
            assert q != p and len(live) == 2
    assert len(live) == 1  # one of the two is kept
    with s.staging(1 << 18) as (q, _):
        assert list(live) == [q]
    with s.staging((1 << 18) + 1) as (q, block):
        assert list(live) == [q] and len(block) == 1 << 19
    with pytest.raises(RuntimeError):
        with s.staging(5) as (q, _):
            raise RuntimeError
    assert not live
    with s.staging(5):
        pass
    s.close()
    assert not live and s.handle is None


class FakeMemory:
    """The runtime's side of a queue whose memory is the host's: what is allocated now, and how large its blocks were."""

    def __init__(self):
        self.live, self.sizes, self.can_pin = {}, [], True

    def gpuMemAlloc(self, handle, nbytes, alignment, shared):
        buf = C.create_string_buffer(nbytes)
        self.live[C.addressof(buf)] = buf
        self.sizes.append((nbytes, shared))
        return C.addressof(buf)

    def imexHipTrySharedAlloc(self, handle, nbytes):
        return self.gpuMemAlloc(handle, nbytes, 64, 1) if self.can_pin else None

    def gpuMemFree(self, handle, ptr):
        del self.live[ptr]

    def imexHipSharedFree(self, ptr):
        del self.live[ptr]

    def gpuMemCopy(self, handle, dst, src, nbytes):
        C.memmove(dst, src, nbytes)

    def gpuCreateStream(self, device, context):
        return 1

    def gpuStreamDestroy(self, handle):
        assert not self.live

    def gpuWait(self, handle):
        pass


@pytest.fixture
def fake_stream(host, monkeypatch):
    """A queue on fake memory, whose launches call `on_launch` in place of a kernel."""
    monkeypatch.setattr(host, "runtime", lambda rt=FakeMemory(): rt)
    stream = host.Stream()
    stream.on_launch = lambda: None
    stream.launch = lambda *args: stream.on_launch()
    yield stream
    stream.close()


def pinned(stream):
    """Bytes of pinned blocks that the queue has asked for, one entry each."""
    return [n for n, shared in stream.rt.sizes if shared]


def test_staged_operators_pin_no_more_than_they_say(host, fake_stream):
    """Operands that are within _STAGED_BYTES only without the space between them would get a block of twice that."""
    fake_stream.staging_pays = lambda nbytes: True
    for n in (2796201, 2796202):
        x = np.zeros(n, np.float32)
        for _ in range(2):
            host.maximum(fake_stream, x, x)
        assert max(pinned(fake_stream), default=0) <= host._STAGED_BYTES, n
    assert 12 * 2796202 <= host._STAGED_BYTES


def test_staged_operators_share_one_block(host, fake_stream):
    """A second thread's call goes through device buffers while the first one's has the queue's block."""
    x, calls = np.zeros(1000, np.float32), []

    def second():
        fake_stream.on_launch = lambda: None
        before = len(pinned(fake_stream))
        thread = threading.Thread(target=lambda: calls.append(host.relu(fake_stream, x)))
        thread.start()
        thread.join()
        assert len(pinned(fake_stream)) == before
    for _ in range(8):
        host.relu(fake_stream, x)
    fake_stream.on_launch = second
    host.relu(fake_stream, x)
    assert len(calls) == 1 and len(fake_stream._staging) == 1 and len(pinned(fake_stream)) == 1


def test_staged_operators_beside_a_thread_that_takes_the_block(host, fake_stream):
    """`staging` of another thread may take the kept block at any moment: between a look whether there is one and a look
    at it, or before it is given back for a larger one."""
    class Taken(list):  # as a list from which the one block goes right after the look
        def __bool__(self):
            return True

        def __len__(self):
            return 1
    small, large = np.zeros(100, np.float32), np.zeros(1 << 19, np.float32)
    for x in [small] * 3 + [large] * 11:
        fake_stream._staging = Taken()
        assert np.array_equal(host.relu(fake_stream, x), x)
        while list.__len__(fake_stream._staging):
            fake_stream.free(fake_stream._staging.pop()[0])
    fake_stream._staging = []


@pytest.mark.parametrize("n,waits", [(1, 1), (1 << 16, 1), (1 << 17, 2), ((1 << 17) + 1, 5), (1 << 20, 20), (1 << 22, 80)])
def test_staged_operators_wait_for_a_block(host, fake_stream, n, waits):
    """A queue's first calls go through device buffers, five for every two MiB of the pinned block that they would get:
    one call on 32 MiB paid 11 ms for it, 60 times what it gained."""
    x = np.zeros(n, np.float32)
    for call in range(waits):
        host.relu(fake_stream, x)
        assert not pinned(fake_stream), call
    for _ in range(3):
        host.relu(fake_stream, x)
    assert len(pinned(fake_stream)) == 1 and pinned(fake_stream)[0] >= 8 * n


def test_staged_operators_grow_their_block_by_the_same_rule(host, fake_stream):
    """Smaller calls take the block that is kept and do not bring a larger one any nearer."""
    small, large = np.zeros(100, np.float32), np.zeros(1 << 19, np.float32)  # 4 MiB for the larger
    for _ in range(40):
        host.relu(fake_stream, small)
    assert pinned(fake_stream) == [1 << 18]
    for _ in range(10):
        host.relu(fake_stream, large)
        host.relu(fake_stream, small)
    assert pinned(fake_stream) == [1 << 18]
    host.relu(fake_stream, large)
    assert pinned(fake_stream) == [1 << 18, 1 << 22] and len(fake_stream._staging) == 1


def test_staged_operators_do_without_pinned_memory(host, fake_stream):
    """Where none is to be had every call goes through device buffers, as it did before there was a block, and a smaller
    block that is kept stays."""
    small, large = np.zeros(100, np.float32), np.zeros(1 << 19, np.float32)
    fake_stream.rt.can_pin = False
    for _ in range(9):
        host.relu(fake_stream, small)
    assert not pinned(fake_stream) and not fake_stream._staging
    fake_stream.rt.can_pin = True
    for _ in range(2):
        host.relu(fake_stream, small)
    fake_stream.rt.can_pin = False
    for _ in range(30):
        host.relu(fake_stream, large)
    assert pinned(fake_stream) == [len(fake_stream._staging[0][1])] == [1 << 18]
    host.relu(fake_stream, small)


def test_queues_that_nobody_closes_give_their_block_back(host, monkeypatch):
    """The pinned block goes with the object, without its queue; a queue that was closed has freed it already."""
    rt = FakeMemory()
    monkeypatch.setattr(host, "runtime", lambda: rt)
    monkeypatch.setattr(host.Stream, "launch", lambda *args: None)
    x = np.zeros(1000, np.float32)
    for closed in (False, True):
        s = host.Stream()
        for _ in range(3):
            host.relu(s, x)
        assert len(rt.live) == 1
        if closed:
            s.close()
        else:
            rt.gpuMemFree = None
        del s
        assert not rt.live
        vars(rt).pop("gpuMemFree", None)


class _Way(Exception):
    """Raised in place of the work by the queue of `way_of`."""


def way_of(host, op, shape, dtype="f32"):
    """"staged" or "device": where the host function `op` puts operands of this shape."""
    class Queue:
        _staging_lock = threading.Lock()

        def staging_pays(self, nbytes):
            raise _Way("staged")

        def to_device(self, array):
            raise _Way("device")
    x = np.empty(shape, np.float32 if dtype == "f32" else np.uint16)
    typed = {} if op in ("maximum", "rowsum", "rowmean", "transpose2d", "transpose3d") else {"dtype": dtype}
    with pytest.raises(_Way) as way:
        getattr(host, op)(Queue(), *[x] * (1 + (op in ("maximum", "loop_fusion", "input_fusion"))), **typed)
    return str(way.value)


@pytest.mark.parametrize("dtype,kept", [("f32", 16384), ("f16", 32768), ("bf16", 32768)])
def test_softmax_staging_rule(host, dtype, kept):
    """Rows that a workgroup cannot keep in registers and that are no whole vectors go through device buffers unless there
    are many of them: read twice over the link, element by element, one of them took up to 1.8 times as long."""
    way = lambda rows, cols: way_of(host, "softmax", (rows, cols), dtype)
    for rows in (1, 10, 63):
        assert way(rows, kept) == way(rows, kept - 1) == way(rows, kept + 8) == way(rows, 65536) == "staged"
        assert way(rows, kept + 1) == way(rows, 40001) == way(rows, 65535) == way(rows, 65537) == "device"
    assert way(64, kept + 1) == way(64, 40001) == "staged" and way(64, 65537) == way(1, 262144) == "device"


def test_transpose_staging_rule(host):
    """Transposes with runs of a few elements on either side, over the link up to four times as slow, and the largest of few
    columns go through device buffers."""
    way = lambda *shape: way_of(host, "transpose%dd" % len(shape), shape)
    assert way(12288, 128) == way(6144, 256) == way(16384, 256) == way(1, 1000000) == "staged"
    assert way(12289, 128) == way(16384, 255) == way(63715, 65) == way(16385, 256) == "device"
    assert way(12288, 1, 128) == "staged" and way(12289, 1, 128) == "device"
    for flip in (1, -1):
        assert way(*(64, 1024, 64)[::flip]) == way(*(1000, 32, 32)[::flip]) == way(*(1024, 4, 8)[::flip]) == "staged"
        assert way(*(64, 1024, 65)[::flip]) == way(*(1025, 32, 32)[::flip]) == way(*(1025, 4, 8)[::flip]) == "device"
        assert way(*(1, 4, 118937)[::flip]) == way(*(4, 4, 147889)[::flip]) == way(*(7, 36, 79)[::flip]) == "device"
        assert way(*(2, 4, 512)[::flip]) == "staged"


def test_sums_staging_rule(host):
    """Column sums and the fused chain with them: through pinned host memory on one side of measured lines, through device
    buffers on the other, where the link made them up to 2.8 times as slow."""
    way = lambda op, *shape: way_of(host, op, shape)
    assert way("reduce_outer", 512, 1024) == way("reduce_outer", 511, 1280) == way("reduce_outer", 512, 128) == "staged"
    assert way("reduce_outer", 512, 1280) == way("reduce_outer", 513, 1024) == way("reduce_outer", 1600, 600) == "device"
    assert way("reduce_outer", 1023, 256) == way("reduce_outer", 8191, 1) == "staged"
    assert way("reduce_outer", 1024, 256) == way("reduce_outer", 200, 127) == "device"
    assert way("input_fusion", 128, 2000) == way("input_fusion", 4, 70000) == way("input_fusion", 5000, 6) == "staged"
    assert way("input_fusion", 15, 2000) == way("input_fusion", 60, 540) == "staged"
    for shape in ((127, 1784), (125, 1557), (12, 31117), (5, 15846), (63, 1494), (64, 540), (128, 511), (128, 2600)):
        assert way("input_fusion", *shape) == "device", shape


def test_profiler_stats_vs_oracle(host, orc):
    rng = np.random.default_rng(3)
    for n in (1, 2, 3, 4, 7, 100, 1000):
        v = (rng.random(n) * 2).astype(np.float32)
        s = host.compute_stats(list(v))
        for mine, theirs in (("avg", "avg"), ("min", "min"), ("max", "max"), ("median", "median_textbook"),
                             ("stddev", "stddev"), ("variance", "variance"), ("p95", "p95"), ("p5", "p5"),
                             ("middle_third_avg", "middle_third_avg")):
            assert s[mine] == orc.stat(theirs, v), (mine, n)


# ---- error convention: message on stdout, then abort() ------------------------------
def _run_snippet(code):
    prog = ("import sys; sys.path.insert(0, %r)\nimport __graft_entry__ as e\nhost = e.load_package().host\n"
            "rt = host.runtime()\nimport ctypes as C\n" % REPO) + code
    return subprocess.run([sys.executable, "-c", prog], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                          timeout=120)


def test_spirv_blob_is_rejected_before_any_gpu_call():
    r = _run_snippet("blob = C.create_string_buffer(b'\\x03\\x02\\x23\\x07' + b'\\0' * 60)\n"
                     "rt.gpuModuleLoad(None, blob, 64)\nprint('survived')\n")
    assert r.returncode == -6  # SIGABRT
    assert "An exception was thrown: gpuModuleLoad: blob is SPIR-V" in r.stdout
    assert "survived" not in r.stdout


def test_garbage_and_null_blobs_abort():
    r = _run_snippet("blob = C.create_string_buffer(b'garbage!' * 8)\nrt.gpuModuleLoad(None, blob, 64)\n")
    assert r.returncode == -6 and "not a code object" in r.stdout
    # an ELF for another machine (x86-64 = 62) is refused by its header, before any HIP call
    r = _run_snippet("blob = C.create_string_buffer(b'\\x7fELF' + bytes(14) + bytes([62, 0]) + bytes(44))\nrt.gpuModuleLoad(None, blob, 64)\n")
    assert r.returncode == -6 and "not an AMDGPU code object" in r.stdout
    r = _run_snippet("rt.gpuModuleLoad(None, None, 0)\n")
    assert r.returncode == -6 and "null module data" in r.stdout
    r = _run_snippet("rt.gpuKernelGet(None, None, b'k')\n")
    assert r.returncode == -6 and "gpuKernelGet: null module" in r.stdout
    r = _run_snippet("rt.gpuLaunchKernel(None, None, 1,1,1, 1,1,1, 0, None, None)\n")
    assert r.returncode == -6 and "null stream" in r.stdout


def test_null_free_is_ignored_and_unload_is_noop():
    r = _run_snippet("rt.gpuMemFree(None, None)\nrt.gpuModuleUnload(None, None)\nrt.mgpuModuleUnload(None)\nprint('ok')\n")
    assert r.returncode == 0 and "ok" in r.stdout


# ---- runner utilities ------------------------------------------------------------------
class Desc2D(C.Structure):
    _fields_ = [("allocated", C.c_void_p), ("aligned", C.c_void_p), ("offset", C.c_int64),
                ("sizes", C.c_int64 * 2), ("strides", C.c_int64 * 2)]


class Unranked(C.Structure):
    _fields_ = [("rank", C.c_int64), ("descriptor", C.c_void_p)]


def memref2d(a):
    d = Desc2D(a.ctypes.data, a.ctypes.data, 0, (C.c_int64 * 2)(*a.shape), (C.c_int64 * 2)(a.shape[1], 1))
    u = Unranked(2, C.cast(C.pointer(d), C.c_void_p))
    return u, d


def test_runner_utils_gemm_matches_oracle_and_golden(host, orc):
    ru = host.runner_utils()
    a = orc.fill_uniform(24 * 40, "f16", 1, -1, 1).reshape(24, 40)
    b = orc.fill_uniform(40 * 16, "f16", 2, -1, 1).reshape(40, 16)
    c = np.zeros((24, 16), np.float32)
    (ua, da), (ub, db), (uc, dc) = memref2d(a), memref2d(b), memref2d(c)
    ru._mlir_ciface_gemmF16F16F32(C.byref(ua), C.byref(ub), C.byref(uc))
    assert np.array_equal(c, orc.gemm(a, b, "f16"))
    ab = orc.fill_uniform(24 * 40, "bf16", 3, -1, 1).reshape(24, 40)
    bb = orc.fill_uniform(40 * 16, "bf16", 4, -1, 1).reshape(40, 16)
    c2 = np.ones((24, 16), np.float32)
    (ua, da), (ub, db), (uc, dc) = memref2d(ab), memref2d(bb), memref2d(c2)
    ru._mlir_ciface_gemmBF16BF16F32(C.byref(ua), C.byref(ub), C.byref(uc))
    assert np.array_equal(c2, orc.gemm(ab, bb, "bf16", c=np.ones((24, 16), np.float32)))
    c3 = np.zeros((24, 16), np.float32)
    (ua, da), (ub, db), (uc, dc) = memref2d(a), memref2d(b), memref2d(c3)
    ru._mlir_ciface_gemmF16F16F16(C.byref(ua), C.byref(ub), C.byref(uc))
    assert np.array_equal(c3, orc.gemm(a, b, "f16", out_round="f16"))


def test_runner_utils_allclose_and_fill(host, orc):
    ru = host.runner_utils()
    ref = orc.fill_uniform(64, "f32", 5, -2, 2).reshape(8, 8)
    near = (ref * np.float32(1.0005)).astype(np.float32)
    far = ref.copy()
    far[3, 3] += 0.01
    (ur, dr), (un, dn), (uf, df) = memref2d(ref), memref2d(near), memref2d(far)
    assert ru._mlir_ciface_allcloseF32(C.byref(un), C.byref(ur)) is True
    assert ru._mlir_ciface_allcloseF32(C.byref(uf), C.byref(ur)) is False
    assert orc.allclose_f32(near, ref) and not orc.allclose_f32(far, ref)
    h = orc.float_to_half(ref)
    (uh, dh) = memref2d(h)
    assert ru._mlir_ciface_allcloseF16(C.byref(uh), C.byref(ur)) == orc.allclose_f32(orc.half_to_float(h), ref)
    buf = np.zeros((4, 6), np.uint16)
    (ub, db) = memref2d(buf)
    ru._mlir_ciface_fillResource1DBF16.argtypes = [C.c_void_p, C.c_float]
    ru._mlir_ciface_fillResource1DBF16(C.byref(ub), 1.5)
    assert np.all(buf == 0x3fc0)
    os.environ["IMEX_RANDOM_SEED"] = "7"
    r1 = np.zeros((5, 5), np.float32)
    (u1, d1) = memref2d(r1)
    ru._mlir_ciface_fillResource1DRandomF32.argtypes = [C.c_void_p, C.c_float, C.c_float, C.c_bool]
    ru._mlir_ciface_fillResource1DRandomF32(C.byref(u1), -0.5, 0.5, False)
    assert r1.min() >= -0.5 and r1.max() < 0.5 and len(np.unique(r1)) > 20
    del os.environ["IMEX_RANDOM_SEED"]


def test_runner_utils_conversions_exhaustive(host, orc):
    """allcloseF16 / allcloseBF16 widen with the library's own converters: compare
    all 65536 patterns against the oracle by filling through the library."""
    ru = host.runner_utils()
    vals = orc.half_to_float(np.arange(0x7c00, dtype=np.uint16)).reshape(-1, 64)
    out = np.zeros(vals.shape, np.uint16)
    ref = np.ascontiguousarray(vals)
    (uo, do), (ur, dr) = memref2d(out), memref2d(ref)
    # every finite half survives f32 -> f16 through the library: allclose with itself is exact
    for i, v in enumerate(ref.ravel()[:: 997]):
        one = np.zeros((1, 1), np.uint16)
        (u1, d1) = memref2d(one)
        ru._mlir_ciface_fillResource1DF16.argtypes = [C.c_void_p, C.c_float]
        ru._mlir_ciface_fillResource1DF16(C.byref(u1), float(v))
        assert one[0, 0] == orc.float_to_half(np.array([v], np.float32))[0]


def test_print_helpers(host, orc, capfd):
    ru = host.runner_utils()
    g = np.array([[14.1, 14.8, 14.6], [11, 13, 10.5], [13.9, 19.9, 12.4]], np.float32)
    h = orc.float_to_half(g)
    (uh, dh), (ug, dg) = memref2d(h), memref2d(g)
    ru._mlir_ciface_printAllcloseF16(C.byref(uh), C.byref(ug))
    ru._mlir_ciface_printMemrefF16(C.byref(uh))
    ru._mlir_ciface_printMaxErrorF32(C.byref(ug), C.byref(ug))
    C.CDLL(None).fflush(None)  # the library prints through C++ iostreams
    out = capfd.readouterr().out
    assert "[ALLCLOSE: TRUE]" in out
    assert "sizes = [3, 3] strides = [3, 1] data =" in out
    assert "[11,   13,   10.5]" in out
    assert "Max absolute error 0" in out


def test_driver_command_line():
    """Parts of the C++ driver that need no GPU: the workload list, bench_imex's -c
    (not offered) and an unknown workload name."""
    import subprocess
    exe = os.path.join(REPO, "mlir-extensions_amd", "lib", "imex-hip-bench")
    r = subprocess.run([exe, "--list"], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0
    names = [l.split()[0] for l in r.stdout.splitlines() if l.strip()]
    assert "gemm_f16_4096" in names and "flash_attention_f16_2x2x4096x64" in names and len(names) >= 11
    r = subprocess.run([exe, "-c", "all"], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 1 and "CPU lowering" in r.stderr
    r = subprocess.run([exe, "no_such_workload"], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 2 and "unknown workload" in r.stderr


def test_launch_shapes_cover_the_problem(host):
    """For the kernels that do not stride over their work (element-wise, reductions,
    fused chains, tiled GEMM) the catalogue's grid must cover every element; checked
    over random problem sizes against each kernel's work per workgroup."""
    from hypothesis import given, settings, strategies as st
    ls = host.launch_shape

    @settings(max_examples=300, deadline=None)
    @given(n=st.integers(1, 1 << 34))
    def eltwise(n):
        small = n < (1 << 22)
        for name, per in (("imex_relu_f32", 4096), ("imex_silu_f32", 1024 if small else 4096), ("imex_relu_bf16", 8192),
                          ("imex_loop_fusion_f32", 1024 if small else 4096),
                          ("imex_loop_fusion_f16", 2048 if small else 8192)):
            (gx, gy, gz), block, _ = ls(name, [n])
            assert block == (256, 1, 1) and gy == gz == 1
            assert (gx - 1) * per < n <= gx * per

    @settings(max_examples=300, deadline=None)
    @given(rows=st.integers(1, 1 << 20), cols=st.integers(1, 1 << 14))
    def rowwise(rows, cols):
        (gx, _, _), _, _ = ls("imex_rowsum_f32", [rows, cols])
        assert gx == rows if cols > 2048 else gx * 4 >= rows
        (gx, _, _), _, _ = ls("imex_reduce_outer_f32", [rows, cols])
        assert gx >= 1 and gx * 8192 >= cols  # the kernel strides over whatever the grid leaves
        (gx, _, _), _, _ = ls("imex_input_fusion_f32", [rows, cols])
        assert gx * 64 >= cols
        (gx, _, _), _, _ = ls("imex_softmax_f16", [rows, cols])
        assert gx >= 1 and (gx == min(-(-rows // 4), 2048) if cols <= 1024 else gx >= min(rows, 1048560))
        (gx, _, _), _, _ = ls("imex_softmax_bf16", [rows, cols])
        assert gx >= 1 and (gx * (8 if rows >= 16384 else 4) >= rows if cols <= 1024 else gx >= min(rows, 1048560))

    @settings(max_examples=300, deadline=None)
    @given(M=st.integers(1, 20000), N=st.integers(1, 20000), k=st.integers(1, 512), round_n=st.booleans(),
           round_k=st.booleans())
    def gemm(M, N, k, round_n, round_k):
        N = (N + 7) // 8 * 8 if round_n else N
        K = k * 8 if round_k else k * 7 + 5
        for name in ("imex_gemm_f16_f16_f32", "imex_gemm_f16_f16_f32_ta", "imex_gemm_f16_f16_f32_tb",
                     "imex_gemm_bf16_bias_silu_bf16"):
            (gx, gy, gz), block, _ = ls(name, [M, N, K])
            assert block == (512, 1, 1) and gy == gz == 1
            tileable = K % 8 == 0 and (name.endswith("_tb") or N % 8 == 0) and (not name.endswith("_ta") or M % 8 == 0)
            assert gx == (-(-M // 256) * -(-N // 256) if tileable else -(-M // 128) * -(-N // 128))

    eltwise()
    rowwise()
    gemm()
