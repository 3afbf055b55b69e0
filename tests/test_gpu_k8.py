"""Pre-shuffled weights (direct_b_k8) through LDS, K over waves and tiles 128 columns wide, at the edges of their
tiles, panels and K loops: against the CPU oracle; the same bits on a second run and from a plan of the selected
id; the kernel of the variant's name still runs by its first id."""
import numpy as np
import pytest

from aster_amd import gemm as AG
from aster_amd.kittens_helpers import (shuffle_scales_e8m0_lanes, shuffle_scales_e8m0_lanes128, shuffle_weight_bytes,
                                       shuffle_weight_k8)
from oracle import gemm as G
from test_gpu_parity import _DT, REL_L2_BAR, _variant_id, check, operands, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype_ab,tile", [
    # K over waves: every tile height, fewer K-steps than wave groups, ranges of steps that are no whole rounds,
    # panels of 16 ... 128 rows with short last ones
    (8, 16, 64, "bf16", (16, 16)), (16, 4096, 4096, "f16", (16, 16)), (16, 6160, 1088, "bf16", (16, 32)),
    (8, 11008, 640, "bf16", (16, 48)), (16, 14352, 192, "f16", (16, 64)), (64, 8208, 832, "bf16", (64, 48)),
    (96, 28672, 320, "bf16", (128, 128)), (88, 14336, 2048, "bf16", (96, 64)), (160, 1040, 8192, "f16", (16, 48)),
    (504, 4096, 1984, "bf16", (64, 128)), (120, 4096, 4096, "bf16", (32, 64)),
    (16, 1024, 8192, "fp8_e4m3", (16, 16)), (80, 14336, 1152, "fp8_e4m3", (96, 64)), (72, 1040, 128, "fp8_e4m3", (16, 32)),
    (8, 1024, 512, "mxfp4", (16, 16)), (40, 4096, 4096, "mxfp4", (32, 32)), (80, 14336, 1024, "mxfp4", (96, 64)),
    (136, 8192, 2560, "mxfp4", (96, 64)), (200, 1088, 4608, "mxfp4", (32, 64)), (488, 4096, 2048, "mxfp4", (64, 128)),
    # tiles: one round and two, edge tiles, fewer K-steps than stages, one K-step
    (136, 14352, 64, "bf16", (128, 128)), (128, 28672, 256, "f16", (128, 128)), (328, 14336, 1024, "bf16", (192, 128)),
    (640, 14320, 192, "bf16", (192, 128)), (504, 14336, 576, "f16", (256, 128)), (4096, 4112, 128, "bf16", (192, 128)),
    (200, 8208, 128, "fp8_e4m3", (128, 128)), (328, 14336, 640, "fp8_e4m3", (192, 128)),
    (1280, 4096, 1152, "fp8_e4m3", (192, 128)), (968, 8176, 256, "fp8_e4m3", (256, 128)),
    # 256 x 256 tiles: one round, two of long rows, three; edge tiles
    (1912, 14336, 2048, "bf16", (256, 256)),
    (1000, 11008, 192, "bf16", (256, 256)), (4096, 11024, 64, "f16", (256, 256)), (2040, 8176, 704, "bf16", (256, 256)),
    # none of them: the own kernel
    (320, 14336, 1024, "mxfp4", (128, 256)), (4096, 8192, 256, "fp8_e4m3", (128, 256)), (640, 11008, 128, "bf16", (128, 256)),
    (1912, 14336, 1984, "bf16", (128, 256)),
])
@pytest.mark.parametrize("dtype_c", ["f32", "bf16"])
def test_pre_shuffled_weights_through_lds(gpu, M, N, K, dtype_ab, tile, dtype_c):
    a, b, extra = operands(M, N, K, dtype_ab, seed=M + K, b_std=0.05)
    rng = np.random.default_rng(M)
    how = dict(operand_path="direct_b_k8", bias=rng.standard_normal(N).astype(np.float32), ldc=N + 8)
    dev = dict(extra)
    if dtype_ab == "mxfp4":      # spread the block scales: a wrong byte must not go unnoticed
        for key in extra:
            extra[key] = (extra[key].astype(np.int32) + rng.integers(-3, 4, extra[key].shape)).astype(np.uint8)
        dev = dict(mx_a=shuffle_scales_e8m0_lanes128(extra["mx_a"]), mx_b=shuffle_scales_e8m0_lanes(extra["mx_b"]))
        how["mx_a_layout"] = "lanes128"
    w = shuffle_weight_k8(np.ascontiguousarray(b).view(np.uint16)) if dtype_ab in ("bf16", "f16") else shuffle_weight_bytes(b)
    info = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, has_bias=True, operand_path="direct_b_k8",
                              mx_a_layout=how.get("mx_a_layout", "rows")).info
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (info.name, info.wg_tile_m, info.wg_tile_n)
    out, name = run_gemm(a, w, M, N, K, dtype_ab, dtype_c, **how, **dev)
    again, _ = run_gemm(a, w, M, N, K, dtype_ab, dtype_c, **how, **dev)
    assert np.array_equal(out.view(np.uint8), again.view(np.uint8))
    pinned, _ = run_gemm(a, w, M, N, K, dtype_ab, dtype_c, variant=info.variant, **how, **dev)
    assert np.array_equal(out.view(np.uint8), pinned.view(np.uint8))
    pad = out[:, N:]
    assert np.isnan(pad).all() if dtype_c == "f32" else (pad == 0x7FC1).all()
    if dtype_ab == "mxfp4":
        want = G.gemm_mxfp4(a, extra["mx_a"], b, extra["mx_b"], out_dtype=_DT[dtype_c], bias=how["bias"])
    else:
        want = G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=how["bias"], **extra)
    bar = (1e-4 if dtype_ab == "fp8_e4m3" else 1e-5) if dtype_c == "f32" else REL_L2_BAR
    check(out, want, dtype_c, N, bar=bar)
    named, _ = run_gemm(a, w, M, N, K, dtype_ab, dtype_c, variant=_variant_id(name), **how, **dev)
    check(named, want, dtype_c, N, bar=bar)
    if dtype_ab == "fp8_e4m3" and tile[1] == 128 and tile[0] >= 128:  # the same products in the same order
        assert np.array_equal(out.view(np.uint8), named.view(np.uint8))
