"""Two 128 x 128 tiles of a CU run as one of 256 x 128, and K loops that start at different steps on different
XCDs: against the CPU oracle; the same bits on a second run and from a plan of the selected id; the kernel by its
name has the bits of the 128 x 128 one."""
import numpy as np
import pytest

from aster_amd import gemm as AG
from oracle import gemm as G
from test_gpu_parity import _DT, REL_L2_BAR, _variant_id, check, operands, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype_ab,dtype_c,tile", [
    (512, 14336, 1024, "bf16", "bf16", (256, 128)),      # 7/8 of the chip, the shortest rows
    (512, 16384, 1160, "f16", "f32", (256, 128)),        # all of it, a K tail
    (1152, 6528, 1088, "bf16", "f16", (256, 128)),       # an odd number of 128-row tiles
    (2048, 4096, 1024, "f16", "f32", (128, 128)),        # fp32 outputs of rows under 18 K-steps
    (1024, 7040, 1024, "bf16", "bf16", (256, 128)),      # one tile column below 7/8: the 256 x 128 variant itself
    (1000, 7048, 1032, "bf16", "bf16", (256, 128)),      # 16 K-steps and a tail, started two apart
    (1000, 4096, 2080, "f16", "bf16", (128, 128)),       # the nine-slot ring, 32 K-steps and a tail
    (500, 7168, 2048, "fp8_e4m3", "bf16", (128, 128)),   # fp8, 16 K-steps
    (300, 4096, 14336, "fp8_e4m3", "f32", (256, 128)),   # split K: 28 K-steps a range, starts 3 and 4 apart
])
def test_pairs_of_tiles(gpu, M, N, K, dtype_ab, dtype_c, tile):
    a, b, extra = operands(M, N, K, dtype_ab, seed=K, b_std=0.05)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    info = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, has_bias=True).info
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (info.name, info.wg_tile_m, info.wg_tile_n)
    out, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8, **extra)
    again, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8, **extra)
    assert np.array_equal(out.view(np.uint8), again.view(np.uint8))
    pinned, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8, variant=info.variant, **extra)
    assert np.array_equal(out.view(np.uint8), pinned.view(np.uint8))
    want = G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=bias, **extra)
    check(out, want, dtype_c, N, bar=(1e-4 if dtype_ab == "fp8_e4m3" else 1e-5) if dtype_c == "f32" else REL_L2_BAR)
    if dtype_ab != "fp8_e4m3":  # by name and by tile size: no pairs, and the K loops start at step 0
        named, square = (run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8, **how)[0]
                         for how in (dict(variant=_variant_id(info.name.decode())), dict(wg_tile=(128, 128))))
        assert np.array_equal(named.view(np.uint8), square.view(np.uint8))
        check(named, want, dtype_c, N, bar=1e-5 if dtype_c == "f32" else REL_L2_BAR)
