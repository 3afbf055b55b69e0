"""Two 128 x 128 tiles of a CU run as one of 256 x 128: against the kernel that the plan names, bit for bit,
and the CPU oracle."""
import numpy as np
import pytest

from aster_amd import gemm as AG
from oracle import gemm as G
from test_gpu_parity import _DT, REL_L2_BAR, check, operands, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype_ab,dtype_c,tile", [
    (512, 14336, 1024, "bf16", "bf16", (256, 128)),      # 7/8 of the chip, the shortest rows
    (512, 16384, 1160, "f16", "f32", (256, 128)),        # all of it, a K tail
    (1152, 6528, 1088, "bf16", "f16", (256, 128)),       # an odd number of 128-row tiles
    (2048, 4096, 1024, "f16", "f32", (128, 128)),        # fp32 outputs of rows under 18 K-steps
    (1024, 7040, 1024, "bf16", "bf16", (256, 128)),      # one tile column below 7/8: the 256 x 128 variant itself
])
def test_pairs_of_tiles(gpu, M, N, K, dtype_ab, dtype_c, tile):
    a, b, _ = operands(M, N, K, dtype_ab, seed=K, b_std=0.05)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    info = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, has_bias=True).info
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (info.name, info.wg_tile_m, info.wg_tile_n)
    out, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8)
    named, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 8, variant=info.variant)
    assert np.array_equal(out.view(np.uint8), named.view(np.uint8))
    want = G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=bias)
    check(out, want, dtype_c, N, bar=1e-5 if dtype_c == "f32" else REL_L2_BAR)
