"""K ranges of the 128 x 128 split kernels on XCDs of their own: every number of ranges, tile counts that divide among a
range's XCDs and ones that do not, against the CPU oracle."""
import numpy as np
import pytest

from aster_amd import _capi, gemm as AG
from oracle import gemm as G
from test_gpu_parity import _DT, REL_L2_BAR, check, operands, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype_ab", [
    (640, 1024, 8192, "bf16"),      # 40 tiles, 4 ranges on two XCDs each
    (1152, 1024, 8192, "f16"),      # 72 tiles, two ranges of 64 steps as four
    (904, 904, 8192, "bf16"),       # 64 tiles, edge tiles in both directions
    (520, 640, 8192, "bf16"),       # 25 tiles, 8 ranges: one XCD each, 25 and 3 rest in the tile order
    (136, 904, 8192, "f16"),        # 16 tiles, 16 ranges: two on an XCD
    (392, 648, 10240, "bf16"),      # 24 tiles, 10 ranges: no power of two
    (264, 392, 14336, "bf16"),      # 12 tiles, 16 ranges
    (1000, 520, 12288, "bf16"),     # 40 tiles, 6 ranges
    (520, 904, 8192, "fp8_e4m3"),   # 40 tiles of bytes, 4 ranges
    (136, 648, 16384, "fp8_e4m3"),  # 12 tiles, 16 ranges
])
def test_ranges_on_their_xcds(gpu, M, N, K, dtype_ab):
    a, b, extra = operands(M, N, K, dtype_ab, seed=M, b_std=0.05)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    prefix = "splitk_" + ("fp8" if dtype_ab == "fp8_e4m3" else dtype_ab) + "_128x128_w2x2_f32"
    lib, cfg, info = _capi.load(), _capi.Config(), _capi.KernelInfo()
    cfg.M = cfg.N = cfg.K = 8192
    ids = [i + 1 for i in range(lib.astergemm_variant_count())
           if lib.astergemm_variant_info(i, cfg, info) == 0 and info.name.decode() == prefix]
    how = dict(bias=bias, ldc=N + 8, variant=ids[0], **extra)   # by its first id: the split kernel whatever AUTO takes
    out, _ = run_gemm(a, b, M, N, K, dtype_ab, "f32", **how)
    again, _ = run_gemm(a, b, M, N, K, dtype_ab, "f32", **how)
    assert np.array_equal(out.view(np.uint8), again.view(np.uint8))
    check(out, G.gemm(a, b, _DT[dtype_ab], _DT["f32"], bias=bias, **extra), "f32", N,
          bar=1e-4 if dtype_ab == "fp8_e4m3" else 1e-5)
