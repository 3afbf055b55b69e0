"""Every id describes every config: what the launchers' rules say with a chip's CU count in hand, on sizes that no
kernel takes as well.  A stand-in for the two device queries gives the count, so nothing here needs a GPU; in a process
of its own, which an arithmetic fault would end."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

QUERIES = """
#include <hip/hip_runtime.h>
#include <cstring>
extern "C" hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
extern "C" hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
"""

WALK = """
import ctypes
from aster_amd import _capi
lib, info, c, n = _capi.load(), _capi.KernelInfo(), _capi.Config(), 0
c.M, c.N, c.K = 80, 4096, 4096                 # the stand-in is heard: K over waves on 256 CUs
c.dtype_ab = c.dtype_c = _capi.BF16
c.operand_path = _capi.OPERAND_DIRECT_B_K8
assert lib.astergemm_select(ctypes.byref(c), ctypes.byref(info)) == 0 and info.wg_tile_m < 128, info.wg_tile_m
for M, N, K in ((0, 0, 64), (0, 4096, 4096), (4096, 0, 4096), (-8, 16, 64), (16, -16, 64), (1, 1, 1), (8, 16, 0),
                (0, 1 << 31, 512), (1 << 40, 16, 512)):
    c = _capi.Config()
    c.M, c.N, c.K = M, N, K
    for i in range(lib.astergemm_variant_count()):
        print(i, M, N, K, flush=True)
        assert lib.astergemm_variant_info(i, ctypes.byref(c), ctypes.byref(info)) == 0
        n += 1
print("described", n)
"""


@pytest.fixture(scope="module")
def queries(tmp_path_factory):
    where = tmp_path_factory.mktemp("queries")
    (where / "queries.cpp").write_text(QUERIES)
    subprocess.run(["g++", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(where / "queries.cpp"), "-o", str(where / "queries.so")], check=True)
    preload = [str(where / "queries.so")] + os.environ.get("LD_PRELOAD", "").split()   # before what is preloaded already
    return dict(os.environ, LD_PRELOAD=" ".join(preload))


def test_every_id_describes_sizes_that_no_kernel_takes(queries):
    p = subprocess.run([sys.executable, "-c", WALK], cwd=ROOT, env=queries,
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and "described" in p.stdout, (p.returncode, p.stdout[-200:], p.stderr[-2000:])


TILES = """
import ctypes
from aster_amd import _capi
lib, info = _capi.load(), _capi.KernelInfo()
for M, N, K, dtype, tile in %r:
    c = _capi.Config()
    c.M, c.N, c.K = M, N, K
    c.dtype_ab, c.dtype_c, c.scale_mode = dtype, _capi.BF16, int(dtype == _capi.FP8_E4M3)
    c.operand_path = _capi.OPERAND_DIRECT_B_K8
    assert lib.astergemm_select(ctypes.byref(c), ctypes.byref(info)) == 0
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (M, N, K, dtype, info.wg_tile_m, info.wg_tile_n)
print("selected")
"""


OWN, BF16, FP8 = (128, 256), 1, 2


@pytest.mark.parametrize("cases", [
    [(128, 73728, 1024, BF16, (128, 128)), (128, 73728, 960, BF16, OWN),
     (1416, 11008, 4096, BF16, (192, 128)), (1400, 11008, 4096, BF16, OWN),     # 516 and 473 tiles of the own kernel
     (720, 28672, 4096, BF16, (256, 128)), (1664, 13120, 3584, BF16, OWN), (2552, 8192, 28672, BF16, OWN),
     (1264, 14208, 7680, BF16, OWN), (1520, 12928, 14336, BF16, (256, 128)),     # 555 and 606 tiles
     (1288, 14336, 4096, BF16, OWN), (872, 11008, 4096, BF16, (192, 128))],     # four rounds and two of 192 x 128
    [(320, 22016, 2048, FP8, (192, 128)), (320, 22016, 1920, FP8, OWN), (344, 14336, 128, FP8, (192, 128)),
     (640, 14320, 192, BF16, (192, 128)), (640, 14320, 128, BF16, (256, 256)),
     (1568, 9344, 8192, BF16, (256, 128)), (1568, 9344, 8128, BF16, OWN), (3128, 4992, 14336, BF16, OWN)],
    [(1912, 14336, 2048, BF16, (256, 256)), (880, 27648, 3072, BF16, OWN),      # 448 and 432 places of 512
     (5216, 14848, 1536, BF16, (256, 256)), (5216, 14848, 1472, BF16, OWN), (5496, 14912, 1024, BF16, OWN)],
    [(768, 10240, 8192, FP8, (256, 128)), (896, 8192, 8192, FP8, OWN), (968, 8176, 256, FP8, (256, 128)),
     (640, 8192, 8192, FP8, (192, 128))],
], ids=["third", "second", "squares", "first"])
def test_rounds_of_tiles_on_pre_shuffled_weights(queries, cases):
    p = subprocess.run([sys.executable, "-c", TILES % cases], cwd=ROOT, env=queries,
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and "selected" in p.stdout, (p.returncode, p.stderr[-2000:])
