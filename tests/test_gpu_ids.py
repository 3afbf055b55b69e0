"""Variant ids and what runs under them: astergemm_variant_info describes what a plan of its id launches."""
import ctypes

import pytest

from aster_amd import _capi, gemm as AG

pytestmark = pytest.mark.gpu

# one problem per kind of launcher with more than one kernel or K order: decode (resident activations, K ranges),
# few tokens, the nine-slot ring, 192 x 128, pairs of 128 x 128, both split kernels, eight waves, small products
PROBLEMS = [(64, 14336, 4096, "bf16"), (64, 4096, 14336, "bf16"), (40, 300, 1984, "f16"), (128, 4096, 4096, "bf16"),
            (80, 14336, 4096, "f16"), (256, 14336, 4096, "bf16"), (333, 14336, 4096, "bf16"),
            (2048, 4096, 4096, "f16"), (333, 4096, 14336, "bf16"), (128, 1024, 8192, "bf16"),
            (16, 4096, 14336, "fp8_e4m3"), (500, 7168, 2048, "fp8_e4m3"), (9, 4096, 11008, "fp8_e4m3"),
            (100, 300, 4096, "fp8_e4m3"), (16, 4096, 14336, "mxfp4"), (128, 4096, 4096, "mxfp4"),
            (300, 300, 2048, "bf16")]


def facts(info):
    return {f: getattr(info, f) for f, _ in info._fields_}


@pytest.mark.parametrize("M,N,K,dtype", PROBLEMS)
def test_every_id_is_described_as_a_plan_of_it_is(gpu, M, N, K, dtype):
    lib, info, seen = _capi.load(), _capi.KernelInfo(), 0
    auto = AG.GemmPlan.create(M, N, K, dtype, "f32")
    for i in range(lib.astergemm_variant_count()):
        _capi.check(lib.astergemm_variant_info(i, ctypes.byref(auto.config), ctypes.byref(info)))
        try:
            named = AG.GemmPlan.create(M, N, K, dtype, "f32", variant=i + 1)
        except _capi.AsterGemmError:
            continue
        seen += 1
        assert facts(info) == facts(named.info)
    assert seen > 0
