"""Variant ids and what runs under them: a plan of the id that AUTO reports runs AUTO's kernel with AUTO's bits,
astergemm_variant_info describes what a plan of its id launches, and astergemm_tune times that."""
import ctypes
import re

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


def device_operands(M, N, K, dtype):
    """(positional pointers without dC, keyword pointers, the tensors that own them)"""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    if dtype == "mxfp4":
        draw = lambda r: torch.randint(0, 256, (r, K // 2), generator=g, device="cuda", dtype=torch.uint8)
        mx = [torch.randint(118, 123, (r, K // 32), generator=g, device="cuda", dtype=torch.uint8) for r in (M, N)]
        keep = [draw(M), draw(N), *mx]
        kw = dict(mx_a=mx[0].data_ptr(), mx_b=mx[1].data_ptr())
    else:
        to = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8_e4m3": torch.float8_e4m3fn}[dtype]
        keep = [(torch.randn(r, K, generator=g, device="cuda") * s).to(to) for r, s in ((M, 1.0), (N, 0.05))]
        kw = {}
        if dtype == "fp8_e4m3":
            keep.append(torch.tensor([0.5, 0.25], device="cuda"))
            kw = dict(scale_a=keep[2].data_ptr(), scale_b=keep[2].data_ptr() + 4)
    return (keep[0].data_ptr(), keep[1].data_ptr()), kw, keep


def bits(plan, ptrs, kw, M, N):
    import torch
    c = torch.full((M, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    print(f"{plan.info.name.decode()} variant={plan.config.variant} M={M} N={N} K={plan.config.K}", flush=True)
    plan.run(*ptrs, c.data_ptr(), **kw)
    torch.cuda.synchronize()
    return c.view(torch.int32)


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


@pytest.mark.parametrize("M,N,K,dtype", PROBLEMS)
def test_a_plan_of_the_selected_id_is_the_selected_kernel(gpu, M, N, K, dtype):
    """The same launch and the same bits, whatever AUTO runs in place of the kernel its variant is named for; the
    name alone says that it is AUTO's form."""
    import torch
    auto = AG.GemmPlan.create(M, N, K, dtype, "f32")
    named = AG.GemmPlan.create(M, N, K, dtype, "f32", variant=auto.info.variant)
    a, n = facts(auto.info), facts(named.info)
    stem, out = a.pop("name").decode().rsplit("_", 1)
    assert n.pop("name").decode() in (f"{stem}_{out}", f"{stem}_auto_{out}") and a == n
    assert auto.workspace_bytes() == named.workspace_bytes()
    ptrs, kw, keep = device_operands(M, N, K, dtype)
    want, got = bits(auto, ptrs, kw, M, N), bits(named, ptrs, kw, M, N)
    assert bool((got == want).all()) and bool(want.view(torch.float32).isfinite().all())


@pytest.mark.parametrize("M,N,K,dtype", PROBLEMS)
@pytest.mark.parametrize("family", [_capi.KERNEL_AUTO, _capi.KERNEL_TILE])
def test_tune_launches_what_the_plan_of_an_id_runs(gpu, M, N, K, dtype, family):
    """dC holds the last candidate's product: the bits of the plan of its id."""
    import torch
    count = _capi.load().astergemm_variant_count()
    auto = AG.GemmPlan.create(M, N, K, dtype, "f32", family=family)
    last = None
    for v in range(count, 0, -1):
        try:
            last = AG.GemmPlan.create(M, N, K, dtype, "f32", variant=v)
        except _capi.AsterGemmError:
            continue
        rows = re.search(r"_m(\d+)", last.info.name.decode())   # activation rows of a decode kernel
        if (family == _capi.KERNEL_AUTO or last.info.family == family) and (rows is None or int(rows[1]) >= M):
            break
    ptrs, kw, keep = device_operands(M, N, K, dtype)
    c = torch.full((M, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    print(f"tune {dtype} M={M} N={N} K={K} family={family}", flush=True)
    tuned = auto.tune(*ptrs, c.data_ptr(), iters=2, **kw)
    torch.cuda.synchronize()
    assert bool((c.view(torch.int32) == bits(last, ptrs, kw, M, N)).all()), last.info.name
    assert tuned.config.variant == tuned.info.variant > 0
