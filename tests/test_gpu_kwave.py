"""The kernels that split K over the waves of a workgroup, at the edges of their tiles, panels and K
loops: against the CPU oracle, with the bars of test_gpu_parity."""
import numpy as np
import pytest

from aster_amd import _capi, gemm as AG
from oracle import formats as F, gemm as G
from test_gpu_ids import PROBLEMS, device_operands
from test_gpu_parity import _DT, REL_L2_BAR, check, operands, run_gemm

pytestmark = pytest.mark.gpu


# waves over a tile's rows and columns: the others of a workgroup share K
_TILE_WAVES = {(16, 16): 1, (16, 32): 1, (16, 48): 1, (16, 64): 1, (32, 16): 2, (32, 32): 2, (32, 64): 2, (32, 128): 4,
               (64, 32): 2, (64, 48): 2, (64, 64): 4, (64, 128): 4, (96, 64): 4, (128, 64): 4, (128, 128): 8}


def ring_bytes(info, dtype_ab):
    """LDS of the kernel that splits K over waves: the ring of every wave group.  The kernels it stands in for have
    other sizes (resident activations 128 KiB, 128 x 128 tiles 80 or 144 KiB in rings of whole tiles)."""
    tile = (info.wg_tile_m, info.wg_tile_n)
    scales = (sum(tile) + 31) // 32 * 256 if dtype_ab == "mxfp4" else 0
    return info.pipeline_stages * (info.block_x // 64 // _TILE_WAVES[tile]) * (sum(tile) * 128 + scales)


@pytest.mark.parametrize("M,N,K,dtype_ab,tile", [
    # decoding: one panel per CU, panels of 8 ... 128 rows, short last panels, two tile rows, K ranges
    (1, 4096, 4096, "bf16", (16, 16)), (16, 520, 14336, "f16", (16, 16)), (7, 4104, 11008, "bf16", (16, 32)),
    (16, 11009, 4096, "bf16", (16, 48)), (15, 14336, 2048, "f16", (16, 64)), (17, 4096, 2304, "bf16", (32, 16)),
    (31, 7000, 4096, "f16", (32, 32)), (24, 14337, 2048, "bf16", (32, 64)), (32, 28672, 2560, "bf16", (32, 128)),
    (48, 1000, 8192, "f16", (16, 16)), (33, 4096, 4096, "bf16", (32, 32)), (64, 8191, 4096, "bf16", (64, 32)),
    (50, 11008, 4096, "f16", (64, 48)), (64, 14336, 4352, "bf16", (64, 64)), (63, 20000, 2048, "bf16", (64, 128)),
    (64, 4096, 14336, "bf16", (64, 64)), (29, 4100, 11008, "f16", (32, 64)), (33, 2700, 16384, "bf16", (64, 64)),
    (16, 14336, 4096, "fp8_e4m3", (16, 64)), (3, 1000, 12288, "fp8_e4m3", (16, 16)),
    (50, 4100, 4608, "fp8_e4m3", (64, 32)), (64, 8192, 28672, "fp8_e4m3", (64, 64)),
    (16, 4096, 14336, "mxfp4", (16, 16)), (9, 7000, 4608, "mxfp4", (16, 32)), (33, 8200, 4096, "mxfp4", (64, 48)),
    (64, 4100, 8192, "mxfp4", (64, 32)),
    # rows that the kernels with resident activations do not take
    (9, 4096, 11008, "fp8_e4m3", (16, 16)), (1, 1024, 4112, "fp8_e4m3", (16, 16)),
    (64, 2056, 4208, "fp8_e4m3", (32, 32)), (5, 1030, 4352, "mxfp4", (16, 16)), (64, 4096, 11008, "mxfp4", (32, 32)),
    (40, 300, 1984, "bf16", (16, 16)), (64, 1000, 992, "f16", (16, 16)), (1, 17, 32, "bf16", (16, 16)),
    # prompts of few tokens: panels of exact rows under every tile height, ragged M, short last panels
    (65, 4096, 4096, "bf16", (32, 64)), (128, 14336, 4096, "f16", (128, 64)), (96, 11008, 4096, "bf16", (96, 64)),
    (100, 28672, 2304, "bf16", (128, 128)), (330, 4096, 4096, "f16", (96, 64)), (511, 4096, 4096, "bf16", (64, 128)),
    (400, 4096, 4096, "bf16", (64, 128)),
    (128, 1024, 8192, "f16", (32, 16)), (72, 8, 4096, "bf16", (32, 16)), (128, 8192, 8192, "fp8_e4m3", (64, 64)),
    (250, 1032, 8192, "fp8_e4m3", (32, 64)), (128, 4096, 4096, "mxfp4", (32, 64)),
    (256, 8192, 8192, "mxfp4", (64, 128)), (80, 14336, 4096, "mxfp4", (96, 64)), (304, 1000, 8192, "mxfp4", (32, 64)),
    # small products: the smallest tile in one round, K tails of 1 and 7 granules, fewer steps than stages
    (100, 100, 520, "bf16", (16, 16)), (300, 300, 2048, "f16", (32, 32)), (65, 130, 1080, "bf16", (16, 16)),
    (600, 599, 1544, "bf16", (32, 64)), (780, 599, 1032, "bf16", (32, 64)), (1200, 33, 2040, "f16", (16, 16)),
    (100, 4095, 4096, "fp8_e4m3", (32, 64)), (70, 1000, 2064, "fp8_e4m3", (32, 32)),
])
@pytest.mark.parametrize("dtype_c", ["f32", "bf16"])
def test_k_over_waves(gpu, M, N, K, dtype_ab, dtype_c, tile):
    a, b, extra = operands(M, N, K, dtype_ab, seed=M + K, b_std=0.05)
    if dtype_ab == "mxfp4":      # spread the block scales: a wrong byte must not go unnoticed
        rng = np.random.default_rng(M)
        for key in extra:
            extra[key] = (extra[key].astype(np.int32) + rng.integers(-3, 4, extra[key].shape)).astype(np.uint8)
    bias = np.random.default_rng(N).standard_normal(N).astype(np.float32)
    info = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, has_bias=True).info
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (info.name, info.wg_tile_m, info.wg_tile_n)
    assert info.lds_bytes == ring_bytes(info, dtype_ab)
    out, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 3, **extra)
    want = G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=bias, **extra)
    f32_bar = 1e-4 if dtype_ab == "fp8_e4m3" else 1e-5
    if dtype_c == "f32" or M * N >= 4096:
        check(out, want, dtype_c, N, bar=f32_bar if dtype_c == "f32" else REL_L2_BAR)
    else:                        # few outputs: two units of the bf16 output each, and the sums' own bar
        got, ref = G.output_to_f32(out[:, :N], _DT[dtype_c]), G.output_to_f32(want, _DT[dtype_c])
        assert np.all(np.abs(got - ref) <= 2.0 ** -6 * np.abs(ref) + f32_bar * np.abs(ref).max())
    pad = out[:, N:]
    assert np.isnan(pad).all() if dtype_c == "f32" else (pad == 0x7FC1).all()
    again, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 3, **extra)
    assert np.array_equal(out.view(np.uint8), again.view(np.uint8))


@pytest.mark.parametrize("M,N,K,dtype_ab,tile", [
    (560, 1024, 8192, "fp8_e4m3", (64, 48)), (901, 1024, 8192, "fp8_e4m3", (64, 64)),
    (1194, 1024, 8192, "fp8_e4m3", (96, 64)), (513, 2048, 8192, "fp8_e4m3", (96, 64)),
    (1000, 1024, 4096, "mxfp4", (64, 64)), (1401, 1016, 8192, "mxfp4", (96, 64)),
    (2047, 1024, 8192, "mxfp4", (64, 128)), (3000, 512, 8192, "mxfp4", (96, 64)), (600, 2048, 4096, "mxfp4", (64, 128)),
])
def test_k_over_waves_past_512_rows(gpu, M, N, K, dtype_ab, tile):
    test_k_over_waves(gpu, M, N, K, dtype_ab, "bf16", tile)


@pytest.mark.parametrize("M,N,K,dtype_ab", [
    (3000, 64, 14336, "mxfp4"), (4096, 64, 8192, "mxfp4"), (2047, 256, 14336, "mxfp4"), (2560, 16, 8192, "mxfp4"),
    (4096, 64, 4096, "mxfp4"), (1400, 64, 14336, "mxfp4"), (631, 1904, 9216, "fp8_e4m3"), (762, 1256, 9216, "fp8_e4m3"),
])
def test_past_512_rows_where_splitting_k_over_waves_is_behind(gpu, M, N, K, dtype_ab):
    """Few columns, whose planes weigh nothing, and rows too long for one round: 128 x 128 tiles."""
    info = AG.GemmPlan.create(M, N, K, dtype_ab, "bf16").info
    assert (info.wg_tile_m, info.wg_tile_n) == (128, 128), (info.name, info.wg_tile_m, info.wg_tile_n)


@pytest.mark.parametrize("M,N,K", [(16, 4096, 14336), (50, 1000, 2304), (100, 200, 1032)])
def test_non_finite_rows_stay_in_their_row(gpu, M, N, K):
    """The rows past M and N repeat the last one; a NaN there, and an infinity, reach their own row only."""
    a, b, _ = operands(M, N, K, "bf16", seed=5, b_std=0.05)
    a = np.array(a, copy=True)
    a[M - 1, K - 1], a[0, 0] = 0x7FC0, 0x7F80       # NaN, +inf
    out, _ = run_gemm(a, b, M, N, K, "bf16", "f32")
    assert np.isnan(out[M - 1]).all() and not np.isfinite(out[0]).any()
    assert np.isfinite(out[1:M - 1]).all()


@pytest.mark.parametrize("first,then", [((16, 14336, 4096), (48, 4096, 4096)), ((16, 60000, 4096), (8, 4096, 4096)),
                                        ((8, 4096, 4096), (16, 60000, 4096)), ((1000, 1000, 2048), (100, 100, 2048))])
def test_a_captured_config_finds_its_kernel_ready(gpu, first, then):
    """One eager call of a decode (small) problem of the same types readies the kernels of all of them, those
    with resident activations included; several replays with eager work between them have the eager bits."""
    import torch
    torch.manual_seed(3)
    stream = torch.cuda.Stream()
    plans = [AG.GemmPlan.create(*s, "f16", "f16") for s in (first, then)]
    sets = [[(torch.randn(r, s[2], device="cuda") * 0.1).half() for r in s[:2]]
            + [torch.zeros(s[0], s[1], device="cuda", dtype=torch.float16)] for s in (first, then)]
    torch.cuda.synchronize()
    call = lambda i, c=None: plans[i].run(sets[i][0].data_ptr(), sets[i][1].data_ptr(),
                                          (sets[i][2] if c is None else c).data_ptr(), stream=stream.cuda_stream)
    print(first, then, flush=True)
    call(0)
    stream.synchronize()
    graph, got = torch.cuda.CUDAGraph(), torch.zeros_like(sets[1][2])
    with torch.cuda.graph(graph, stream=stream):
        call(1, got)
    call(1)
    torch.cuda.synchronize()
    for _ in range(3):
        got.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, sets[1][2])
        call(0)


def test_a_named_tile_keeps_the_kernels_it_had():
    for (M, N, K), wg in (((300, 300, 2048), (64, 64)), ((16, 4096, 4096), (16, 16))):
        info = AG.GemmPlan.create(M, N, K, "bf16", "bf16", wg_tile=wg).info
        assert (info.wg_tile_m, info.wg_tile_n) == wg and b"kwave" not in info.name
    assert info.lds_bytes == 128 * 1024 != ring_bytes(info, "bf16")      # resident activations


@pytest.mark.parametrize("dtype_c", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,N,K,dtype_ab", PROBLEMS + [(100, 100, 520, "bf16"), (70, 1000, 2064, "fp8_e4m3"),
                                                       (1000, 4096, 2080, "f16"), (1000, 7048, 1032, "bf16")])
def test_row_pitches_above_k(gpu, M, N, K, dtype_ab, dtype_c):
    """A and B with pitches of their own, the gaps full of NaN codes (MXFP4: -6): the bits of packed
    operands, and nothing written past column N."""
    import torch
    (pa, pb), kw, keep = device_operands(M, N, K, dtype_ab)
    per = {"mxfp4": 2, "fp8_e4m3": 1}.get(dtype_ab, 0.5)          # elements of a byte
    row = int(K / per)
    wide = [torch.full((r, row + pad), 0xFF, dtype=torch.uint8, device="cuda") for r, pad in ((M, 16), (N, 144))]
    for w, t in zip(wide, keep):
        w[:, :row] = t.view(torch.uint8)
    ldc, out = N + (3 if M <= 64 else 8), {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dtype_c]
    lda, ldb = K + int(16 * per), K + int(144 * per)
    packed = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, ldc=ldc)
    padded = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, lda=lda, ldb=ldb, ldc=ldc)
    want, got = (torch.full((M, ldc), float("nan"), dtype=out, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    print(f"{padded.info.name.decode()} M={M} N={N} K={K}", flush=True)
    packed.run(pa, pb, want.data_ptr(), **kw)
    padded.run(wide[0].data_ptr(), wide[1].data_ptr(), got.data_ptr(), **kw)
    torch.cuda.synchronize()
    assert padded.info.variant == packed.info.variant
    assert torch.equal(got[:, :N], want[:, :N]) and bool(torch.isfinite(want[:, :N]).all())
    assert bool(torch.isnan(got[:, N:]).all())


@pytest.mark.parametrize("M,N,K,dtype_ab,tile", [
    # one round of small tiles whatever the row: one K-step and less, fewer than wave groups, exact rounds of them
    (256, 256, 256, "f16", (16, 16)), (17, 26, 40, "bf16", (16, 16)), (65, 16, 8, "f16", (16, 16)),
    (512, 500, 64, "bf16", (32, 32)), (300, 300, 512, "f16", (32, 32)), (1024, 250, 320, "bf16", (32, 32)),
    # 32 x 64 tiles: from three K-steps on, from nine with whole panels on an XCD only
    (500, 1000, 136, "bf16", (32, 64)), (500, 1000, 128, "bf16", (64, 64)), (2000, 200, 512, "f16", (32, 64)),
    (256, 2000, 800, "bf16", (32, 64)), (2000, 200, 520, "bf16", (64, 64)),
])
@pytest.mark.parametrize("dtype_c", ["f32", "bf16"])
def test_small_products_of_short_rows(gpu, M, N, K, dtype_ab, dtype_c, tile):
    a, b, _ = operands(M, N, K, dtype_ab, seed=M + K, b_std=0.05)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    info = AG.GemmPlan.create(M, N, K, dtype_ab, dtype_c, has_bias=True).info
    assert (info.wg_tile_m, info.wg_tile_n) == tile, (info.name, info.wg_tile_m, info.wg_tile_n)
    out, _ = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 3)
    check(out, G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=bias), dtype_c, N,
          bar=1e-5 if dtype_c == "f32" else REL_L2_BAR)
    pad = out[:, N:]
    assert np.isnan(pad).all() if dtype_c == "f32" else (pad == 0x7FC1).all()


@pytest.mark.parametrize("wg_tile", [(0, 0), (64, 64), (128, 128)])
@pytest.mark.parametrize("scale_mode", ["none", "tensor"])
def test_row_pitches_past_32_bits(gpu, wg_tile, scale_mode):
    """Everything a packed launch argument holds at its widest: rows of C 2^32 + 24 elements apart, padded rows of A
    and B, tensor scales on 16-bit operands, bias."""
    import torch
    M, N, K, lda, ldb, ldc = 2, 40, 72, 4096, 88, 2 ** 32 + 24
    a, b, _ = operands(M, N, K, "bf16", seed=9, b_std=0.05)
    dev = torch.device("cuda:0")
    ta, tb = torch.zeros(M, lda, dtype=torch.int16, device=dev), torch.zeros(N, ldb, dtype=torch.int16, device=dev)
    ta[:, :K] = torch.from_numpy(a.view(np.int16)).to(dev)
    tb[:, :K] = torch.from_numpy(b.view(np.int16)).to(dev)
    bias = torch.arange(N, dtype=torch.float32, device=dev) * 0.25
    scales = torch.tensor([0.5, 3.0], device=dev)
    out = torch.empty(ldc + 64, dtype=torch.int16, device=dev)
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16", scale_mode=scale_mode, has_bias=True, lda=lda, ldb=ldb, ldc=ldc,
                              wg_tile=wg_tile, family=_capi.KERNEL_TILE)
    kw = dict(scale_a=scales.data_ptr(), scale_b=scales.data_ptr() + 4) if scale_mode == "tensor" else {}
    torch.cuda.synchronize()
    print("launch", plan.info.name.decode(), flush=True)
    plan.run(ta.data_ptr(), tb.data_ptr(), out.data_ptr(), bias=bias.data_ptr(), **kw)
    torch.cuda.synchronize()
    got = np.stack([out[m * ldc:m * ldc + N].cpu().numpy().view(np.uint16) for m in range(M)])
    s = dict(scale_a=0.5, scale_b=3.0) if kw else {}
    want = F.bf16_bits_to_f32(a) @ F.bf16_bits_to_f32(b).T * (1.5 if s else 1.0) + bias.cpu().numpy()
    assert G.rel_l2(F.bf16_bits_to_f32(got), want) <= 4e-3   # one bf16 rounding: 2^-9 of each value at most


@pytest.mark.parametrize("M,N,K,dtype_ab", [
    (1000, 1000, 256, "bf16"), (1000, 1030, 256, "f16"),      # 256 and 272 tiles of four K-steps
    (1024, 1000, 264, "bf16"), (1001, 1000, 200, "f16"),      # five, and four with a tail
    (2040, 1000, 40, "bf16"), (2060, 1000, 40, "f16"),        # 512 and 528 tiles of one
    (520, 1000, 72, "bf16"),
])
@pytest.mark.parametrize("dtype_c", ["f32", "bf16"])
def test_either_form_of_the_general_kernels_arguments(gpu, M, N, K, dtype_ab, dtype_c):
    """64 x 64 tiles on both sides of the line up to which 16-bit operands have their arguments packed."""
    a, b, _ = operands(M, N, K, dtype_ab, seed=M + K, b_std=0.05)
    bias = np.random.default_rng(K).standard_normal(N).astype(np.float32)
    out, info = run_gemm(a, b, M, N, K, dtype_ab, dtype_c, bias=bias, ldc=N + 3, wg_tile=(64, 64))
    check(out, G.gemm(a, b, _DT[dtype_ab], _DT[dtype_c], bias=bias), dtype_c, N,
          bar=1e-5 if dtype_c == "f32" else REL_L2_BAR)
    pad = out[:, N:]
    assert np.isnan(pad).all() if dtype_c == "f32" else (pad == 0x7FC1).all()
