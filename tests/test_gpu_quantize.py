"""GPU parity of the operand quantisers: bytes out of the HIP kernels (through the C-ABI)
must equal the oracle's, bit for bit: e4m3 codes and the fp32 tensor scale; e2m1 nibbles and
e8m0 block scale bytes.  The e4m3 oracle is itself pinned against the converter vectors of
the reference's tests (tests/test_oracle_formats.py)."""
import numpy as np
import pytest

from aster_amd import _capi, gemm as AG, quantize as Q
from aster_amd.execution import GpuBuffer
from oracle import formats as F, gemm as G

pytestmark = pytest.mark.gpu


def _special_f32():
    codes = F.e4m3_decode(np.arange(256, dtype=np.uint8)).astype(np.float32)
    fin = np.unique(codes[np.isfinite(codes)])
    mids = ((fin[:-1].astype(np.float64) + fin[1:]) / 2).astype(np.float32)
    up, dn = np.nextafter(mids, np.float32(np.inf)), np.nextafter(mids, np.float32(-np.inf))
    return np.concatenate([fin, mids, up, dn]).astype(np.float32)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 1023, 4096, 65537, 1 << 20])
def test_fp8_tensor_quantiser_matches_oracle(n):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * rng.choice([1e-3, 0.05, 1.0, 40.0], n)).astype(np.float32)
    print(f"quantize_fp8_tensor n={n}", flush=True)
    q, s = Q.quantize_fp8_tensor(x)
    qo, so = F.quantize_fp8_tensor(x)
    assert np.float32(s).tobytes() == np.float32(so).tobytes()
    assert np.array_equal(q, qo)


def test_fp8_tensor_quantiser_rounding_cases():
    # absmax 448 -> scale exactly 1: every code, every midpoint between codes and both
    # neighbours of each midpoint go through the encoder unscaled
    sp = _special_f32()
    x = np.concatenate([sp, -sp, np.array([0.0, -0.0, 2.0 ** -10, 2.0 ** -11, 1.5 * 2.0 ** -10,
                                           1e-45, -1e-45, 1e-40], np.float32)])
    assert np.max(np.abs(x)) == 448.0
    print(f"quantize_fp8_tensor rounding cases n={x.size}", flush=True)
    q, s = Q.quantize_fp8_tensor(x)
    qo, so = F.quantize_fp8_tensor(x)
    assert s == 1.0 and so == 1.0
    assert np.array_equal(q, qo)
    # signed zeros and the tie at half the smallest subnormal
    assert q[x.size - 8] == 0x00 and q[x.size - 7] == 0x80 and q[x.size - 6] == 0x00


@pytest.mark.parametrize("case", ["zeros", "nan", "inf", "empty", "huge", "tiny"])
def test_fp8_tensor_quantiser_edge_tensors(case):
    rng = np.random.default_rng(5)
    x = rng.standard_normal(1000).astype(np.float32)
    if case == "zeros":
        x[:] = 0
        x[3] = -0.0
    elif case == "nan":
        x[17] = np.nan
    elif case == "inf":
        x[99] = -np.inf
    elif case == "empty":
        x = x[:0]
    elif case == "huge":
        x *= np.float32(1e37)
    elif case == "tiny":
        x *= np.float32(1e-41)
    print(f"quantize_fp8_tensor edge {case}", flush=True)
    q, s = Q.quantize_fp8_tensor(x)
    with np.errstate(all="ignore"):
        qo, so = F.quantize_fp8_tensor(x)
    assert np.float32(s).tobytes() == np.float32(so).tobytes()
    assert np.array_equal(q, qo)


def test_absmax_matches_numpy():
    rng = np.random.default_rng(7)
    for n in (0, 1, 7, 1000, 300001):
        x = rng.standard_normal(n).astype(np.float32)
        if n > 5:
            x[n // 2] = -77.25
        src, out = GpuBuffer(max(x.nbytes, 16)), GpuBuffer(4)
        src.copy_from_host(x)
        print(f"absmax n={n}", flush=True)
        Q.absmax_device(src.ptr_value, n, out.ptr_value)
        got = np.empty(1, np.float32)
        out.copy_to_host(got)
        assert got[0] == (np.max(np.abs(x)) if n else 0.0)


def _mx_input(rows, K, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    # every block its own magnitude, over the whole fp32 exponent range
    e = rng.integers(-140, 126, size=(rows, K // 32))
    x = (x.astype(np.float64) * np.ldexp(1.0, np.repeat(e, 32, axis=1))).astype(np.float32)
    return x


@pytest.mark.parametrize("rows,K", [(1, 32), (3, 64), (16, 4096), (257, 1024), (64, 14336)])
def test_mxfp4_quantiser_matches_oracle(rows, K):
    x = _mx_input(rows, K, rows * 7 + K)
    print(f"quantize_mxfp4 rows={rows} K={K}", flush=True)
    p, s = Q.quantize_mxfp4(x)
    po, so = F.quantize_mxfp4(x)
    assert np.array_equal(s, so)
    assert np.array_equal(p, po)


def test_mxfp4_quantiser_special_blocks():
    rng = np.random.default_rng(11)
    x = rng.standard_normal((8, 256)).astype(np.float32)
    x[0, 0:32] = 0.0                       # all-zero block -> scale byte 127, zero nibbles
    x[0, 5] = -0.0
    x[1, 32:64] = np.nan                   # NaN block -> 0xFF
    x[2, 64:96][3] = np.inf                # inf element -> 0xFF
    x[3, 0:32] *= np.float32(1e-44)        # fp32-subnormal block
    x[3, 32:64] = np.float32(2.0 ** -149)
    x[4, 0:32] *= np.float32(3e38)         # top of the fp32 range (may overflow to inf)
    x[4, 32:64] = np.float32(2.0 ** 127)
    # ties of the e2m1 grid with absmax 6 (scale 1): .25 .75 1.25 1.75 2.5 3.5 5 and neighbours
    t = np.array([6, .25, .75, 1.25, 1.75, 2.5, 3.5, 5, -.25, -.75, -1.25, -1.75, -2.5, -3.5, -5,
                  .5, 1, 1.5, 2, 3, 4, 0.2499999, 0.2500001, 5.0000005, 4.9999995, 0, -0.0,
                  7.9, 1e-30, -1e-30, 0.7499999, 0.7500001], np.float32)
    assert t.size == 32
    x[5, 0:32] = t
    x[5, 32:64] = t * np.float32(2.0 ** -20)
    x[6, 0:32] = 7.9999995                 # absmax just below 8 -> exponent 0, saturates to 6
    x[6, 32:64] = 8.0
    print("quantize_mxfp4 special blocks", flush=True)
    p, s = Q.quantize_mxfp4(x)
    with np.errstate(all="ignore"):
        po, so = F.quantize_mxfp4(x)
    assert np.array_equal(s, so)
    assert np.array_equal(p, po)
    assert s[0, 0] == 127 and p[0, 2] == 0x80 and not np.delete(p[0, :16], 2).any()
    assert s[1, 1] == 0xFF and s[2, 2] == 0xFF


def test_mxfp4_quantiser_strided_source_and_bad_arguments():
    rows, K, ld = 5, 96, 128
    x = _mx_input(rows, ld, 3)
    src, pk, sc = GpuBuffer(x.nbytes), GpuBuffer(rows * K // 2), GpuBuffer(rows * K // 32)
    src.copy_from_host(x)
    print("quantize_mxfp4 strided", flush=True)
    Q.quantize_mxfp4_device(src.ptr_value, rows, K, pk.ptr_value, sc.ptr_value, ld_src=ld)
    p, s = np.empty((rows, K // 2), np.uint8), np.empty((rows, K // 32), np.uint8)
    pk.copy_to_host(p)
    sc.copy_to_host(s)
    po, so = F.quantize_mxfp4(np.ascontiguousarray(x[:, :K]))
    assert np.array_equal(p, po) and np.array_equal(s, so)
    with pytest.raises(_capi.AsterGemmError, match="K % 32"):
        Q.quantize_mxfp4_device(src.ptr_value, rows, 48, pk.ptr_value, sc.ptr_value)
    with pytest.raises(_capi.AsterGemmError, match="ld_src"):
        Q.quantize_mxfp4_device(src.ptr_value, rows, K, pk.ptr_value, sc.ptr_value, ld_src=64)
    with pytest.raises(_capi.AsterGemmError, match="aligned"):
        Q.quantize_mxfp4_device(src.ptr_value + 4, rows, K, pk.ptr_value, sc.ptr_value)
    with pytest.raises(_capi.AsterGemmError, match="aligned"):
        Q.quantize_fp8_tensor_device(src.ptr_value + 4, 8, pk.ptr_value, sc.ptr_value)


def test_quantise_then_gemm_on_device_fp8():
    """fp32 operands in HBM -> device quantiser -> fp8 GEMM, nothing through the host; the
    result equals the oracle's GEMM on the oracle's quantised operands."""
    M, N, K = 256, 512, 1024
    rng = np.random.default_rng(21)
    xa = rng.standard_normal((M, K)).astype(np.float32)
    xb = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    fa, fb = GpuBuffer(xa.nbytes), GpuBuffer(xb.nbytes)
    qa, qb, sa, sb = GpuBuffer(M * K), GpuBuffer(N * K), GpuBuffer(4), GpuBuffer(4)
    dc = GpuBuffer(M * N * 2)
    fa.copy_from_host(xa)
    fb.copy_from_host(xb)
    print("quantise + gemm fp8", flush=True)
    Q.quantize_fp8_tensor_device(fa.ptr_value, M * K, qa.ptr_value, sa.ptr_value)
    Q.quantize_fp8_tensor_device(fb.ptr_value, N * K, qb.ptr_value, sb.ptr_value)
    plan = AG.GemmPlan.create(M, N, K, "fp8_e4m3", "bf16")
    plan.run(qa.ptr_value, qb.ptr_value, dc.ptr_value, scale_a=sa.ptr_value, scale_b=sb.ptr_value)
    out = np.empty((M, N), np.uint16)
    dc.copy_to_host(out)
    a_q, s_a = F.quantize_fp8_tensor(xa)
    b_q, s_b = F.quantize_fp8_tensor(xb)
    want = G.gemm_fp8(a_q, b_q, s_a, s_b, out_dtype=G.BF16)
    rel = G.rel_l2(G.output_to_f32(out, G.BF16), G.output_to_f32(want, G.BF16))
    assert rel <= 1e-3, rel
    # and the quantised GEMM stays near the fp32 product (e4m3 has 3 mantissa bits)
    assert G.rel_l2(G.output_to_f32(out, G.BF16), G.gemm_f32(xa, xb)) < 0.06


def test_quantise_then_gemm_on_device_mxfp4():
    M, N, K = 256, 256, 1024
    rng = np.random.default_rng(22)
    xa = rng.standard_normal((M, K)).astype(np.float32)
    xb = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    fa, fb = GpuBuffer(xa.nbytes), GpuBuffer(xb.nbytes)
    pa, pb = GpuBuffer(M * K // 2), GpuBuffer(N * K // 2)
    ma, mb = GpuBuffer(M * K // 32), GpuBuffer(N * K // 32)
    dc = GpuBuffer(M * N * 4)
    fa.copy_from_host(xa)
    fb.copy_from_host(xb)
    print("quantise + gemm mxfp4", flush=True)
    Q.quantize_mxfp4_device(fa.ptr_value, M, K, pa.ptr_value, ma.ptr_value)
    Q.quantize_mxfp4_device(fb.ptr_value, N, K, pb.ptr_value, mb.ptr_value)
    plan = AG.GemmPlan.create(M, N, K, "mxfp4", "f32")
    plan.run(pa.ptr_value, pb.ptr_value, dc.ptr_value, mx_a=ma.ptr_value, mx_b=mb.ptr_value)
    out = np.empty((M, N), np.float32)
    dc.copy_to_host(out)
    a_p, a_s = F.quantize_mxfp4(xa)
    b_p, b_s = F.quantize_mxfp4(xb)
    want = G.gemm_mxfp4(a_p, a_s, b_p, b_s, out_dtype=G.F32)
    rel = G.rel_l2(out, G.output_to_f32(want, G.F32))
    assert rel <= 1e-3, rel


@pytest.mark.parametrize("src", ["bf16", "f16"])
def test_quantisers_take_16_bit_sources(src):
    """bf16 / f16 sources (what a GEMM of this library writes) give the bytes of the widened
    values, bit for bit."""
    rng = np.random.default_rng(91)
    x32 = (rng.standard_normal((48, 4096)) * rng.choice([1e-3, 0.1, 1.0, 30.0], (48, 1))).astype(np.float32)
    if src == "bf16":
        bits = F.f32_to_bf16_bits(x32)
        wide = F.bf16_bits_to_f32(bits)
        host = bits
    else:
        host = x32.astype(np.float16)
        wide = host.astype(np.float32)
    host[0, :40] = 0                                   # an all-zero block and signed zeros
    wide[0, :40] = 0
    print(f"quantisers from {src}", flush=True)
    q, s = Q.quantize_fp8_tensor(host, src)
    qo, so = F.quantize_fp8_tensor(wide)
    assert np.float32(s).tobytes() == np.float32(so).tobytes() and np.array_equal(q, qo)
    p, sc = Q.quantize_mxfp4(host, src)
    po, sco = F.quantize_mxfp4(wide)
    assert np.array_equal(sc, sco) and np.array_equal(p, po)
    # odd lengths take the scalar tail
    q, s = Q.quantize_fp8_tensor(host.reshape(-1)[:1003], src)
    qo, so = F.quantize_fp8_tensor(wide.reshape(-1)[:1003])
    assert np.float32(s).tobytes() == np.float32(so).tobytes() and np.array_equal(q, qo)


def test_gemm_output_feeds_the_next_quantised_gemm():
    """bf16 GEMM -> MXFP4 quantiser on its bf16 output -> MXFP4 decode GEMM, all on the device."""
    M, K1, K2, N = 16, 1024, 4096, 512
    rng = np.random.default_rng(92)
    x = F.f32_to_bf16_bits(rng.standard_normal((M, K1)).astype(np.float32))
    w1 = F.f32_to_bf16_bits((rng.standard_normal((K2, K1)) * 0.03).astype(np.float32))
    w2 = (rng.standard_normal((N, K2)) * 0.05).astype(np.float32)
    w2p, w2s = F.quantize_mxfp4(w2)
    bufs = {k: GpuBuffer(v.nbytes) for k, v in dict(x=x, w1=w1, w2p=w2p, w2s=w2s).items()}
    for k, v in dict(x=x, w1=w1, w2p=w2p, w2s=w2s).items():
        bufs[k].copy_from_host(np.ascontiguousarray(v))
    h, hp, hs, y = GpuBuffer(M * K2 * 2), GpuBuffer(M * K2 // 2), GpuBuffer(M * K2 // 32), GpuBuffer(M * N * 4)
    print("bf16 gemm -> mxfp4 quantise -> mxfp4 gemm", flush=True)
    AG.GemmPlan.create(M, K2, K1, "bf16", "bf16").run(bufs["x"].ptr_value, bufs["w1"].ptr_value, h.ptr_value)
    Q.quantize_mxfp4_device(h.ptr_value, M, K2, hp.ptr_value, hs.ptr_value, src_dtype="bf16")
    plan = AG.GemmPlan.create(M, N, K2, "mxfp4", "f32")
    assert plan.info.name.decode().startswith("skinnyx_mxfp4")
    plan.run(hp.ptr_value, bufs["w2p"].ptr_value, y.ptr_value, mx_a=hs.ptr_value,
             mx_b=bufs["w2s"].ptr_value)
    out = np.empty((M, N), np.float32)
    y.copy_to_host(out)
    # oracle: the device's own bf16 intermediate, quantised and multiplied on the CPU
    hb = np.empty((M, K2), np.uint16)
    h.copy_to_host(hb)
    hq, hsc = F.quantize_mxfp4(F.bf16_bits_to_f32(hb))
    want = G.gemm_mxfp4(hq, hsc, w2p, w2s, out_dtype=G.F32)
    assert G.rel_l2(out, G.output_to_f32(want, G.F32)) <= 1e-5


@pytest.mark.parametrize("dtype_ab,path", [("bf16", "direct_b"), ("f16", "direct_b_k8"), ("fp8_e4m3", "direct_b"),
                                           ("fp8_e4m3", "direct_b_k8"), ("mxfp4", "direct_b"),
                                           ("mxfp4", "direct_b_k8")])
def test_preshuffle_on_the_device_writes_the_bytes_of_the_host_functions(gpu, dtype_ab, path):
    # the five pre-shuffled layouts, device to device, against kittens_helpers (which the C host
    # functions are tested against): same bytes; N, K with several row blocks and steps
    from aster_amd import kittens_helpers as H
    from aster_amd.execution import GpuBuffer
    N, K = 192, 1280
    rng = np.random.default_rng(8)
    mx = rng.integers(0, 256, (N, K // 32)).astype(np.uint8)
    if dtype_ab in ("bf16", "f16"):
        b = rng.integers(0, 65536, (N, K)).astype(np.uint16)
        want = (H.shuffle_weight if path == "direct_b" else H.shuffle_weight_k8)(b)
    else:
        b = rng.integers(0, 256, (N, K if dtype_ab == "fp8_e4m3" else K // 2)).astype(np.uint8)
        want = H.shuffle_weight_bytes(b)
    want_mx = (H.shuffle_scales_e8m0 if path == "direct_b" else H.shuffle_scales_e8m0_lanes)(mx)
    d_b, d_o, d_mx, d_mo = GpuBuffer(b.nbytes), GpuBuffer(b.nbytes), GpuBuffer(mx.nbytes), GpuBuffer(mx.nbytes)
    d_b.copy_from_host(b)
    d_mx.copy_from_host(mx)
    d_o.copy_from_host(np.zeros_like(b))
    d_mo.copy_from_host(np.zeros_like(mx))
    print(f"preshuffle {dtype_ab} {path}", flush=True)
    Q.preshuffle_device(d_b.ptr_value, d_o.ptr_value, N, K, dtype_ab, path,
                        d_mx_src=d_mx.ptr_value, d_mx_dst=d_mo.ptr_value)
    got, got_mx = np.zeros_like(b), np.zeros_like(mx)
    d_o.copy_to_host(got)
    d_mo.copy_to_host(got_mx)
    assert np.array_equal(got, want)
    if dtype_ab == "mxfp4":
        assert np.array_equal(got_mx, want_mx)
    else:
        assert not got_mx.any()     # no scale plane for these types: left alone
    with pytest.raises(_capi.AsterGemmError):   # in place is refused
        Q.preshuffle_device(d_b.ptr_value, d_b.ptr_value, N, K, dtype_ab, path,
                            d_mx_src=d_mx.ptr_value, d_mx_dst=d_mo.ptr_value)
    for bf in (d_b, d_o, d_mx, d_mo):
        bf.free()


@pytest.mark.parametrize("n", [7, 8, 9, 8191, 131072, 131073, 131080, 262144, 262149, 300007, 524288, 524296, 2097159])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_fp8_quantiser_one_and_two_launch_forms(n, dtype):
    """Both sides of the one-launch limit and of 64 workgroups (65 count on two levels), whole and broken 16-byte groups, every source type, with
    signed zeros and the maximum in the last element; nothing behind the n codes is written."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    x[n // 3] = -0.0
    x[-1] = -9.5
    src = x if dtype == "f32" else x.astype(np.float16) if dtype == "f16" else (x.view(np.uint32) >> 16).astype(np.uint16)
    wide = (src.astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else src.astype(np.float32)
    a, q, sc = GpuBuffer(src.nbytes + 16), GpuBuffer(n + 64), GpuBuffer(4)
    a.copy_from_host(src)
    q.copy_from_host(np.full(n + 64, 0xAB, np.uint8))
    print(f"quantize_fp8_tensor {dtype} n={n}", flush=True)
    Q.quantize_fp8_tensor_device(a.ptr_value, n, q.ptr_value, sc.ptr_value, src_dtype=dtype)
    got, s = np.empty(n + 64, np.uint8), np.empty(1, np.float32)
    q.copy_to_host(got)
    sc.copy_to_host(s)
    qo, so = F.quantize_fp8_tensor(wide)
    assert s[0].tobytes() == np.float32(so).tobytes()
    assert np.array_equal(got[:n], qo) and (got[n:] == 0xAB).all()


@pytest.mark.parametrize("n", [114688, 114689, 131071])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_fp8_quantiser_round_its_first_line(n, dtype):
    """Every workgroup reads the whole tensor, and one past that its part, outside a capture."""
    test_fp8_quantiser_one_and_two_launch_forms(n, dtype)


@pytest.mark.parametrize("n", [2 ** 25 - 1, 2 ** 25, 2 ** 25 + 1029])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_fp8_quantiser_with_two_workgroups_per_cu(n, dtype):
    """2^25 elements and more: 512 workgroups, 32 on each counter; one below, 256."""
    test_fp8_quantiser_one_and_two_launch_forms(n, dtype)


@pytest.mark.parametrize("case", ["zeros", "nan", "inf", "huge", "tiny", "subnormal", "2^60", "2^-60"])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_fp8_quantiser_two_launch_edges(case, dtype):
    """Tensors past the one-launch limit whose scale is no ordinary one (absmax zero, NaN, infinite, scales on
    either side of 2^-60 and 2^60): the codes of every path of the encoder, the special element among the
    elements whose place holds the partial maxima, in the middle and behind the last whole group."""
    n = 131072 + 5003
    x = np.random.default_rng(17).standard_normal(n).astype(np.float32)
    with np.errstate(all="ignore"):
        if case == "zeros":
            x[:] = 0.0
            x[::7] = -0.0
        elif case in ("huge", "tiny", "subnormal"):
            x *= np.float32({"huge": 6e37, "tiny": 1e-30, "subnormal": 1e-41}[case] if dtype != "f16" else
                            {"huge": 1e4, "tiny": 1e-5, "subnormal": 1e-7}[case])
        elif case.startswith("2^"):
            if dtype == "f16":
                pytest.skip("not in the range of f16")
            # 448 * 2^+-60 is the largest (smallest) absmax of the plain path; some tensors beyond it
            x = x / np.abs(x).max() * np.float32(448.0 * 2.0 ** int(case[2:]) * (1.01 if case == "2^60" else 0.99))
        src = (x if dtype == "f32" else x.astype(np.float16) if dtype == "f16"
               else (x.view(np.uint32) >> 16).astype(np.uint16))
    for at in ((3, n // 2, n - 1) if case in ("nan", "inf") else (0,)):
        y = src.copy()
        if case in ("nan", "inf"):
            y[at] = {"f32": {"nan": np.nan, "inf": -np.inf}, "f16": {"nan": np.nan, "inf": -np.inf},
                     "bf16": {"nan": 0x7FC0, "inf": 0xFF80}}[dtype][case]
        wide = (y.astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else y.astype(np.float32)
        a, q, sc = GpuBuffer(y.nbytes + 16), GpuBuffer(n), GpuBuffer(4)
        a.copy_from_host(y)
        print(f"quantize_fp8_tensor {dtype} {case} at {at}", flush=True)
        Q.quantize_fp8_tensor_device(a.ptr_value, n, q.ptr_value, sc.ptr_value, src_dtype=dtype)
        got, s = np.empty(n, np.uint8), np.empty(1, np.float32)
        q.copy_to_host(got)
        sc.copy_to_host(s)
        with np.errstate(all="ignore"):
            qo, so = F.quantize_fp8_tensor(wide)
        assert s[0].tobytes() == np.float32(so).tobytes()
        assert np.array_equal(got, qo)
        for bf in (a, q, sc):
            bf.free()


def _fp8_forms_sizes():
    """Past the one-launch limit and both sides of every count of groups per thread (16-byte groups of 256 workgroups),
    elements behind the last whole group among them."""
    for dtype, per in (("bf16", 8), ("f16", 8), ("f32", 4)):
        yield dtype, 131073
        for u in (1, 2, 4, 8, 16, 24, 32):
            if dtype == "f16" and u > 2:
                continue
            groups = 256 * 512 * u
            yield dtype, groups * per
            yield dtype, (groups + 1) * per + 3
    yield "bf16", 2 ** 26 + 70001


@pytest.mark.parametrize("dtype,n", _fp8_forms_sizes())
def test_fp8_quantiser_forms_agree(dtype, n):
    """The form that keeps the tensor in registers, the same without patience for the other maxima, and the two
    launches a capture gets (replayed, with eager calls between): the same codes and scale, with the maximum in the
    first, a middle and the last element, and equal to torch's conversion of the quotients."""
    import torch
    src = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(n, generator=g, device="cuda").to(src)
    q = [torch.full((n + 16,), 0xAB, device="cuda", dtype=torch.uint8) for _ in range(3)]
    s = [torch.zeros(1, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        Q.quantize_fp8_tensor_device(x.data_ptr(), n, q[2].data_ptr(), s[2].data_ptr(), src_dtype=dtype,
                                     stream=stream.cuda_stream)
    for turn, at in enumerate((0, n // 2 + 5, n - 1)):
        x[at] = -(9.0 + turn)
        print(f"quantize_fp8_tensor {dtype} n={n} maximum at {at}", flush=True)
        torch.cuda.synchronize()
        graph.replay()
        Q.quantize_fp8_tensor_device(x.data_ptr(), n, q[0].data_ptr(), s[0].data_ptr(), src_dtype=dtype)
        patience = (0, 100, 5000)[turn]
        _capi.check(_capi.load().astergemm_diag_quantize_fp8(
            x.data_ptr(), _capi.DTYPE_NAMES[dtype], n, q[1].data_ptr(), s[1].data_ptr(), patience, None))
        torch.cuda.synchronize()
        scale = np.float32(9.0 + turn) / np.float32(448)
        assert [v.item() for v in s] == [scale] * 3
        want = torch.div(x.float(), torch.tensor(scale, device="cuda")).to(torch.float8_e4m3fn).view(torch.uint8)
        for v in q:
            assert torch.equal(v[:n], want) and bool((v[n:] == 0xAB).all())
            v[:n].zero_()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_fp8_quantiser_sets_of_maxima_in_turn(dtype):
    """More launches than there are sets of maxima, none waited for, of two sizes in turn and on two streams: every one has
    its own maximum."""
    import torch
    src = torch.float32 if dtype == "f32" else torch.bfloat16
    streams, sizes, count = [torch.cuda.Stream(), torch.cuda.Stream()], (140000, 600003), 150
    x = [torch.randn(n, device="cuda").clamp(-3, 3).to(src) for n in sizes]
    xs = [x[i % 2].clone() for i in range(count)]
    for i, v in enumerate(xs):
        v[(i * 977) % v.numel()] = 4.0 + i
    qs, ss = [torch.zeros(v.numel(), device="cuda", dtype=torch.uint8) for v in xs], torch.zeros(count, device="cuda")
    torch.cuda.synchronize()
    print(f"quantize_fp8_tensor {dtype} {count} launches on two streams", flush=True)
    for i, v in enumerate(xs):
        Q.quantize_fp8_tensor_device(v.data_ptr(), v.numel(), qs[i].data_ptr(), ss.data_ptr() + 4 * i, src_dtype=dtype,
                                     stream=streams[(i // 2) % 2].cuda_stream)
    torch.cuda.synchronize()
    # 4 ... 153 in bf16: whole numbers, exact
    assert ss.cpu().numpy().tolist() == [np.float32(4.0 + i) / np.float32(448) for i in range(count)]
    for i, v in enumerate(xs):
        want = torch.div(v.float(), ss[i]).to(torch.float8_e4m3fn).view(torch.uint8)
        assert torch.equal(qs[i], want)


@pytest.mark.parametrize("patience", [0, 5000])
@pytest.mark.parametrize("dtype,n", [
    ("bf16", 114689), ("f32", 114691), ("f16", 131072),           # from the first size on that the form takes
    ("bf16", 1 << 20), ("f32", (1 << 21) + 3), ("bf16", (1 << 23) + 7), ("bf16", (1 << 24) + 5),    # 1 ... 16 groups
    ("bf16", 3 * (1 << 23)), ("f32", 1 << 24), ("bf16", (1 << 26) + 70003), ("f32", (1 << 25) + 70001),  # 1024 threads
])
def test_fp8_quantiser_looks_up_the_maximum_anywhere(dtype, n, patience):
    """A maximum, an infinity and a NaN in the first, a middle and the last element, in the last whole group and, of a
    tensor that the registers do not hold, behind what they hold; without patience, so that workgroups look the shares
    up, and with it: the bytes of the two launches (one up to 131072 elements) of a capture."""
    import torch
    src = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    per = 4 if dtype == "f32" else 8
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(n, generator=g, device="cuda").clamp(-5, 5).to(src)
    q = [torch.full((n + 16,), 0xAB, device="cuda", dtype=torch.uint8) for _ in range(2)]
    s = [torch.zeros(1, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        Q.quantize_fp8_tensor_device(x.data_ptr(), n, q[1].data_ptr(), s[1].data_ptr(), src_dtype=dtype,
                                     stream=stream.cuda_stream)
    held = 14 * 256 * 1024 * per
    for at in [0, n // 2 + 5, n // per * per - 1, n - 1] + ([held + 9, (held + n) // 2] if n > 1 << 25 else []):
        kept = x[at].clone()
        for value, scale in ((-9.0, np.float32(9) / np.float32(448)), (float("-inf"), np.inf), (float("nan"), 1.0)):
            x[at] = value
            print(f"quantize_fp8_tensor {dtype} n={n} {value} at {at} patience {patience}", flush=True)
            torch.cuda.synchronize()
            graph.replay()
            _capi.check(_capi.load().astergemm_diag_quantize_fp8(
                x.data_ptr(), _capi.DTYPE_NAMES[dtype], n, q[0].data_ptr(), s[0].data_ptr(), patience, None))
            torch.cuda.synchronize()
            assert [v.item() for v in s] == [scale] * 2
            assert torch.equal(q[0], q[1]) and bool((q[0][n:] == 0xAB).all())
            q[0][:n].zero_()
        x[at] = kept


@pytest.fixture
def captured(monkeypatch):
    """Q.quantize_fp8_tensor_device as a captured call, replayed: one launch up to 131072 elements, two past that,
    which is what devices of fewer than 256 CUs run as well."""
    import torch
    eager = Q.quantize_fp8_tensor_device
    graphs = []

    def call(*args, **kw):
        torch.cuda.synchronize()
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            eager(*args, stream=stream.cuda_stream, **kw)
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
        graphs.append(graph)

    monkeypatch.setattr(Q, "quantize_fp8_tensor_device", call)
    return graphs


@pytest.mark.parametrize("n", [114688, 114689, 131072, 131073, 131080, 262144, 262149, 300007, 524288, 524296, 2097159])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_fp8_quantiser_sizes_of_the_captured_forms(captured, n, dtype):
    """Round the limit of the one launch in which every workgroup reads the whole tensor, of 64 workgroups of the second
    launch (65 count on two levels: past 524288 16-bit elements, 262144 of fp32), whole and broken groups."""
    test_fp8_quantiser_one_and_two_launch_forms(n, dtype)
    assert len(captured) == 1


@pytest.mark.parametrize("n", [2 ** 25 - 1, 2 ** 25, 2 ** 25 + 1029])
def test_fp8_quantiser_captured_with_two_workgroups_per_cu(captured, n):
    """2^25 elements and more: 512 workgroups in the second launch, 32 on each counter; one below, 256."""
    test_fp8_quantiser_one_and_two_launch_forms(n, "bf16")
    assert len(captured) == 1


@pytest.mark.parametrize("case", ["zeros", "nan", "inf", "huge", "tiny", "subnormal", "2^60", "2^-60"])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_fp8_quantiser_two_launch_edges_captured(captured, case, dtype):
    """Scales that are no ordinary ones, the special element in the place of the partial maxima, in the middle and
    behind the last whole group."""
    test_fp8_quantiser_two_launch_edges(case, dtype)
    assert captured


def test_the_diagnostic_entry_takes_what_the_form_takes():
    import torch
    x, s = torch.ones(114689, device="cuda"), torch.zeros(1, device="cuda")
    q = torch.zeros(114692, device="cuda", dtype=torch.uint8)
    run = lambda n: _capi.load().astergemm_diag_quantize_fp8(x.data_ptr(), _capi.DTYPE_NAMES["f32"], n, q.data_ptr(),
                                                             s.data_ptr(), 100, None)
    assert run(114688) == -22 and run(114689) == 0
    torch.cuda.synchronize()
    assert s.item() == np.float32(1) / np.float32(448) and bool((q[:114689] == 0x7E).all())


def test_fp8_quantiser_beside_a_kernel_that_holds_most_cus():
    """A product keeps 224 CUs for longer than the quantiser runs: the workgroups that find a place look up the maxima of
    the others between them, once, and not each for itself.  Against the two launches of a capture, which wait for nobody
    (1.5 times as long as those; 30 times where every workgroup reads all missing shares); the bytes are the same."""
    import torch
    from time import perf_counter
    n, (M, N, K) = 1 << 24, (3584, 4096, 65536)
    a, b = (torch.zeros(r, K, device="cuda", dtype=torch.bfloat16) for r in (M, N))
    c = torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    assert plan.info.grid_x == 224 and plan.info.lds_bytes == 160 * 1024
    x = torch.randn(n, device="cuda").to(torch.bfloat16)
    q = [torch.zeros(n, device="cuda", dtype=torch.uint8) for _ in range(2)]
    s = torch.zeros(2, device="cuda")
    busy, stream, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    call = lambda i: Q.quantize_fp8_tensor_device(x.data_ptr(), n, q[i].data_ptr(), s.data_ptr() + 4 * i, src_dtype="bf16",
                                                  stream=stream.cuda_stream)
    with torch.cuda.graph(graph, stream=stream):
        call(1)

    def replay():
        with torch.cuda.stream(stream):
            graph.replay()

    def took(what):
        torch.cuda.synchronize()
        plan.run(a.data_ptr(), b.data_ptr(), c.data_ptr(), stream=busy.cuda_stream)
        began = perf_counter()
        while perf_counter() - began < 150e-6:      # the product's workgroups have their CUs
            pass
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record(stream)
        what()
        e[1].record(stream)
        torch.cuda.synchronize()
        return e[0].elapsed_time(e[1])

    print("quantize_fp8_tensor beside a product", flush=True)
    eager, captured = (min(took(f) for _ in range(6)) for f in (lambda: call(0), replay))
    assert torch.equal(q[0], q[1]) and s[0] == s[1]
    assert eager <= 4 * captured, (eager, captured)


@pytest.mark.parametrize("rows", [1, 15, 127, 128, 129, 300])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_mxfp4_quantiser_lane_order_edges(rows, dtype):
    """Row counts round the 128-row groups of the lane order: the plane equals the shuffled
    row-major one, bytes of rows past the end stay as they are, the nibbles are the same."""
    from aster_amd.kittens_helpers import shuffle_scales_e8m0_lanes128
    K = 512
    x = np.random.default_rng(rows).standard_normal((rows, K)).astype(np.float32)
    src = x if dtype == "f32" else x.astype(np.float16) if dtype == "f16" else (x.view(np.uint32) >> 16).astype(np.uint16)
    wide = (src.astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else src.astype(np.float32)
    padded = (rows + 127) // 128 * 128
    a, p, sc = GpuBuffer(src.nbytes), GpuBuffer(rows * K // 2), GpuBuffer(padded * K // 32)
    a.copy_from_host(src)
    sc.copy_from_host(np.full(padded * K // 32, 0xAB, np.uint8))
    print(f"quantize_mxfp4 lanes128 {dtype} rows={rows}", flush=True)
    Q.quantize_mxfp4_device(a.ptr_value, rows, K, p.ptr_value, sc.ptr_value, src_dtype=dtype,
                            scales_layout="lanes128")
    got_p, got_s = np.empty((rows, K // 2), np.uint8), np.empty(padded * K // 32, np.uint8)
    p.copy_to_host(got_p)
    sc.copy_to_host(got_s)
    po, so = F.quantize_mxfp4(wide)
    plane = np.full((padded, K // 32), 0xAB, np.uint8)
    plane[:rows] = so
    assert np.array_equal(got_p, po)
    assert np.array_equal(got_s, np.asarray(shuffle_scales_e8m0_lanes128(plane)).reshape(-1))


@pytest.mark.parametrize("rows,K,ld,dtype,layout", [
    (1024, 4096, 0, "bf16", "rows"), (1025, 4096, 0, "bf16", "rows"),          # 2^19 groups of 16 bytes, and past them
    (1024, 4096, 4104, "f16", "rows"), (1025, 4096, 4104, "bf16", "rows"), (513, 4096, 0, "f32", "rows"),
    (1024, 4096, 0, "bf16", "lanes128"), (1025, 4096, 0, "bf16", "lanes128"),  # 2^22 elements, and past them
    (1025, 4096, 0, "f32", "lanes128"), (100, 4096, 4104, "f16", "lanes128"),
])
def test_mxfp4_quantiser_sizes_of_its_forms(rows, K, ld, dtype, layout):
    """Both sides of the lines between one and two groups per lane and between the two workgroup sizes."""
    from aster_amd.kittens_helpers import shuffle_scales_e8m0_lanes128
    x = np.random.default_rng(rows).standard_normal((rows, ld or K)).astype(np.float32) * 3
    src = x if dtype == "f32" else x.astype(np.float16) if dtype == "f16" else (x.view(np.uint32) >> 16).astype(np.uint16)
    wide = (src.astype(np.uint32) << 16).view(np.float32) if dtype == "bf16" else src.astype(np.float32)
    plane = (rows + 127) // 128 * 128 * (K // 32) if layout == "lanes128" else rows * (K // 32)
    a, p, sc = GpuBuffer(src.nbytes), GpuBuffer(rows * K // 2), GpuBuffer(plane)
    a.copy_from_host(src)
    sc.copy_from_host(np.full(plane, 127, np.uint8))
    print(f"quantize_mxfp4 {layout} {dtype} {rows}x{K} ld={ld}", flush=True)
    Q.quantize_mxfp4_device(a.ptr_value, rows, K, p.ptr_value, sc.ptr_value, src_dtype=dtype, ld_src=ld,
                            scales_layout=layout)
    packed, scales = np.empty((rows, K // 2), np.uint8), np.empty(plane, np.uint8)
    p.copy_to_host(packed)
    sc.copy_to_host(scales)
    want, want_s = F.quantize_mxfp4(np.ascontiguousarray(wide[:, :K]))
    assert np.array_equal(packed, want)
    if layout == "lanes128":
        want_s = shuffle_scales_e8m0_lanes128(want_s)
    assert np.array_equal(scales, np.asarray(want_s).reshape(-1))
    for bf in (a, p, sc):
        bf.free()


@pytest.mark.parametrize("rows,K,ld,dtype,layout", [
    (1, 256, 0, "f32", "lanes128"), (32, 256, 0, "f32", "lanes128"), (33, 512, 520, "f32", "lanes128"),  # 256 threads, 1024
    (48, 256, 264, "bf16", "lanes128"), (49, 512, 0, "f16", "lanes128"),
    (2417, 4096, 0, "bf16", "rows"), (3000, 4096, 0, "f16", "rows"), (3195, 4096, 0, "bf16", "rows"),  # two, four, two
    (1500, 4096, 0, "f32", "rows"),
    (2457, 4096, 4104, "bf16", "rows"), (2458, 4096, 4104, "bf16", "rows"), (4096, 4096, 4104, "f16", "rows"),
    (4097, 4096, 4104, "bf16", "rows"), (1300, 4096, 4224, "f32", "rows"), (2049, 4096, 4104, "f32", "rows"),
])
def test_mxfp4_quantiser_lines_between_its_forms(rows, K, ld, dtype, layout):
    """Few rows in lane order, and two groups per lane or four."""
    test_mxfp4_quantiser_sizes_of_its_forms(rows, K, ld, dtype, layout)
