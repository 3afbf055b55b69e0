"""The entry point that allocates nothing (`astergemm_run_noalloc`) against `astergemm_run`.

Shapes whose rows are cut into K ranges keep their fp32 partial sums in a scratch array built
into the library instead of an allocated workspace; the results must be the same bits.  Two calls
in a row share the array, the second smaller than the first; a shape that needs no workspace and
one that needs more than the array holds are covered as well, and so is a HIP graph that holds
two launches of it and is replayed on fresh activations.
"""
import ctypes
import os

import numpy as np
import pytest

from aster_amd import _capi, gemm as AG
from aster_amd.execution import GpuBuffer
from oracle import formats as F, gemm as G

pytestmark = pytest.mark.gpu


def _bf16(rng, shape, std):
    return F.f32_to_bf16_bits((rng.standard_normal(shape) * std).astype(np.float32))


def _both_ways(M, N, K, seed):
    rng = np.random.default_rng(seed)
    a, b = _bf16(rng, (M, K), 1.0), _bf16(rng, (N, K), 0.02)
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    bufs = [GpuBuffer(a.nbytes), GpuBuffer(b.nbytes), GpuBuffer(M * N * 2), GpuBuffer(M * N * 2)]
    bufs[0].copy_from_host(a)
    bufs[1].copy_from_host(b)
    outs = []
    for i, run in enumerate((plan.run, plan.run_noalloc)):
        out = np.full((M, N), 0x7FC1, np.uint16)
        bufs[2 + i].copy_from_host(out)
        print(f"{run.__name__} {plan.info.name.decode()} M={M} N={N} K={K} "
              f"workspace={plan.workspace_bytes()}", flush=True)
        run(bufs[0].ptr_value, bufs[1].ptr_value, bufs[2 + i].ptr_value)
        bufs[2 + i].copy_to_host(out)
        outs.append(out)
    for bf in bufs:
        bf.free()
    want = G.gemm(a, b, G.BF16, G.BF16)
    return plan, outs[0], outs[1], want


def test_noalloc_matches_run_on_two_calls_in_a_row(gpu):
    # split K on the 128 x 128 kernel: 8 K ranges x 128 x 4096 x 4 bytes = the whole 16 MiB array
    plan, ref, got, want = _both_ways(128, 4096, 14336, seed=7)
    assert plan.workspace_bytes() == _capi.NOALLOC_SCRATCH_BYTES
    assert np.array_equal(ref, got)
    assert G.rel_l2(F.bf16_bits_to_f32(got), F.bf16_bits_to_f32(want)) <= 1e-3
    # then a smaller one through the same array: a decode shape in K ranges
    plan, ref, got, want = _both_ways(16, 520, 14336, seed=8)
    assert 0 < plan.workspace_bytes() < _capi.NOALLOC_SCRATCH_BYTES
    assert np.array_equal(ref, got)
    assert G.rel_l2(F.bf16_bits_to_f32(got), F.bf16_bits_to_f32(want)) <= 1e-3
    # and a shape without K ranges: the array is not touched at all
    plan, ref, got, want = _both_ways(264, 520, 512, seed=9)
    assert plan.workspace_bytes() == 0
    assert np.array_equal(ref, got)


def test_noalloc_refuses_what_the_scratch_cannot_hold(gpu):
    plan = AG.GemmPlan.create(512, 4096, 14336, "bf16", "bf16")
    assert plan.workspace_bytes() > _capi.NOALLOC_SCRATCH_BYTES
    with pytest.raises(_capi.AsterGemmError) as err:
        plan.run_noalloc(256, 256, 256)     # refused before any pointer is used
    assert err.value.code == -22 and "scratch" in str(err.value)


@pytest.mark.parametrize("M,N,K", [(333, 4096, 14336), (130, 1032, 8192)])
def test_split_configs_without_scratch_of_their_own(gpu, M, N, K):
    """AUTO cuts these into K ranges where the library's buffer may be used; the entry point without
    allocations and a capture (several replays, eager work between them) run the other kernel."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    ref = a.float() @ b.float().T
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    assert plan.workspace_bytes() > 0
    c = torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)

    def check():
        torch.cuda.synchronize()
        rel = float((c.float() - ref).norm() / ref.norm())
        c.zero_()
        assert rel <= 4e-3, rel      # bf16 rounding of the output, 1.7e-3, and the order of fp32 sums

    ptrs = (a.data_ptr(), b.data_ptr(), c.data_ptr())
    print(f"{plan.info.name.decode()} M={M} N={N} K={K}", flush=True)
    torch.cuda.synchronize()
    plan.run(*ptrs)
    check()
    plan.run_noalloc(*ptrs)
    check()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.run(*ptrs, stream=torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        graph.replay()
        check()
        plan.run(*ptrs)
        check()


@pytest.mark.parametrize("M,N,K", [(333, 4096, 14336), (130, 1032, 8192), (512, 4096, 14336)])
def test_a_workspace_of_the_stated_size_gives_the_eager_bits_under_capture(gpu, M, N, K):
    """Configs with an optional split: with a caller's workspace a captured call runs the kernel an eager one
    does, several replays with eager work between them; so does a plan that names the kernel."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    eager, got = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    pinned = AG.GemmPlan.create(M, N, K, "bf16", "bf16", variant=plan.info.variant)
    need = plan.workspace_bytes()
    ws = torch.zeros(need, device="cuda", dtype=torch.uint8)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    print(f"{plan.info.name.decode()} M={M} N={N} K={K}", flush=True)
    plan.run(a.data_ptr(), b.data_ptr(), eager.data_ptr(), stream=stream.cuda_stream)
    stream.synchronize()
    for p, extra in ((plan, dict(workspace=ws.data_ptr(), workspace_bytes=need)), (pinned, {})):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            p.run(a.data_ptr(), b.data_ptr(), got.data_ptr(), stream=stream.cuda_stream, **extra)
        for _ in range(3):
            got.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, eager)
            plan.run(a.data_ptr(), b.data_ptr(), eager.data_ptr(), stream=stream.cuda_stream)
            torch.cuda.synchronize()


@pytest.mark.parametrize("M,N,K", [(96, 1000, 16384),      # one launch: K over waves, the workspace left unused
                                   (128, 4096, 14336)])    # 128 x 128 tiles in eight K ranges
def test_caller_workspace_matches_the_library_workspace(gpu, M, N, K):
    rng = np.random.default_rng(11)
    a, b = _bf16(rng, (M, K), 1.0), _bf16(rng, (N, K), 0.02)
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    need = plan.workspace_bytes()
    assert need > 0 and ((plan.info.wg_tile_m, plan.info.wg_tile_n) == (128, 128)) == (N == 4096)
    bufs = [GpuBuffer(a.nbytes), GpuBuffer(b.nbytes), GpuBuffer(M * N * 2), GpuBuffer(need)]
    bufs[0].copy_from_host(a)
    bufs[1].copy_from_host(b)
    out_lib, out_own = np.zeros((M, N), np.uint16), np.zeros((M, N), np.uint16)
    plan.run(bufs[0].ptr_value, bufs[1].ptr_value, bufs[2].ptr_value)
    bufs[2].copy_to_host(out_lib)
    plan.run(bufs[0].ptr_value, bufs[1].ptr_value, bufs[2].ptr_value, workspace=bufs[3].ptr_value,
             workspace_bytes=need)
    bufs[2].copy_to_host(out_own)
    assert np.array_equal(out_lib, out_own)
    with pytest.raises(_capi.AsterGemmError):
        plan.run(bufs[0].ptr_value, bufs[1].ptr_value, bufs[2].ptr_value,
                 workspace=bufs[3].ptr_value, workspace_bytes=need - 4)
    for bf in bufs:
        bf.free()


@pytest.mark.parametrize("M,N,K,dtype,kernel,planes", [
    # AUTO: K over waves in fewer ranges than the kernel it stands in for, whose planes the workspace is sized for
    (64, 4096, 14336, "bf16", None, 4), (29, 4100, 11008, "f16", None, 3), (64, 8192, 28672, "fp8_e4m3", None, 2),
    # by name: the kernels with K ranges themselves
    (96, 1000, 16384, "bf16", "splitk_bf16_128x128_w2x2_bf16", 0),
    (128, 1024, 8192, "f16", "splitk_f16_128x128_w2x2_bf16", 0),
    (50, 1032, 28672, "bf16", "skinnyx_bf16_m64_bf16", 0), (16, 4096, 14336, "fp8_e4m3", "skinnyx_fp8_m64_bf16", 0)])
def test_partial_sums_go_to_the_memory_of_the_call(gpu, M, N, K, dtype, kernel, planes):
    """The library's buffer, a caller's, the built-in scratch, each eagerly and captured (several replays with eager
    work between): the same bits; of a caller's buffer the planes are written and nothing else."""
    import torch
    from test_gpu_ids import device_operands
    from test_gpu_parity import _variant_id
    plan = AG.GemmPlan.create(M, N, K, dtype, "bf16", variant=_variant_id(kernel) if kernel else 0)
    need, own = plan.workspace_bytes(), planes or plan.workspace_bytes() // (4 * M * N)
    assert (planes or 2) * 4 * M * N <= need <= _capi.NOALLOC_SCRATCH_BYTES
    (pa, pb), kw, keep = device_operands(M, N, K, dtype)
    want, got = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ws = torch.full((need // 4 + 64,), float("nan"), device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    print(f"{plan.info.name.decode()} M={M} N={N} K={K}", flush=True)
    plan.run(pa, pb, want.data_ptr(), stream=stream.cuda_stream, **kw)
    stream.synchronize()
    ref = keep[0].float() @ keep[1].float().T * (0.125 if dtype == "fp8_e4m3" else 1.0)
    assert float((want.float() - ref).norm() / ref.norm()) <= 4e-3   # bf16 rounding, 1.7e-3, and the sums' order
    small = dict(workspace=ws.data_ptr(), workspace_bytes=need - 4)
    with pytest.raises(_capi.AsterGemmError, match="workspace of"):
        plan.run(pa, pb, got.data_ptr(), **kw, **small)
    for call, extra in ((plan.run, {}), (plan.run, dict(workspace=ws.data_ptr(), workspace_bytes=need)),
                        (plan.run_noalloc, {})):
        ws.fill_(float("nan"))
        got.zero_()
        torch.cuda.synchronize()
        call(pa, pb, got.data_ptr(), stream=stream.cuda_stream, **kw, **extra)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        written = ~torch.isnan(ws)
        assert int(written.sum()) == (own * M * N if extra else 0) and (not extra or bool(written[:own * M * N].all()))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(pa, pb, got.data_ptr(), stream=stream.cuda_stream, **kw, **extra)
        for _ in range(3):
            got.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            plan.run(pa, pb, want.data_ptr(), stream=stream.cuda_stream, **kw)
            torch.cuda.synchronize()


def test_an_eager_split_call_readies_its_stream_for_a_capture_of_the_same_config(gpu):
    """512 x 4096 x 14336: an eager call runs split K on 256 x 128 tiles , a captured one on 128 x 128,
    whose planes go to the library's buffer of the stream, which cannot grow inside a capture.  Every replay
    has the bits of that kernel, with eager calls between the replays; a call that succeeds leaves the
    thread's last error as it was."""
    import torch
    M, N, K = 512, 4096, 14336
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    eager, got, want = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
    assert plan.info.name.decode() == "splitk_bf16_256x128_w4x2_bf16"
    lib, info = _capi.load(), _capi.KernelInfo()
    for i in range(lib.astergemm_variant_count()):
        _capi.check(lib.astergemm_variant_info(i, ctypes.byref(plan.config), ctypes.byref(info)))
        if info.name.decode() == "splitk_bf16_128x128_w2x2_bf16":
            square = AG.GemmPlan.create(M, N, K, "bf16", "bf16", variant=info.variant)
    assert 0 < square.workspace_bytes() <= plan.workspace_bytes()
    stream = torch.cuda.Stream()
    with pytest.raises(_capi.AsterGemmError, match="non-null"):
        plan.run(None, None, None)
    torch.cuda.synchronize()
    print("eager, capture, replays", flush=True)
    plan.run(a.data_ptr(), b.data_ptr(), eager.data_ptr(), stream=stream.cuda_stream)
    assert "non-null" in _capi.last_error()
    stream.synchronize()
    first = eager.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        plan.run(a.data_ptr(), b.data_ptr(), got.data_ptr(), stream=stream.cuda_stream)
    square.run(a.data_ptr(), b.data_ptr(), want.data_ptr())
    torch.cuda.synchronize()
    for _ in range(3):
        got.zero_()
        eager.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        plan.run(a.data_ptr(), b.data_ptr(), eager.data_ptr(), stream=stream.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(eager, first)


@pytest.mark.parametrize("M,N,K,dtype,kernel", [
    (128, 1024, 8192, "bf16", "splitk_bf16_128x128_w2x2_bf16"),
    (129, 1032, 8192, "bf16", "splitk_bf16_256x128_w4x2_bf16"),
    (50, 1032, 28672, "bf16", "skinnyx_bf16_m64_bf16"), (16, 520, 14336, "mxfp4", "skinnyx_mxfp4_m64_bf16"),
    (64, 2048, 14336, "bf16", None), (64, 4096, 14336, "bf16", None)])    # AUTO: K over waves in four ranges
def test_two_host_threads_on_one_stream_keep_products_and_sums_in_pairs(gpu, M, N, K, dtype, kernel):
    """Split K and the K ranges of the decode kernels: two threads enqueue different activations on one
    stream and share the partial sums' memory (the library's buffer, the built-in scratch, a caller's
    buffer); each call's product and sum stay together, so every output has the bits of the call alone."""
    import threading
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    if dtype == "mxfp4":
        draw = lambda rows: torch.randint(0, 256, (rows, K // 2), generator=g, device="cuda", dtype=torch.uint8)
        mx = lambda rows: torch.randint(118, 123, (rows, K // 32), generator=g, device="cuda", dtype=torch.uint8)
        mb, mas = mx(N), [mx(M) for _ in range(2)]
        scales = [dict(mx_a=m.data_ptr(), mx_b=mb.data_ptr()) for m in mas]
    else:
        draw = lambda rows: torch.randn(rows, K, generator=g, device="cuda").to(torch.bfloat16)
        scales = [{}, {}]
    w, xs = draw(N), [draw(M) for _ in range(2)]
    lib, info = _capi.load(), _capi.KernelInfo()
    plan = AG.GemmPlan.create(M, N, K, dtype, "bf16")
    for i in range(lib.astergemm_variant_count()):
        _capi.check(lib.astergemm_variant_info(i, ctypes.byref(plan.config), ctypes.byref(info)))
        if info.name.decode() == kernel:
            plan = AG.GemmPlan.create(M, N, K, dtype, "bf16", variant=info.variant)
    if kernel is None:
        assert (plan.info.wg_tile_m, plan.info.wg_tile_n) == (64, 64) and plan.info.grid_x == N // 64 * 4
    else:
        assert plan.info.name.decode() == kernel
    need = plan.workspace_bytes()
    assert 0 < need <= _capi.NOALLOC_SCRATCH_BYTES
    own = torch.zeros(need, device="cuda", dtype=torch.uint8)
    want = torch.zeros(2, M, N, device="cuda", dtype=torch.bfloat16)
    n = 100
    outs = torch.zeros(2, n, M, N, device="cuda", dtype=torch.bfloat16)
    torch.cuda.synchronize()
    for i in range(2):
        plan.run(xs[i].data_ptr(), w.data_ptr(), want[i].data_ptr(), **scales[i])
    assert not torch.equal(want[0], want[1])
    for way in ("run", "run_noalloc", "caller"):
        print(f"{way} {plan.info.name.decode()} M={M} N={N} K={K}", flush=True)
        outs.zero_()
        torch.cuda.synchronize()
        call = plan.run_noalloc if way == "run_noalloc" else plan.run
        extra = dict(workspace=own.data_ptr(), workspace_bytes=need) if way == "caller" else {}
        start, failed = threading.Barrier(2), []

        def work(i):
            try:
                start.wait(30)
                for r in range(n):
                    call(xs[i].data_ptr(), w.data_ptr(), outs[i, r].data_ptr(), **scales[i], **extra)
            except Exception as exc:
                failed.append(exc)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not failed, failed
        for i in range(2):
            assert torch.equal(outs[i], want[i].expand(n, M, N)), way


def _hip():
    # the HIP runtime the library itself is linked against, found through the library's own handle
    # (another copy of libamdhip64 may be loaded in this process, e.g. the one torch ships, and a
    # stream of one runtime means nothing to the other)
    lib = _capi.load()
    for name, args in (("hipStreamBeginCapture", [ctypes.c_void_p, ctypes.c_int]),
                       ("hipStreamEndCapture", [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]),
                       ("hipGraphInstantiate", [ctypes.POINTER(ctypes.c_void_p), ctypes.c_void_p,
                                                ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]),
                       ("hipGraphLaunch", [ctypes.c_void_p, ctypes.c_void_p]),
                       ("hipGraphExecDestroy", [ctypes.c_void_p]),
                       ("hipGraphDestroy", [ctypes.c_void_p])):
        fn = getattr(lib, name)
        fn.argtypes, fn.restype = args, ctypes.c_int
    return lib


def test_noalloc_launches_replay_from_a_graph(gpu):
    # two decode projections in a row, h = x W1^T (no K ranges) and y = h W2^T (rows cut into K
    # ranges: partial sums in the built-in scratch array), captured once in global capture mode
    # (a hipMalloc or a synchronizing call inside the capture would fail it) and replayed on
    # three different x, with eager launches and synchronizations in between; every replay must
    # give the bits of the eager pair on the same x
    M, H, D = 16, 4096, 14336
    rng = np.random.default_rng(21)
    w1, w2 = _bf16(rng, (D, H), 0.02), _bf16(rng, (H, D), 0.02)
    xs = [_bf16(rng, (M, H), 1.0) for _ in range(3)]
    up = AG.GemmPlan.create(M, D, H, "bf16", "bf16")
    down = AG.GemmPlan.create(M, H, D, "bf16", "bf16")
    assert up.workspace_bytes() == 0 and 0 < down.workspace_bytes() <= _capi.NOALLOC_SCRATCH_BYTES
    dx, dw1, dw2 = GpuBuffer(xs[0].nbytes), GpuBuffer(w1.nbytes), GpuBuffer(w2.nbytes)
    dh, dy = GpuBuffer(M * D * 2), GpuBuffer(M * H * 2)
    dw1.copy_from_host(w1)
    dw2.copy_from_host(w2)
    rt, hip = _capi.load(), _hip()

    def eager_pair(x):
        dx.copy_from_host(x)
        up.run(dx.ptr_value, dw1.ptr_value, dh.ptr_value)
        down.run(dh.ptr_value, dw2.ptr_value, dy.ptr_value)
        y = np.zeros((M, H), np.uint16)
        dy.copy_to_host(y)
        return y

    want = [eager_pair(x) for x in xs]
    assert not np.array_equal(want[0], want[1])
    # the eager calls above were also the first calls on this device: set-up is behind us
    up.run_noalloc(dx.ptr_value, dw1.ptr_value, dh.ptr_value)
    down.run_noalloc(dh.ptr_value, dw2.ptr_value, dy.ptr_value)
    _capi.check(rt.aster_rt_device_synchronize())

    stream, graph, gexec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    _capi.check(rt.aster_rt_stream_create(ctypes.byref(stream)))
    print("capture", up.info.name.decode(), down.info.name.decode(), flush=True)
    assert hip.hipStreamBeginCapture(stream, 0) == 0        # hipStreamCaptureModeGlobal
    try:
        up.run_noalloc(dx.ptr_value, dw1.ptr_value, dh.ptr_value, stream=stream.value)
        down.run_noalloc(dh.ptr_value, dw2.ptr_value, dy.ptr_value, stream=stream.value)
    finally:
        rc = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert rc == 0 and graph.value
    assert hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0) == 0
    try:
        for i in (2, 0, 1):
            # eager work between the replays: another x through the allocating entry point
            assert np.array_equal(eager_pair(xs[(i + 1) % 3]), want[(i + 1) % 3])
            dx.copy_from_host(xs[i])
            dy.copy_from_host(np.full((M, H), 0x7FC1, np.uint16))
            print("replay on x", i, flush=True)
            assert hip.hipGraphLaunch(gexec, stream) == 0
            _capi.check(rt.aster_rt_stream_synchronize(stream))
            y = np.zeros((M, H), np.uint16)
            dy.copy_to_host(y)
            assert np.array_equal(y, want[i]), f"replay on x{i}"
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)
        _capi.check(rt.aster_rt_stream_destroy(stream))
        for bf in (dx, dw1, dw2, dh, dy):
            bf.free()


_PLANES_CHILD = r"""
import ctypes
import torch
from aster_amd import _capi, gemm as AG
_capi.check(_capi.load().aster_rt_init())
M, N, K = 333, 1032, 1024                      # AUTO: a stream kernel; planes off 16 bytes: the general tile kernel
g = torch.Generator(device="cuda").manual_seed(1)
draw = lambda rows: torch.randint(0, 256, (rows, K // 2), generator=g, device="cuda", dtype=torch.uint8)
mx = lambda rows: torch.randint(118, 123, (rows * K // 32 + 8,), generator=g, device="cuda", dtype=torch.uint8)
a, b, ma, mb = draw(M), draw(N), mx(M), mx(N)
got, want = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
plan = AG.GemmPlan.create(M, N, K, "mxfp4", "bf16")
plan.prepare()
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
args = lambda c: (a.data_ptr(), b.data_ptr(), c.data_ptr())
planes = dict(mx_a=ma.data_ptr() + 8, mx_b=mb.data_ptr() + 8)
with torch.cuda.graph(graph):
    plan.run(*args(got), stream=torch.cuda.current_stream().cuda_stream, **planes)
plan.run(*args(want), **planes)
for _ in range(3):
    got.zero_()
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(got, want) and float(want.float().abs().max()) > 0
print("PLANES-OK", flush=True)
"""


def test_prepare_readies_the_kernel_of_planes_on_8_byte_boundaries(gpu):
    # in a process of its own, where nothing has launched the general tile kernel yet
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    print("child process: prepare, capture with planes off 16 bytes, replays", flush=True)
    proc = subprocess.run([sys.executable, "-c", _PLANES_CHILD], cwd=root, capture_output=True, text=True,
                          timeout=110)
    assert proc.returncode == 0 and "PLANES-OK" in proc.stdout, proc.stdout[-2000:] + proc.stderr[-2000:]


_CAPTURE_CHILD = r"""
import ctypes, sys
import numpy as np
from aster_amd import _capi, gemm as AG
from aster_amd.execution import GpuBuffer

lib = _capi.load()
for name, args in (("hipStreamBeginCapture", [ctypes.c_void_p, ctypes.c_int]),
                   ("hipStreamEndCapture", [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]),
                   ("hipGraphInstantiate", [ctypes.POINTER(ctypes.c_void_p), ctypes.c_void_p,
                                            ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]),
                   ("hipGraphLaunch", [ctypes.c_void_p, ctypes.c_void_p])):
    fn = getattr(lib, name)
    fn.argtypes, fn.restype = args, ctypes.c_int
_capi.check(lib.aster_rt_init())
M, N, K = 16, 4096, 14336                      # rows cut into K ranges: partial sums in the scratch
rng = np.random.default_rng(3)
x = (rng.standard_normal((M, K)).astype(np.float32)).view(np.uint32) >> 16
w = (rng.standard_normal((N, K)).astype(np.float32) * 0.02).view(np.uint32) >> 16
x, w = x.astype(np.uint16), w.astype(np.uint16)
dx, dw, dy = GpuBuffer(x.nbytes), GpuBuffer(w.nbytes), GpuBuffer(M * N * 2)
dx.copy_from_host(x)
dw.copy_from_host(w)
plan = AG.GemmPlan.create(M, N, K, "bf16", "bf16")
stream, graph, gexec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
_capi.check(lib.aster_rt_stream_create(ctypes.byref(stream)))

# 1. nothing of this config has run in this process: its first launch inside a capture is refused
assert lib.hipStreamBeginCapture(stream, 0) == 0
try:
    plan.run_noalloc(dx.ptr_value, dw.ptr_value, dy.ptr_value, stream=stream.value)
    refused = None
except _capi.AsterGemmError as exc:
    refused = str(exc)
rc = lib.hipStreamEndCapture(stream, ctypes.byref(graph))
assert refused and "astergemm_prepare" in refused, refused
print("refused:", refused, flush=True)

# 2. after astergemm_prepare the same capture goes through, and the replay gives the eager bits
plan.prepare()
assert lib.hipStreamBeginCapture(stream, 0) == 0
plan.run_noalloc(dx.ptr_value, dw.ptr_value, dy.ptr_value, stream=stream.value)
assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0 and graph.value
assert lib.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0) == 0
got = []
for _ in range(2):
    dy.copy_from_host(np.full((M, N), 0x7FC1, np.uint16))
    assert lib.hipGraphLaunch(gexec, stream) == 0
    _capi.check(lib.aster_rt_stream_synchronize(stream))
    y = np.zeros((M, N), np.uint16)
    dy.copy_to_host(y)
    got.append(y)
plan.run(dx.ptr_value, dw.ptr_value, dy.ptr_value)
_capi.check(lib.aster_rt_device_synchronize())
eager = np.zeros((M, N), np.uint16)
dy.copy_to_host(eager)
assert np.array_equal(got[0], eager) and np.array_equal(got[1], eager)
print("CAPTURE-OK", flush=True)
"""


def test_first_launch_inside_a_capture_is_refused_until_prepared(gpu):
    # in a process of its own, so that no earlier test has launched the kernel: the first launch of
    # a kernel on a device sets a function attribute, which must not happen inside a capture; the
    # library refuses it and astergemm_prepare does that step ahead of time
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    print("child process: capture before / after astergemm_prepare", flush=True)
    proc = subprocess.run([sys.executable, "-c", _CAPTURE_CHILD], cwd=root, capture_output=True, text=True,
                          timeout=110)
    assert proc.returncode == 0 and "CAPTURE-OK" in proc.stdout, proc.stdout[-2000:] + proc.stderr[-2000:]
