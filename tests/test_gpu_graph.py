"""HIP graph capture of the decode path, through the C ABI.

The entry points launch kernels only once their per-stream workspaces exist
(no allocation, copy, memset or synchronization on a warm stream), so a
caller can capture them.  Each case runs the work eagerly twice on a side
stream (growing that stream's workspaces), captures it once on that stream
(torch.cuda.CUDAGraph), then replays the graph three times with eager work on
another stream and synchronizations between the replays.  The outputs are
filled with NaN before every replay, and every replay and every eager run
must reproduce the first eager result bit for bit.

Cases: embedding + a three-layer kcmm_decode_layers_on_stream call + logits
(bf16 and fp8-e4m3 pools; the fp8 page writer's zero-restored counters are
replayed too), standalone paged decode attention (bf16, fp8), and a
split-K projection with its reduction kernel."""
import concurrent.futures
import ctypes as C
import functools

import numpy as np
import pytest

import oracle as O
from lattice_amd.bindings import KV_BF16, KV_FP8, hip, memcpy_dtoh
from lattice_amd.workload import build_decode_case
from tests.test_gpu_glue import _layer_weights, bf16_dev

pytestmark = pytest.mark.gpu


def _check_replays(torch, run, outputs, replays=3):
    """run(stream_ptr) launches the work; outputs() lists the result tensors."""
    gs = torch.cuda.Stream()
    torch.cuda.synchronize()
    run(gs.cuda_stream)
    run(gs.cuda_stream)
    torch.cuda.synchronize()
    ref = [t.clone() for t in outputs()]
    assert all(bool(torch.isfinite(t.float()).all()) for t in ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=gs):
        run(gs.cuda_stream)
    torch.cuda.synchronize()
    main = torch.cuda.current_stream().cuda_stream
    for r in range(replays):
        for t in outputs():
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for i, (t, e) in enumerate(zip(outputs(), ref)):
            assert torch.equal(t, e), f"replay {r}: output {i} differs from the eager run"
        run(main)                       # eager work between the replays
        torch.cuda.synchronize()
        for i, (t, e) in enumerate(zip(outputs(), ref)):
            assert torch.equal(t, e), f"eager run after replay {r}: output {i} differs"
    del graph


@pytest.mark.parametrize("dtype", [KV_BF16, KV_FP8])
def test_decode_step_graph_replays(gpu_lib, dtype):
    import torch
    hq, hkv, d, h, inter, vocab, nl = 32, 8, 128, 4096, 1024, 1024, 3
    lens = [1, 16, 17, 130, 700]
    case = build_decode_case(gpu_lib, batch=len(lens), num_q_heads=hq, kv_heads=hkv, head_dim=d,
                             block_size=16, ctx_lens=lens, dtype=dtype, seed=3, num_layers=nl)
    try:
        rng = np.random.default_rng(21)
        ws = [_layer_weights(torch, rng, h, inter, hq, hkv, d) for _ in range(nl)]
        embed = bf16_dev(torch, O.encode(O.BF16, rng.standard_normal((vocab, h))))
        head = bf16_dev(torch, O.encode(O.BF16, rng.standard_normal((vocab, h)) * 0.02))
        fnorm = bf16_dev(torch, O.encode(O.BF16, 1.0 + 0.1 * rng.standard_normal(h)))
        ids = torch.tensor(rng.integers(0, vocab, size=len(lens)), dtype=torch.int32, device="cuda")
        hidden = torch.empty((len(lens), h), dtype=torch.bfloat16, device="cuda")
        logits = torch.empty((len(lens), vocab), dtype=torch.bfloat16, device="cuda")
        invd = torch.from_numpy(O.default_inv_freq(500000.0, d).astype(np.float32)).cuda()
        dv = case.dev
        B = len(lens)

        def run(s):
            gpu_lib.embed_tokens_bf16(embed.data_ptr(), ids.data_ptr(), hidden.data_ptr(), B, h,
                                      vocab, s)
            case.pool.decode_layers(first_layer=0, weights=[w[2] for w in ws],
                                    hidden_ptr=hidden.data_ptr(),
                                    block_tables_ptr=dv["bt"].data_ptr(),
                                    seq_lens_ptr=dv["sl"].data_ptr(),
                                    block_offsets_f16_ptr=dv["offs"].data_ptr(),
                                    inv_freq_ptr=invd.data_ptr(), batch=B, hidden_size=h,
                                    num_q_heads=hq, intermediate_size=inter,
                                    max_blocks_per_seq=case.mbps, rms_eps=1e-5, stream_ptr=s)
            gpu_lib.decode_logits_bf16(hidden.data_ptr(), fnorm.data_ptr(), head.data_ptr(),
                                       logits.data_ptr(), B, h, vocab, 1e-5, s)

        _check_replays(torch, run, lambda: [hidden, logits])
        # the appended K/V rows are the same bytes in every run
        mb = case.geometry["mapped_bytes"]
        regions = [memcpy_dtoh(case.pool.va_k(l), mb) for l in range(nl)]
        run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert all(np.array_equal(r, memcpy_dtoh(case.pool.va_k(l), mb))
                   for l, r in enumerate(regions))
    finally:
        case.pool.destroy()


@pytest.mark.parametrize("dtype", [KV_BF16, KV_FP8])
def test_attention_graph_replays(gpu_lib, dtype):
    import torch
    hq, hkv, d = 32, 8, 128
    lens = [2500, 1, 0, 1025, 4096, 37, 300, 2049]
    case = build_decode_case(gpu_lib, batch=len(lens), num_q_heads=hq, kv_heads=hkv, head_dim=d,
                             block_size=16, ctx_lens=lens, dtype=dtype, seed=4)
    try:
        dv = case.dev
        out = torch.empty((len(lens), hq, d), dtype=torch.bfloat16, device="cuda")

        def run(s):
            case.pool.paged_attn_decode(layer_idx=0, query_ptr=dv["q"].data_ptr(),
                                        out_ptr=out.data_ptr(), block_tables_ptr=dv["bt"].data_ptr(),
                                        seq_lens_ptr=dv["sl"].data_ptr(),
                                        block_offsets_f16_ptr=dv["offs"].data_ptr(),
                                        batch=len(lens), num_q_heads=hq, kv_heads=hkv, head_dim=d,
                                        block_size=16, max_blocks_per_seq=case.mbps,
                                        scale=1.0 / np.sqrt(d), stream_ptr=s)

        _check_replays(torch, run, lambda: [out])
    finally:
        case.pool.destroy()


def test_split_gemm_graph_replays(gpu_lib):
    import torch
    m, n, k = 64, 4096, 4096
    assert gpu_lib.gemm_plan(m, n, k)["splits"] > 1     # partials + the reduction kernel
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    r = torch.randn((m, n), generator=g, device="cuda").to(torch.bfloat16)
    y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")

    def run(s):
        gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), r.data_ptr(), y.data_ptr(), m, n, k, s)

    _check_replays(torch, run, lambda: [y])


def in_new_thread(test):
    """Runs a test in a thread of its own: workspaces belong to (stream, host
    thread), so every stream is a cold one there, whichever tests ran before."""
    @functools.wraps(test)
    def run(*args, **kw):
        with concurrent.futures.ThreadPoolExecutor(1) as ex:
            return ex.submit(test, *args, **kw).result()
    return run


class _KernelNode(C.Structure):   # hipKernelNodeParams
    _fields_ = [("block", C.c_uint32 * 3), ("extra", C.c_void_p), ("func", C.c_void_p),
                ("grid", C.c_uint32 * 3), ("params", C.c_void_p), ("shared", C.c_uint32)]


def _captured_kernels(run, warm=None):
    """(grid, block) of the kernels that run(stream) leaves in a graph captured on a
    stream which ran warm(stream) before."""
    h = hip()
    st = C.c_void_p()
    graph = C.c_void_p()
    n = C.c_size_t()
    assert h.hipStreamCreateWithFlags(C.byref(st), C.c_uint(1)) == 0
    try:
        if warm is not None:
            warm(st.value)
        assert h.hipStreamSynchronize(st) == 0
        assert h.hipStreamBeginCapture(st, C.c_int(1)) == 0
        try:
            run(st.value)
        finally:
            rc = h.hipStreamEndCapture(st, C.byref(graph))
        assert rc == 0
        assert h.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        nodes = (C.c_void_p * n.value)()
        assert h.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
        kernels = []
        for node in nodes:
            kp = _KernelNode()
            assert h.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(kp)) == 0
            kernels.append((tuple(kp.grid), tuple(kp.block)))
        assert h.hipGraphDestroy(graph) == 0
        return kernels
    finally:
        h.hipStreamDestroy(st)


def _scratch_free_work(torch, lib, what):
    """(run, run_more, output, close): a call that can run without scratch
    but takes some when run eagerly, and one that makes the stream's buffer
    of that slot grow."""
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    if what == "prefill":
        case = build_decode_case(lib, batch=2, num_q_heads=32, kv_heads=8, head_dim=128,
                                 block_size=16, ctx_lens=[4000, 900], dtype=KV_BF16, seed=3)
        q = torch.randn((300, 32, 128), generator=g, device="cuda").to(torch.bfloat16)
        out = torch.empty_like(q)
        dv = case.dev

        def prefill(lens, mbps):
            qsl = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32,
                               device="cuda")
            bt = dv["bt"][:, :mbps].contiguous()
            sl = torch.clamp(dv["sl"], max=mbps * 16)

            def run(s):
                case.pool.paged_attn_prefill(
                    layer_idx=0, query_ptr=q.data_ptr(), out_ptr=out.data_ptr(),
                    block_tables_ptr=bt.data_ptr(), seq_lens_ptr=sl.data_ptr(),
                    query_start_loc_ptr=qsl.data_ptr(), block_offsets_f16_ptr=dv["offs"].data_ptr(),
                    batch=2, total_query_tokens=int(sum(lens)), num_q_heads=32, kv_heads=8,
                    head_dim=128, block_size=16, max_blocks_per_seq=mbps,
                    scale=1 / np.sqrt(128), stream_ptr=s)
            return run

        return prefill([30, 20], 70), prefill([200, 100], 250), out[:50], case.pool.destroy
    m, n, k, fp8 = dict(uneven=(5, 320, 11008, False), uneven_fp8=(5, 320, 11008, True),
                        wide=(777, 6144, 4096, False))[what]
    assert lib.gemm_plan(m, n, k, fp8_weights=fp8)["splits"] > 1
    # the larger call: four times the rows, or the down projection (four splits of 777 x 4096)
    more = (777, 4096, 14336) if what == "wide" else (4 * m, n, k)
    x = torch.randn((more[0], more[2]), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn((more[1], more[2]), generator=g, device="cuda") * 0.02
    w = w.to(torch.float8_e4m3fn).view(torch.uint8) if fp8 else w.to(torch.bfloat16)
    scale = torch.full((n,), 0.5, device="cuda")
    y = torch.empty((max(m * n, more[0] * more[1]),), device="cuda", dtype=torch.bfloat16)

    def product(m, n, k):
        def run(s):
            if fp8:
                lib.gemm_fp8w_bf16(x.data_ptr(), w.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n,
                                   k, s)
            else:
                lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, s)
        return run

    return product(m, n, k), product(*more), y[:m * n], lambda: None


@pytest.mark.parametrize("what", ["prefill", "uneven", "uneven_fp8", "wide"])
@in_new_thread
def test_captures_hold_no_optional_scratch(gpu_lib, what):
    """Calls that can run without scratch do so under every capture, on a warm
    stream too: one kernel with the whole key range or K in each workgroup
    (grid.y 1), so that the graph holds no address of a buffer which a later,
    larger call on the stream frees.  The replays after such a call, and on
    another stream, equal those of a graph captured on a cold stream."""
    import torch
    run, run_more, out, close = _scratch_free_work(torch, gpu_lib, what)
    try:
        kernels = _captured_kernels(run, warm=run)
        assert len(kernels) == 1 and kernels[0][0][1] == 1, kernels
        graphs = []
        for warm in (False, True):
            st = torch.cuda.Stream()
            graph = torch.cuda.CUDAGraph()
            if warm:
                run(st.cuda_stream)
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=st):
                run(st.cuda_stream)
            graphs.append((graph, st))
        run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        eager = out.clone()
        run_more(graphs[1][1].cuda_stream)               # the slot grows
        torch.cuda.synchronize()
        seen = []
        for _ in range(2):
            for graph, _st in graphs:
                out.fill_(float("nan"))
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                seen.append(out.clone())
                run_more(torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
        assert all(torch.equal(s, seen[0]) for s in seen)
        # another order of the same fp32 sums, rounded to bf16
        d = (seen[0].double() - eager.double()).norm() / eager.double().norm()
        print(f"captured / eager {what}: {float(d):.2e}", flush=True)
        assert float(d) <= 1e-2
    finally:
        close()


@pytest.mark.parametrize("m,n,k,slot,kernels", [
    (777, 4096, 14336, 0, 1),    # both kernels split it (4 and 2 ways): unsplit on a cold stream
    (777, 6144, 4096, 0, 1),     # only the wide kernel splits it
    (300, 4096, 14336, 4, 2),    # the slot holds the tiled kernel's 4 splits, not the wide one's 8
    (300, 4096, 14336, 3, 1)])   # nor those
@in_new_thread
def test_wide_splits_under_capture(gpu_lib, tunables, m, n, k, slot, kernels):
    """A product whose split partials do not fit the stream's workspace is
    captured with fewer splits, or none, instead of allocating in the capture.
    Its replays equal each other and the float64 product (bound: fp32 sums of
    k products, 2^-24 each, and one rounding to bf16)."""
    import torch
    assert gpu_lib.gemm_plan(m, n, k)["splits"] > 1
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    y = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
    small = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)

    def run(s):
        gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, s)

    def warm(s):   # a slot of `slot` splits' partials (buffers get a quarter more than asked for)
        rows = m * slot // 4 * 4 // 5
        if slot == 0:
            return
        tunables.setenv("KCMM_GEMM_TILE", "9")
        tunables.setenv("KCMM_GEMM_SPLITS", "4")
        gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), small.data_ptr(), rows, n, k, s)
        tunables.delenv("KCMM_GEMM_TILE")
        tunables.delenv("KCMM_GEMM_SPLITS")

    assert len(_captured_kernels(run, warm)) == kernels
    st = torch.cuda.Stream()
    warm(st.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        run(st.cuda_stream)
    seen = []
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        seen.append(y.clone())
        run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    assert all(torch.equal(s, seen[0]) for s in seen)
    ref = x.double() @ w.double().t().contiguous()
    mag = x.double().abs() @ w.double().abs().t().contiguous()
    tol = k * 2.0 ** -24 * mag + 2.0 ** -8 * ref.abs() * 1.01
    for got in (seen[0], y):
        assert float(((got.double() - ref).abs() / tol).max()) <= 1.0


@pytest.mark.parametrize("dtype,ctx,tokens,waves", [
    (KV_BF16, [600] * 64, 4800, 1),      # 9728 (kv head, tile) entries, 76800 in the wide table
    (KV_FP8, [1456], 32768, 1),          # 368 and 8192
    (KV_FP8, [600] * 64, 4800, 8)])
def test_decode_workgroups_in_wide_tables(gpu_lib, dtype, ctx, tokens, waves):
    """A table wider than its sequences, as a server keeps it at its maximum
    length, gets the workgroups of a narrow one and the same result."""
    import torch
    case = build_decode_case(gpu_lib, batch=len(ctx), num_q_heads=32, kv_heads=8, head_dim=128,
                             block_size=16, ctx_lens=ctx, dtype=dtype, seed=len(ctx))
    try:
        dv = case.dev
        wide = torch.nn.functional.pad(dv["bt"], (0, tokens // 16 - case.mbps)).contiguous()
        seen = []
        for bt in (dv["bt"], wide):
            out = torch.full((len(ctx), 32, 128), float("nan"), dtype=torch.bfloat16, device="cuda")

            def run(s):
                case.pool.paged_attn_decode(layer_idx=0, query_ptr=dv["q"].data_ptr(),
                                            out_ptr=out.data_ptr(), block_tables_ptr=bt.data_ptr(),
                                            seq_lens_ptr=dv["sl"].data_ptr(),
                                            block_offsets_f16_ptr=dv["offs"].data_ptr(),
                                            batch=len(ctx), num_q_heads=32, kv_heads=8,
                                            head_dim=128, block_size=16,
                                            max_blocks_per_seq=bt.shape[1],
                                            scale=1.0 / np.sqrt(128), stream_ptr=s)

            assert _captured_kernels(run, warm=run)[0][1] == (64 * waves, 1, 1)
            run(torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            seen.append(out)
        assert torch.isfinite(seen[0].float()).all() and torch.equal(seen[0], seen[1])
    finally:
        case.pool.destroy()


@pytest.mark.parametrize("what", ["prefill", "uneven", "wide"])
def test_first_call_beside_another_threads_capture(gpu_lib, what):
    """A thread's first calls on its stream (its scratch grows twice), while another thread captures a
    graph (in the mode that forbids allocations on all threads): the scratch
    that it would take is no reason to fail or to break that capture."""
    import threading
    import torch
    run, run_more, out, close = _scratch_free_work(torch, gpu_lib, what)
    try:
        x = torch.zeros(64, device="cuda")
        (x + 1.0).sum()                                   # torch's kernels are loaded
        st, gs = torch.cuda.Stream(), torch.cuda.Stream()
        run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        want = out.clone()
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        failed = []
        run_more(torch.cuda.current_stream().cuda_stream)   # (every kernel is loaded)
        torch.cuda.synchronize()

        def first_call():
            try:
                for call in (run, run_more, run):
                    call(st.cuda_stream)
            except Exception as e:                        # noqa: BLE001 (re-raised below)
                failed.append(e)

        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=gs, capture_error_mode="global"):
            x.add_(1.0)
            t = threading.Thread(target=first_call)
            t.start()
            t.join()
            x.add_(1.0)
        assert not failed, failed
        torch.cuda.synchronize()
        for _ in range(3):
            graph.replay()
        torch.cuda.synchronize()
        assert float(x[0]) == 6.0
        d = (out.double() - want.double()).norm() / want.double().norm()
        assert float(d) <= 1e-2                           # (maybe in another order of the sums)
    finally:
        close()


@pytest.mark.parametrize("m,inter,k,wide", [(200, 64, 14336, False), (300, 512, 4096, False),
                                            (129, 2816, 8192, False), (777, 2816, 1024, True),
                                            (4096, 1024, 4096, True), (150, 14336, 4096, True)])
@in_new_thread
def test_swiglu_kernel_choice(gpu_lib, tunables, m, inter, k, wide):
    """Gate/up products above 128 tokens: few tiles of long rows take the
    weight-stream kernel with K splits (two kernels on a warm stream, the wide
    one under a capture without scratch), others the wide kernel; both against
    float64 (bound: the bf16 roundings of gate, up, silu and the product, and
    fp32 sums of k terms, through silu's slope of at most 1.1)."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(m + inter)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((2 * inter, k), generator=g, device="cuda") / k ** 0.5).to(torch.bfloat16)
    act = torch.full((m, inter), float("nan"), device="cuda", dtype=torch.bfloat16)

    def run(s):
        gpu_lib.gemm_bf16_swiglu(x.data_ptr(), w.data_ptr(), act.data_ptr(), m, inter, k, s)

    assert len(_captured_kernels(run)) == 1
    assert len(_captured_kernels(run, warm=run)) == (1 if wide else 2)
    gu = x.double() @ w.double().t().contiguous()
    mag = x.double().abs() @ w.double().abs().t().contiguous() * (k * 2.0 ** -24)
    gate, up = gu[:, :inter], gu[:, inter:]
    silu = torch.nn.functional.silu(gate)
    dg, du = (2.0 ** -8 * v.abs() + mag[:, i * inter:(i + 1) * inter] for i, v in enumerate((gate, up)))
    bound = ((1.1 * dg + 2.0 ** -8 * silu.abs()) * (up.abs() + du) + silu.abs() * du +
             2.0 ** -8 * (silu * up).abs()) * 1.05 + 1e-30
    for graph in (False, True):
        act.fill_(float("nan"))
        if graph:
            st = torch.cuda.Stream()
            cg = torch.cuda.CUDAGraph()
            torch.cuda.synchronize()
            with torch.cuda.graph(cg, stream=st):
                run(st.cuda_stream)
            cg.replay()
        else:
            run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        worst = float(((act.double() - silu * up).abs() / bound).max())
        print(f"swiglu {m}x{inter}x{k} graph={graph} worst {worst:.3f} of the bound", flush=True)
        assert worst <= 1.0
