"""Projection GEMM Y = X W^T (bf16, fp32 accumulate) on the GPU vs the
oracle (fp64) on small shapes and vs a torch fp32 matmul at the Llama-3-8B
decode shapes.  Tolerance: max|Y-ref| / max|ref| <= 1e-2 (bf16)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rel_err(got, ref):
    return float(np.abs(got - ref).max() / np.abs(ref).max())


@pytest.fixture(params=["tiled", "stream"])
def backend(request, tunables):
    """kcmm_gemm_bf16 runs products with M > 128 on the LDS-tiled MFMA
    kernel; KCMM_GEMM_TILED=0 keeps them on the weight-stream kernel.  Both
    are checked."""
    tunables.setenv("KCMM_GEMM_TILED", "1" if request.param == "tiled" else "0")
    return request.param


def run(gpu_lib, x, w):
    import torch
    m, k = x.shape
    n = w.shape[0]
    y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k,
                      torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (17, 192, 512), (64, 256, 1024),
                                   (100, 128, 768), (256, 320, 2048), (129, 192, 512),
                                   (300, 1024, 256), (513, 640, 1024)])
def test_vs_oracle(gpu_lib, backend, m, n, k):
    import torch
    if backend == "tiled" and m <= 128:
        pytest.skip("M <= 128 always runs the weight-stream kernel")
    rng = np.random.default_rng(m + n + k)
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    wb = O.encode(O.BF16, rng.standard_normal((n, k)) * 0.02)
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    w = torch.from_numpy(wb.view(np.int16)).view(torch.bfloat16).cuda()
    y = run(gpu_lib, x, w)
    got = O.decode(O.BF16, y.cpu().view(torch.int16).numpy().view(np.uint16))
    err = rel_err(got, O.gemm_bf16_f64(xb, wb))
    print(f"gemm {backend} {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("m", [64, 256])
@pytest.mark.parametrize("n,k", [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)])
def test_llama3_8b_projections(gpu_lib, backend, m, n, k):
    import torch
    if backend == "tiled" and m <= 128:
        pytest.skip("M <= 128 always runs the weight-stream kernel")
    g = torch.Generator(device="cuda")
    g.manual_seed(m * 7 + n + k)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    y = run(gpu_lib, x, w).float()
    ref = x.float() @ w.float().t()
    err = float((y - ref).abs().max() / ref.abs().max())
    print(f"gemm {backend} {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("target", ["1", "64", "256", "100000"])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (17, 384, 512), (33, 1280, 2304),
                                   (64, 256, 14336), (64, 6144, 4096), (48, 64, 1024)])
def test_split_k_choices(gpu_lib, tunables, target, m, n, k):
    """The K split chosen for a target workgroup count (1 = never split,
    100000 = as many splits as chunks allow) gives the same product: split
    partials and their reduction are exact up to fp32 rounding."""
    import torch
    tunables.setenv("KCMM_GEMM_WGS", target)
    g = torch.Generator(device="cuda")
    g.manual_seed(m * 31 + n + k + len(target))
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    y = run(gpu_lib, x, w).float()
    ref = x.float() @ w.float().t()
    err = float((y - ref).abs().max() / ref.abs().max())
    print(f"gemm target={target} {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("m,n,k", [(64, 16384, 1024), (1, 16384, 512), (100, 16384, 768),
                                   (64, 128256, 4096)])
@pytest.mark.parametrize("residual", [False, True])
def test_eight_wave_workgroups(gpu_lib, tunables, m, n, k, residual):
    """Unsplit plain products in 8-wave workgroups (KCMM_GEMM_WAVES=8: 128
    weight rows share one staged activation chunk; the last shape is the
    Llama-3-8B lm_head at the decode batch) give the same bits as 4-wave
    workgroups, each output being summed by one wave in the same k order;
    both against a torch fp32 product."""
    import torch
    assert gpu_lib.gemm_plan(m, n, k)["splits"] == 1
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k + residual)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    r = torch.randn((m, n), generator=g, device="cuda").to(torch.bfloat16)
    s = torch.cuda.current_stream().cuda_stream
    outs = {}
    for waves in ("4", "8"):
        tunables.setenv("KCMM_GEMM_WAVES", waves)
        if residual:
            y = r.clone()
            gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), y.data_ptr(), y.data_ptr(), m, n, k, s)
        else:
            y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, s)
        torch.cuda.synchronize()
        outs[waves] = y
    assert torch.equal(outs["4"], outs["8"])
    prod = x.float() @ w.float().t()
    ref = prod.to(torch.bfloat16).float() + r.float() if residual else prod
    err = float((outs["8"].float() - ref).abs().max() / ref.abs().max())
    print(f"8-wave gemm {m}x{n}x{k} residual={residual} err={err:.3e}", flush=True)
    assert err <= 1e-2


def test_eight_wave_swiglu(gpu_lib, tunables):
    """The fused gate/up + SwiGLU product at the Llama-3-8B decode shape
    (unsplit, 224 workgroups of 8 waves) gives the same bits as 4-wave
    workgroups; against silu(g)*u of a torch fp32 product.  (fp8 weights
    reach this kernel through the layer driver: tests/test_gpu_glue.py.)"""
    import torch
    m, inter, k = 64, 14336, 4096
    assert gpu_lib.gemm_plan(m, 2 * inter, k)["splits"] == 1
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((2 * inter, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    s = torch.cuda.current_stream().cuda_stream
    outs = {}
    for waves in ("4", "8"):
        tunables.setenv("KCMM_GEMM_WAVES", waves)
        act = torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device="cuda")
        gpu_lib.gemm_bf16_swiglu(x.data_ptr(), w.data_ptr(), act.data_ptr(), m, inter, k, s)
        torch.cuda.synchronize()
        outs[waves] = act
    assert torch.equal(outs["4"], outs["8"])
    gu = (x.float() @ w.float().t()).to(torch.bfloat16).float()
    gate, up = gu[:, :inter], gu[:, inter:]
    ref = (gate * torch.sigmoid(gate)).to(torch.bfloat16).float() * up
    err = float((outs["8"].float() - ref).abs().max() / ref.abs().max())
    print(f"8-wave swiglu err={err:.3e}", flush=True)
    assert err <= 1e-2


def test_eight_wave_workgroups_fp8_weights(gpu_lib, tunables):
    """The same for fp8-e4m3 weights (row scales applied in the store)."""
    import torch
    m, n, k = 64, 16384, 2048
    assert gpu_lib.gemm_plan(m, n, k, fp8_weights=True)["splits"] == 1
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    wf = torch.randn((n, k), generator=g, device="cuda") * 0.02
    sc = (wf.abs().amax(dim=1) / 448.0).clamp_min(1e-12)
    w8 = (wf / sc[:, None]).to(torch.float8_e4m3fn)
    s = torch.cuda.current_stream().cuda_stream
    outs = {}
    for waves in ("4", "8"):
        tunables.setenv("KCMM_GEMM_WAVES", waves)
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8.view(torch.uint8).data_ptr(), sc.data_ptr(),
                               y.data_ptr(), m, n, k, s)
        torch.cuda.synchronize()
        outs[waves] = y
    assert torch.equal(outs["4"], outs["8"])
    ref = x.float() @ (w8.float() * sc[:, None]).t()
    err = float((outs["8"].float() - ref).abs().max() / ref.abs().max())
    print(f"8-wave fp8w gemm {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("tile", [str(i) for i in range(11)])
@pytest.mark.parametrize("splits", ["1", "2", "4"])
@pytest.mark.parametrize("residual", [False, True])
def test_tiled_tiles_splits_residual(gpu_lib, tunables, tile, splits, residual):
    """Every configuration of the tiled kernel (tiles 128x256, 128x128,
    128x64, 64x128, 64x64, 128x256 on 4 waves, 256x128, 128x256 with 2
    stages) with 1, 2 or 4 K splits, M not a multiple of the tile, with and
    without a residual (in place: R == Y), against the fp64 oracle; two
    calls in a row give the same bits."""
    import torch
    tunables.setenv("KCMM_GEMM_TILE", tile)
    tunables.setenv("KCMM_GEMM_SPLITS", splits)
    m, n, k = 300, 768, 1024
    rng = np.random.default_rng(int(tile) * 10 + int(splits) + residual)
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    wb = O.encode(O.BF16, rng.standard_normal((n, k)) * 0.02)
    rb = O.encode(O.BF16, rng.standard_normal((m, n)))
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    w = torch.from_numpy(wb.view(np.int16)).view(torch.bfloat16).cuda()
    outs = []
    for _ in range(2):
        y = torch.from_numpy(rb.view(np.int16)).view(torch.bfloat16).cuda().clone()
        if residual:
            gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), y.data_ptr(), y.data_ptr(), m, n, k,
                                  torch.cuda.current_stream().cuda_stream)
        else:
            gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k,
                              torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs.append(y.cpu().view(torch.int16).numpy().view(np.uint16))
    assert np.array_equal(outs[0], outs[1])
    got = O.decode(O.BF16, outs[0]).astype(np.float64)
    prod = O.gemm_bf16_f64(xb, wb)
    ref = (O.decode(O.BF16, O.encode(O.BF16, prod)).astype(np.float64) +
           O.decode(O.BF16, rb)) if residual else prod
    err = rel_err(got, ref)
    print(f"tiled tile={tile} splits={splits} residual={residual} err={err:.3e}", flush=True)
    assert err <= 1e-2


def _fp8_weights(torch, rng, n, k, std):
    w8, s = O.quantize_fp8_rows(rng.standard_normal((n, k)).astype(np.float32) * std)
    return w8, s, torch.from_numpy(w8).cuda(), torch.from_numpy(s).cuda()


@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (17, 192, 512), (64, 256, 1024),
                                   (100, 128, 768), (129, 192, 512), (256, 640, 2048)])
def test_fp8_weights_vs_oracle(gpu_lib, m, n, k):
    """kcmm_gemm_fp8w_bf16: e4m3 weights with per-row scales against the fp64
    oracle (relative 1e-2, the bf16 output's tolerance); a second call gives
    the same bits."""
    import torch
    rng = np.random.default_rng(m * 3 + n + k)
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    w8, s, w8d, sd = _fp8_weights(torch, rng, n, k, 0.02)
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    outs = []
    for _ in range(2):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8d.data_ptr(), sd.data_ptr(), y.data_ptr(), m, n, k,
                               torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs.append(y.cpu().view(torch.int16).numpy().view(np.uint16))
    assert np.array_equal(outs[0], outs[1])
    got = O.decode(O.BF16, outs[0]).astype(np.float64)
    err = rel_err(got, O.gemm_fp8w_f64(xb, w8, s))
    print(f"fp8w gemm {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("m", [64, 128, 256])
@pytest.mark.parametrize("n,k", [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)])
def test_fp8_weights_llama3_8b_projections(gpu_lib, m, n, k):
    """The four Llama-3-8B projections with fp8 weights vs a torch fp32 product
    of the dequantized weights."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn((n, k), generator=g, device="cuda") * 0.02
    s = (w.abs().amax(dim=1) / 448.0).clamp_min(1e-30)
    w8 = (w / s[:, None]).to(torch.float8_e4m3fn)
    y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8.view(torch.uint8).data_ptr(), s.data_ptr(),
                           y.data_ptr(), m, n, k, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref = x.float() @ (w8.float() * s[:, None]).t()
    err = float((y.float() - ref).abs().max() / ref.abs().max())
    print(f"fp8w gemm {m}x{n}x{k} err={err:.3e}", flush=True)
    assert err <= 1e-2


@pytest.mark.parametrize("tile", [str(i) for i in range(11)])
@pytest.mark.parametrize("splits", ["1", "2", "4"])
def test_fp8_weights_tiled(gpu_lib, tunables, tile, splits):
    """fp8 weights with more than 128 tokens take the LDS-tiled kernel (codes
    staged in 64-byte LDS rows, converted to bf16 as they are read): every
    tiling with 1, 2 or 4 K splits, M not a multiple of the tile, against the
    fp64 oracle; two calls give the same bits; the weight-stream kernel
    (KCMM_GEMM_TILED=0) agrees within the same tolerance."""
    import torch
    tunables.setenv("KCMM_GEMM_TILE", tile)
    tunables.setenv("KCMM_GEMM_SPLITS", splits)
    m, n, k = 300, 768, 1024
    rng = np.random.default_rng(int(tile) * 10 + int(splits) + 5)
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    w8, s, w8d, sd = _fp8_weights(torch, rng, n, k, 0.02)
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    assert gpu_lib.gemm_plan(m, n, k, fp8_weights=True)["kernel"] == "tiled"
    outs = []
    for _ in range(2):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8d.data_ptr(), sd.data_ptr(), y.data_ptr(), m, n, k,
                               torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs.append(y.cpu().view(torch.int16).numpy().view(np.uint16))
    assert np.array_equal(outs[0], outs[1])
    got = O.decode(O.BF16, outs[0]).astype(np.float64)
    ref = O.gemm_fp8w_f64(xb, w8, s)
    err = rel_err(got, ref)
    print(f"fp8w tiled tile={tile} splits={splits} err={err:.3e}", flush=True)
    assert err <= 1e-2
    tunables.setenv("KCMM_GEMM_TILED", "0")
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8d.data_ptr(), sd.data_ptr(), y.data_ptr(), m, n, k,
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    stream = O.decode(O.BF16, y.cpu().view(torch.int16).numpy().view(np.uint16)).astype(np.float64)
    assert rel_err(stream, ref) <= 1e-2


@pytest.mark.parametrize("splits", ["1", "2", "4", "8"])
def test_fp8_weights_split_k(gpu_lib, tunables, splits):
    import torch
    tunables.setenv("KCMM_GEMM_SPLITS", splits)
    rng = np.random.default_rng(int(splits))
    m, n, k = 64, 512, 4096
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    w8, s, w8d, sd = _fp8_weights(torch, rng, n, k, 0.02)
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w8d.data_ptr(), sd.data_ptr(), y.data_ptr(), m, n, k,
                           torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = O.decode(O.BF16, y.cpu().view(torch.int16).numpy().view(np.uint16)).astype(np.float64)
    assert rel_err(got, O.gemm_fp8w_f64(xb, w8, s)) <= 1e-2


def test_workspace_two_host_threads(gpu_lib):
    """Two host threads launch split-K GEMMs on the same (null) stream with
    growing shapes: each thread has its own split-partial workspace, so one
    thread growing (and freeing) its buffer never frees the buffer the other
    is about to launch with.  Every product is checked."""
    import threading
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    shapes = [(64, n, 4096) for n in (256, 512, 1024, 2048, 3072)]
    data = {}
    for m, n, k in shapes:
        x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
        w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
        data[n] = (x, w, (x.float() @ w.float().t()))
    torch.cuda.synchronize()
    errors = []

    def worker(order):
        try:
            torch.cuda.set_device(0)
            for rep in range(3):
                for n in order:
                    x, w, ref = data[n]
                    y = torch.empty((64, n), dtype=torch.bfloat16, device="cuda")
                    gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), 64, n, 4096, 0)
                    torch.cuda.synchronize()
                    err = float((y.float() - ref).abs().max() / ref.abs().max())
                    if not err <= 1e-2:
                        errors.append((n, rep, err))
        except Exception as e:          # reported below
            errors.append(repr(e))

    ns = [n for _, n, _ in shapes]
    threads = [threading.Thread(target=worker, args=(ns,)),
               threading.Thread(target=worker, args=(ns[::-1],))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=120)
    assert not any(t.is_alive() for t in threads)
    assert errors == []


def test_gemm_plan(gpu_lib, tunables):
    """kcmm_gemm_plan reports what the product entry points run."""
    p = gpu_lib.gemm_plan(64, 6144, 4096)
    assert p["kernel"] == "stream" and p["tile"] == -1
    assert p["partial_bytes"] == (p["splits"] * 64 * 6144 * 4 if p["splits"] > 1 else 0)
    assert gpu_lib.gemm_plan(256, 6144, 4096)["kernel"] == "tiled"
    assert gpu_lib.gemm_plan(256, 6144, 4096, fp8_weights=True)["kernel"] == "tiled"
    assert gpu_lib.gemm_plan(128, 6144, 4096, fp8_weights=True)["kernel"] == "stream"
    tunables.setenv("KCMM_GEMM_SPLITS", "2")
    assert gpu_lib.gemm_plan(64, 512, 4096)["splits"] == 2
    tunables.setenv("KCMM_GEMM_TILED", "0")
    assert gpu_lib.gemm_plan(256, 6144, 4096)["kernel"] == "stream"
    with pytest.raises(Exception):
        gpu_lib.gemm_plan(64, 100, 4096)          # n not a multiple of 64


@pytest.mark.parametrize("tile", [101, 102, 103, 104, 124, 131])
@pytest.mark.parametrize("m,n,k,splits", [(129, 320, 256, 1), (257, 576, 256, 1), (320, 64, 512, 2),
                                          (513, 1344, 1024, 4), (700, 192, 512, 1)])
def test_wide_kernel(gpu_lib, tunables, tile, m, n, k, splits):
    """Every token-tile height of the wide kernel (KCMM_GEMM_TILE = 100 + fb0
    [+ 10 fb1 for the second half of the weight tiles]: 64 fb tokens, ragged
    last tiles of every height), weight tiles past N, the shortest K per
    split, the residual in place and the SwiGLU store.  Bound: bf16 rounding
    of the product (8 significant bits, to nearest: half a step of 2^-7, so
    2^-8 of it; twice with the residual) plus fp32 sums of k terms (2^-23 k
    sum|x||w|).  SwiGLU: the same bits as the plain product of
    [gate; up] followed by silu_mul (the same sum order per output)."""
    import torch
    tunables.setenv("KCMM_GEMM_TILE", str(tile))
    tunables.setenv("KCMM_GEMM_SPLITS", str(splits))
    plan = gpu_lib.gemm_plan(m, n, k)
    assert plan["tile"] == 100 + tile % 10 and plan["splits"] == splits
    rng = np.random.default_rng(m + n + k + tile)
    xb = O.encode(O.BF16, rng.standard_normal((m, k)))
    wb = O.encode(O.BF16, rng.standard_normal((2 * n, k)) * 0.02)
    rb = O.encode(O.BF16, rng.standard_normal((m, n)))
    x = torch.from_numpy(xb.view(np.int16)).view(torch.bfloat16).cuda()
    w = torch.from_numpy(wb.view(np.int16)).view(torch.bfloat16).cuda()
    y = torch.from_numpy(rb.view(np.int16)).view(torch.bfloat16).cuda()
    s = torch.cuda.current_stream().cuda_stream
    gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), y.data_ptr(), y.data_ptr(), m, n, k, s)
    z = run(gpu_lib, x, w[:n])
    prod = O.gemm_bf16_f64(xb, wb[:n])
    terms = k * 2.0 ** -23 * (np.abs(O.decode(O.BF16, xb)).astype(np.float64) @
                              np.abs(O.decode(O.BF16, wb[:n])).astype(np.float64).T)
    res = O.decode(O.BF16, rb).astype(np.float64)
    u = 2.0 ** -8
    for got, ref, bound in ((z, prod, u * np.abs(prod)),
                            (y, prod + res, u * (np.abs(prod) + np.abs(prod + res)) * (1 + u))):
        got = O.decode(O.BF16, got.cpu().view(torch.int16).numpy().view(np.uint16)).astype(np.float64)
        worst = float((np.abs(got - ref) / (bound + (1 + u) * terms + 1e-30)).max())
        print(f"wide {tile} {m}x{n}x{k}/{splits} worst {worst:.3f} of the bound", flush=True)
        assert np.isfinite(got).all() and worst <= 1.0
    if splits == 1:
        act = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        ref = torch.empty_like(act)
        gu = run(gpu_lib, x, w)
        gpu_lib.silu_mul_bf16(gu.data_ptr(), ref.data_ptr(), m, n, s)
        gpu_lib.gemm_bf16_swiglu(x.data_ptr(), w.data_ptr(), act.data_ptr(), m, n, k, s)
        torch.cuda.synchronize()
        assert torch.equal(act.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("m,n,k,wide", [(1, 98304, 4096, True), (16, 98304, 256, False),
                                        (17, 98304, 256, True), (64, 98240, 512, False),
                                        (64, 98368, 512, True), (65, 49152, 256, True),
                                        (65, 49088, 256, False), (128, 49216, 768, True)])
@pytest.mark.parametrize("residual", [False, True])
def test_long_weights(gpu_lib, tunables, m, n, k, wide, residual):
    """Both sides of the rule that gives decode-sized products over long
    weight matrices to the wide kernel: the same bits as the weight-stream
    kernel (KCMM_GEMM_TILED=0), each output being one sum in the same k
    order; the plan names the kernel that runs."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    r = torch.randn((m, n), generator=g, device="cuda").to(torch.bfloat16)
    s = torch.cuda.current_stream().cuda_stream
    outs = []
    for tiled in ("0", "1"):
        tunables.setenv("KCMM_GEMM_TILED", tiled)
        y = r.clone() if residual else torch.full_like(r, float("nan"))
        if residual:
            gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), y.data_ptr(), y.data_ptr(), m, n, k, s)
        else:
            gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, s)
        torch.cuda.synchronize()
        outs.append(y)
        plan = gpu_lib.gemm_plan(m, n, k)
        assert plan["kernel"] == ("tiled" if wide and tiled == "1" else "stream"), plan
        assert plan["splits"] == 1
    assert bool(torch.isfinite(outs[1].float()).all())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("m", [1, 17, 64, 128])
@pytest.mark.parametrize("n,k,fp8", [(128, 1792, False), (64, 2816, True), (320, 11008, False),
                                     (64, 5632, True), (1024, 4864, False),
                                     (5120, 3072, False), (8192, 2816, True)])
def test_uneven_splits(gpu_lib, tunables, m, n, k, fp8):
    """Where the divisors of the chunk count leave the chip empty, the last K
    split is shorter than the others: plain products, with and without a
    residual, against float64, within the fp32 rounding of k products summed
    in any order plus the bf16 roundings."""
    import torch
    plan = gpu_lib.gemm_plan(m, n, k, fp8_weights=fp8)
    chunk = 128 if m > 64 else 512 if fp8 and m <= 16 and k % 512 == 0 else 256
    per = -(-(k // chunk) // plan["splits"])
    assert plan["splits"] > 1 and (plan["splits"] - 1) * per < k // chunk
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    r = torch.randn((m, n), generator=g, device="cuda").to(torch.bfloat16)
    if fp8:
        w = torch.randint(0, 120, (n, k), generator=g, device="cuda", dtype=torch.uint8)
        scale = torch.rand(n, generator=g, device="cuda") * 0.01
        wd = w.cpu().view(torch.float8_e4m3fn).double() * scale.cpu().double()[:, None]
    else:
        w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
        wd = w.cpu().double()
    ref = x.cpu().double() @ wd.t()
    mag = x.cpu().double().abs() @ wd.abs().t()
    st = torch.cuda.current_stream().cuda_stream
    for residual in (0, 1):
        y = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
        want = ref
        if residual and fp8:
            continue
        if residual:
            gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), r.data_ptr(), y.data_ptr(), m, n, k, st)
            want = ref + r.cpu().double()
        elif fp8:
            gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n,
                                   k, st)
        else:
            gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, st)
        # fp32 sums of k products: at most k roundings of 2^-24 of the magnitude
        # sum; bf16: 2^-8 of each value rounded (the product, and its sum with
        # the residual)
        tol = k * 2.0 ** -24 * mag + 2.0 ** -8 * (want.abs() + residual * ref.abs()) * 1.01
        worst = float(((y.cpu().double() - want).abs() / tol).max())
        print(f"uneven {m}x{n}x{k} fp8={fp8} residual={residual} splits={plan['splits']} "
              f"worst {worst:.3f}", flush=True)
        assert worst <= 1.0


@pytest.mark.parametrize("fp8", [False, True])
def test_uneven_splits_under_capture(gpu_lib, fp8):
    """An unevenly split product captured on a stream that never ran it: the
    capture may not allocate the partials, so it runs unsplit; its replays
    equal each other and the eager split call up to fp32 rounding."""
    import torch
    m, n, k = 5, 320, 11008
    assert gpu_lib.gemm_plan(m, n, k, fp8_weights=fp8)["splits"] > 1
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randint(0, 120, (n, k), generator=g, device="cuda", dtype=torch.uint8) if fp8
         else (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16))
    scale = torch.full((n,), 1e-3, device="cuda")
    y = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)

    def run(sp):
        if fp8:
            gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w.data_ptr(), scale.data_ptr(), y.data_ptr(), m, n,
                                   k, sp)
        else:
            gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, sp)

    run(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    eager = y.double()
    graph = torch.cuda.CUDAGraph()
    st = torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=st):
        run(st.cuda_stream)
    seen = []
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        seen.append(y.clone())
        run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    assert all(torch.equal(s, seen[0]) for s in seen)
    # two fp32 sums of the same k products, each rounded to bf16 (2^-8)
    wd = w.cpu().view(torch.float8_e4m3fn).double() * 1e-3 if fp8 else w.cpu().double()
    mag = x.cpu().double().abs() @ wd.abs().t()
    tol = 2 * k * 2.0 ** -24 * mag + 2 * 2.0 ** -8 * eager.cpu().abs() * 1.01
    assert float(((seen[0].double() - eager).abs().cpu() / tol).max()) <= 1.0


@pytest.mark.parametrize("tile", ["100", "105", "110", "999"])
def test_tilings_that_do_not_exist_force_nothing(gpu_lib, tunables, tile):
    """KCMM_GEMM_TILE above 100 without a token-tile height of 1..4: plain and
    SwiGLU products run as with the variable unset."""
    import torch
    m, n, k = 130, 320, 512
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((2 * n, k), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    s = torch.cuda.current_stream().cuda_stream
    seen = []
    for value in (None, tile):
        if value:
            tunables.setenv("KCMM_GEMM_TILE", value)
        act = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
        gpu_lib.gemm_bf16_swiglu(x.data_ptr(), w.data_ptr(), act.data_ptr(), m, n, k, s)
        torch.cuda.synchronize()
        seen.append((act, run(gpu_lib, x, w), gpu_lib.gemm_plan(m, 2 * n, k)))
    assert torch.isfinite(seen[0][0].float()).all()
    assert torch.equal(seen[0][0], seen[1][0]) and torch.equal(seen[0][1], seen[1][1])
    assert seen[0][2] == seen[1][2]


@pytest.mark.parametrize("m,n,k", [(256, 320, 256), (1, 98304, 4096)])
def test_wide_kernel_special_values(gpu_lib, tunables, m, n, k):
    """NaN of any sign and payload, infinities and signed zeros in the
    residual, the tokens and the weights: the wide kernel's bits are the
    weight-stream kernel's (every NaN as 0x7fc0), in the residual and the
    SwiGLU stores."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    special = torch.tensor([0x7fc0, 0xffc1 - 65536, 0x7f81, 0xff93 - 65536, 0x7f80, 0xff80 - 65536,
                            0x8000 - 65536, 0x0001], dtype=torch.int16, device="cuda")

    def normal(shape, scale=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale).to(torch.bfloat16)

    def sprinkle(t, every):
        flat = t.view(torch.int16).view(-1)
        at = torch.arange(3, flat.numel(), every, device="cuda")
        flat[at] = special[torch.arange(at.numel(), device="cuda") % 8]
        return t

    s = torch.cuda.current_stream().cuda_stream
    x, w, r = normal((m, k)), normal((n, k), 0.02), sprinkle(normal((m, n)), 37)
    if m > 1:
        sprinkle(x[m // 2:], 8 * k + 5)   # some tokens and some weight rows
        sprinkle(w[n // 2:], 16 * k + 3)
        tunables.setenv("KCMM_GEMM_TILE", "104")
        tunables.setenv("KCMM_GEMM_SPLITS", "1")
    seen = []
    for tiled in ("0", "1"):
        tunables.setenv("KCMM_GEMM_TILED", tiled)
        y = r.clone()
        gpu_lib.gemm_bf16_add(x.data_ptr(), w.data_ptr(), y.data_ptr(), y.data_ptr(), m, n, k, s)
        act = torch.zeros((m, n // 2), dtype=torch.bfloat16, device="cuda")
        gpu_lib.gemm_bf16_swiglu(x.data_ptr(), w.data_ptr(), act.data_ptr(), m, n // 2, k, s)
        torch.cuda.synchronize()
        seen.append((y.view(torch.int16), act.view(torch.int16)))
    (y0, a0), (y1, a1) = seen
    print(f"special values {m}x{n}x{k}: {int((y0 != y1).sum())} and {int((a0 != a1).sum())} differ",
          flush=True)
    assert bool(y0.view(torch.bfloat16).isnan().any()) and bool((y0 == 0x7fc0).any())
    assert torch.equal(y0, y1) and torch.equal(a0, a1)


@pytest.mark.parametrize("m,n,k,fp8,splits", [
    (1, 4096, 11008, False, 4),      # 43 chunks, 64 tiles: uneven splits in one round
    (1, 11008, 11008, False, 1),     # 172 tiles: a second round would eat the gain
    (17, 9024, 768, True, 1),        # 3 chunks: the split sum costs more than it gains
    (32, 4416, 768, False, 1),
    (65, 384, 5120, True, 10),       # 14 uneven splits of 3 chunks against 10 of 4
    (65, 2048, 14336, False, 8),     # 8 splits meet the target: not the 7 below it
    (1, 5120, 3072, False, 3),       # 4 would go past it
    (2, 2048, 2048, True, 4)])       # 512-element chunks would leave 2
def test_split_rules(gpu_lib, m, n, k, fp8, splits):
    """Both sides of the rules that choose K splits, and a product with each
    against float64."""
    import torch
    assert gpu_lib.gemm_plan(m, n, k, fp8_weights=fp8)["splits"] == splits
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn((n, k), generator=g, device="cuda") * 0.02
    w = w.to(torch.float8_e4m3fn) if fp8 else w.to(torch.bfloat16)
    one = torch.ones(n, device="cuda")
    y = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    s = torch.cuda.current_stream().cuda_stream
    if fp8:
        gpu_lib.gemm_fp8w_bf16(x.data_ptr(), w.data_ptr(), one.data_ptr(), y.data_ptr(), m, n, k, s)
    else:
        gpu_lib.gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, s)
    ref = x.double() @ w.double().t().contiguous()
    mag = x.double().abs() @ w.double().abs().t().contiguous()
    tol = k * 2.0 ** -24 * mag + 2.0 ** -8 * ref.abs() * 1.01
    assert float(((y.double() - ref).abs() / tol).max()) <= 1.0
