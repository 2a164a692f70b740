"""The work that a serving program has this framework do, as measurable cases.

A program that serves a Llama-type model through libkcmm makes five kinds of
call, and every case here is one of them, through the public entry points of
lattice_amd.bindings:

  decode   paged decode attention of one layer (one new token per sequence);
  prefill  causal chunked-prefill attention of one layer over the same pages;
  append   a prompt chunk's (or a decode step's) K/V rows written into pages
           through device slot ids;
  gemm     one projection: plain, with the residual add, with SwiGLU in its
           store, or with residual add and RMSNorm; bf16 or fp8-e4m3 weights;
  step     a whole decode step: token embedding, decoder layers, final norm
           and lm_head to logits.

Shapes are those of this repository's configurations, tests and benchmark
(Llama-3-8B: 32/8 heads of 128, hidden 4096, intermediate 14336, vocabulary
128256; the smaller 64-wide-head shapes of the reference's own engine runs),
from one short sequence to the largest batches.  Page types: bf16, f16,
fp8-e4m3 with per-(page, head) scales, fp32.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from lattice_amd.bindings import (KV_BF16, KV_F16, KV_F32, KV_FP8, KcmmLayerWeights,
                                  KcmmLayerWeightsFp8, KcmmLibrary, make_config, memset_d8)
from lattice_amd.workload import (build_decode_case, build_prefix_shared_case, elem_bytes,
                                  rope_inv_freq, torch_io_dtype)

DTYPES = {"bf16": KV_BF16, "f16": KV_F16, "fp8": KV_FP8, "f32": KV_F32}
# hidden, intermediate, q heads, kv heads, head_dim, vocabulary
MODELS = {
    "8b": (4096, 14336, 32, 8, 128, 128256),     # the benchmark's model
    "1b": (2048, 8192, 32, 8, 64, 32000),        # a 64-wide-head model
    "small": (1024, 2816, 16, 4, 64, 32000),     # the reference's own engine run: 1024, 16/4, 64
}
EPS = 1e-5
THETA = 500000.0


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # one user's chat turn: the shortest call, launches and latency count
        dict(name="decode_one_short", kind="decode", dtype="bf16", batch=1, hq=32, hkv=8, d=128,
             bs=16, lo=700, hi=900, tail=0, lens=1),
        # the reference configuration's oracle shape: fp32 pages, 8 heads of 64
        dict(name="decode_f32_small", kind="decode", dtype="f32", batch=4, hq=8, hkv=8, d=64,
             bs=16, lo=2, hi=513, tail=0, lens=2),
        # the headline batch: 64 sequences, context 512..4096 plus the new token
        dict(name="decode_batch64", kind="decode", dtype="bf16", batch=64, hq=32, hkv=8, d=128,
             bs=16, lo=513, hi=4097, tail=0, lens=3),
        # two long documents on an f16 pool: few sequences, many pages each
        dict(name="decode_long_f16", kind="decode", dtype="f16", batch=2, hq=32, hkv=8, d=128,
             bs=16, lo=24001, hi=49999, tail=0, lens=4),
        # beam-search sized batch on fp8 pages, long-tailed contexts
        dict(name="decode_batch128_fp8", kind="decode", dtype="fp8", batch=128, hq=32, hkv=8,
             d=128, bs=16, lo=1024, hi=8192, tail=1, lens=5),
        # 16 requests behind one shared 1024-token prefix, 256 tokens each
        dict(name="prefill_shared_prefix", kind="prefill", dtype="bf16", batch=16, hq=32, hkv=8,
             d=128, bs=16, prefix=1024, lo=256, hi=256, lens=6, shared=1),
        # ragged prompts on fp8 pages, the later chunk of each
        dict(name="prefill_ragged_fp8", kind="prefill", dtype="fp8", batch=3, hq=32, hkv=8,
             d=128, bs=16, prefix=1111, lo=300, hi=1900, lens=7, shared=0),
        # the same prompts' K/V going into fp8 pages
        dict(name="append_prompt_fp8", kind="append", dtype="fp8", batch=3, hkv=8, d=128, bs=16,
             first=0, lo=300, hi=1900, lens=7),
        # gate/up of a 2048-token prompt chunk, SwiGLU in the store
        dict(name="gemm_swiglu_2048", kind="gemm", op="swiglu", weights="bf16", m=2048, n=14336,
             k=4096),
        # down projection with its residual for a ragged few hundred tokens
        dict(name="gemm_down_add_777", kind="gemm", op="add", weights="bf16", m=777, n=4096,
             k=14336),
        # a whole decode step of a full batch (two of the model's layers, and its head)
        dict(name="step_batch64", kind="step", model="8b", weights="bf16", dtype="bf16", batch=64,
             layers=2, lo=512, hi=2048, lens=8),
        # a whole decode step of one sequence with fp8 weights and pages
        dict(name="step_one_fp8", kind="step", model="8b", weights="fp8", dtype="fp8", batch=1,
             layers=2, lo=1024, hi=2048, lens=9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


HEADS = [(32, 8, 128), (32, 8, 64), (16, 4, 64), (8, 8, 64), (32, 4, 128), (16, 8, 128)]


def draw(rng):
    """One more case: the kind as often as it is listed, sizes over the log
    of their range, contexts ragged."""
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 2 + ["append"] + ["gemm"] * 4 + ["step"] * 2)
    lens = rng.randrange(1 << 30)
    if kind == "decode":
        dtype = rng.choice(["bf16", "bf16", "f16", "fp8", "f32"])
        hq, hkv, d = rng.choice(HEADS)
        if dtype == "fp8":
            d = 128
        if dtype == "f32":
            hq, hkv, d = 8, 8, 64
        batch = _log_int(rng, 1, 8 if dtype == "f32" else 128)
        most = 1024 if dtype == "f32" else 400_000   # tokens over the batch
        hi = _log_int(rng, 32, min(32768, most // batch))
        return dict(kind=kind, dtype=dtype, batch=batch, hq=hq, hkv=hkv, d=d,
                    bs=rng.choice([16, 16, 32]), lo=max(1, hi // 4), hi=hi, tail=0, lens=lens)
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "f16", "fp8"])
        hq, hkv, d = rng.choice(HEADS)
        if dtype == "fp8":
            d = 128
        batch = _log_int(rng, 1, 16)
        hi = _log_int(rng, 16, 4096 // batch)
        return dict(kind=kind, dtype=dtype, batch=batch, hq=hq, hkv=hkv, d=d,
                    bs=rng.choice([16, 16, 32]), prefix=rng.choice([0, _log_int(rng, 16, 2048)]),
                    lo=max(1, hi // 4), hi=hi, lens=lens, shared=0)
    if kind == "append":
        batch = _log_int(rng, 1, 128)
        hi = _log_int(rng, 1, max(1, 4096 // batch))
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16", "fp8", "fp8"]), batch=batch,
                    hkv=8, d=128, bs=rng.choice([16, 16, 32]),
                    first=rng.choice([0, rng.randrange(1, 200)]), lo=max(1, hi // 4), hi=hi,
                    lens=lens)
    if kind == "gemm":
        hidden, inter, hq, hkv, d, _ = MODELS[rng.choice(["8b", "8b", "1b", "small"])]
        op = rng.choice(["plain", "add", "swiglu", "add_rmsnorm"])
        weights = rng.choice(["bf16", "bf16", "fp8"]) if op == "plain" else "bf16"
        if op == "plain":
            n, k = rng.choice([((hq + 2 * hkv) * d, hidden), (2 * inter, hidden), (hidden, inter)])
        elif op == "add":
            n, k = rng.choice([(hidden, hq * d), (hidden, inter)])
        elif op == "swiglu":
            n, k = inter, hidden
        else:
            n, k = hidden, hq * d
        return dict(kind=kind, op=op, weights=weights, m=_log_int(rng, 1, 2048), n=n, k=k)
    weights = rng.choice(["bf16", "bf16", "fp8"])
    model = rng.choice(["8b", "1b", "small"])
    dtype = rng.choice(["bf16", "fp8"]) if model == "8b" else "bf16"
    hi = _log_int(rng, 32, 2048)
    return dict(kind="step", model=model, weights=weights, dtype=dtype,
                batch=_log_int(rng, 1, 64), layers=2, lo=max(1, hi // 4), hi=hi, lens=lens)


def _lens(case):
    """The sequences' lengths: uniform in [lo, hi]; tail: one in five long
    (16384..32768), as a beam-search service sees them."""
    r = np.random.default_rng(case["lens"])
    n = r.integers(case["lo"], case["hi"] + 1, size=case["batch"])
    if case.get("tail"):
        n = np.where(r.random(case["batch"]) < 0.2, r.integers(16384, 32769, size=case["batch"]), n)
    return n.astype(np.int64)


# ---- inputs ------------------------------------------------------------------------------------

_lib = None


def _library():
    global _lib
    if _lib is None:
        _lib = KcmmLibrary()
    return _lib


class _Pool:
    """Frees the pool's memory with the state that holds it."""

    def __init__(self, pool):
        self.pool = pool

    def __del__(self):
        self.pool.destroy()


class _Region:
    """Device memory of the pool, for torch to see it in place.  The tensor
    made from it keeps it, and with it the pool, alive."""

    def __init__(self, owner, ptr, nbytes):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1",
                                         "data": (ptr, False), "version": 3}


def _region(owner, ptr, nbytes):
    return torch.as_tensor(_Region(owner, ptr, nbytes), device="cuda")


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, scale=1.0, dtype=torch.bfloat16):
    """N(0, scale), made in pieces (a float32 copy of the whole would be twice its size)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 26):
        m = min(1 << 26, flat.numel() - i)
        flat[i:i + m] = (torch.randn(m, generator=g, device="cuda") * scale).to(dtype)
    return out


def _quantize_rows(w):
    """fp8-e4m3 codes and one fp32 scale per row (amax / 448)."""
    codes = torch.empty(w.shape, dtype=torch.uint8, device="cuda")
    scale = torch.empty(w.shape[0], dtype=torch.float32, device="cuda")
    for i in range(0, w.shape[0], 16384):
        x = w[i:i + 16384].float()
        s = x.abs().amax(dim=1) / 448.0
        codes[i:i + 16384] = (x / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8)
        scale[i:i + 16384] = s
    return codes, scale


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _attention_args(c, q, out):
    dev = c.dev
    return dict(query_ptr=q.data_ptr(), out_ptr=out.data_ptr(),
                block_tables_ptr=dev["bt"].data_ptr(),
                block_offsets_f16_ptr=dev["offs"].data_ptr(), num_q_heads=c.num_q_heads,
                kv_heads=c.kv_heads, head_dim=c.head_dim, block_size=c.block_size,
                max_blocks_per_seq=c.mbps, scale=1.0 / math.sqrt(c.head_dim))


def _prepare_decode(case, seed):
    c = build_decode_case(_library(), batch=case["batch"], num_q_heads=case["hq"],
                          kv_heads=case["hkv"], head_dim=case["d"], block_size=case["bs"],
                          ctx_lens=_lens(case), dtype=DTYPES[case["dtype"]], seed=seed,
                          host_mirror=False)
    args = _attention_args(c, c.dev["q"], c.dev["out"])
    return dict(kind="decode", case=c, keep=_Pool(c.pool), pool=c.pool, out=c.dev["out"],
                args=dict(args, layer_idx=0, seq_lens_ptr=c.dev["sl"].data_ptr(),
                          batch=case["batch"]))


def _prepare_prefill(case, seed):
    dtype = DTYPES[case["dtype"]]
    chunk = _lens(case)
    if case["shared"]:
        c = build_prefix_shared_case(_library(), batch=case["batch"], prefix_tokens=case["prefix"],
                                     suffix_tokens=case["lo"], chunk=case["lo"],
                                     num_q_heads=case["hq"], kv_heads=case["hkv"],
                                     head_dim=case["d"], block_size=case["bs"], dtype=dtype,
                                     seed=seed)
        qsl, q, out = c.dev["qsl"], c.dev["q"], c.dev["out"]
        rows = int(c.qsl[-1])
    else:
        c = build_decode_case(_library(), batch=case["batch"], num_q_heads=case["hq"],
                              kv_heads=case["hkv"], head_dim=case["d"], block_size=case["bs"],
                              ctx_lens=chunk + case["prefix"], dtype=dtype, seed=seed,
                              host_mirror=False)
        rows = int(chunk.sum())
        qsl = torch.from_numpy(np.concatenate([[0], np.cumsum(chunk)]).astype(np.int32)).cuda()
        q = _randn(_generator(seed + 1), (rows, case["hq"], case["d"]), dtype=torch_io_dtype(dtype))
        out = torch.zeros_like(q)
    args = _attention_args(c, q, out)
    return dict(kind="prefill", case=c, keep=_Pool(c.pool), pool=c.pool, out=out, q=q, qsl=qsl,
                args=dict(args, layer_idx=0, seq_lens_ptr=c.dev["sl"].data_ptr(),
                          query_start_loc_ptr=qsl.data_ptr(), batch=case["batch"],
                          total_query_tokens=rows, stream_ptr=_stream()))


def _prepare_append(case, seed):
    dtype = DTYPES[case["dtype"]]
    bs, lens = case["bs"], _lens(case)
    total = lens + case["first"]
    pages = -(-total // bs)
    cfg = make_config(num_layers=1, kv_heads=case["hkv"], head_dim=case["d"],
                      max_batch=case["batch"], max_seq_len=int(total.max()), block_size=bs)
    pool = _library().create_pool(cfg, dtype)
    ids = np.random.default_rng(seed).permutation(np.asarray(pool.alloc_blocks(int(pages.sum()))))
    slots, at = [], 0
    for n, t, p in zip(lens, total, pages):
        table = ids[at:at + p]
        at += p
        pool.update_seq_len(pool.register_sequence(table.tolist()), int(t))
        pos = np.arange(case["first"], t)
        slots.append(table[pos // bs] * bs + pos % bs)
    nbytes = pool.stats()["superblock_count"] * 2 * 1024 * 1024
    for base in (pool.va_k(0), pool.va_v(0)):
        memset_d8(base, 0, nbytes)
    g = _generator(seed)
    row = (int(lens.sum()), case["hkv"] * case["d"])
    src = torch_io_dtype(dtype)
    dev = dict(slots=torch.from_numpy(np.concatenate(slots).astype(np.int64)).cuda(),
               offs=torch.from_numpy(np.asarray(pool.all_block_offsets_f16(), dtype=np.uint64)
                                     .view(np.int64)).cuda(),
               valid=torch.from_numpy(np.asarray(pool.all_block_valid_flags(), np.uint8)).cuda(),
               status=torch.zeros(1, dtype=torch.int32, device="cuda"),
               k=_randn(g, row, dtype=src), v=_randn(g, row, dtype=src))
    args = dict(layer_idx=0, slot_mapping_ptr=dev["slots"].data_ptr(),
                block_offsets_f16_ptr=dev["offs"].data_ptr(),
                valid_blocks_ptr=dev["valid"].data_ptr(),
                block_offsets_f16_len=dev["offs"].numel(), batch=row[0],
                k_src_ptr=dev["k"].data_ptr(), v_src_ptr=dev["v"].data_ptr(),
                status_ptr=dev["status"].data_ptr(), stream_ptr=_stream())
    keep = _Pool(pool)
    return dict(kind="append", keep=keep, pool=pool, dev=dev, args=args,
                out=dict(k=_region(keep, pool.va_k(0), nbytes),
                         v=_region(keep, pool.va_v(0), nbytes), status=dev["status"]))


def _prepare_gemm(case, seed):
    g = _generator(seed)
    m, n, k, op = case["m"], case["n"], case["k"], case["op"]
    s = dict(kind="gemm", op=op, m=m, n=n, k=k, lib=_library(), x=_randn(g, (m, k)),
             y=torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), fp8=None)
    w = _randn(g, (2 * n if op == "swiglu" else n, k), 0.02)
    if case["weights"] == "fp8":
        s["w"], s["fp8"] = _quantize_rows(w)
    else:
        s["w"] = w
    if op in ("add", "add_rmsnorm"):
        s["r"] = _randn(g, (m, n))
    if op == "add_rmsnorm":
        # the call adds into the hidden state in place: every pass starts from
        # its own rows, as the attention before it leaves them to the model
        s["norm"] = (1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")).to(torch.bfloat16)
        s["hidden"] = s["r"].clone()
    return s


def _prepare_step(case, seed):
    hidden, inter, hq, hkv, d, vocab = MODELS[case["model"]]
    dtype, fp8w = DTYPES[case["dtype"]], case["weights"] == "fp8"
    c = build_decode_case(_library(), batch=case["batch"], num_q_heads=hq, kv_heads=hkv,
                          head_dim=d, block_size=16, ctx_lens=_lens(case), dtype=dtype,
                          num_layers=case["layers"], seed=seed, host_mirror=False)
    g = _generator(seed + 1)
    shapes = dict(qkv=((hq + 2 * hkv) * d, hidden), o=(hidden, hq * d), gate_up=(2 * inter, hidden),
                  down=(hidden, inter))
    layers, structs = [], []
    for _ in range(case["layers"]):
        w = {}
        for name, shape in shapes.items():
            w[name] = _randn(g, shape, 0.02)
            if fp8w:
                w[name], w[name + "_scale"] = _quantize_rows(w[name])
        for name in ("attn_norm", "mlp_norm"):
            w[name] = (1.0 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(torch.bfloat16)
        layers.append(w)
        kind = KcmmLayerWeightsFp8 if fp8w else KcmmLayerWeights
        structs.append(kind(**{name: t.data_ptr() for name, t in w.items()}))
    batch = case["batch"]
    dev = dict(embed=_randn(g, (vocab, hidden)), head=_randn(g, (vocab, hidden), 0.02),
               norm=(1.0 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(torch.bfloat16),
               ids=torch.randint(0, vocab, (batch,), generator=g, device="cuda", dtype=torch.int32),
               inv=torch.from_numpy(rope_inv_freq(THETA, d)).cuda(),
               hidden=torch.zeros((batch, hidden), dtype=torch.bfloat16, device="cuda"),
               logits=torch.zeros((batch, vocab), dtype=torch.bfloat16, device="cuda"))
    nbytes, keep = c.geometry["mapped_bytes"], _Pool(c.pool)
    out = dict(logits=dev["logits"], hidden=dev["hidden"])
    for i in range(case["layers"]):
        for name, base in (("k%d" % i, c.pool.va_k(i)), ("v%d" % i, c.pool.va_v(i))):
            r = _region(keep, base, nbytes)
            out[name] = r if dtype == KV_FP8 else r.view(torch_io_dtype(dtype))
    args = dict(first_layer=0, weights=structs, hidden_ptr=dev["hidden"].data_ptr(),
                block_tables_ptr=c.dev["bt"].data_ptr(), seq_lens_ptr=c.dev["sl"].data_ptr(),
                block_offsets_f16_ptr=c.dev["offs"].data_ptr(), inv_freq_ptr=dev["inv"].data_ptr(),
                batch=batch, hidden_size=hidden, num_q_heads=hq, intermediate_size=inter,
                max_blocks_per_seq=c.mbps, rms_eps=EPS, stream_ptr=_stream())
    return dict(kind="step", lib=_library(), case=c, keep=keep, pool=c.pool,
                layers=layers, dev=dev, args=args, out=out, fp8w=fp8w, vocab=vocab)


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "append": _prepare_append,
            "gemm": _prepare_gemm, "step": _prepare_step}[case["kind"]](case, seed)


# ---- one pass ----------------------------------------------------------------------------------

def _run_gemm(s):
    lib, m, n, k, st = s["lib"], s["m"], s["n"], s["k"], _stream()
    x, w, y = s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr()
    if s["op"] == "add":
        lib.gemm_bf16_add(x, w, s["r"].data_ptr(), y, m, n, k, st)
    elif s["op"] == "swiglu":
        lib.gemm_bf16_swiglu(x, w, y, m, n, k, st)
    elif s["op"] == "add_rmsnorm":
        s["hidden"].copy_(s["r"])
        lib.gemm_bf16_add_rmsnorm(x, w, s["hidden"].data_ptr(), s["norm"].data_ptr(), y, m, n, k,
                                  EPS, st)
        return [s["y"], s["hidden"]]
    elif s["fp8"] is not None:
        lib.gemm_fp8w_bf16(x, w, s["fp8"].data_ptr(), y, m, n, k, st)
    else:
        lib.gemm_bf16(x, w, y, m, n, k, st)
    return s["y"]


def _run_step(s):
    lib, dev, a = s["lib"], s["dev"], s["args"]
    b, h = a["batch"], a["hidden_size"]
    hid = dev["hidden"].data_ptr()
    lib.embed_tokens_bf16(dev["embed"].data_ptr(), dev["ids"].data_ptr(), hid, b, h, s["vocab"],
                          a["stream_ptr"])
    (s["pool"].decode_layers_fp8w if s["fp8w"] else s["pool"].decode_layers)(**a)
    lib.decode_logits_bf16(hid, dev["norm"].data_ptr(), dev["head"].data_ptr(),
                           dev["logits"].data_ptr(), b, h, s["vocab"], EPS, a["stream_ptr"])
    return s["out"]


def run(state):
    kind = state["kind"]
    if kind == "gemm":
        return _run_gemm(state)
    if kind == "step":
        return _run_step(state)
    if kind == "decode":
        state["pool"].paged_attn_decode(stream_ptr=_stream(), **state["args"])
    elif kind == "prefill":
        state["pool"].paged_attn_prefill(**state["args"])
    else:
        state["pool"].append_kv_device_slots_on_stream(**state["args"])
    return state["out"]


# ---- what a pass cannot do without -------------------------------------------------------------

def _kv_token_bytes(hkv, d, dtype, bs):
    """K and V bytes of one token of one layer (fp8: with its share of the page's scales)."""
    return 2 * hkv * (d * elem_bytes(dtype) + (4 / bs if dtype == KV_FP8 else 0))


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        rows = 2 * n if case["op"] == "swiglu" else n
        rw = {"plain": 1, "swiglu": 1, "add": 2, "add_rmsnorm": 3}[case["op"]]
        weight = rows * k * (1 if case["weights"] == "fp8" else 2)
        return dict(bytes=weight + 2 * m * k + 2 * rw * m * n, flops=2 * m * rows * k)
    n = _lens(case)
    if kind == "step":
        hidden, inter, hq, hkv, d, vocab = MODELS[case["model"]]
        per = (hq + 2 * hkv) * d * hidden + hidden * hq * d + 3 * hidden * inter
        kv = _kv_token_bytes(hkv, d, DTYPES[case["dtype"]], 16) * int(n.sum())
        wb = 1 if case["weights"] == "fp8" else 2
        b = case["batch"]
        return dict(bytes=case["layers"] * (per * wb + kv) + 2 * vocab * hidden + 2 * b * vocab +
                    4 * b * hidden,
                    flops=2 * b * (case["layers"] * per + vocab * hidden) +
                    case["layers"] * 4 * hq * d * int(n.sum()))
    dtype = DTYPES[case["dtype"]]
    tok = _kv_token_bytes(case["hkv"], case["d"], dtype, case["bs"])
    if kind == "append":
        src = 2 * case["hkv"] * case["d"] * (2 if dtype == KV_FP8 else elem_bytes(dtype))
        return dict(bytes=int(n.sum()) * (src + tok + 8), flops=0)
    io = 2 * case["hq"] * case["d"] * (4 if dtype == KV_F32 else 2)
    if kind == "decode":
        return dict(bytes=int(n.sum()) * tok + case["batch"] * io,
                    flops=4 * case["hq"] * case["d"] * int(n.sum()))
    kv_tokens = case["prefix"] + int(n.sum()) if case["shared"] else int((n + case["prefix"]).sum())
    keys = sum(int(x) * case["prefix"] + int(x) * (int(x) + 1) // 2 for x in n)
    return dict(bytes=kv_tokens * tok + int(n.sum()) * io, flops=4 * case["hq"] * case["d"] * keys)


def tolerance(case):
    """About four times what the path and its 64-bit form differ by."""
    kind = case["kind"]
    if kind == "append":
        return "exact"           # bytes
    if kind == "decode":
        return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "fp8": 1e-2, "f32": 4e-6}[case["dtype"]]}
    if kind == "prefill":
        return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "fp8": 1.4e-2}[case["dtype"]]}
    if kind == "gemm":
        return {"rel": 1e-2 if case["op"] == "swiglu" else 8e-3}
    # two bf16 layers and the head; fp8 page codes may fall to a neighbour
    return {"rel": 3e-2, "max": 0.9, "differ": 1e-3}


# ---- the same in 64 bits -----------------------------------------------------------------------

def _pages(base, c, table, length):
    """[length][hkv][d] in float64: the tokens of one sequence, from its pages."""
    st = c.pool.stats()
    bb, nsb = st["block_bytes"], st["superblock_count"]
    raw = _region(c, base, nsb * 2 * 1024 * 1024)
    n = -(-length // c.block_size)
    off = torch.from_numpy(c.offsets_f16[table[:n]].astype(np.int64) * 2).cuda()
    idx = off[:, None] + torch.arange(bb, device="cuda")[None, :]
    page = raw[idx]
    eb = elem_bytes(c.dtype)
    data = c.block_size * c.kv_heads * c.head_dim * eb
    x = page[:, :data].contiguous()
    shape = (n, c.block_size, c.kv_heads, c.head_dim)
    if c.dtype == KV_FP8:
        x = x.view(torch.float8_e4m3fn).to(torch.float64).view(shape)
        scale = page[:, data:data + 4 * c.kv_heads].contiguous().view(torch.float32).double()
        x = x * scale[:, None, :, None]
    else:
        x = x.view(torch_io_dtype(c.dtype)).double().view(shape)
    return x.reshape(-1, c.kv_heads, c.head_dim)[:length]


def _attend(q, k, v, positions):
    """q [n][hq][d] at the given positions over keys 0..position, float64."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.empty_like(q)
    late = torch.arange(k.shape[0], device="cuda")[None, :] > positions[:, None]
    for h in range(hq):
        g = h * hkv // hq
        s = q[:, h].contiguous() @ k[:, g].t().contiguous() / math.sqrt(d)
        s.masked_fill_(late, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ v[:, g].contiguous()
    return out


def _rmsnorm(x, w):
    return w.double() * x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _weight(w, name):
    if name + "_scale" in w:
        return w[name].view(torch.float8_e4m3fn).to(torch.float64) * w[name + "_scale"].double()[:, None]
    return w[name].double()


def _product(x, w):
    return x @ w.t().contiguous()


def _exact_step(s):
    c, dev, a = s["case"], s["dev"], s["args"]
    b, d, hq, hkv = a["batch"], c.head_dim, c.num_q_heads, c.kv_heads
    inter = a["intermediate_size"]
    x = dev["embed"][dev["ids"].long()].double()
    pos = torch.from_numpy(c.seq_lens.astype(np.int64) - 1).cuda()
    ang = pos.double()[:, None] * dev["inv"].double()[None, :]
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def rope(t):
        u, v = t[..., :d // 2], t[..., d // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], dim=-1)

    for i, w in enumerate(s["layers"]):
        qkv = _product(_rmsnorm(x, w["attn_norm"]), _weight(w, "qkv")).view(b, hq + 2 * hkv, d)
        q, k, v = rope(qkv[:, :hq]), rope(qkv[:, hq:hq + hkv]), qkv[:, hq + hkv:]
        att = torch.empty_like(q)
        for j in range(b):
            n = int(c.seq_lens[j])
            keys = _pages(c.pool.va_k(i), c, c.block_tables[j], n)
            vals = _pages(c.pool.va_v(i), c, c.block_tables[j], n)
            keys[n - 1], vals[n - 1] = k[j], v[j]
            att[j:j + 1] = _attend(q[j:j + 1], keys, vals, pos[j:j + 1])
        x = x + _product(att.reshape(b, hq * d), _weight(w, "o"))
        gu = _product(_rmsnorm(x, w["mlp_norm"]), _weight(w, "gate_up"))
        act = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
        x = x + _product(act, _weight(w, "down"))
    out = {name: None for name in s["out"]}
    return dict(out, hidden=x, logits=_product(_rmsnorm(x, dev["norm"]), dev["head"].double()))


def exact(case, seed):
    if case["kind"] == "append":
        return None              # bytes: the page writer's own encoding
    s = prepare(case, seed)
    if case["kind"] == "gemm":
        w = _weight(dict(w=s["w"], w_scale=s["fp8"]) if s["fp8"] is not None else dict(w=s["w"]), "w")
        y = _product(s["x"].double(), w)
        if case["op"] == "swiglu":
            return torch.nn.functional.silu(y[:, :s["n"]]) * y[:, s["n"]:]
        if case["op"] in ("add", "add_rmsnorm"):
            y = y + s["r"].double()
        return [_rmsnorm(y, s["norm"]), y] if case["op"] == "add_rmsnorm" else y
    if case["kind"] == "step":
        return _exact_step(s)
    c = s["case"]
    if case["kind"] == "decode":
        q = c.dev["q"].double()
        first = torch.arange(len(q) + 1)
    else:
        q = s["q"].double()
        first = s["qsl"].cpu().long()
    out = torch.empty_like(q)
    for b in range(case["batch"]):
        lo, hi, n = int(first[b]), int(first[b + 1]), int(c.seq_lens[b])
        k = _pages(c.pool.va_k(0), c, c.block_tables[b], n)
        v = _pages(c.pool.va_v(0), c, c.block_tables[b], n)
        pos = torch.arange(n - (hi - lo), n, device="cuda")
        out[lo:hi] = _attend(q[lo:hi], k, v, pos)
    return out
