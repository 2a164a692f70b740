// Projection GEMM for prompt-sized token counts on gfx950: Y[M][N] = X[M][K]
// * W[N][K]^T, bf16 operands, fp32 accumulation (the product the reference
// hands to cuBLAS, ref runtime.rs:17-41), with the plain / residual / SwiGLU /
// split-partial stores.
//
// At a few hundred tokens and more the product is bound by the matrix cores,
// and what keeps them from their rate is the LDS port and the waits around
// it, so:
//  * workgroup = 8 waves on 256 weight rows x BM = 64 * FB tokens (FB 1..4),
//    each wave on two 32-row halves by two halves of 16 * FB tokens.  At BM =
//    256 the LDS port moves 64 KiB in and 192 KiB out per 64-element k chunk,
//    1280 of the 2048 cycles that the chunk's MFMAs take (a 64 x 64 wave tile,
//    as in gemm_tiled.hip, needs 1800);
//  * waves 0-3 and 4-7 (one of each on a SIMD) run half a phase apart: while
//    one group's 8 * FB MFMAs run, the other reads the fragments of its next
//    phase (all weights and one token half, then the other token half) and
//    issues its loads, with a barrier at each change, so that the matrix
//    cores always have a wave whose operands are in registers;
//  * chunks reach LDS by direct loads (global_load_lds_dwordx4) into a ring of
//    two weight and three token tiles (160 KiB at BM = 256), each load into
//    the place whose last reader was one phase ago, so that 1.25 .. 1.75
//    chunks are in flight and a wave waits for its loads once per chunk;
//  * LDS rows are 128 bytes of eight 16-byte pieces, piece p of row r at slot
//    p ^ s(r); W rows are dealt to MFMA rows so that a lane ends with 8
//    consecutive output columns (16-byte stores), and s() follows that order
//    so that the lanes of an LDS cycle hit distinct banks;
//  * workgroup i runs on XCD i % 8: tiles are numbered so that an XCD's
//    concurrent tiles are a block of few weight tiles x up to 8 token tiles.
// Measured (MI355X): 8192^3 776 us = 1.42 PFLOP/s (2.18 without the loads,
// 1.35 in four phases of 16 MFMAs, 1.36 with the loads issued between the
// MFMAs; the 128 x 256 tile 1.06); gate/up + SwiGLU of 2048 tokens at the
// Llama-3-8B shape 690 us on the weight-stream kernel, 357 here (1.35
// PFLOP/s); down + residual of 777 tokens 130 -> 100 us.
#include <algorithm>
#include <string>
#include <type_traits>

#include "../device_api.hpp"
#include "common.hpp"

namespace kcmm {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

// 16 bytes per lane from global memory straight into LDS at lds + 16 * lane
// (lds is wave-uniform).
__device__ __forceinline__ void load_lds16(const uint8_t* g, uint8_t* lds) {
    __builtin_amdgcn_global_load_lds(g, (lds_ptr)lds, 16, 0, 0);
}

// The same, nontemporal (weights that one token tile reads once).
__device__ __forceinline__ void load_lds16_nt(const uint8_t* g, uint8_t* lds) {
    __builtin_amdgcn_global_load_lds(g, (lds_ptr)lds, 16, 0, 2);
}

// s_waitcnt vmcnt(N) lgkmcnt(0) (gfx9 encoding: vmcnt bits 3:0 and 15:14,
// expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("" ::: "memory");   // the LDS reads before it stay before it
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// A bare barrier (a fenced one would wait for the loads in flight), which no
// memory access moves across.
__device__ __forceinline__ void phase_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

struct WideParams {
    const uint8_t* X;    // [M][K] bf16
    const uint8_t* W;    // [N][K] bf16 (SwiGLU: [2 I][K], gate rows then up rows)
    uint16_t* Y;         // [M][N] (SwiGLU: [M][I])
    const uint16_t* R;   // residual [M][N] or null (may equal Y)
    float* part;         // non-null: fp32 partials [split][M][N]
    int M, N, K, klen;   // N: output columns (SwiGLU: I); klen: K per split
    // The grid's x range: zone 0's full token tiles, zone 1's, then the
    // ragged last token tile of every weight tile of zone 0 and zone 1.  Zone
    // z covers nw[z] weight tiles (zone 0 first) with full[z] token tiles of
    // 64 * fb[z] and, when rag[z] > 0, one of 64 * rag[z].
    int nw[2], full[2], fb[2], rag[2];
};

constexpr int kWidePlain = 0;
constexpr int kWideSwiglu = 1;
constexpr int kWideLds = 160 * 1024;

// One tile: 256 weight rows of weight tile tn by BM = 64 * FB tokens from m0.
template <int EPI, int FB, bool WNT>
__device__ __forceinline__ void wide_tile(const WideParams& p, uint8_t* lds, int tn, int m0) {
    constexpr int BM = 64 * FB;
    constexpr int BN = EPI == kWideSwiglu ? 128 : 256;   // output columns
    constexpr int WT = 256 * 128, XT = BM * 128;         // bytes of a chunk's W and X tiles
    static_assert(2 * WT + 3 * XT <= kWideLds, "LDS");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    // wave (wn, wm): weight rows wn*32 .. of each 128-row half, tokens
    // wm*16*FB .. of each half; the two groups of waves are wm = 0 and 1
    const int wn = wave & 3, wm = wave >> 2;
    const int n0 = tn * BN;
    const int kbeg = blockIdx.y * p.klen;
    const int nchunks = p.klen >> 6;
    const uint32_t rowb = static_cast<uint32_t>(p.K) * 2;

    // Direct loads: instruction i of wave w fills LDS rows 8*(8*i + w) .. +8
    // of a tile; lane l writes slot l & 7 of row 8*(8*i + w) + (l >> 3), from
    // piece slot ^ s(row): s(r) = (r & 3) | bit 3 of r, shifted to bit 2, for
    // W rows; r & 7 for X rows.  Rows past N or M are clamped, unused.
    const int lrow = lane >> 3;
    const int wpiece = (lane & 7) ^ ((lrow & 3) | ((wave & 1) << 2));
    const int xpiece = (lane & 7) ^ lrow;
    uint32_t wof[4], xof[FB];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * (8 * i + wave) + lrow;
        int row;
        if constexpr (EPI == kWideSwiglu) row = min(n0 + (r & 127), p.N - 1) + (i >> 1) * p.N;
        else row = min(n0 + r, p.N - 1);
        wof[i] = static_cast<uint32_t>(row) * rowb + wpiece * 16;
    }
#pragma unroll
    for (int i = 0; i < FB; ++i) {
        const int r = min(m0 + 8 * (8 * i + wave) + lrow, p.M - 1);
        xof[i] = static_cast<uint32_t>(r) * rowb + xpiece * 16;
    }
    const uint8_t* wk = p.W + static_cast<size_t>(kbeg) * 2;
    const uint8_t* xk = p.X + static_cast<size_t>(kbeg) * 2;
    auto issue_w = [&](int c) {
        uint8_t* dst = lds + (c & 1) * WT + wave * 1024;
        const uint8_t* src = wk + static_cast<size_t>(c) * 128;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (WNT) load_lds16_nt(src + wof[i], dst + i * 8192);
            else load_lds16(src + wof[i], dst + i * 8192);
        }
    };
    auto issue_x = [&](int c, int slot) {
        uint8_t* dst = lds + 2 * WT + slot * XT + wave * 1024;
        const uint8_t* src = xk + static_cast<size_t>(c) * 128;
#pragma unroll
        for (int i = 0; i < FB; ++i) load_lds16(src + xof[i], dst + i * 8192);
    };

    f32x4 acc[2][2][2][FB];   // [weight half][block][token half][block]
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int j = 0; j < FB; ++j) acc[a][i][b][j] = f32x4{0, 0, 0, 0};

    // Fragment reads.  MFMA row a of W block i is weight row 8*(a >> 2) + 4*i
    // + (a & 3) of the wave's 32, so D row 4*lg + r of block i is row 8*lg +
    // 4*i + r: a lane's two blocks are 8 consecutive output columns.
    const int a_lane = (wn * 32 + 8 * (ln >> 2) + (ln & 3)) * 128;
    const int b_lane = 2 * WT + (wm * 16 * FB + ln) * 128;
    const int sw0 = ((0 + lg) ^ (ln & 7)) * 16, sw1 = ((4 + lg) ^ (ln & 7)) * 16;
    u32x4 a[2][2][2], b[2][FB];   // [k-step][half][block], [k-step][block]
    auto read_a = [&](int c) {
        const uint8_t* st = lds + (c & 1) * WT + a_lane;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[0][h][i] = *reinterpret_cast<const u32x4*>(st + sw0 + h * 16384 + i * 512);
                a[1][h][i] = *reinterpret_cast<const u32x4*>(st + sw1 + h * 16384 + i * 512);
            }
    };
    auto read_b = [&](int h, int slot) {
        const uint8_t* st = lds + slot * XT + b_lane + h * (XT / 2);
#pragma unroll
        for (int j = 0; j < FB; ++j) {
            b[0][j] = *reinterpret_cast<const u32x4*>(st + sw0 + j * 2048);
            b[1][j] = *reinterpret_cast<const u32x4*>(st + sw1 + j * 2048);
        }
    };
    auto mfmas = [&](int bh) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < FB; ++j)
                        acc[h][i][bh][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, a[ks][h][i]), __builtin_bit_cast(bf16x8, b[ks][j]),
                            acc[h][i][bh][j], 0, 0, 0);
    };
    // One chunk, two phases.  Before the first barrier of a phase a wave
    // reads the phase's fragments and issues loads into a place whose last
    // readers (both groups) finished before the previous barrier: the token
    // tile of chunk c - 1, then the weight tile of chunk c, take chunk c + 2.
    // Chunk c + 1 must have landed when the second phase's barrier lets a
    // group go on to it; what was issued since for chunk c + 2 stays in
    // flight (near the end nothing is issued, and the wait is for all).
    int sx = 0;   // X slot of chunk c (c % 3)
    auto chunk = [&](int c, auto steady_tag) {
        constexpr bool ST = decltype(steady_tag)::value;
        const int sn = sx == 0 ? 2 : sx - 1;   // slot of chunk c + 2
        read_b(0, sx);
        read_a(c);
        if constexpr (ST) issue_x(c + 2, sn);
        wait_vm_lgkm0<63>();   // the fragments only
        phase_barrier();
        __builtin_amdgcn_s_setprio(1);
        mfmas(0);
        __builtin_amdgcn_s_setprio(0);
        phase_barrier();
        read_b(1, sx);
        if constexpr (ST) issue_w(c + 2);
        wait_vm_lgkm0<ST ? FB + 4 : 0>();
        phase_barrier();
        __builtin_amdgcn_s_setprio(1);
        mfmas(1);
        __builtin_amdgcn_s_setprio(0);
        phase_barrier();
        sx = sx == 2 ? 0 : sx + 1;
    };

    // nchunks >= 2 (the launcher's choice of klen)
    issue_x(0, 0);
    issue_w(0);
    issue_x(1, 1);
    issue_w(1);
    wait_vm_lgkm0<FB + 4>();
    phase_barrier();
    if (wm == 1) phase_barrier();   // half a phase behind
    int c = 0;
    for (; c < nchunks - 2; ++c) chunk(c, std::true_type{});
    for (; c < nchunks; ++c) chunk(c, std::false_type{});
    if (wm == 0) phase_barrier();

    // Stores: acc[ah][i][bh][j][r] = token m0 + bh*BM/2 + wm*16*FB + 16j + ln,
    // weight row (of half ah) wn*32 + 8*lg + 4*i + r; SwiGLU: half 0 holds
    // gate rows, half 1 the up rows of the same columns.
#pragma unroll
    for (int bh = 0; bh < 2; ++bh)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
            const int m = m0 + bh * (BM / 2) + wm * 16 * FB + 16 * j + ln;
            if (m >= p.M) continue;
            if constexpr (EPI == kWideSwiglu) {
                const int n = n0 + wn * 32 + 8 * lg;
                if (n >= p.N) continue;
                float v[8];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        v[4 * i + r] = swiglu_product(bf16_round_hw(acc[0][i][bh][j][r]),
                                                      bf16_round_hw(acc[1][i][bh][j][r]),
                                                      [](float x) { return bf16_round_hw(x); });
                *reinterpret_cast<u32x4*>(p.Y + static_cast<size_t>(m) * p.N + n) = pack_bf16x8(v);
            } else {
#pragma unroll
                for (int ah = 0; ah < 2; ++ah) {
                    const int n = n0 + ah * 128 + wn * 32 + 8 * lg;
                    if (n >= p.N) continue;
                    const size_t at = static_cast<size_t>(m) * p.N + n;
                    if (p.part != nullptr) {
                        f32x4* d = reinterpret_cast<f32x4*>(
                            p.part + static_cast<size_t>(blockIdx.y) * p.M * p.N + at);
                        d[0] = acc[ah][0][bh][j];
                        d[1] = acc[ah][1][bh][j];
                        continue;
                    }
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[4 * i + r] = acc[ah][i][bh][j][r];
                    if (p.R != nullptr) {
                        const u32x4 rr = *reinterpret_cast<const u32x4*>(p.R + at);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            v[2 * e] = bf16_round_hw(v[2 * e]) + __uint_as_float(rr[e] << 16);
                            v[2 * e + 1] = bf16_round_hw(v[2 * e + 1]) + __uint_as_float(rr[e] & 0xffff0000u);
                        }
                    }
                    *reinterpret_cast<u32x4*>(p.Y + at) = pack_bf16x8(v);
                }
            }
        }
}

// The idx-th tile of a run of n workgroups, so that each XCD (workgroup i of
// a grid runs on XCD i % 8) takes a contiguous piece of the tile list.
__device__ __forceinline__ int xcd_order(int idx, int n) {
    const int x = idx & 7, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + (idx >> 3);
}

template <int EPI, bool WNT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_wide_kernel(WideParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kWideLds];
    int i = blockIdx.x, fb = 0, tn = 0, m0 = 0;
#pragma unroll
    for (int z = 0; z < 2; ++z) {
        const int n = p.nw[z] * p.full[z];
        if (fb == 0 && i < n) {
            // blocks of 8 token tiles, token tiles fastest
            const int t = xcd_order(i, n);
            const int mg = t / (8 * p.nw[z]), rem = t - mg * 8 * p.nw[z];
            const int gm = min(8, p.full[z] - mg * 8);
            tn = rem / gm;
            m0 = (mg * 8 + rem - tn * gm) * 64 * p.fb[z];
            fb = p.fb[z];
            if (z) tn += p.nw[0];
        }
        i -= n;
    }
#pragma unroll
    for (int z = 0; z < 2; ++z) {
        const int n = p.rag[z] > 0 ? p.nw[z] : 0;
        if (fb == 0 && i < n) {
            tn = xcd_order(i, n) + (z ? p.nw[0] : 0);
            m0 = p.full[z] * 64 * p.fb[z];
            fb = p.rag[z];
        }
        i -= n;
    }
    switch (fb) {
        case 1: wide_tile<EPI, 1, WNT>(p, lds, tn, m0); break;
        case 2: wide_tile<EPI, 2, WNT>(p, lds, tn, m0); break;
        case 3: wide_tile<EPI, 3, WNT>(p, lds, tn, m0); break;
        case 4: wide_tile<EPI, 4, WNT>(p, lds, tn, m0); break;
        default: break;
    }
}

// Finish time of workgroups dealt in order to 256 CUs (one at a time each):
// kMax groups of equal free times, earliest first.
struct Cus {
    static constexpr int kMax = 12;
    double t[kMax];
    int cnt[kMax], n = 1;
    Cus() { t[0] = 0.0; cnt[0] = 256; }
    void deal(int tiles, double us) {
        if (n == 1 && tiles >= 256) {   // whole rounds
            t[0] += tiles / 256 * us;
            tiles %= 256;
        }
        while (tiles > 0) {
            int g = 0;
            for (int i = 1; i < n; ++i)
                if (t[i] < t[g]) g = i;
            const int take = std::min(tiles, cnt[g]);
            tiles -= take;
            if (take < cnt[g] && n < kMax) {
                t[n] = t[g];
                cnt[n++] = cnt[g] - take;
                cnt[g] = take;
            }
            t[g] += us;
        }
    }
    double last() const { return *std::max_element(t, t + n); }
};

// Modelled time of a plan: a workgroup takes chunks x kChunk + kFixed us by
// its token tile's height (fitted to timings of the 15 products and 12 token
// counts of M 129 .. 2048, N 1024 .. 28672, K 1024 .. 14336: within 5% at the
// median, 12% for nine in ten), or the weights and the partials at 4.2 TB/s
// where that is more; the split sum adds its launch and the partials' way.
double wide_us(const dev::GemmWidePlan& c, int M, int N, int K, bool swiglu) {
    constexpr double kChunk[5] = {0, 0.686, 0.755, 0.860, 1.025};
    auto us = [&](int fb) { return K / 64.0 / c.splits * kChunk[fb] + 2.7 + 1.7 * (fb - 1); };
    const int bn = swiglu ? 128 : 256;
    const int tiles_n = (N + bn - 1) / bn;
    const int nw[2] = {tiles_n - c.nw1, c.nw1}, fb[2] = {c.fb0, c.fb1};
    Cus cus;
    for (int z = 0; z < 2; ++z)
        if (nw[z] > 0) cus.deal(nw[z] * (M / (64 * fb[z])) * c.splits, us(fb[z]));
    for (int z = 0; z < 2; ++z) {
        const int rag = nw[z] > 0 ? (M % (64 * fb[z]) + 63) / 64 : 0;
        if (rag > 0) cus.deal(nw[z] * c.splits, us(rag));
    }
    const double part = c.splits > 1 ? 4.0 * c.splits * M * N : 0.0;
    const double bytes = 2.0 * (swiglu ? 2 : 1) * N * K + part;
    double t = 0.5 + std::max(cus.last(), bytes / 4.2e6);
    if (c.splits > 1) t += 4.2 + 0.31e-6 * part;
    return t;
}

}  // namespace

namespace dev {

// (fb0 is 1..4; any other value above 100 forces nothing)
int gemm_wide_forced() {
    const int f = tunable_or(Tun::kGemmTile, -1) - 100;
    return f > 0 && f % 10 >= 1 && f % 10 <= 4 ? f : 0;
}

// The plan of least modelled time: token tiles of 64 .. 256 (a ragged last
// tile only as high as it needs), K splits of at least 4 chunks for plain
// products, and -- when whole rounds of tiles leave a partly filled last round
// -- lower token tiles for the weight tiles of that round (gate/up of 2048
// tokens, 3.5 rounds of 256-token tiles: 369 -> 357 us with the last half
// round on 128-token tiles).  A split counts 5% more than its model, whose
// error is larger there.  KCMM_GEMM_SPLITS forces the split (0 splits in the
// result: it cannot be had); KCMM_GEMM_TILE = 100 + fb0 the token tiles'
// height, 100 + 10 fb1 + fb0 two heights, half of the weight tiles each.
GemmWidePlan gemm_wide_plan(uint32_t m, uint32_t n, uint32_t k, bool swiglu, int max_splits) {
    const int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k);
    const int forced = gemm_wide_forced();
    const int forced_splits = swiglu ? 1 : tunable_or(Tun::kGemmSplits, 0);
    const int bn = swiglu ? 128 : 256;
    const int tiles_n = (N + bn - 1) / bn, chunks = K / 64;
    GemmWidePlan best;
    best.splits = 0;
    auto take = [&](GemmWidePlan c) {
        c.us = wide_us(c, M, N, K, swiglu) * (c.splits > 1 ? 1.05 : 1.0);
        if (best.splits == 0 || c.us < best.us) best = c;
    };
    for (int fb = 1; fb <= 4; ++fb) {
        if (forced ? fb != forced % 10 : fb > 1 && 64 * (fb - 1) >= M) continue;
        for (int s = 1; s <= (swiglu ? 1 : max_splits); s *= 2) {
            if (chunks % s || chunks / s < (s > 1 ? 4 : 2)) break;
            if (forced_splits > 0 && s != forced_splits) continue;
            GemmWidePlan c;
            c.fb0 = c.fb1 = fb;
            c.splits = s;
            if (forced >= 10) {
                c.fb1 = std::min(4, forced / 10);
                c.nw1 = tiles_n / 2;
            }
            take(c);
            const int full = M / (64 * fb);
            if (s > 1 || forced || fb == 1 || tiles_n * full < 256) continue;
            c.nw1 = tiles_n - tiles_n * full / 256 * 256 / full;
            for (c.fb1 = 1; c.nw1 > 0 && c.fb1 < fb; ++c.fb1) take(c);
        }
    }
    return best;
}

bool gemm_wide(const GemmWideArgs& a, std::string* err) {
    WideParams p{};
    p.X = reinterpret_cast<const uint8_t*>(a.x);
    p.W = reinterpret_cast<const uint8_t*>(a.w);
    p.Y = reinterpret_cast<uint16_t*>(a.y);
    p.R = reinterpret_cast<const uint16_t*>(a.residual);
    p.M = static_cast<int>(a.m);
    p.N = static_cast<int>(a.n);
    p.K = static_cast<int>(a.k);
    const GemmWidePlan& c = a.plan;
    if (a.m == 0 || a.n == 0 || a.n % 32 != 0 || c.splits < 1 || a.k % (64u * c.splits) != 0 ||
        a.k / (64u * c.splits) < 2 || (a.swiglu && c.splits != 1) ||
        (c.splits > 1 && a.part == nullptr)) {
        *err = "wide gemm: n % 32 == 0 and at least two whole 64-element chunks per K split";
        return false;
    }
    p.klen = p.K / c.splits;
    p.part = c.splits > 1 ? a.part : nullptr;
    const int bn = a.swiglu ? 128 : 256;
    const int tiles_n = (p.N + bn - 1) / bn;
    const int fb[2] = {c.fb0, c.fb1};
    p.nw[1] = std::min(c.nw1, tiles_n);
    p.nw[0] = tiles_n - p.nw[1];
    int grid = 0;
    for (int z = 0; z < 2; ++z) {
        if (fb[z] < 1 || fb[z] > 4) {
            *err = "wide gemm: token tiles are 64, 128, 192 or 256 high";
            return false;
        }
        p.fb[z] = fb[z];
        p.full[z] = p.M / (64 * fb[z]);
        p.rag[z] = (p.M - p.full[z] * 64 * fb[z] + 63) / 64;
        grid += p.nw[z] * (p.full[z] + (p.rag[z] > 0));
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(a.stream);
    const dim3 g(grid, c.splits);
    const bool once = p.M <= 64 * c.fb0 && c.nw1 == 0;   // one token tile
    auto launch = [&](auto epi, auto nt) {
        hipLaunchKernelGGL((gemm_wide_kernel<decltype(epi)::value, decltype(nt)::value>), g,
                           dim3(512), 0, s, p);
    };
    using P = std::integral_constant<int, kWidePlain>;
    using S = std::integral_constant<int, kWideSwiglu>;
    if (a.swiglu && once) launch(S{}, std::true_type{});
    else if (a.swiglu) launch(S{}, std::false_type{});
    else if (once) launch(P{}, std::true_type{});
    else launch(P{}, std::false_type{});
    KCMM_HIP_CHECK(hipGetLastError(), err);
    return true;
}

}  // namespace dev
}  // namespace kcmm
