// fp8-e4m3 page write (device side), shared by the append kernels and the
// decode step's RoPE + append.
#pragma once
#include "common.hpp"

namespace kcmm {
namespace {

// fp32 -> OCP e4m3fn, round to nearest even, saturating to +-448.
__device__ __forceinline__ uint32_t f32_to_fp8e4m3(float x) {
    const uint32_t bits = __float_as_uint(x);
    const uint32_t sign = (bits >> 24) & 0x80u;
    const float a = fabsf(x);
    if (a != a) return sign | 0x7fu;
    if (a >= 448.0f) return sign | 0x7eu;
    if (a < 0.015625f) {  // below 2^-6: subnormal grid of 2^-9
        return sign | static_cast<uint32_t>(rintf(a * 512.0f));
    }
    const uint32_t ab = __float_as_uint(a);
    int e = static_cast<int>(ab >> 23) - 127;
    const uint32_t mant = ab & 0x7fffffu;
    uint32_t q = mant >> 20;
    const uint32_t rem = mant & 0xfffffu;
    if (rem > 0x80000u || (rem == 0x80000u && (q & 1u))) ++q;
    if (q == 8) {
        q = 0;
        ++e;
    }
    uint32_t code = (static_cast<uint32_t>(e + 7) << 3) | q;
    if (code > 0x7eu) code = 0x7eu;
    return sign | code;
}

// x / scale clamped to the e4m3 range, for scales in the range below, r = 1 /
// scale and x not NaN: x * r with one residual step is the correctly rounded
// quotient wherever it matters to four significant bits (Markstein's division;
// tests/test_fp8_quotient.py sweeps it against x / scale).  Its callers pass
// any bf16 value up to 448 * scale, or a stored code's value times an older,
// smaller scale -- 24 significant bits, so the residual of a quotient of 2^-11
// and more has bits down to 2^-57 * scale, which the lower bound keeps above
// the smallest float (at 2^-100 a few codes fell to the neighbour of a tie).
// The hardware conversion gives the bits of f32_to_fp8e4m3 (the two agree on
// every float but NaN, whose sign the hardware does not keep).
constexpr float kFp8QuotientMin = 0x1p-80f, kFp8QuotientMax = 0x1p100f;
__device__ __forceinline__ float fp8_quotient(float x, float scale, float r) {
    const float q = x * r;
    return __builtin_amdgcn_fmed3f(copysignf(fmaf(fmaf(-q, scale, x), r, q), x), -448.0f, 448.0f);
}

// 8 bf16 elements (4 dwords, no NaN) / scale as e4m3 bytes.
__device__ __forceinline__ u32x2 fp8_encode8(const u32x4& x, float scale, float r) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        v[i] = fp8_quotient(__uint_as_float((i & 1) ? x[i >> 1] & 0xffff0000u : x[i >> 1] << 16),
                            scale, r);
    u32x2 o;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * w], v[4 * w + 1], 0, false);
        o[w] = static_cast<uint32_t>(
            __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * w + 2], v[4 * w + 3], lo, true));
    }
    return o;
}

// fp8 page write of one (page, kv head) for one call.  `row_of` (bs entries,
// LDS) gives, for each token slot, the source row this call writes there (the
// call's last row for that slot), or -1.  The rows a call writes into a page
// are applied as one set, so the bytes do not depend on their order:
//   amax  = max |x| over the written rows of this kv head;
//   fresh = the call writes slot 0, or the footer scale is not a finite
//           positive number (a page never started);
//   fresh:  scale = amax / 448 (1 for amax 0); the slots the call does not
//           write are left as they are and are undefined from then on;
//   else:   scale = old, raised to amax / 448 when amax > 448 * old, and then
//           every slot the call does not write is re-encoded from old to the
//           new scale (e4m3(decode(code) * old / scale));
// and each written row is stored as e4m3(x / scale).  One wavefront.  With
// head_dim % 8 == 0 and 16-byte aligned source rows, lanes take 16-byte
// pieces of the rows, 256 pieces (16 rows of 128) per pass with every load
// in flight at once; a page of at most 256 pieces is read once.
__device__ __forceinline__ void fp8_write_page_head(uint8_t* page, uint32_t kvh,
                                                    const uint16_t* src_base, const int32_t* row_of,
                                                    uint32_t bs, uint32_t kv_heads,
                                                    uint32_t head_dim, uint32_t row_bytes,
                                                    uint32_t data_bytes) {
    const int lane = threadIdx.x & 63;
    float* sp = reinterpret_cast<float*>(page + data_bytes) + kvh;
    const float old = *sp;
    const bool vec = (head_dim & 7) == 0 && (reinterpret_cast<uintptr_t>(src_base) & 15) == 0;
    constexpr uint32_t PASS = 4;              // pieces per lane per pass
    const uint32_t C = head_dim / 8;          // pieces per row (vec: 1..32)
    const uint32_t total = bs * C, rcp = vec ? 65536u / C + 1 : 0;
    const uint32_t step = vec ? (64 * PASS / C) * C : 0;   // whole rows per pass
    u32x4 x[PASS];
    int32_t at[PASS];                         // slot * C + piece, or -1
    auto load_pass = [&](uint32_t q0) {
#pragma unroll
        for (uint32_t i = 0; i < PASS; ++i) {
            const uint32_t q = lane + 64 * i, u = (q * rcp) >> 16;   // q / C (q < 256)
            at[i] = -1;
            x[i] = u32x4{0, 0, 0, 0};
            const uint32_t slot = q0 / C + u;
            if (q >= step || slot >= bs) continue;
            const int32_t r = row_of[slot];
            if (r < 0) continue;
            at[i] = static_cast<int32_t>(q0 + q);
            x[i] = *reinterpret_cast<const u32x4*>(
                src_base + (static_cast<uint64_t>(r) * kv_heads + kvh) * head_dim + (q - u * C) * 8);
        }
    };
    float amax = 0.0f;
    bool nan = false;
    if (vec) {
#pragma unroll 1
        for (uint32_t q0 = 0; q0 < total; q0 += step) {
            load_pass(q0);
#pragma unroll
            for (uint32_t i = 0; i < PASS; ++i)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float lo = __uint_as_float(x[i][w] << 16);
                    const float hi = __uint_as_float(x[i][w] & 0xffff0000u);
                    amax = fmaxf(amax, fmaxf(fabsf(lo), fabsf(hi)));
                    nan |= lo != lo || hi != hi;
                }
        }
    } else {
#pragma unroll 1
        for (uint32_t u = 0; u < bs; ++u) {
            const int32_t r = row_of[u];
            if (r < 0) continue;
            const uint16_t* src = src_base + (static_cast<uint64_t>(r) * kv_heads + kvh) * head_dim;
#pragma unroll
            for (int i = 0; i < 4; ++i) {   // head_dim <= 256
                const uint32_t d = lane + 64 * i;
                if (d < head_dim) amax = fmaxf(amax, fabsf(bf16_bits_to_f32(src[d])));
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    const bool fresh = row_of[0] >= 0 || !(old > 0.0f && old <= 3.40282347e38f);
    float scale;
    if (fresh) {
        scale = amax > 0.0f ? amax / 448.0f : 1.0f;
    } else {
        scale = old;
        if (amax > 448.0f * old) {
            scale = amax / 448.0f;
            if ((head_dim & 15) == 0 && (row_bytes & 15) == 0 && scale >= kFp8QuotientMin &&
                scale <= kFp8QuotientMax) {
                // 16-byte pieces of all unwritten slots at once: one memory
                // round trip for the page instead of one per slot
                const uint32_t pieces = head_dim / 16;
                const float r = 1.0f / scale;
#pragma unroll 1
                for (uint32_t c = lane; c < bs * pieces; c += 64) {
                    const uint32_t u = c / pieces;
                    if (row_of[u] >= 0) continue;
                    uint8_t* q = page + static_cast<uint64_t>(u) * row_bytes + kvh * head_dim +
                                 (c - u * pieces) * 16;
                    const u32x4 v = *reinterpret_cast<const u32x4*>(q);
                    u32x4 o;
                    bool nan_code = false;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const uint32_t m = v[w] & 0x7f7f7f7fu;   // a byte of 0x7f carries into bit 7
                        nan_code |= ((m + 0x01010101u) & 0x80808080u) != 0;
                        const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(v[w]), false);
                        const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(v[w]), true);
                        const int p0 = __builtin_amdgcn_cvt_pk_fp8_f32(
                            fp8_quotient(lo[0] * old, scale, r), fp8_quotient(lo[1] * old, scale, r),
                            0, false);
                        o[w] = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(
                            fp8_quotient(hi[0] * old, scale, r), fp8_quotient(hi[1] * old, scale, r),
                            p0, true));
                    }
                    if (!nan_code) {
                        *reinterpret_cast<u32x4*>(q) = o;
                        continue;
                    }
#pragma unroll 1
                    for (int i = 0; i < 16; ++i)
                        q[i] = static_cast<uint8_t>(f32_to_fp8e4m3(fp8e4m3_to_f32(q[i]) * old / scale));
                }
            } else {
#pragma unroll 1
                for (uint32_t u = 0; u < bs; ++u) {
                    if (row_of[u] >= 0) continue;
                    uint8_t* row = page + static_cast<uint64_t>(u) * row_bytes + kvh * head_dim;
#pragma unroll 1
                    for (uint32_t d = lane; d < head_dim; d += 64) {
                        const float y = fp8e4m3_to_f32(row[d]) * old;
                        row[d] = static_cast<uint8_t>(f32_to_fp8e4m3(y / scale));
                    }
                }
            }
        }
    }
    if (vec && !__any(nan) && scale >= kFp8QuotientMin && scale <= kFp8QuotientMax) {
        const float r = 1.0f / scale;
        uint8_t* base = page + kvh * head_dim;
#pragma unroll 1
        for (uint32_t q0 = 0; q0 < total; q0 += step) {
            if (total > step) load_pass(q0);
#pragma unroll
            for (uint32_t i = 0; i < PASS; ++i) {
                if (at[i] < 0) continue;
                const uint32_t q = at[i], u = q / C;
                u32x2* d = reinterpret_cast<u32x2*>(base + static_cast<uint64_t>(u) * row_bytes +
                                                    (q - u * C) * 8);
                *d = fp8_encode8(x[i], scale, r);
            }
        }
    } else {
#pragma unroll 1
        for (uint32_t u = 0; u < bs; ++u) {
            const int32_t r = row_of[u];
            if (r < 0) continue;
            const uint16_t* src = src_base + (static_cast<uint64_t>(r) * kv_heads + kvh) * head_dim;
            uint8_t* row = page + static_cast<uint64_t>(u) * row_bytes + kvh * head_dim;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t d = lane + 64 * i;
                if (d < head_dim)
                    row[d] = static_cast<uint8_t>(f32_to_fp8e4m3(bf16_bits_to_f32(src[d]) / scale));
            }
        }
    }
    if (lane == 0) *sp = scale;
}

// Waves per fp8 writer workgroup: one per (kv head, K|V) pair, at most 16.
constexpr int kFp8MaxWaves = 16;
// Token slots per page the fp8 writer handles (its slot table lives in LDS).
constexpr uint32_t kFp8MaxBlockSize = 4096;

}  // namespace
}  // namespace kcmm
