// KV append (reshape-and-cache) kernels for gfx950.
//
// Reference semantics: a source row b of [batch][kv_heads*head_dim] lands at
// region + page_offset + slot*row_bytes for both K and V (ref pool.rs:1036-1098,
// ffi.rs:1088-1383), or -- with device slot ids -- at
// region + offsets_f16[slot/bs]*2 + (slot%bs)*row_bytes with the status word
// of ref kcmm_vllm_kv_write.cu:8-66 (1 = id past the table, 2 = inactive id).
// The reference issues two driver memcpys per row (host paths) or one thread
// per 16-bit element (device path); here one launch moves every row with
// 16-byte vector copies.
//
// fp8-e4m3 pools take bf16 source rows and quantize per (page, kv head) with
// one fp32 scale in the page footer.  The rows one call writes into a page
// are applied as a set (the call's last row for each slot), so the result
// does not depend on their order: a call that writes slot 0 starts the page
// with scale amax/448 over its rows (1 if all zero); a later call raises the
// scale to amax/448 when its rows exceed 448*scale and re-encodes every slot
// it does not write, so no value is ever clipped (fp8_write_page_head).
// Encoding is round-to-nearest-even with saturation to +-448.
#include <algorithm>
#include <cmath>
#include <vector>

#include "../device_api.hpp"
#include "common.hpp"
#include "fp8_page.hpp"

namespace kcmm {
namespace {

constexpr int kRowsPerLaunch = 64;

struct RowBatch {
    uint64_t dst[kRowsPerLaunch];  // byte offset of the destination row in a region
    uint32_t src[kRowsPerLaunch];  // source row index
};

// 16-bit pools: plain row copies.
__global__ __launch_bounds__(256) void kv_rows_copy(RowBatch rb, uint8_t* k_base, uint8_t* v_base,
                                                     const uint8_t* k_src, const uint8_t* v_src,
                                                     uint32_t row_bytes) {
    const int r = blockIdx.x;
    const uint64_t d = rb.dst[r];
    const uint64_t s = static_cast<uint64_t>(rb.src[r]) * row_bytes;
    if ((row_bytes & 15u) == 0) {
        for (uint32_t i = threadIdx.x * 16; i < row_bytes; i += 256 * 16) {
            *reinterpret_cast<u32x4*>(k_base + d + i) = *reinterpret_cast<const u32x4*>(k_src + s + i);
            *reinterpret_cast<u32x4*>(v_base + d + i) = *reinterpret_cast<const u32x4*>(v_src + s + i);
        }
    } else {
        for (uint32_t i = threadIdx.x * 2; i < row_bytes; i += 256 * 2) {
            *reinterpret_cast<uint16_t*>(k_base + d + i) = *reinterpret_cast<const uint16_t*>(k_src + s + i);
            *reinterpret_cast<uint16_t*>(v_base + d + i) = *reinterpret_cast<const uint16_t*>(v_src + s + i);
        }
    }
}

// Host-resolved fp8 rows grouped by page: rows start[g] .. start[g+1]-1 of the
// batch target one page, in call order.  A page's rows never span launches.
struct Fp8RowBatch {
    uint64_t page[kRowsPerLaunch];
    uint32_t slot[kRowsPerLaunch];
    uint32_t src[kRowsPerLaunch];
    uint16_t start[kRowsPerLaunch + 1];
};

// grid (groups), dynamic LDS bs * 4 bytes; wave w takes the (kv head, K|V)
// pairs w, w + waves, ...
__global__ __launch_bounds__(64 * kFp8MaxWaves) void kv_rows_fp8(
    Fp8RowBatch rb, uint8_t* k_base, uint8_t* v_base, const uint16_t* k_src,
    const uint16_t* v_src, uint32_t bs, uint32_t kv_heads, uint32_t head_dim, uint32_t row_bytes,
    uint32_t data_bytes) {
    extern __shared__ int32_t row_of[];
    const uint32_t g = blockIdx.x;
    const uint32_t r0 = rb.start[g], r1 = rb.start[g + 1];
    for (uint32_t u = threadIdx.x; u < bs; u += blockDim.x) row_of[u] = -1;
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t r = r0; r < r1; ++r) row_of[rb.slot[r]] = static_cast<int32_t>(rb.src[r]);
    __syncthreads();
    const uint32_t waves = blockDim.x >> 6;
    for (uint32_t j = threadIdx.x >> 6; j < 2 * kv_heads; j += waves) {
        const bool is_v = j & 1;
        fp8_write_page_head((is_v ? v_base : k_base) + rb.page[r0], j >> 1, is_v ? v_src : k_src,
                            row_of, bs, kv_heads, head_dim, row_bytes, data_bytes);
    }
}

struct SlotArgs {
    const int64_t* slots;
    const uint64_t* offsets_f16;
    const uint8_t* valid;
    int32_t* status;
    uint8_t* k_base;
    uint8_t* v_base;
    const uint8_t* k_src;
    const uint8_t* v_src;
    uint32_t offsets_len, block_size, row_bytes, src_row_bytes, kv_heads, head_dim, data_bytes;
    int bs_shift;
};

// Resolves row r's slot; returns false (after recording the status) when the
// row is padding or invalid.
__device__ __forceinline__ bool resolve_slot(const SlotArgs& a, uint32_t r, uint64_t* page,
                                             uint32_t* slot_in_page) {
    const int64_t slot = a.slots[r];
    if (slot < 0) return false;
    const int64_t id = slot / a.block_size;
    if (id >= static_cast<int64_t>(a.offsets_len)) {
        if (a.status && threadIdx.x == 0) atomicCAS(a.status, 0, 1);
        return false;
    }
    if (a.valid && a.valid[id] == 0) {
        if (a.status && threadIdx.x == 0) atomicCAS(a.status, 0, 2);
        return false;
    }
    *page = a.offsets_f16[id] * 2ull;
    *slot_in_page = static_cast<uint32_t>(slot % a.block_size);
    return true;
}

__global__ __launch_bounds__(256) void kv_slots_copy(SlotArgs a) {
    const uint32_t r = blockIdx.x;
    uint64_t page;
    uint32_t sl;
    if (!resolve_slot(a, r, &page, &sl)) return;
    const uint64_t d = page + static_cast<uint64_t>(sl) * a.row_bytes;
    const uint64_t s = static_cast<uint64_t>(r) * a.row_bytes;
    if ((a.row_bytes & 15u) == 0) {
        for (uint32_t i = threadIdx.x * 16; i < a.row_bytes; i += 256 * 16) {
            *reinterpret_cast<u32x4*>(a.k_base + d + i) = *reinterpret_cast<const u32x4*>(a.k_src + s + i);
            *reinterpret_cast<u32x4*>(a.v_base + d + i) = *reinterpret_cast<const u32x4*>(a.v_src + s + i);
        }
    } else {
        for (uint32_t i = threadIdx.x * 2; i < a.row_bytes; i += 256 * 2) {
            *reinterpret_cast<uint16_t*>(a.k_base + d + i) = *reinterpret_cast<const uint16_t*>(a.k_src + s + i);
            *reinterpret_cast<uint16_t*>(a.v_base + d + i) = *reinterpret_cast<const uint16_t*>(a.v_src + s + i);
        }
    }
}

// Block id of a slot (bs_shift: log2 of a power-of-two block size, else -1).
__device__ __forceinline__ int64_t block_of(const SlotArgs& a, int64_t slot) {
    if (a.bs_shift >= 0) return slot >> a.bs_shift;
    if (slot >> 32) return slot / a.block_size;
    return static_cast<uint32_t>(slot) / a.block_size;
}

// fp8 pages through device slot ids.  All rows of a page are applied as one
// set by one workgroup (fp8_write_page_head), the one that holds the page's
// first row of the call.  A workgroup holds R consecutive rows: it resolves
// them (status as above), lists the distinct pages they name, and walks the
// call's slot ids once, 1024 at a time, entering every row of those pages
// into the pages' slot tables in LDS (the last row for a slot wins, in call
// order) and dropping a page that an earlier row names.  The waves then take
// the (page, kv head, K|V) triples of the pages left.
//
// R gives every CU one workgroup of up to 16 waves: a prompt's rows fill a page
// each and want R near the page's rows, a decode step's have a page each and
// want as many waves as the chip holds, and the host cannot tell them apart.
// One workgroup per row, a serial walk over a page's rows and a pass that
// counted them (9 us) before / R = 16 with 8 waves above 512 rows / so, us, 8 kv
// heads, 16-slot pages: 600 prompt rows 57 / 15.9 / 9.6, 2400 290 / 13.1 / 11.2,
// 4500 359 / 21.1 / 18.3, 8100 648 / 27.0 / 24.7; one row per page, 600 rows 27.5
// / 79 / 16.8, 2000 66 / 84 / 37, 8000 237 / 162 / 128 (2 kv heads 58 / 82 / 44).
// The pages are found through a hash table: comparing each slot id with up to
// 32 of them took most of the time of 8000 rows (2 kv heads 86 us).
//
// A call of more than kFp8ScanRows rows would spend its time walking the
// slot ids (every workgroup walks all): `lead` / `cnt` (int32 per block id,
// zero between calls) then collect, per page, batch - (first row) and the
// number of rows, and a workgroup walks from its own rows on until it has
// them all; R = 12 with 4 waves there (9000 rows with a page each, 8 / 2 kv
// heads: 146 / 48 us, with 16 and 8 183 / 70; 12000 prompt rows 39 and 37).
constexpr uint32_t kFp8ScanRows = 8192;
constexpr uint32_t kFp8RowsPerGroup = 32;
constexpr uint32_t kFp8Slots = 256;   // of the hash table that finds a workgroup's pages by block id
__device__ __forceinline__ uint32_t fp8_hash(int32_t id) {
    return (static_cast<uint32_t>(id) * 0x9E3779B1u) >> 24;
}

__global__ __launch_bounds__(256) void kv_slots_fp8_collect(SlotArgs a, uint32_t batch,
                                                            int32_t* lead, int32_t* cnt) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= batch) return;
    const int64_t slot = a.slots[r];
    if (slot < 0) return;
    const int64_t id = block_of(a, slot);
    if (id >= static_cast<int64_t>(a.offsets_len)) return;
    if (a.valid && a.valid[id] == 0) return;
    atomicMax(lead + id, static_cast<int32_t>(batch - r));
    atomicAdd(cnt + id, 1);
}

// grid (ceil(batch / R)); 64 * waves threads; dynamic LDS R * block_size * 4.
__global__ __launch_bounds__(64 * kFp8MaxWaves) void kv_slots_fp8_write(SlotArgs a,
                                                                         uint32_t batch, uint32_t R,
                                                                         int32_t* lead,
                                                                         int32_t* cnt) {
    extern __shared__ int32_t row_of[];                  // [page of the list][block_size]
    __shared__ int32_t s_id[kFp8RowsPerGroup];           // the list: block ids
    __shared__ int32_t s_left[kFp8RowsPerGroup];         // collected: rows not found yet
    __shared__ int32_t s_dead[kFp8RowsPerGroup];         // an earlier row leads the page
    __shared__ int32_t s_key[kFp8Slots], s_page[kFp8Slots];   // block id (-1: free) -> place in the list
    __shared__ int32_t s_pages;
    const uint32_t r0 = blockIdx.x * R, t = threadIdx.x;
    const uint32_t bs = a.block_size;
    if (t < 64) {
        // this workgroup's rows, one per lane: status, then the distinct pages
        const int64_t slot = t < R && r0 + t < batch ? a.slots[r0 + t] : -1;
        const int64_t b = block_of(a, slot < 0 ? 0 : slot);
        const bool row = slot >= 0, past = b >= static_cast<int64_t>(a.offsets_len);
        bool active = row && !past;
        if (active && a.valid != nullptr) active = a.valid[b] != 0;
        if (a.status != nullptr && row && !active) atomicCAS(a.status, 0, past ? 1 : 2);
        const int32_t id = active ? static_cast<int32_t>(b) : -1;   // (offsets_len <= 2^28)
        bool first = id >= 0;
        for (uint32_t j = 0; j + 1 < R; ++j) {
            const int32_t other = __shfl(id, j);
            first &= j >= t || other != id;
        }
        int32_t rows = 0;
        if (lead != nullptr && first) {
            first = __atomic_load_n(lead + id, __ATOMIC_RELAXED) == static_cast<int32_t>(batch - r0 - t);
            if (first) rows = __atomic_load_n(cnt + id, __ATOMIC_RELAXED);
        }
        for (uint32_t i = t; R > 1 && i < kFp8Slots; i += 64) s_key[i] = -1;
        __builtin_amdgcn_wave_barrier();
        const uint64_t m = __ballot(first);
        if (first) {
            const int at = __popcll(m & ((1ull << t) - 1));
            s_id[at] = id;
            s_left[at] = rows;
            s_dead[at] = 0;
            if (R > 1) {
                uint32_t h = fp8_hash(id);   // (at most kFp8RowsPerGroup of them: a free one is near)
                while (atomicCAS(s_key + h, -1, id) != -1) h = (h + 1) % kFp8Slots;
                s_page[h] = at;
            }
        }
        if (t == 0) s_pages = __popcll(m);
    }
    for (uint32_t i = t; i < R * bs; i += blockDim.x) row_of[i] = -1;
    __syncthreads();
    const int pages = s_pages;
    if (pages == 0) return;   // (uniform)
    // Walk the slot ids, kAhead per thread in flight together.
    constexpr uint32_t kAhead = 4;
    const uint32_t nt = blockDim.x;
    for (uint32_t base = lead != nullptr ? r0 : 0; base < batch; base += nt * kAhead) {
        int64_t slot[kAhead];
#pragma unroll
        for (uint32_t i = 0; i < kAhead; ++i) {
            const uint32_t rr = base + t + i * nt;
            slot[i] = a.slots[min(rr, batch - 1)];
            if (rr >= batch) slot[i] = -1;
        }
#pragma unroll
        for (uint32_t i = 0; i < kAhead; ++i) {
            if (slot[i] < 0) continue;
            const uint32_t rr = base + t + i * nt;
            const int64_t id = block_of(a, slot[i]);
            if (id >= static_cast<int64_t>(a.offsets_len)) continue;
            int j = 0;
            if (R == 1) {
                if (id != s_id[0]) continue;
            } else {
                uint32_t h = fp8_hash(static_cast<int32_t>(id));
                int32_t key = s_key[h];
                while (key != id && key != -1) key = s_key[h = (h + 1) % kFp8Slots];
                if (key == -1) continue;
                j = s_page[h];
            }
            // (a page dropped here may still be entered by others: its table
            // is not used)
            if (rr < r0) s_dead[j] = 1;
            atomicMax(row_of + j * bs + static_cast<uint32_t>(slot[i] - id * bs),
                      static_cast<int32_t>(rr));
            if (lead != nullptr) atomicSub(s_left + j, 1);
        }
        if (lead != nullptr) {
            __syncthreads();
            int left = 0;
            for (int j = 0; j < pages; ++j) left += s_left[j];
            __syncthreads();
            if (left == 0) break;   // (uniform)
        }
    }
    __syncthreads();
    const uint32_t waves = nt >> 6, units = 2 * a.kv_heads;
    uint32_t w = t >> 6;   // wave w takes triples w, w + waves, ... of the live pages
    for (int j = 0; j < pages; ++j) {
        if (s_dead[j]) continue;
        const uint64_t page = a.offsets_f16[s_id[j]] * 2ull;
        for (; w < units; w += waves) {
            const bool is_v = w & 1;
            fp8_write_page_head((is_v ? a.v_base : a.k_base) + page, w >> 1,
                                reinterpret_cast<const uint16_t*>(is_v ? a.v_src : a.k_src),
                                row_of + j * bs, bs, a.kv_heads, a.head_dim, a.row_bytes,
                                a.data_bytes);
        }
        w -= units;
    }
    if (lead != nullptr && t < static_cast<uint32_t>(pages)) {
        // (every workgroup that names the page compares lead with a row of
        // its own: zero never matches)
        lead[s_id[t]] = 0;
        cnt[s_id[t]] = 0;
    }
}

}  // namespace

namespace dev {

// Row indices sorted by (page, slot), keeping only the last row of the call
// for each (page, slot): a call that names a slot twice stores its last row
// there, as the reference's sequential row copies do (ref pool.rs:1084-1091).
static std::vector<uint32_t> last_row_per_slot(const RowDst* rows, size_t n) {
    std::vector<uint32_t> order(n);
    for (size_t i = 0; i < n; ++i) order[i] = static_cast<uint32_t>(i);
    std::sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
        if (rows[x].page_offset != rows[y].page_offset)
            return rows[x].page_offset < rows[y].page_offset;
        if (rows[x].slot != rows[y].slot) return rows[x].slot < rows[y].slot;
        return x < y;
    });
    size_t m = 0;
    for (size_t i = 0; i < n; ++i) {
        const bool superseded = i + 1 < n && rows[order[i]].page_offset == rows[order[i + 1]].page_offset &&
                                rows[order[i]].slot == rows[order[i + 1]].slot;
        if (!superseded) order[m++] = order[i];
    }
    order.resize(m);
    return order;
}

bool kv_write_rows(const KvRowsArgs& a, std::string* err) {
    hipStream_t s = reinterpret_cast<hipStream_t>(a.stream);
    auto* kb = reinterpret_cast<uint8_t*>(a.k_base);
    auto* vb = reinterpret_cast<uint8_t*>(a.v_base);
    const std::vector<uint32_t> order = last_row_per_slot(a.rows, a.num_rows);
    const size_t num = order.size();
    if (a.dtype == kDtFP8) {
        if (a.head_dim > 256) {
            *err = "fp8 KV write supports head_dim <= 256";
            return false;
        }
        if (a.block_size == 0 || a.block_size > kFp8MaxBlockSize) {
            *err = "fp8 KV write supports block_size <= 4096";
            return false;
        }
        // One workgroup per page; a page's rows (distinct slots) go to one
        // launch, whole groups packed kRowsPerLaunch rows at a time.
        const int waves = static_cast<int>(std::min<uint32_t>(2 * a.kv_heads, kFp8MaxWaves));
        const size_t lds = static_cast<size_t>(a.block_size) * 4;
        size_t i = 0;
        while (i < num) {
            Fp8RowBatch rb{};
            uint32_t groups = 0, n = 0;
            while (i < num) {
                size_t j = i;
                while (j < num && a.rows[order[j]].page_offset == a.rows[order[i]].page_offset) ++j;
                if (j - i > static_cast<size_t>(kRowsPerLaunch)) {
                    *err = "fp8 KV write: more than 64 rows into one page in one call";
                    return false;
                }
                if (n + (j - i) > static_cast<size_t>(kRowsPerLaunch)) break;
                rb.start[groups++] = static_cast<uint16_t>(n);
                for (; i < j; ++i, ++n) {
                    const RowDst& r = a.rows[order[i]];
                    rb.page[n] = r.page_offset;
                    rb.slot[n] = r.slot;
                    rb.src[n] = r.src_row;
                }
            }
            rb.start[groups] = static_cast<uint16_t>(n);
            hipLaunchKernelGGL(kv_rows_fp8, dim3(groups), dim3(64 * waves), lds, s, rb, kb, vb,
                               reinterpret_cast<const uint16_t*>(a.k_src),
                               reinterpret_cast<const uint16_t*>(a.v_src), a.block_size,
                               a.kv_heads, a.head_dim, a.row_bytes, a.data_bytes);
            KCMM_HIP_CHECK(hipGetLastError(), err);
        }
        return true;
    }
    for (size_t base = 0; base < num; base += kRowsPerLaunch) {
        const size_t n = std::min<size_t>(kRowsPerLaunch, num - base);
        RowBatch rb{};
        for (size_t i = 0; i < n; ++i) {
            const RowDst& r = a.rows[order[base + i]];
            rb.dst[i] = r.page_offset + static_cast<uint64_t>(r.slot) * a.row_bytes;
            rb.src[i] = r.src_row;
        }
        hipLaunchKernelGGL(kv_rows_copy, dim3(n), dim3(256), 0, s, rb, kb, vb,
                           reinterpret_cast<const uint8_t*>(a.k_src),
                           reinterpret_cast<const uint8_t*>(a.v_src), a.row_bytes);
        KCMM_HIP_CHECK(hipGetLastError(), err);
    }
    return true;
}

bool kv_write_device_slots(const KvDeviceSlotsArgs& a, std::string* err) {
    hipStream_t s = reinterpret_cast<hipStream_t>(a.stream);
    SlotArgs sa{};
    sa.slots = reinterpret_cast<const int64_t*>(a.slot_mapping);
    sa.offsets_f16 = reinterpret_cast<const uint64_t*>(a.offsets_f16);
    sa.valid = reinterpret_cast<const uint8_t*>(a.valid_blocks);
    sa.status = reinterpret_cast<int32_t*>(a.status);
    sa.k_base = reinterpret_cast<uint8_t*>(a.k_base);
    sa.v_base = reinterpret_cast<uint8_t*>(a.v_base);
    sa.k_src = reinterpret_cast<const uint8_t*>(a.k_src);
    sa.v_src = reinterpret_cast<const uint8_t*>(a.v_src);
    sa.offsets_len = a.offsets_len;
    sa.block_size = a.block_size;
    sa.row_bytes = a.row_bytes;
    sa.kv_heads = a.kv_heads;
    sa.head_dim = a.head_dim;
    sa.data_bytes = a.data_bytes;
    sa.bs_shift = -1;
    if (a.block_size != 0 && (a.block_size & (a.block_size - 1)) == 0)
        sa.bs_shift = __builtin_ctz(a.block_size);
    if (a.dtype == kDtFP8) {
        if (a.head_dim > 256) {
            *err = "fp8 KV write supports head_dim <= 256";
            return false;
        }
        if (a.batch > 0x7FFFFFFFu || a.offsets_len > (1u << 28)) {
            *err = "fp8 KV write: batch or offset table too large";
            return false;
        }
        if (a.block_size == 0 || a.block_size > kFp8MaxBlockSize) {
            *err = "fp8 KV write supports block_size <= 4096";
            return false;
        }
        if (a.batch == 0) return true;
        int32_t *lead = nullptr, *cnt = nullptr;
        if (a.batch > kFp8ScanRows) {
            // per block id: batch - first row, row count (zero between calls)
            void* ws = nullptr;
            if (!stream_workspace(a.stream, 8, static_cast<size_t>(a.offsets_len) * 8, &ws, true, err))
                return false;
            lead = static_cast<int32_t*>(ws);
            cnt = lead + a.offsets_len;
            hipLaunchKernelGGL(kv_slots_fp8_collect, dim3((a.batch + 255) / 256), dim3(256), 0, s,
                               sa, a.batch, lead, cnt);
            KCMM_HIP_CHECK(hipGetLastError(), err);
        }
        // (the slot tables of R pages take the LDS of one page of kFp8MaxBlockSize)
        // Up to 512 rows of at most 4 kv heads the chip holds a workgroup per row.
        const bool single = a.batch <= 512 && a.kv_heads <= 4;
        const uint32_t R = std::max(1u, std::min({lead != nullptr ? 12u : single ? 1u : (a.batch + 255) / 256,
                                                  kFp8RowsPerGroup, kFp8MaxBlockSize / a.block_size}));
        const uint32_t most = lead != nullptr ? 4u : (a.batch + R - 1) / R > 256 ? 8u : kFp8MaxWaves;
        const uint32_t waves = std::min(2 * a.kv_heads * R, most);
        hipLaunchKernelGGL(kv_slots_fp8_write, dim3((a.batch + R - 1) / R), dim3(64 * waves),
                           static_cast<size_t>(R) * a.block_size * 4, s, sa, a.batch, R, lead, cnt);
    } else {
        hipLaunchKernelGGL(kv_slots_copy, dim3(a.batch), dim3(256), 0, s, sa);
    }
    KCMM_HIP_CHECK(hipGetLastError(), err);
    return true;
}

}  // namespace dev
}  // namespace kcmm
