// gdb_group_rows.cpp — a hash-aggregate table's groups in key order, as
// columns, made on the device: what a group-by's result needs instead of the
// whole table copied to the host and its occupied slots sorted there.
//
// Slots are 4 words [key | count << 32, sum, min, max]; the empty key is
// 0xFFFFFFFF. Keys are unique, so the order of the compacted slots does not
// matter and the sort by key makes the result the same every time.

#include "gdb/gdb_hip.h"
#include "gdb/gdb_kernels.h"
#include "gdb_error.h"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace {

typedef unsigned int u32;
typedef unsigned long long u64;

constexpr u32 kEmpty = 0xFFFFFFFFu;
constexpr u32 kSmallRows = GDB_GROUP_ROWS_SMALL;

gdb_status bad(const char* m) { return gdbhip::fail(GDB_ERR_INVALID, m); }

__device__ __forceinline__ u32 lane() { return threadIdx.x & 63u; }
__device__ __forceinline__ u64 lanesBelow() { return (1ull << lane()) - 1ull; }

// --- small tables: one block, everything in LDS ----------------------------
// Bound by latency, not bytes: at 2,048 slots and 700 groups the launch, the
// 4 loads per thread in flight together and 55 bitonic steps. The rows go
// straight to pinned host memory, so the caller waits once and copies nothing.
__device__ __forceinline__ void groupRowsSmall(const u64* __restrict__ tab, u32 slots, u64* __restrict__ out) {
    __shared__ u64 e[kSmallRows];
    __shared__ u32 n_;
    if (threadIdx.x == 0) n_ = 0;
    __syncthreads();
    for (u32 s0 = 0; s0 < slots; s0 += 4096u) {
        u64 w[4];
#pragma unroll
        for (u32 k = 0; k < 4; ++k) {
            const u32 s = s0 + k * 1024u + threadIdx.x;
            w[k] = s < slots ? tab[(u64)s * 4] : (u64)kEmpty;
        }
#pragma unroll
        for (u32 k = 0; k < 4; ++k) {
            const bool occ = (u32)w[k] != kEmpty;
            const u64 m = __ballot(occ);
            if (m == 0) continue;  // the same for the whole wave
            u32 base = 0;
            if (lane() == 0) base = atomicAdd(&n_, (u32)__popcll(m));
            base = (u32)__shfl((int)base, 0, 64);
            const u32 i = base + (u32)__popcll(m & lanesBelow());
            if (occ && i < kSmallRows) e[i] = (w[k] << 32) | (u64)(s0 + k * 1024u + threadIdx.x);
        }
    }
    __syncthreads();
    const u32 n = n_;
    if (n > kSmallRows) {  // the caller takes the general path
        if (threadIdx.x == 0) out[0] = n;
        return;
    }
    u32 P = 2;
    while (P < n) P <<= 1;
    for (u32 i = n + threadIdx.x; i < P; i += 1024u) e[i] = ~0ull;
    __syncthreads();
    for (u32 k = 2; k <= P; k <<= 1) {
        for (u32 j = k >> 1; j > 0; j >>= 1) {
            for (u32 t = threadIdx.x; t < P / 2; t += 1024u) {
                const u32 a = ((t & ~(j - 1u)) << 1) | (t & (j - 1u)), b = a | j;
                const u64 x = e[a], y = e[b];
                if ((x > y) == ((a & k) == 0)) {
                    e[a] = y;
                    e[b] = x;
                }
            }
            __syncthreads();
        }
    }
    u64* const col = out + 8;
    for (u32 i = threadIdx.x; i < n; i += 1024u) {
        const u64* r = tab + (u64)(u32)e[i] * 4;
        col[i] = r[0];
        col[kSmallRows + i] = r[1];
        col[2 * kSmallRows + i] = r[2];
        col[3 * kSmallRows + i] = r[3];
    }
    if (threadIdx.x == 0) out[0] = n;
}
__global__ void __launch_bounds__(1024) groupRowsSmallKernel(const u64* tab, u32 slots, u64* out) {
    groupRowsSmall(tab, slots, out);
}
// Several tables, one block each: they share one launch and one wait, and the
// blocks' latency chains run side by side.
struct GroupTables {
    gdb_group_table t[GDB_GROUP_MANY];
};
__global__ void __launch_bounds__(1024) groupRowsSmallManyKernel(GroupTables all) {
    const gdb_group_table& t = all.t[blockIdx.x];
    groupRowsSmall((const u64*)t.table, (u32)t.slots, (u64*)t.pinned_out);
}

// --- general tables ---------------------------------------------------------
__global__ void clearHeadKernel(u64* head) {
    if (threadIdx.x < 2) head[threadIdx.x] = 0;
}

// Occupied slots as (key << 32 | slot) pairs in any order, their number and
// the largest key. Bound by reading one word of every 32-byte slot, i.e. the
// whole table. Blocks of 8,192 slots: one counter atomic each.
__global__ void __launch_bounds__(1024) groupCompactKernel(const u64* __restrict__ tab, u64 slots,
                                                           u64* __restrict__ pairs, u64* __restrict__ head) {
    __shared__ u32 cnt[16], mx[16];
    __shared__ u64 base_;
    const u32 wave = threadIdx.x >> 6;
    const u64 s0 = (u64)blockIdx.x * 8192u;
    u64 w[8];
#pragma unroll
    for (u32 k = 0; k < 8; ++k) {
        const u64 s = s0 + k * 1024u + threadIdx.x;
        w[k] = s < slots ? __builtin_nontemporal_load(tab + s * 4) : (u64)kEmpty;
    }
    u32 c = 0, m = 0;
#pragma unroll
    for (u32 k = 0; k < 8; ++k) {
        const bool occ = (u32)w[k] != kEmpty;
        c += (u32)__popcll(__ballot(occ));
        if (occ && (u32)w[k] > m) m = (u32)w[k];
    }
#pragma unroll
    for (int d = 32; d; d >>= 1) {
        const u32 o = (u32)__shfl_xor((int)m, d, 64);
        m = o > m ? o : m;
    }
    if (lane() == 0) {
        cnt[wave] = c;
        mx[wave] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 total = 0, top = 0;
        for (u32 i = 0; i < 16; ++i) {
            const u32 x = cnt[i];
            cnt[i] = total;
            total += x;
            top = mx[i] > top ? mx[i] : top;
        }
        base_ = total ? atomicAdd(head, (u64)total) : 0ull;
        if (total) atomicMax(head + 1, (u64)top);
    }
    __syncthreads();
    u64 at = base_ + cnt[wave];
#pragma unroll
    for (u32 k = 0; k < 8; ++k) {
        const bool occ = (u32)w[k] != kEmpty;
        const u64 b = __ballot(occ);
        if (occ) pairs[at + (u32)__popcll(b & lanesBelow())] = (w[k] << 32) | (s0 + k * 1024u + threadIdx.x);
        at += (u32)__popcll(b);
    }
}

// Least-significant-digit radix sort of the pairs by key, 8 bits a pass:
// counts per (digit, tile), their exclusive scan per digit, a stable scatter.
// A tile is 4,096 pairs (256 threads x 16): runs of 16 pairs per digit fill
// 128-byte lines in the scatter. Only the passes the largest key needs run.
constexpr u32 kTile = 4096;

__global__ void __launch_bounds__(256) radixCountKernel(const u64* __restrict__ in, u64 n, int shift, u32 tiles,
                                                        u32* __restrict__ hist) {
    __shared__ u32 h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const u64 b = (u64)blockIdx.x * kTile;
#pragma unroll
    for (u32 k = 0; k < 16; ++k) {
        const u64 i = b + k * 256u + threadIdx.x;
        if (i < n) atomicAdd(&h[(u32)(in[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(u64)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

// Block d: exclusive scan of digit d's counts over the tiles, total last.
__global__ void __launch_bounds__(256) radixScanKernel(u32* __restrict__ hist, u32 tiles, u32* __restrict__ total) {
    __shared__ u32 sum[4];
    u32* const row = hist + (u64)blockIdx.x * tiles;
    u32 carry = 0;
    for (u32 t0 = 0; t0 < tiles; t0 += 256u) {
        const u32 t = t0 + threadIdx.x;
        const u32 v = t < tiles ? row[t] : 0u;
        u32 x = v;  // inclusive over the wave
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const u32 o = (u32)__shfl_up((int)x, d, 64);
            if (lane() >= (u32)d) x += o;
        }
        if (lane() == 63u) sum[threadIdx.x >> 6] = x;
        __syncthreads();
        u32 before = carry, all = 0;
#pragma unroll
        for (u32 i = 0; i < 4; ++i) {
            if (i < (threadIdx.x >> 6)) before += sum[i];
            all += sum[i];
        }
        if (t < tiles) row[t] = before + x - v;
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

__global__ void __launch_bounds__(256) radixScatterKernel(const u64* __restrict__ in, u64 n, int shift, u32 tiles,
                                                          const u32* __restrict__ hist, const u32* __restrict__ total,
                                                          u64* __restrict__ out) {
    __shared__ u32 cnt[4][256];  // per wave and digit: a count, then the next output index
    __shared__ u32 tot[256];
    const u32 wave = threadIdx.x >> 6;
#pragma unroll
    for (u32 i = 0; i < 4; ++i) cnt[i][threadIdx.x] = 0;
    tot[threadIdx.x] = total[threadIdx.x];
    __syncthreads();
    // wave w owns the tile's pairs [1024 w, 1024 w + 1024): row k, then lane
    const u64 b = (u64)blockIdx.x * kTile + wave * 1024u + lane();
    u64 p[16];
    u32 rank[16];
#pragma unroll
    for (u32 k = 0; k < 16; ++k) p[k] = b + k * 64u < n ? in[b + k * 64u] : 0ull;
#pragma unroll
    for (u32 k = 0; k < 16; ++k) {
        const bool ok = b + k * 64u < n;
        const u32 d = (u32)(p[k] >> shift) & 255u;
        u64 same = __ballot(ok);
#pragma unroll
        for (u32 bit = 0; bit < 8; ++bit) {
            const u64 m = __ballot((d >> bit) & 1u);
            same &= (d >> bit) & 1u ? m : ~m;
        }
        const u32 old = cnt[wave][d];
        rank[k] = old + (u32)__popcll(same & lanesBelow());
        __builtin_amdgcn_wave_barrier();
        if (ok && (same & lanesBelow()) == 0) cnt[wave][d] = old + (u32)__popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // digit d (= this thread): where its pairs begin over all digits and tiles
    u32 x = tot[threadIdx.x];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const u32 o = (u32)__shfl_up((int)x, d, 64);
        if (lane() >= (u32)d) x += o;
    }
    __shared__ u32 sum[4];
    if (lane() == 63u) sum[wave] = x;
    __syncthreads();
    u32 at = x - tot[threadIdx.x] + hist[(u64)threadIdx.x * tiles + blockIdx.x];
    for (u32 i = 0; i < wave; ++i) at += sum[i];
#pragma unroll
    for (u32 i = 0; i < 4; ++i) {
        const u32 c = cnt[i][threadIdx.x];
        cnt[i][threadIdx.x] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (u32 k = 0; k < 16; ++k)
        if (b + k * 64u < n) out[cnt[wave][(u32)(p[k] >> shift) & 255u] + rank[k]] = p[k];
}

// Row i of the result: the slot of pair i, its words split into columns
// (32-byte reads at random slots, coalesced writes).
__global__ void __launch_bounds__(256) groupColumnsKernel(const u64* __restrict__ tab, const u64* __restrict__ pairs,
                                                          u64 n, u32* __restrict__ key, u32* __restrict__ count,
                                                          u64* __restrict__ sum, u64* __restrict__ mn,
                                                          u64* __restrict__ mx) {
    const u64 i = (u64)blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const ulonglong2* r = reinterpret_cast<const ulonglong2*>(tab + (u64)(u32)pairs[i] * 4);
    const ulonglong2 a = r[0], b = r[1];
    key[i] = (u32)a.x;
    count[i] = (u32)(a.x >> 32);
    sum[i] = a.y;
    mn[i] = b.x;
    mx[i] = b.y;
}

u32 tilesOf(uint64_t n) { return (u32)((n + kTile - 1) / kTile); }
size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

extern "C" {

gdb_status gdb_group_rows_small(const uint64_t* table, uint64_t slots, uint64_t* pinned_out, gdb_stream s) {
    if (!table || !pinned_out) return bad("gdb_group_rows_small: null argument");
    if (slots > 2 * (uint64_t)kSmallRows) return bad("gdb_group_rows_small: too many slots");
    hipLaunchKernelGGL(groupRowsSmallKernel, dim3(1), dim3(1024), 0, (hipStream_t)s, (const u64*)table, (u32)slots,
                       (u64*)pinned_out);
    return gdbhip::launchCheck("groupRowsSmallKernel");
}

gdb_status gdb_group_rows_small_many(const gdb_group_table* tables, int n, gdb_stream s) {
    if (n < 0 || (n > 0 && !tables)) return bad("gdb_group_rows_small_many: null argument");
    for (int i = 0; i < n; ++i) {
        if (!tables[i].table || !tables[i].pinned_out) return bad("gdb_group_rows_small_many: null argument");
        if (tables[i].slots > 2 * (uint64_t)kSmallRows) return bad("gdb_group_rows_small_many: too many slots");
    }
    for (int i = 0; i < n; i += GDB_GROUP_MANY) {
        GroupTables all{};
        const int m = std::min(n - i, GDB_GROUP_MANY);
        std::copy(tables + i, tables + i + m, all.t);
        hipLaunchKernelGGL(groupRowsSmallManyKernel, dim3((u32)m), dim3(1024), 0, (hipStream_t)s, all);
    }
    return gdbhip::launchCheck("groupRowsSmallManyKernel");
}

gdb_status gdb_group_rows_compact(const uint64_t* table, uint64_t slots, uint64_t* pairs, uint64_t* head, gdb_stream s) {
    if (!table || !pairs || !head) return bad("gdb_group_rows_compact: null argument");
    if (slots > (1ull << 31)) return bad("gdb_group_rows_compact: more than 2^31 slots");
    hipLaunchKernelGGL(clearHeadKernel, dim3(1), dim3(64), 0, (hipStream_t)s, (u64*)head);
    if (slots)
        hipLaunchKernelGGL(groupCompactKernel, dim3((u32)((slots + 8191) / 8192)), dim3(1024), 0, (hipStream_t)s,
                           (const u64*)table, (u64)slots, (u64*)pairs, (u64*)head);
    return gdbhip::launchCheck("groupCompactKernel");
}

size_t gdb_group_rows_scratch_bytes(uint64_t n) {
    return up256((size_t)n * 8) + up256((size_t)256 * tilesOf(n) * 4) + 1024;
}

gdb_status gdb_group_rows_sort(const uint64_t* table, uint64_t* pairs, uint64_t n, uint64_t max_key, void* scratch,
                               uint32_t* key, uint32_t* count, int64_t* sum, int64_t* mn, int64_t* mx, gdb_stream s) {
    if (n == 0) return GDB_OK;
    if (!table || !pairs || !scratch || !key || !count || !sum || !mn || !mx)
        return bad("gdb_group_rows_sort: null argument");
    if (n > (1ull << 31)) return bad("gdb_group_rows_sort: more than 2^31 groups");
    const u32 tiles = tilesOf(n);
    u64* a = (u64*)pairs;
    u64* b = (u64*)scratch;
    u32* hist = (u32*)((char*)scratch + up256((size_t)n * 8));
    u32* total = (u32*)((char*)hist + up256((size_t)256 * tiles * 4));
    for (int bit = 0; bit < 32 && (bit == 0 || (max_key >> bit) != 0); bit += 8) {
        hipLaunchKernelGGL(radixCountKernel, dim3(tiles), dim3(256), 0, (hipStream_t)s, a, (u64)n, 32 + bit, tiles, hist);
        hipLaunchKernelGGL(radixScanKernel, dim3(256), dim3(256), 0, (hipStream_t)s, hist, tiles, total);
        hipLaunchKernelGGL(radixScatterKernel, dim3(tiles), dim3(256), 0, (hipStream_t)s, a, (u64)n, 32 + bit, tiles,
                           hist, total, b);
        u64* t = a;
        a = b;
        b = t;
    }
    hipLaunchKernelGGL(groupColumnsKernel, dim3((u32)((n + 255) / 256)), dim3(256), 0, (hipStream_t)s, (const u64*)table,
                       (const u64*)a, (u64)n, key, count, (u64*)sum, (u64*)mn, (u64*)mx);
    return gdbhip::launchCheck("groupColumnsKernel");
}

}  // extern "C"
