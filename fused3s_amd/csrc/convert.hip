// convert.hip -- CSR -> 16x16 block-sparse conversion on the GPU.
//
// Semantics of convert_csr_to_block_sparse (src/converter.cu:13-44): W =
// ceil(n/16) row windows (:15); for window w the ascending unique set of
// c/16 over the edges (u, c) of rows [16w, min(16w+16, n)) (:19-36);
// window_offsets = exclusive prefix of the set sizes (:39).  New output: the
// 16 row masks of each tile (bit c of row r <=> edge (16w+r, 16b+c)).
//
// Design (no sort; LDS bitmaps with one bit per block column):
//   * list_hubs, the first launch of either pass, lists the hub windows (more
//     than kLightEdges edges);
//   * convert_waves, the main launch: its first workgroups take a hub window
//     each (hub_window: a bitmap sized to the graph, the edges read in chunks
//     of kHubChunk), the others a window per wave, with no workgroup barrier:
//     the edges stay in registers, the bitmap is kept in two levels (a bit
//     per bitmap word, and the words in use side by side), a tile's output
//     rank is the tiles before its word plus the set bits below its own, and
//     row masks and block columns are put together in LDS and leave in
//     coalesced stores;
//   * convert_wide: graphs too wide for that (W > kLightMaxW) take a
//     workgroup per window, the bitmap swept in column slices of kSliceCols
//     block columns (only slices holding an edge of the window are visited).
//     Each thread owns a contiguous run of the window's edges and merges
//     consecutive edges that hit the same LDS word before its atomic; windows
//     with more than NT * kEPT edges re-read them from memory and OR their
//     masks straight into the zeroed output.
// The per-window work is O(E); the output is deterministic and does not
// depend on the order of columns in a row.  Counts become window_offsets
// through counts_to_offsets (two launches).
#include <algorithm>

#include "f3s_common.hpp"
#include "f3s_device.hpp"

namespace f3s {

constexpr int kConvThreads = 256;                 // every main launch's workgroup
constexpr int kBitWords = 2048;                  // bitmap words per column slice
constexpr int kSumWords = kBitWords / 32;         // summary: one bit per bitmap word
constexpr int kSliceCols = kBitWords * 32;        // block columns per slice
constexpr int kMaxSlices = 2048;                  // >= ceil(2^27 / kSliceCols)
constexpr int kEPT = 8;                           // edges per thread kept in registers
constexpr int kHubBatch = 4;                      // edge loads in flight per thread, wide windows
static_assert(kSumWords == kWave, "the summary is scanned by one wave");

// Error flags of a call, one word each: in pinned host memory, cleared by the
// host before the launch, so that a kernel only ever stores to them (an atomic
// OR there would cross PCIe) and no launch clears or copies them.
enum ConvErr : int { kErrRowPtr = 0, kErrCol = 1, kErrCount = 2, kErrWords = 3 };
__device__ __forceinline__ void raise_error(int32_t* err, ConvErr e) { err[e] = 1; }

// The count pass needs only the bitmap; its LDS stays small for occupancy.
// MT tile masks are staged at once (one per thread of the workgroup).
template <bool FILL, int MT>
struct ConvLds {
    uint32_t bits[kBitWords];                  // block columns of the current slice
    uint32_t base[FILL ? kBitWords : 1];       // tiles before each non-empty word
    uint32_t masks[FILL ? MT * 8 : 1];         // row masks of tiles [ms, ms + MT)
    uint16_t list[FILL ? kBitWords : 2];       // non-empty words, ascending
    uint32_t summary[FILL ? kSumWords : 1];    // non-empty bitmap words
    uint32_t slices[kMaxSlices / 32];          // slices holding at least one edge
    int32_t rp[17];
    int32_t scan[MT / kWave];
    int32_t nlist;
    int32_t bad;
};

struct WindowRows {
    int32_t u0, nrows;
    int64_t e0, E;
};

// Loads the window's row pointers into LDS and validates them (threads 0-16).
__device__ __forceinline__ WindowRows load_window_rows(const int32_t* __restrict__ row_ptr,
                                                       int32_t n, int64_t nnz, int32_t w,
                                                       int32_t* rp, int32_t* err)
{
    WindowRows wr;
    wr.u0 = w * 16;
    wr.nrows = min(16, n - wr.u0);
    if ((int)threadIdx.x <= wr.nrows) rp[threadIdx.x] = row_ptr[wr.u0 + threadIdx.x];
    __syncthreads();
    if ((int)threadIdx.x < wr.nrows) {
        int32_t a = rp[threadIdx.x], b = rp[threadIdx.x + 1];
        if (a < 0 || b < a || b > nnz) raise_error(err, kErrRowPtr);
    }
    wr.e0 = rp[0];
    wr.E = (int64_t)rp[wr.nrows] - wr.e0;
    return wr;
}

// Row of the window that holds edge e: the last r < nrows with rp[r] <= e
// (an empty row r has rp[r] == rp[r + 1], so the search passes over it).
__device__ __forceinline__ int row_of_edge(const int32_t* rp, int nrows, int32_t e)
{
    int r = 0;
#pragma unroll
    for (int step = 8; step > 0; step >>= 1)
        if (r + step < nrows && rp[r + step] <= e) r += step;
    return r;
}

// One window by one workgroup of NT threads, any edge count (convert_wide).  Pass kind: COUNT
// writes counts[w]; FILL
// writes block_col / tile_mask at window_offsets[w] and checks the count
// against the offsets.
template <bool FILL, int NT>
__device__ __forceinline__ void
convert_one_window(ConvLds<FILL, NT>& L, int32_t w, const int32_t* __restrict__ row_ptr,
                   const int32_t* __restrict__ col_idx, int32_t n, int64_t nnz, int32_t W,
                   int32_t* __restrict__ counts, const int32_t* __restrict__ window_offsets,
                   int32_t* __restrict__ block_col, uint16_t* __restrict__ tile_mask,
                   int32_t* __restrict__ err)
{
    const int tid = threadIdx.x;
    __syncthreads();   // the previous window of this workgroup is done with L
    if (tid == 0) L.bad = 0;
    if (tid < kMaxSlices / 32) L.slices[tid] = 0u;
    for (int g = tid; g < kBitWords / 4; g += NT)
        *reinterpret_cast<uint4*>(&L.bits[4 * g]) = make_uint4(0u, 0u, 0u, 0u);
    if constexpr (FILL) {
        if (tid < kSumWords) L.summary[tid] = 0u;
    }
    WindowRows wr = load_window_rows(row_ptr, n, nnz, w, L.rp, err);
    __syncthreads();
    if (wr.E < 0 || wr.e0 < 0 || wr.e0 + wr.E > nnz) {
        if (tid == 0) raise_error(err, kErrRowPtr);
        return;
    }
    int32_t out_base = 0, expect = 0;
    if (FILL) {
        // The caller's offsets must describe this CSR (checked against the
        // tile count found below) and stay inside [0, window_offsets[W]],
        // the size of block_col / tile_mask.
        const int32_t total = window_offsets[W];
        out_base = window_offsets[w];
        expect = window_offsets[w + 1] - out_base;
        if (out_base < 0 || expect < 0 || out_base > total - expect) {
            if (tid == 0) raise_error(err, kErrCount);
            return;
        }
    }
    constexpr int kRegEdgesNT = NT * kEPT;
    const int E = (int)wr.E;
    const int32_t e0 = (int32_t)wr.e0;
    const int nrows = wr.nrows;
    // This thread's run of edges: e0 + [i0, i1).
    const int per = (E + NT - 1) / NT;
    const int i0 = min(E, tid * per), i1 = min(E, i0 + per);
    const bool in_regs = E <= kRegEdgesNT;   // i.e. per <= kEPT

    // Visits the run's valid edges (column c, row r) in order.
    int32_t col[kEPT];
    uint32_t rows = 0;
    auto for_each_edge = [&](auto&& fn) {
        if (in_regs) {
#pragma unroll
            for (int j = 0; j < kEPT; ++j)
                if (col[j] >= 0) fn(col[j], (int)((rows >> (4 * j)) & 15u));
        } else {
            // kHubBatch loads in flight per thread, then their edges in order
            int r = i0 < i1 ? row_of_edge(L.rp, nrows, e0 + i0) : 0;
            for (int i = i0; i < i1; i += kHubBatch) {
                int32_t cb[kHubBatch];
#pragma unroll
                for (int j = 0; j < kHubBatch; ++j)
                    cb[j] = i + j < i1 ? col_idx[e0 + i + j] : -1;
#pragma unroll
                for (int j = 0; j < kHubBatch; ++j) {
                    if (i + j < i1) {
                        while (r + 1 < nrows && e0 + i + j >= L.rp[r + 1]) ++r;
                        if (cb[j] >= 0 && cb[j] < n) fn(cb[j], r);
                    }
                }
            }
        }
    };

    // ---- load (registers) or validate (hub), and mark the slices in use ----
    {
        int32_t last_sl = -1;
        auto mark = [&](int32_t c) {
            const int32_t sl = (c >> 4) / kSliceCols;
            if (sl != last_sl) {
                atomicOr(&L.slices[sl >> 5], 1u << (sl & 31));
                last_sl = sl;
            }
        };
        int r = i0 < i1 ? row_of_edge(L.rp, nrows, e0 + i0) : 0;
        if (in_regs) {
#pragma unroll
            for (int j = 0; j < kEPT; ++j) {
                const int i = i0 + j;
                int32_t c = -1;
                if (i < i1) {
                    while (r + 1 < nrows && e0 + i >= L.rp[r + 1]) ++r;
                    c = col_idx[e0 + i];
                    if (c < 0 || c >= n) {
                        L.bad = 1;
                        c = -1;
                    } else {
                        mark(c);
                    }
                }
                col[j] = c;
                rows |= (uint32_t)r << (4 * j);
            }
        } else {
            for (int i = i0; i < i1; i += kHubBatch) {
                int32_t cb[kHubBatch];
#pragma unroll
                for (int j = 0; j < kHubBatch; ++j)
                    cb[j] = i + j < i1 ? col_idx[e0 + i + j] : 0;
#pragma unroll
                for (int j = 0; j < kHubBatch; ++j) {
                    if (cb[j] < 0 || cb[j] >= n)
                        L.bad = 1;
                    else
                        mark(cb[j]);
                }
            }
        }
    }
    __syncthreads();

    const int32_t nslices = (W + kSliceCols - 1) / kSliceCols;
    int32_t running = 0;   // tiles of the slices already done
    for (int32_t sl = 0; sl < nslices; ++sl) {
        if (!((L.slices[sl >> 5] >> (sl & 31)) & 1u)) continue;   // block-uniform
        const int32_t lo = sl * kSliceCols;

        // ---- mark block columns; newly set bits are new tiles ----
        int32_t fresh = 0;
        {
            int32_t cur = -1;
            uint32_t acc = 0;
            auto flush = [&]() {
                if (cur < 0) return;
                const uint32_t old = atomicOr(&L.bits[cur], acc);
                fresh += __popc(acc & ~old);
                if constexpr (FILL) {
                    if (old == 0u) atomicOr(&L.summary[cur >> 5], 1u << (cur & 31));
                }
            };
            for_each_edge([&](int32_t c, int) {
                const int32_t q = (c >> 4) - lo;
                if (q < 0 || q >= kSliceCols) return;
                const int32_t wi = q >> 5;
                if (wi != cur) {
                    flush();
                    cur = wi;
                    acc = 0u;
                }
                acc |= 1u << (q & 31);
            });
            flush();
        }
        int32_t total;
        (void)block_exclusive_scan<NT>(fresh, L.scan, total);   // barriers inside

        if constexpr (FILL) {
            if (running + total <= expect) {
                // ---- ascending list of the non-empty words (one wave) ----
                if (tid < kSumWords) {
                    uint32_t sm = L.summary[tid];
                    const int cnt = __popc(sm);
                    const int incl = wave_inclusive_scan(cnt);
                    int pos = incl - cnt;
                    while (sm) {
                        const int b = __builtin_ctz(sm);
                        sm &= sm - 1u;
                        L.list[pos++] = (uint16_t)(tid * 32 + b);
                    }
                    if (tid == kSumWords - 1) L.nlist = incl;
                }
                __syncthreads();
                // ---- word bases and block columns, contiguous list entries ----
                const int nl = L.nlist;
                const int lper = (nl + NT - 1) / NT;
                const int a0 = min(nl, tid * lper), a1 = min(nl, a0 + lper);
                int32_t loc = 0;
                for (int a = a0; a < a1; ++a) loc += __popc(L.bits[L.list[a]]);
                int32_t tot2;
                int32_t t = block_exclusive_scan<NT>(loc, L.scan, tot2);
                for (int a = a0; a < a1; ++a) {
                    const int wi = L.list[a];
                    L.base[wi] = (uint32_t)t;
                    uint32_t m = L.bits[wi];
                    while (m) {
                        const int b = __builtin_ctz(m);
                        m &= m - 1u;
                        block_col[(int64_t)out_base + running + t] = lo + wi * 32 + b;
                        ++t;
                    }
                }
                __syncthreads();   // bases complete
                if (!in_regs) {
                    // ---- hub window: OR the edge bits straight into the zeroed
                    // output masks (one pass over the edges, not one per round) ----
                    if (tile_mask) {
                        uint4* dst = reinterpret_cast<uint4*>(
                            tile_mask + ((int64_t)out_base + running) * 16);
                        for (int i = tid; i < 2 * total; i += NT)
                            dst[i] = make_uint4(0u, 0u, 0u, 0u);
                        // the zeros reach L2, where the atomics act, before any OR
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                        __syncthreads();
                        uint32_t* gm = reinterpret_cast<uint32_t*>(
                            tile_mask + ((int64_t)out_base + running) * 16);
                        int32_t cur = -1;
                        uint32_t acc = 0;
                        for_each_edge([&](int32_t c, int r) {
                            const int32_t q = (c >> 4) - lo;
                            if (q < 0 || q >= kSliceCols) return;
                            const int32_t wi = q >> 5;
                            const uint32_t below = (1u << (q & 31)) - 1u;
                            const int32_t idx =
                                (int32_t)(L.base[wi] + __popc(L.bits[wi] & below)) * 8 + (r >> 1);
                            if (idx != cur) {
                                if (cur >= 0) atomicOr(&gm[cur], acc);
                                cur = idx;
                                acc = 0u;
                            }
                            acc |= (1u << (c & 15)) << (16 * (r & 1));
                        });
                        if (cur >= 0) atomicOr(&gm[cur], acc);
                    }
                    __syncthreads();
                }
                // ---- tile masks, NT at a time ----
                for (int32_t ms = 0; in_regs && ms < total; ms += NT) {
                    for (int i = tid; i < NT * 2; i += NT)
                        *reinterpret_cast<uint4*>(&L.masks[4 * i]) = make_uint4(0u, 0u, 0u, 0u);
                    __syncthreads();
                    int32_t cur = -1;
                    uint32_t acc = 0;
                    for_each_edge([&](int32_t c, int r) {
                        const int32_t q = (c >> 4) - lo;
                        if (q < 0 || q >= kSliceCols) return;
                        const int32_t wi = q >> 5;
                        const uint32_t below = (1u << (q & 31)) - 1u;
                        const int32_t t2 =
                            (int32_t)(L.base[wi] + __popc(L.bits[wi] & below)) - ms;
                        if (t2 < 0 || t2 >= NT) return;
                        const int32_t idx = t2 * 8 + (r >> 1);
                        if (idx != cur) {
                            if (cur >= 0) atomicOr(&L.masks[cur], acc);
                            cur = idx;
                            acc = 0u;
                        }
                        acc |= (1u << (c & 15)) << (16 * (r & 1));
                    });
                    if (cur >= 0) atomicOr(&L.masks[cur], acc);
                    __syncthreads();
                    if (tile_mask) {
                        const int32_t nt = min(NT, total - ms);
                        for (int t3 = tid; t3 < nt; t3 += NT) {
                            const uint4* src = reinterpret_cast<const uint4*>(&L.masks[t3 * 8]);
                            uint4* dst = reinterpret_cast<uint4*>(
                                tile_mask + ((int64_t)out_base + running + ms + t3) * 16);
                            dst[0] = src[0];
                            dst[1] = src[1];
                        }
                    }
                    __syncthreads();   // masks are cleared by the next round
                }
            }
            if (tid < kSumWords) L.summary[tid] = 0u;
        }
        // ---- leave the bitmap clear for the next slice ----
        for_each_edge([&](int32_t c, int) {
            const int32_t q = (c >> 4) - lo;
            if (q >= 0 && q < kSliceCols) L.bits[q >> 5] = 0u;
        });
        running += total;
        __syncthreads();
    }
    if (tid == 0) {
        if (L.bad) raise_error(err, kErrCol);
        if (FILL) {
            if (running != expect) raise_error(err, kErrCount);
        } else {
            counts[w] = running;
        }
    }
}

// Every window of a graph too wide for convert_waves, a workgroup per window.
template <bool FILL>
__global__ void __launch_bounds__(kConvThreads)
convert_wide(const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ col_idx,
             int32_t n, int64_t nnz, int32_t W, int32_t* __restrict__ counts,
             const int32_t* __restrict__ window_offsets, int32_t* __restrict__ block_col,
             uint16_t* __restrict__ tile_mask, int32_t* __restrict__ err)
{
    __shared__ ConvLds<FILL, kConvThreads> L;
    for (int32_t w = blockIdx.x; w < W; w += gridDim.x)
        convert_one_window<FILL, kConvThreads>(L, w, row_ptr, col_idx, n, nnz, W, counts,
                                               window_offsets, block_col, tile_mask, err);
}

// ---------------------------------------------------------------------------
// Hub windows (more than kLightEdges edges).  list_hubs, the first launch of
// either pass, lists them per block of kListBlock windows: the heavy ones
// (more than kHeavyEdges edges) from the front of the block's part of
// `hubs`, the others from its back, and both counts in seg[block] -- no
// counter to clear first.  (Up to kFindW windows each hub workgroup looks
// through the row pointers itself instead: a launch less.)  The first
// workgroups of the main launch take one listed window each, heavy ones
// first, so that the longest chains start first and the light windows fill
// in behind them (hub workgroups dealt out between the light ones: 8 to 36 us
// slower on 1 M nodes with 1,310 hubs).
// ---------------------------------------------------------------------------
constexpr int kLightEdges = 1024;
constexpr int kHeavyEdges = 4096;
constexpr int kListBlock = 1024;
constexpr int kHubLaunch = 2048;   // hub workgroups of a launch at most (they loop over the list)
constexpr int kLightMaxW = 262144; // windows of the widest graph convert_waves takes
static_assert(kLightMaxW / kListBlock <= kConvThreads, "one thread per block of the list");
constexpr int kFindPer = 8;        // windows a thread looks at
constexpr int kFindW = kConvThreads * kFindPer;

// The window's edges as the main launch counts them too.
__device__ __forceinline__ int32_t window_edges(int32_t first, int32_t end)
{
    return (int32_t)((uint32_t)end - (uint32_t)first);
}

__global__ void __launch_bounds__(kListBlock)
list_hubs(const int32_t* __restrict__ row_ptr, int32_t n, int32_t W, int2* __restrict__ seg,
          int32_t* __restrict__ hubs)
{
    __shared__ int2 part[kListBlock / kWave];
    const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
    const int32_t w = blockIdx.x * kListBlock + t;
    int32_t E = 0;
    if (w < W) E = window_edges(row_ptr[(int64_t)w * 16], row_ptr[min((int64_t)w * 16 + 16, (int64_t)n)]);
    const bool heavy = E > kHeavyEdges, other = E > kLightEdges && !heavy;
    const uint64_t mh = __ballot(heavy), mo = __ballot(other);
    if (lane == 0) part[wid] = make_int2(__popcll(mh), __popcll(mo));
    __syncthreads();
    int2 before = make_int2(0, 0), all = make_int2(0, 0);
#pragma unroll
    for (int i = 0; i < kListBlock / kWave; ++i) {
        const int2 p = part[i];
        if (i < wid) before = make_int2(before.x + p.x, before.y + p.y);
        all = make_int2(all.x + p.x, all.y + p.y);
    }
    const uint64_t below = (1ull << lane) - 1ull;
    int32_t* dst = hubs + (int64_t)blockIdx.x * kListBlock;
    if (heavy) dst[before.x + __popcll(mh & below)] = w;
    if (other) dst[kListBlock - 1 - (before.y + __popcll(mo & below))] = w;
    if (t == 0) seg[blockIdx.x] = all;
}

// Window of hub i (heavy windows first), or -1 past the last: from the list,
// or (seg == NULL) from the row pointers.  Every thread of the workgroup calls
// it; `lds` needs kConvThreads / 64 + 1 int64.
__device__ __forceinline__ int32_t hub_entry(int32_t i, int32_t n, int32_t W,
                                             const int32_t* __restrict__ row_ptr,
                                             const int2* __restrict__ seg,
                                             const int32_t* __restrict__ hubs, int64_t* lds)
{
    const int t = threadIdx.x;
    int32_t* found = reinterpret_cast<int32_t*>(lds + kConvThreads / kWave);
    int2 s = make_int2(0, 0);   // heavy and other hubs of this thread's part
    uint32_t heavy = 0, other = 0;
    if (seg) {
        if (t < (W + kListBlock - 1) / kListBlock) s = seg[t];
    } else {
        int32_t e[kFindPer + 1];
#pragma unroll
        for (int k = 0; k <= kFindPer; ++k)
            e[k] = row_ptr[min(16 * (int64_t)(t * kFindPer + k), (int64_t)n)];
#pragma unroll
        for (int k = 0; k < kFindPer; ++k) {
            const int32_t E = window_edges(e[k], e[k + 1]);
            if (t * kFindPer + k >= W || E <= kLightEdges) continue;
            (E > kHeavyEdges ? heavy : other) |= 1u << k;
        }
        s = make_int2(__popc(heavy), __popc(other));
    }
    if (t == 0) *found = -1;
    int64_t all;
    const int64_t ex = block_exclusive_scan<kConvThreads>(
        (int64_t)s.x | ((int64_t)s.y << 32), lds, all);   // barriers inside
    int32_t h = i - (int32_t)(ex & 0xffffffff);
    int32_t o = i - (int32_t)(all & 0xffffffff) - (int32_t)(ex >> 32);
    if (h >= s.x) h = -1;
    if (i < (int32_t)(all & 0xffffffff) || o >= s.y) o = -1;
    if (h >= 0 || o >= 0) {   // one thread at most
        if (seg) {
            *found = hubs[t * kListBlock + (h >= 0 ? h : kListBlock - 1 - o)];
        } else {
            uint32_t m = h >= 0 ? heavy : other;
            for (int32_t k = max(h, o); k > 0; --k) m &= m - 1u;
            *found = t * kFindPer + __builtin_ctz(m);
        }
    }
    __syncthreads();
    const int32_t w = *found;
    __syncthreads();
    return w;
}

extern __shared__ __align__(16) unsigned char conv_lds[];

__host__ __device__ inline uint32_t align16(uint32_t x) { return (x + 15u) & ~15u; }

// Hub window w by a workgroup of kConvThreads.  Every edge ORs its block
// column's bit into an LDS bitmap sized to the graph; edges are read in
// coalesced chunks of kHubChunk, all loads of a chunk in flight at once.
// Counting, the bits set for the first time are the tiles.  Filling, each
// thread scans a run of bitmap words, and a tile's rank is `chunk` (tiles
// before its run) plus `base` (in the run, before its word) plus the bits
// below its own.  A window of one chunk keeps its edges in registers and
// stages its tiles in LDS, over the bitmap, once their ranks are known; a
// heavier one of few tiles stages them beside it, and one of many ORs its
// edges' bits into its zeroed output.
constexpr int kHubEPT = 16;
constexpr int kHubChunk = kConvThreads * kHubEPT;
static_assert(kHubChunk == kHeavyEdges, "heavy windows are those of more than one chunk");

struct HubHead {
    int64_t scan[kConvThreads / kWave + 1];
    int32_t rp[17];
    uint32_t chunk[kConvThreads];
};

// log2 of the bitmap words per thread
__host__ __device__ inline int hub_shift(int32_t W)
{
    int s = 0;
    while (((W + 31) / 32) > (kConvThreads << s)) ++s;
    return s;
}
// bytes at least: the bitmap (a multiple of 16 bytes) and, filling, a u16 per word
__host__ __device__ inline uint32_t hub_bits_bytes(int32_t W) { return (uint32_t)((W + 127) / 128 * 16); }
__host__ __device__ inline uint32_t hub_work_bytes(int32_t W, bool fill)
{
    const uint32_t b = hub_bits_bytes(W);
    return align16(fill ? b + b / 2 : b);
}

// Staged row masks to the output, coalesced.  `stream` (the output may be
// larger than the Infinity Cache, kStreamTiles, so nobody finds it there
// afterwards): non-temporal stores, which leave the L2 to the edges and to the
// lines the heavy hubs' atomics work on (the fill of 17 M edges with hubs
// 174 -> 130 us; 122 M edges without hubs 512 -> 517 us).
constexpr int64_t kStreamTiles = ((int64_t)256 << 20) / 32;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_masks(uint4* __restrict__ dst, const uint4* src, int count,
                                            int first, int step, bool stream)
{
    if (stream) {
        for (int k = first; k < count; k += step)
            __builtin_nontemporal_store(__builtin_bit_cast(u32x4, src[k]),
                                        reinterpret_cast<u32x4*>(dst) + k);
    } else {
        for (int k = first; k < count; k += step) dst[k] = src[k];
    }
}

template <bool FILL>
__device__ __forceinline__ void
hub_window(int32_t w, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ col_idx,
           int32_t n, int64_t nnz, int32_t W, int32_t* __restrict__ counts,
           const int32_t* __restrict__ window_offsets, int32_t* __restrict__ block_col,
           uint16_t* __restrict__ tile_mask, int32_t cap, bool stream, HubHead& head,
           unsigned char* work, uint32_t work_bytes, int32_t* __restrict__ err)
{
    constexpr int NT = kConvThreads;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // nothing derived from it is kept across windows
    const int words = (W + 31) / 32;
    uint32_t* bits = reinterpret_cast<uint32_t*>(work);
    uint16_t* base = reinterpret_cast<uint16_t*>(work + hub_bits_bytes(W));
    for (uint32_t g = tid; g < hub_bits_bytes(W) / 16; g += NT)
        reinterpret_cast<uint4*>(bits)[g] = make_uint4(0u, 0u, 0u, 0u);
    const WindowRows wr = load_window_rows(row_ptr, n, nnz, w, head.rp, err);   // a barrier inside
    if (wr.E < 0 || wr.e0 < 0 || wr.e0 + wr.E > nnz) {   // uniform
        if (tid == 0) {
            raise_error(err, kErrRowPtr);
            if (!FILL) counts[w] = 0;
        }
        return;
    }
    const uint32_t E = (uint32_t)wr.E;
    const int32_t* cols = col_idx + wr.e0;

    // ---- mark ----
    int32_t col[kHubEPT];
    int32_t fresh = 0;
    bool bad = false;
    for (uint32_t c0 = 0; c0 < E; c0 += kHubChunk) {
#pragma unroll
        for (int j = 0; j < kHubEPT; ++j) {
            const uint32_t e = c0 + tid + NT * j;
            col[j] = e < E ? cols[e] : 0;
        }
#pragma unroll
        for (int j = 0; j < kHubEPT; ++j) {
            const bool in = c0 + tid + NT * j < E;
            const int32_t c = col[j];
            const bool ok = in && (uint32_t)c < (uint32_t)n;
            bad |= in && !ok;
            col[j] = ok ? c : -1;
            if (ok) {
                const uint32_t bit = 1u << ((c >> 4) & 31);
                if constexpr (FILL)
                    atomicOr(&bits[c >> 9], bit);
                else
                    fresh += (atomicOr(&bits[c >> 9], bit) & bit) == 0u;
            }
        }
    }
    if (__any(bad) && (tid & (kWave - 1)) == 0) raise_error(err, kErrCol);
    if constexpr (!FILL) {
        int64_t T;
        (void)block_exclusive_scan<NT>((int64_t)fresh, head.scan, T);   // barriers inside
        if (tid == 0) counts[w] = (int32_t)T;
        return;
    } else {
        const int32_t out_base = window_offsets[w];
        const int32_t expect = window_offsets[w + 1] - out_base;
        // ---- scan ----
        __syncthreads();   // every mark is done
        const int sh = hub_shift(W);
        const int a0 = min(words, tid << sh), a1 = min(words, (tid + 1) << sh);
        int32_t own = 0;
        for (int a = a0; a < a1; ++a) {
            base[a] = (uint16_t)own;
            own += __popc(bits[a]);
        }
        int64_t all;
        const int64_t before = block_exclusive_scan<NT>((int64_t)own, head.scan, all);
        head.chunk[tid] = (uint32_t)before;
        __syncthreads();
        const int32_t total = (int32_t)all;
        // the caller's offsets have to describe this CSR, and stay inside
        // [0, window_offsets[W]], the size of block_col / tile_mask (or cap)
        const bool fits = out_base >= 0 && expect >= 0 &&
                          out_base <= min(window_offsets[W], cap) - expect && total <= expect;
        if ((!fits || total != expect) && tid == 0) raise_error(err, kErrCount);
        if (!fits) return;   // uniform
        auto rank = [&](int32_t c) __attribute__((always_inline)) -> uint32_t {
            const int32_t wi = c >> 9;
            return head.chunk[wi >> sh] + base[wi] +
                   __popc(bits[wi] & ((1u << ((c >> 4) & 31)) - 1u));
        };
        auto load_chunk = [&](uint32_t c0) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kHubEPT; ++j) {
                const uint32_t e = c0 + tid + NT * j;
                col[j] = e < E ? cols[e] : -1;
            }
        };
        auto row_at = [&](uint32_t c0, int j) __attribute__((always_inline)) -> int {
            return row_of_edge(head.rp, wr.nrows, (int32_t)((uint32_t)wr.e0 + c0 + tid + NT * j));
        };
        auto put = [&](uint32_t t, int r, int32_t c, uint32_t* masks, int32_t* tcol)
                       __attribute__((always_inline)) {
            atomicOr(&masks[t * 8 + (r >> 1)], 1u << ((c & 15) + 16 * (r & 1)));
            tcol[t] = c >> 4;   // every edge of the tile writes the same
        };
        // The window's tiles, st at a time: put together at `at`, then stored.
        auto stage_tiles = [&](int32_t tiles, int32_t out, unsigned char* at, int32_t st,
                               auto&& fill) __attribute__((always_inline)) {
            uint32_t* masks = reinterpret_cast<uint32_t*>(at);
            int32_t* tcol = reinterpret_cast<int32_t*>(masks + 8 * st);
            for (int32_t ms = 0; ms < tiles; ms += st) {
                const int32_t nt = min(st, tiles - ms);
                __syncthreads();   // ranks taken, or the last round's tiles read
                for (int k = tid; k < 2 * nt; k += NT)
                    reinterpret_cast<uint4*>(masks)[k] = make_uint4(0u, 0u, 0u, 0u);
                __syncthreads();
                fill((uint32_t)ms, (uint32_t)nt, masks, tcol);
                __syncthreads();
                const int64_t o = (int64_t)out + ms;
                for (int k = tid; k < nt; k += NT) block_col[o + k] = tcol[k];
                if (tile_mask)
                    store_masks(reinterpret_cast<uint4*>(tile_mask + o * 16),
                                reinterpret_cast<const uint4*>(masks), 2 * nt, tid, NT, stream);
            }
        };
        const uint32_t both = align16(hub_bits_bytes(W) * 3 / 2);
        const int32_t beside = (int32_t)((work_bytes - both) / 36) & ~3;   // tiles
        if (E <= kHubChunk) {
            uint32_t aux[kHubEPT];   // rank, row << 16
#pragma unroll
            for (int j = 0; j < kHubEPT; ++j) {
                asm volatile("" : "+v"(col[j]));   // recompute, do not keep from the marking
                aux[j] = 0xffffu;
                if (col[j] >= 0)
                    aux[j] = rank(col[j]) | ((uint32_t)row_at(0u, j) << 16);
            }
            stage_tiles(total, out_base, work, (int32_t)(work_bytes / 36) & ~3,
                        [&](uint32_t ms, uint32_t nt, uint32_t* masks, int32_t* tcol)
                            __attribute__((always_inline)) {
#pragma unroll
                            for (int j = 0; j < kHubEPT; ++j) {
                                asm volatile("" : "+v"(col[j]), "+v"(aux[j]));
                                const uint32_t t = (aux[j] & 0xffffu) - ms;
                                if (t < nt) put(t, (int)(aux[j] >> 16), col[j], masks, tcol);
                            }
                        });
        } else if (total <= 4 * beside) {
            // few tiles for its edges: a stage beside the bitmap, the edges
            // read again for each of at most four rounds
            stage_tiles(total, out_base, work + both, beside,
                        [&](uint32_t ms, uint32_t nt, uint32_t* masks, int32_t* tcol)
                            __attribute__((always_inline)) {
                            for (uint32_t c0 = 0; c0 < E; c0 += kHubChunk) {
                                load_chunk(c0);
#pragma unroll
                                for (int j = 0; j < kHubEPT; ++j) {
                                    if ((uint32_t)col[j] >= (uint32_t)n) continue;
                                    const uint32_t t = rank(col[j]) - ms;
                                    if (t < nt) put(t, row_at(c0, j), col[j], masks, tcol);
                                }
                            }
                        });
        } else {
            uint32_t* gm = reinterpret_cast<uint32_t*>(tile_mask + (int64_t)out_base * 16);
            if (tile_mask) {
                for (int64_t k = tid; k < 2 * (int64_t)total; k += NT)
                    reinterpret_cast<uint4*>(gm)[k] = make_uint4(0u, 0u, 0u, 0u);
                // the zeros reach the L2, where the atomics act, before any OR
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
            }
            // Edges that share words of the masks: a thread takes consecutive
            // ones and ORs a word's bits at once -- atomics of one instruction
            // to one word run one after another (one node joined to 100 k
            // others, the whole conversion: 550 -> 312 us; without masks the
            // coalesced loads below are the better ones, 263 against 282).
            const bool shared = tile_mask && E > 4 * (uint32_t)total;
            for (uint32_t c0 = 0; shared && c0 < E; c0 += kHubChunk) {
                const uint32_t e = c0 + kHubEPT * tid;
#pragma unroll
                for (int j = 0; j < kHubEPT; ++j) col[j] = e + j < E ? cols[e + j] : -1;
                int r = row_of_edge(head.rp, wr.nrows, (int32_t)((uint32_t)wr.e0 + min(e, E - 1)));
                uint32_t left = (uint32_t)(head.rp[r + 1] - (int32_t)wr.e0) - min(e, E - 1);
                int32_t tile = -1;
                uint32_t t = 0, at = 0, acc = 0;
#pragma unroll
                for (int j = 0; j < kHubEPT; ++j) {
                    const int32_t c = col[j];
                    // (left: the row's edges from this one on)
                    while (left == 0 && r + 1 < wr.nrows) {
                        ++r;
                        left = (uint32_t)(head.rp[r + 1] - head.rp[r]);
                    }
                    --left;
                    if ((uint32_t)c >= (uint32_t)n) continue;
                    if (c >> 4 != tile) {
                        tile = c >> 4;
                        t = rank(c);
                        block_col[(int64_t)out_base + t] = tile;   // every edge of the tile: the same
                    }
                    const uint32_t word = t * 8 + (r >> 1);
                    if (word != at && acc) {
                        atomicOr(&gm[at], acc);
                        acc = 0;
                    }
                    at = word;
                    acc |= 1u << ((c & 15) + 16 * (r & 1));
                }
                if (acc) atomicOr(&gm[at], acc);
            }
            for (uint32_t c0 = 0; !shared && c0 < E; c0 += kHubChunk) {
                load_chunk(c0);
#pragma unroll
                for (int j = 0; j < kHubEPT; ++j) {
                    const int32_t c = col[j];
                    if ((uint32_t)c >= (uint32_t)n) continue;
                    const uint32_t t = rank(c);
                    block_col[(int64_t)out_base + t] = c >> 4;   // every edge of the tile: the same
                    if (tile_mask) {
                        const int r = row_at(c0, j);
                        atomicOr(&gm[(int64_t)t * 8 + (r >> 1)], 1u << ((c & 15) + 16 * (r & 1)));
                    }
                }
            }
        }
        __syncthreads();   // the next window's bitmap goes over this one's
    }
}

// ---------------------------------------------------------------------------
// convert_waves, the main pass of graphs of up to kLightMaxW windows: after
// the hub workgroups (above), one window of up to kLightEdges edges per wave,
// no workgroup barrier, the edges in registers (lane + 64 j).  A window's
// block columns are a sparse set, so its bitmap is kept in two levels: `sp`
// has one bit per bitmap word of the graph (32 block columns) and the words
// that hold an edge sit side by side in `bits`.  Per window:
//   mark   every edge ORs its word's bit into sp (a run of edges in one word
//          once); a scan over sp gives each word's place;
//   words  every edge ORs its block column's bit into its word;
//          counting, the set bits are the tiles;
//   ranks  (fill) a scan over the words gives the tiles before each, and an
//          edge's tile is that plus the set bits below its own;
//   stage  (fill) kStageTiles tiles at a time, row masks and block columns
//          are put together in LDS, over the words, and leave in coalesced
//          stores.
// What bounds it (MI355X): on sparse windows the stores, on full ones the
// VALU and LDS instructions (about 65 and 12 per 64 edges when filling).  The
// fill's launch takes 130 us for 1 M nodes and 17 M edges on random ids (hub
// windows included; 0.68 GB, 5.2 TB/s) and 515 us for 2.4 M nodes in
// communities with 122 M edges (2.7 GB, 5.2 TB/s); the former pass of one
// window per 256-thread workgroup, whose barriers and wave 0's walk over the
// summary set the pace, took 207 + 106 us (hubs in launches of their own) and
// 1,000 us.  Counting takes 35 us (39 + 13) and 217 us (209).
// Several windows per wave, the next one's edges in flight, measured slower
// the more there were (both calls of the second graph: 745 us with one, 806
// with two, 945 with sixteen): a prefetch's wait is also a wait for the
// stores of the window before.
// ---------------------------------------------------------------------------
constexpr int kWaveSlots = kLightEdges / kWave;   // edge slots per lane
constexpr int kWaveGroup = 2;                     // slots per uniform branch
constexpr int kWavesPerWg = kConvThreads / kWave;
constexpr int kStageTiles = 160;                  // tiles staged at once (256: 10 % slower, fewer waves)
// a wave's words (u32 bits, and filling u16 tiles before), or its stage
constexpr uint32_t kFillWork = 6 * kLightEdges, kCountWork = 4 * kLightEdges;
static_assert(kStageTiles * 36 <= (int)kFillWork, "the stage fits over the words");

__host__ __device__ inline uint32_t wave_lds_bytes(int32_t sums, bool fill)
{
    return align16(8u * (uint32_t)sums) + 4 * kWave + (fill ? 4 * 32 + 4 * 16 + kFillWork : kCountWork);
}

constexpr uint32_t kHubHead = (sizeof(HubHead) + 15) / 16 * 16;

__host__ __device__ inline uint32_t convert_lds_bytes(int32_t W, bool fill)
{
    const uint32_t light = kWavesPerWg * wave_lds_bytes((W + 1023) / 1024, fill);
    const uint32_t hub = kHubHead + hub_work_bytes(W, fill);
    return light > hub ? light : hub;
}

template <int V>
struct IntC {
    static constexpr int value = V;
};

template <int G, typename Fn>
__device__ __forceinline__ void for_groups_from(int32_t E, Fn& fn)
{
    if constexpr (G * kWaveGroup < kWaveSlots) {
        if (E <= kWave * kWaveGroup * G) return;
        fn(IntC<G>());
        for_groups_from<G + 1>(E, fn);
    }
}

// Calls fn(slot) for the slots that hold one of E edges, kWaveGroup slots per
// uniform branch; fn masks the lanes past the window's last edge.
template <typename Fn>
__device__ __forceinline__ void for_slots(int32_t E, Fn&& fn)
{
    auto group = [&](auto G) __attribute__((always_inline)) {
#pragma unroll
        for (int j = kWaveGroup * G.value; j < kWaveGroup * (G.value + 1); ++j) fn(j);
    };
    for_groups_from<0>(E, group);
}

template <bool FILL>
__global__ void __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(FILL ? 5 : 8)))
convert_waves(const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ col_idx,
              int32_t n, int64_t nnz, int32_t W, int32_t* __restrict__ counts,
              const int32_t* __restrict__ window_offsets, int32_t* __restrict__ block_col,
              uint16_t* __restrict__ tile_mask, int32_t cap, bool stream, int32_t hub_wgs,
              const int2* __restrict__ seg,
              const int32_t* __restrict__ hubs, int32_t* __restrict__ err,
              int64_t* __restrict__ tiles_out)
{
    if ((int32_t)blockIdx.x < hub_wgs) {
        HubHead& head = *reinterpret_cast<HubHead*>(conv_lds);
        for (int32_t i = blockIdx.x;; i += hub_wgs) {
            const int32_t w = hub_entry(i, n, W, row_ptr, seg, hubs, head.scan);
            if (w < 0 || w >= W) return;   // uniform: past the list's end
            hub_window<FILL>(w, row_ptr, col_idx, n, nnz, W, counts, window_offsets, block_col,
                             tile_mask, cap, stream, head, conv_lds + kHubHead,
                             convert_lds_bytes(W, FILL) - kHubHead, err);
        }
    }
    const int lane = threadIdx.x & (kWave - 1);
    // (read into a scalar register: the compiler then knows that everything
    // about the window is the same for the whole wave)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int32_t w = ((int32_t)blockIdx.x - hub_wgs) * kWavesPerWg + wave;
    if (w >= W) return;
    // lane t <= nrows: row_ptr[16 w + t]; filling, lanes 17 and 18 the
    // window's output offsets, lane 19 the tiles in all
    const int nrows = min(16, n - w * 16);
    int32_t v = 0;
    {
        const int32_t* p = nullptr;
        if (lane <= nrows) p = row_ptr + (int64_t)w * 16 + lane;
        if (FILL && (lane == 17 || lane == 18)) p = window_offsets + w + (lane - 17);
        if (FILL && lane == 19) p = window_offsets + W;
        if (p) v = *p;
    }
    if (FILL && w == 0 && lane == 19) *tiles_out = v;   // for the host
    const int32_t sums = (W + 1023) / 1024;
    unsigned char* lds = conv_lds + wave * wave_lds_bytes(sums, FILL);
    uint2* sp = reinterpret_cast<uint2*>(lds);   // .x words that hold an edge, .y words before
    // lanes with nothing to OR do so here, each in its own word
    uint32_t* dummy = reinterpret_cast<uint32_t*>(lds + align16(8u * (uint32_t)sums));
    uint32_t* start = dummy + kWave;   // (fill) a bit for the first edge of each non-empty row
    uint32_t* rowtab = start + 32;     // (fill) the i-th non-empty row
    uint32_t* bits = dummy + kWave + (FILL ? 32 + 16 : 0);
    uint16_t* base = reinterpret_cast<uint16_t*>(bits + kLightEdges);   // (fill) tiles before a word
    uint32_t* masks = bits;   // (fill) the stage, once the ranks are known
    int32_t* tcol = reinterpret_cast<int32_t*>(bits + kStageTiles * 8);
    for (int i = lane; i < sums; i += kWave) sp[i].x = 0u;
    if (FILL && lane < 32) start[lane] = 0u;

    const int32_t e0 = __builtin_amdgcn_readlane(v, 0);
    const int32_t end = __builtin_amdgcn_readlane(v, nrows);
    const int32_t nxt = __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, false);   // lane + 1's
    const bool in_rows = lane < nrows;
    const uint64_t back = __ballot(in_rows && nxt < v);
    const uint64_t nonempty = __ballot(in_rows && nxt > v);
    const int32_t E = window_edges(e0, end);
    const bool rows_ok = back == 0 && e0 >= 0 && end >= e0 && (int64_t)end <= nnz;
    int32_t out_base = 0, expect = 0;
    bool out_ok = true;
    if constexpr (FILL) {
        const int32_t oe = __builtin_amdgcn_readlane(v, 18);
        out_base = __builtin_amdgcn_readlane(v, 17);
        expect = oe - out_base;
        out_ok = out_base >= 0 && oe >= out_base && oe <= min(__builtin_amdgcn_readlane(v, 19), cap);
    }
    if (rows_ok && E > kLightEdges) return;   // a hub window: list_hubs has it
    if (!rows_ok || !out_ok || E == 0) {
        if (lane == 0) {
            if (!FILL) counts[w] = 0;
            if (!rows_ok)
                raise_error(err, kErrRowPtr);
            else if (FILL && (!out_ok || expect != 0))
                raise_error(err, kErrCount);
        }
        return;
    }

    int32_t col[kWaveSlots];
    const __amdgpu_buffer_rsrc_t er = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int32_t*>(col_idx) + e0, (short)0, 4 * E, 0x00020000);
    for_slots(E, [&](int j) __attribute__((always_inline)) {
        col[j] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(er, 4 * lane + 4 * kWave * j, 0, 0);
    });
    if (FILL && ((nonempty >> lane) & 1ull)) {
        const int32_t pos = v - e0;
        atomicOr(&start[pos >> 5], 1u << (pos & 31));
        rowtab[__builtin_amdgcn_mbcnt_lo((uint32_t)nonempty, 0u)] = (uint32_t)lane;
    }

    // ---- mark ----
    bool bad = false;
    for_slots(E, [&](int j) __attribute__((always_inline)) {
        const bool in = lane < E - kWave * j;   // (a scalar subtraction)
        const int32_t c = col[j];
        const bool ok = in && (uint32_t)c < (uint32_t)n;
        bad |= in && !ok;
        const int32_t wi = ok ? c >> 9 : -1;
        col[j] = ok ? c : -1;
        const int32_t pw = __builtin_amdgcn_update_dpp(-1, wi, 0x111, 0xf, 0xf, false);   // lane - 1's
        uint32_t* p = wi != pw ? &sp[wi >> 5].x : &dummy[lane];
        if (!ok) p = &dummy[lane];
        atomicOr(p, 1u << (wi & 31));
    });
    if (__any(bad) && lane == 0) raise_error(err, kErrCol);
    wave_lds_order();
    int32_t nw = 0;
    for (int s0 = 0; s0 < sums; s0 += kWave) {
        const int sw = s0 + lane;
        const int cnt = sw < sums ? __popc(sp[sw].x) : 0;
        const int incl = wave_scan_incl(cnt);
        if (sw < sums) sp[sw].y = (uint32_t)(nw + incl - cnt);
        nw += __builtin_amdgcn_readlane(incl, kWave - 1);
    }
    // ---- words (nw <= E <= kLightEdges) ----
    for (int k = 0; k < nw; k += kWave) bits[k + lane] = 0u;
    wave_lds_order();
    uint32_t aux[kWaveSlots];   // the edge's word; then its place in the masks
    for_slots(E, [&](int j) __attribute__((always_inline)) {
        asm volatile("" : "+v"(col[j]));   // recompute, do not keep across phases
        const int32_t c = col[j];
        const int32_t wi = max(c, 0) >> 9;
        const uint2 s = sp[wi >> 5];
        const uint32_t ci = s.y + __popc(s.x & ((1u << (wi & 31)) - 1u));
        aux[j] = ci;
        atomicOr(c >= 0 ? &bits[ci] : &dummy[lane], 1u << ((c >> 4) & 31));
    });
    wave_lds_order();
    if constexpr (!FILL) {
        int32_t t = 0;
        for (int k = lane; k < nw; k += kWave) t += __popc(bits[k]);
        t = wave_scan_incl(t);
        if (lane == kWave - 1) counts[w] = t;
    } else {
        // ---- ranks ----
        int32_t total = 0;
        for (int k0 = 0; k0 < nw; k0 += kWave) {
            const int k = k0 + lane;
            const int cnt = k < nw ? __popc(bits[k]) : 0;
            const int incl = wave_scan_incl(cnt);
            base[k] = (uint16_t)(total + incl - cnt);
            total += __builtin_amdgcn_readlane(incl, kWave - 1);
        }
        wave_lds_order();
        if (total != expect) {
            if (lane == 0) raise_error(err, kErrCount);
            if (total > expect) return;
        }
        // an edge's row: the first edges of the non-empty rows up to its own
        const uint32_t starts = start[lane & 31];
        const bool full = nonempty == 0xffffull;   // uniform: every row has an edge
        int32_t rowrun = -1;
        for_slots(E, [&](int j) __attribute__((always_inline)) {
            const uint32_t lo = __builtin_amdgcn_readlane(starts, 2 * j);
            const uint32_t hi = __builtin_amdgcn_readlane(starts, 2 * j + 1);
            const uint64_t m = ((uint64_t)hi << 32) | lo;
            const uint64_t m1 = m >> 1;
            const int32_t idx = (int32_t)__builtin_amdgcn_mbcnt_hi(
                (uint32_t)(m1 >> 32),
                __builtin_amdgcn_mbcnt_lo((uint32_t)m1, (uint32_t)(rowrun + (int32_t)(lo & 1u))));
            rowrun += __popcll(m);
            asm volatile("" : "+v"(col[j]));
            const int32_t c = col[j];
            const uint32_t r = full ? (uint32_t)idx : rowtab[idx];
            const uint32_t ci = aux[j];
            const uint32_t below = (1u << ((c >> 4) & 31)) - 1u;
            const uint32_t t = base[ci] + __popc(bits[ci] & below);
            // byte offset of the (tile, row pair) word, its bit's position above
            aux[j] = c >= 0 ? t * 32 + (r >> 1) * 4 + (((c & 15) + 16 * (r & 1)) << 16) : 0xffffu;
        });
        // ---- stage ----
        for (int32_t ms = 0; ms < total; ms += kStageTiles) {
            wave_lds_order();
            const int32_t nt = min(kStageTiles, total - ms);
            for (int k = lane; k < 2 * nt; k += kWave)
                reinterpret_cast<uint4*>(masks)[k] = make_uint4(0u, 0u, 0u, 0u);
            wave_lds_order();
            for_slots(E, [&](int j) __attribute__((always_inline)) {
                asm volatile("" : "+v"(col[j]), "+v"(aux[j]));
                const uint32_t o = (aux[j] & 0xffffu) - (uint32_t)ms * 32;
                if (o < (uint32_t)nt * 32) {
                    atomicOr(&masks[o >> 2], 1u << (aux[j] >> 16));
                    tcol[o >> 5] = col[j] >> 4;   // every edge of the tile writes the same
                }
            });
            wave_lds_order();
            const int64_t o = (int64_t)out_base + ms;
            for (int k = lane; k < nt; k += kWave) block_col[o + k] = tcol[k];
            if (tile_mask) {
                store_masks(reinterpret_cast<uint4*>(tile_mask + o * 16),
                            reinterpret_cast<const uint4*>(masks), 2 * nt, lane, kWave, stream);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Counts -> window_offsets in two launches: block sums, then each workgroup
// adds up the sums of the blocks before its own (at most kOffsFusedBlocks of
// them; wider graphs scan the sums in one workgroup first; a single block
// needs none), scans its block
// straight into the int32 offsets -- T <= nnz <= INT32_MAX, since a tile
// holds at least one edge -- and its last workgroup writes offsets[W] and the
// total in 64 bits.
// ---------------------------------------------------------------------------
constexpr int kOffsThreads = 256;
constexpr int kOffsPerThread = 8;
constexpr int kOffsTile = kOffsThreads * kOffsPerThread;
constexpr int64_t kOffsFusedBlocks = 1024;

__global__ void __launch_bounds__(kOffsThreads)
offsets_block_sums(const int32_t* __restrict__ counts, int64_t W, int64_t* __restrict__ sums)
{
    __shared__ int64_t lds[kOffsThreads / kWave];
    const int64_t base = (int64_t)blockIdx.x * kOffsTile + (int64_t)threadIdx.x * kOffsPerThread;
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kOffsPerThread; ++i)
        if (base + i < W) s += counts[base + i];
    int64_t total;
    (void)block_exclusive_scan<kOffsThreads>(s, lds, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// One workgroup: the block sums into exclusive prefix sums, in place.
__global__ void __launch_bounds__(kOffsThreads)
offsets_scan_sums(int64_t* __restrict__ sums, int64_t nblocks)
{
    __shared__ int64_t lds[kOffsThreads / kWave];
    int64_t carry = 0;
    for (int64_t b0 = 0; b0 < nblocks; b0 += kOffsThreads) {
        const int64_t i = b0 + threadIdx.x;
        const int64_t v = i < nblocks ? sums[i] : 0;
        int64_t total;
        const int64_t ex = block_exclusive_scan<kOffsThreads>(v, lds, total);
        if (i < nblocks) sums[i] = carry + ex;
        carry += total;
    }
}

__global__ void __launch_bounds__(kOffsThreads)
offsets_apply(const int32_t* __restrict__ counts, int64_t W, const int64_t* __restrict__ sums,
              bool scanned, int32_t* __restrict__ offsets, int64_t* __restrict__ total_out)
{
    __shared__ int64_t lds[kOffsThreads / kWave];
    int64_t before;
    if (scanned) {
        before = sums[blockIdx.x];
    } else {
        int64_t part = 0;
        for (int64_t i = threadIdx.x; i < (int64_t)blockIdx.x; i += kOffsThreads) part += sums[i];
        (void)block_exclusive_scan<kOffsThreads>(part, lds, before);
    }
    const int64_t base = (int64_t)blockIdx.x * kOffsTile + (int64_t)threadIdx.x * kOffsPerThread;
    int64_t v[kOffsPerThread];
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kOffsPerThread; ++i) {
        v[i] = (base + i < W) ? counts[base + i] : 0;
        s += v[i];
    }
    int64_t total;
    int64_t ex = block_exclusive_scan<kOffsThreads>(s, lds, total) + before;
#pragma unroll
    for (int i = 0; i < kOffsPerThread; ++i) {
        if (base + i < W) offsets[base + i] = (int32_t)ex;
        ex += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        offsets[W] = (int32_t)(before + total);
        *total_out = before + total;
    }
}

int64_t offsets_sum_elems(int64_t W) { return W > 0 ? ceil_div(W, kOffsTile) : 1; }

f3s_status counts_to_offsets(const int32_t* counts, int32_t* offsets, int64_t W, int64_t* sums,
                             int64_t* total_out, hipStream_t stream)
{
    const int64_t nb = offsets_sum_elems(W);
    if (nb > 1)
        hipLaunchKernelGGL(offsets_block_sums, dim3((unsigned)nb), dim3(kOffsThreads), 0, stream,
                           counts, W, sums);
    const bool scanned = nb > kOffsFusedBlocks;
    if (scanned)
        hipLaunchKernelGGL(offsets_scan_sums, dim3(1), dim3(kOffsThreads), 0, stream, sums, nb);
    hipLaunchKernelGGL(offsets_apply, dim3((unsigned)nb), dim3(kOffsThreads), 0, stream, counts,
                       W, sums, scanned, offsets, total_out);
    F3S_HIP(hipGetLastError());
    return F3S_OK;
}

// The tile count a fill was given, for the host (convert_waves does it itself).
__global__ void report_tiles(const int32_t* __restrict__ window_offsets, int32_t W,
                             int64_t* __restrict__ tiles_out)
{
    if (threadIdx.x == 0) *tiles_out = window_offsets[W];
}

// What a call reports to the host: the tile count and the error flags.
struct ConvertStatus {
    int64_t tiles;
    int32_t err[kErrWords + 1];
};
static_assert(sizeof(ConvertStatus) <= 16 * sizeof(int64_t), "fits the staging words");

// Per-call workspace of the converter, one allocation: the status where no
// pinned memory was to be had, the hub list and, for the count pass, the
// counts and their scan's block sums.
struct ConvertScratch {
    ConvertStatus* status;
    int2* seg;
    int32_t* hubs;
    int32_t* counts;
    int64_t* tmp;
};

static f3s_status convert_scratch(StreamBuffer& buf, int32_t W, bool count, ConvertScratch& s)
{
    const size_t blocks = W > kFindW && W <= kLightMaxW ? (size_t)ceil_div(W, kListBlock) : 0;
    const size_t seg = sizeof(int2) * blocks;
    const size_t hubs = sizeof(int32_t) * blocks * kListBlock;
    const size_t counts = count ? sizeof(int32_t) * (size_t)W : 0;
    const size_t tmp = count ? sizeof(int64_t) * (size_t)offsets_sum_elems(W) : 0;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    F3S_TRY(buf.reserve(al(sizeof(ConvertStatus)) + al(seg) + al(hubs) + al(counts) + al(tmp)));
    char* p = static_cast<char*>(buf.ptr);
    s.status = reinterpret_cast<ConvertStatus*>(p);
    p += al(sizeof(ConvertStatus));
    s.seg = reinterpret_cast<int2*>(p);
    p += al(seg);
    s.hubs = reinterpret_cast<int32_t*>(p);
    p += al(hubs);
    s.counts = reinterpret_cast<int32_t*>(p);
    p += al(counts);
    s.tmp = reinterpret_cast<int64_t*>(p);
    return F3S_OK;
}

// One pass (count or fill) over all windows: one launch of a workgroup per hub
// window and a wave per other window, on larger graphs after the hub list's. A
// valid CSR of nnz edges has at most nnz / (kLightEdges + 1) hub windows; how
// many it has is known on the device only, so that many hub workgroups (at
// most kHubLaunch) look for theirs and leave if there is none.  Graphs too
// wide for a wave's bitmap run every window through the per-window kernel.
template <bool FILL>
static f3s_status launch_pass(const int32_t* row_ptr, const int32_t* col_idx, int32_t n,
                              int64_t nnz, int32_t W, const int32_t* window_offsets,
                              int32_t* block_col, uint16_t* tile_mask, int32_t cap,
                              const ConvertScratch& s, ConvertStatus* status, hipStream_t stream)
{
    if (W <= 0 || W > kLightMaxW) {
        if (W > 0)
            hipLaunchKernelGGL(convert_wide<FILL>, dim3((unsigned)W), dim3(kConvThreads), 0,
                               stream, row_ptr, col_idx, n, nnz, W, s.counts, window_offsets,
                               block_col, tile_mask, status->err);
        if (FILL)
            hipLaunchKernelGGL(report_tiles, dim3(1), dim3(64), 0, stream, window_offsets, W,
                               &status->tiles);
        F3S_HIP(hipGetLastError());
        return F3S_OK;
    }
    const int64_t most = std::min<int64_t>(nnz / (kLightEdges + 1), W);
    const int32_t hub_wgs = (int32_t)std::min<int64_t>(most, kHubLaunch);
    const bool listed = hub_wgs > 0 && W > kFindW;
    if (listed)
        hipLaunchKernelGGL(list_hubs, dim3((unsigned)ceil_div(W, kListBlock)), dim3(kListBlock), 0,
                           stream, row_ptr, n, W, s.seg, s.hubs);
    hipLaunchKernelGGL(convert_waves<FILL>, dim3((unsigned)(hub_wgs + ceil_div(W, kWavesPerWg))),
                       dim3(kConvThreads), convert_lds_bytes(W, FILL), stream, row_ptr, col_idx,
                       n, nnz, W, s.counts, window_offsets, block_col, tile_mask, cap,
                       nnz > kStreamTiles, hub_wgs, listed ? s.seg : nullptr, s.hubs, status->err,
                       &status->tiles);
    F3S_HIP(hipGetLastError());
    return F3S_OK;
}

// Count call: tile counts and their scan into the caller's offsets.  Fill
// call: the lists.  One host round trip each, for T and the error flags, which
// the kernels write to pinned host memory themselves.  `once`: both at once,
// into lists of min(nnz, W * W) entries, with one round trip -- the offsets of
// a CSR that turns out to be invalid may pass the lists' end, so the fill is
// given it.
static f3s_status convert_impl(const int32_t* row_ptr, const int32_t* col_idx, int32_t n,
                               int64_t nnz, int32_t* window_offsets, int32_t* block_col,
                               uint16_t* tile_mask, bool once, int64_t* T_out, hipStream_t stream)
{
    const int32_t W = (int32_t)ceil_div(n, 16);
    const bool count = once || block_col == nullptr;
    StreamBuffer buf(stream);
    ConvertScratch s;
    F3S_TRY(convert_scratch(buf, W, count, s));
    bool pinned = false;
    ConvertStatus* h = reinterpret_cast<ConvertStatus*>(host_staging(&pinned));
    StagingGuard staging(stream);
    *h = ConvertStatus{};
    ConvertStatus* status = pinned ? h : s.status;
    if (!pinned) F3S_HIP(hipMemsetAsync(status, 0, sizeof(ConvertStatus), stream));
    if (count) {
        F3S_TRY(launch_pass<false>(row_ptr, col_idx, n, nnz, W, nullptr, nullptr, nullptr, 0, s,
                                   status, stream));
        F3S_TRY(counts_to_offsets(s.counts, window_offsets, W, s.tmp, &status->tiles, stream));
    }
    if (block_col)
        F3S_TRY(launch_pass<true>(row_ptr, col_idx, n, nnz, W, window_offsets, block_col,
                                  tile_mask,
                                  once ? (int32_t)std::min<int64_t>(nnz, (int64_t)W * W) : INT32_MAX,
                                  s, status, stream));
    F3S_HIP(hipGetLastError());
    if (!pinned)
        F3S_HIP(hipMemcpyAsync(h, status, sizeof(ConvertStatus), hipMemcpyDeviceToHost, stream));
    F3S_HIP(staging.wait());
    const int32_t* err = h->err;
    const int64_t total = h->tiles;
    if (count) {
        // (on an error the offsets written are meaningless, as documented)
        if (err[kErrRowPtr]) {
            set_error("f3s_convert_csr_to_bsf: row_ptr is not monotone within [0, nnz]");
            return F3S_EDATA;
        }
        if (err[kErrCol]) {
            set_error("f3s_convert_csr_to_bsf: a column index is outside [0, n)");
            return F3S_EDATA;
        }
        if (total > INT32_MAX) {
            set_error("f3s_convert_csr_to_bsf: more than 2^31-1 active tiles");
            return F3S_EUNSUPPORTED;
        }
        if (!once) {
            *T_out = total;
            return F3S_OK;
        }
    }
    if (err[kErrRowPtr] || err[kErrCol]) {
        set_error("f3s_convert_csr_to_bsf: CSR violates the format (row_ptr or column range)");
        return F3S_EDATA;
    }
    if (err[kErrCount]) {
        set_error("f3s_convert_csr_to_bsf: window_offsets do not match this CSR "
                  "(call once with d_block_col = NULL first)");
        return F3S_EINVAL;
    }
    *T_out = total;
    return F3S_OK;
}

__global__ void warm_convert_kernel() {}

hipError_t warm_convert(hipStream_t s)
{
    hipLaunchKernelGGL(warm_convert_kernel, dim3(1), dim3(64), 0, s);
    return hipGetLastError();
}

}  // namespace f3s

extern "C" f3s_status f3s_convert_csr_to_bsf(const int32_t* d_row_ptr, const int32_t* d_col_idx,
                                             int32_t n, int64_t nnz, int32_t* d_window_offsets,
                                             int32_t* d_block_col, uint16_t* d_tile_mask,
                                             int64_t* T_out, void* stream)
{
    using namespace f3s;
    F3S_REQUIRE(n >= 0 && nnz >= 0, "f3s_convert_csr_to_bsf: negative size");
    F3S_REQUIRE(nnz <= INT32_MAX, "f3s_convert_csr_to_bsf: nnz exceeds int32 CSR range");
    F3S_REQUIRE(d_row_ptr && d_window_offsets && T_out, "f3s_convert_csr_to_bsf: NULL pointer");
    F3S_REQUIRE(nnz == 0 || d_col_idx, "f3s_convert_csr_to_bsf: NULL col_idx");
    F3S_REQUIRE(!d_tile_mask || d_block_col,
                "f3s_convert_csr_to_bsf: tile_mask requires block_col");
    F3S_TRY(require_device());
    clear_error();
    return convert_impl(d_row_ptr, d_col_idx, n, nnz, d_window_offsets, d_block_col,
                        d_tile_mask, false, T_out, as_stream(stream));
}

extern "C" f3s_status f3s_convert_csr_to_bsf_once(const int32_t* d_row_ptr,
                                                  const int32_t* d_col_idx, int32_t n, int64_t nnz,
                                                  int32_t* d_window_offsets, int32_t* d_block_col,
                                                  uint16_t* d_tile_mask, int64_t* T_out,
                                                  void* stream)
{
    using namespace f3s;
    F3S_REQUIRE(n >= 0 && nnz >= 0, "f3s_convert_csr_to_bsf_once: negative size");
    F3S_REQUIRE(nnz <= INT32_MAX, "f3s_convert_csr_to_bsf_once: nnz exceeds int32 CSR range");
    F3S_REQUIRE(d_row_ptr && d_window_offsets && d_block_col && T_out,
                "f3s_convert_csr_to_bsf_once: NULL pointer");
    F3S_REQUIRE(nnz == 0 || d_col_idx, "f3s_convert_csr_to_bsf_once: NULL col_idx");
    if (ceil_div(n, 16) > kLightMaxW) {
        set_error("f3s_convert_csr_to_bsf_once: n exceeds 4,194,304");
        return F3S_EUNSUPPORTED;
    }
    F3S_TRY(require_device());
    clear_error();
    return convert_impl(d_row_ptr, d_col_idx, n, nnz, d_window_offsets, d_block_col,
                        d_tile_mask, true, T_out, as_stream(stream));
}
