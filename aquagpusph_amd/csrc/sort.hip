// Stable LSD radix sort (8-bit digits) and the permutation helpers.
//
// Replaces the reference RadixSort tool (aquagpusph/CalcServer/RadixSort.cpp
// :129-303, kernels RadixSort.cl.in:35-323), which sorts 4-bit digits with
// 1024 work-items that each scan a contiguous chunk serially.  Here an array
// of one workgroup's size is sorted by one launch (rs_small); beyond it each
// pass is reduce-then-scan over tiles:
//   1. rs_hist    : per-tile digit histogram (wave-aggregated LDS counters);
//   2. rs_rows    : the first slot of each (digit, tile) within its digit and
//                   the digits' totals (few tiles: rs_scatter adds the table
//                   up itself, RS_DIRECT);
//   3. rs_scatter : ranks the tile's keys, brings them into digit order in
//                   LDS and writes each digit's run; the last pass writes the
//                   inverse permutation as well.
// No kernel waits on another workgroup, so every wave always finishes.
#include <algorithm>

#include "aq_internal.hpp"

namespace aq {

constexpr int RS_BS = 256;  // threads per tile (4 wave64)
constexpr int SC_BS = 256;
constexpr int SC_IPT = 4;
constexpr int SC_TILE = SC_BS * SC_IPT;

__device__ __forceinline__ unsigned lane_id() { return __lane_id(); }

// lanes of the wavefront whose 8-bit digit equals this lane's
__device__ __forceinline__ uint64_t match_digit(uint32_t d, uint64_t active)
{
    uint64_t m = active;
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

// ---- exclusive scan of uint32 ----------------------------------------------
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* ws,
                                                    uint32_t* total)
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) ws[w] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    const int nw = blockDim.x >> 6;
    for (int k = 0; k < nw; k++) {
        if (k < w) off += ws[k];
        tot += ws[k];
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

__global__ void __launch_bounds__(SC_BS)
    scan_reduce(const uint32_t* __restrict__ in, uint32_t m,
                uint32_t* __restrict__ sums)
{
    __shared__ uint32_t ws[SC_BS / 64];
    const size_t base = (size_t)blockIdx.x * SC_TILE + threadIdx.x * SC_IPT;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SC_IPT; k++)
        if (base + k < m) s += in[base + k];
    uint32_t tot;
    block_excl_scan(s, ws, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// single workgroup: exclusive scan of the per-tile sums, any length
__global__ void __launch_bounds__(1024) scan_top(uint32_t* sums, uint32_t nb)
{
    __shared__ uint32_t ws[16];
    uint32_t carry = 0;
    for (uint32_t b = 0; b < nb; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = (i < nb) ? sums[i] : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan(v, ws, &tot);
        if (i < nb) sums[i] = carry + ex;
        carry += tot;
    }
}

__global__ void __launch_bounds__(SC_BS)
    scan_down(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
              uint32_t m, const uint32_t* __restrict__ sums)
{
    __shared__ uint32_t ws[SC_BS / 64];
    const size_t base = (size_t)blockIdx.x * SC_TILE + threadIdx.x * SC_IPT;
    uint32_t v[SC_IPT];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SC_IPT; k++) {
        v[k] = (base + k < m) ? in[base + k] : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t x = block_excl_scan(s, ws, &tot) + sums[blockIdx.x];
#pragma unroll
    for (int k = 0; k < SC_IPT; k++) {
        if (base + k < m) out[base + k] = x;
        x += v[k];
    }
}

// single workgroup: exclusive scan of a short array in chunks of 1024
// (in == out allowed: a chunk is read before any of it is written)
__global__ void __launch_bounds__(1024)
    scan_one(const uint32_t* in, uint32_t* out, uint32_t m)
{
    __shared__ uint32_t ws[16];
    uint32_t carry = 0;
    for (uint32_t b = 0; b < m; b += 1024) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = (i < m) ? in[i] : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan(v, ws, &tot);
        if (i < m) out[i] = carry + ex;
        carry += tot;
    }
}

size_t scan_workspace(uint32_t m) { return (size_t)blocks_for(m, SC_TILE) * 4; }

void exclusive_scan(const uint32_t* in, uint32_t* out, uint32_t m,
                    uint32_t* sums, hipStream_t s)
{
    if (m <= 16384) {
        // one launch for short arrays (the blocked cell order's counts)
        if (m) hipLaunchKernelGGL(scan_one, dim3(1), dim3(1024), 0, s, in, out, m);
        return;
    }
    const unsigned nb = blocks_for(m, SC_TILE);
    hipLaunchKernelGGL(scan_reduce, dim3(nb), dim3(SC_BS), 0, s, in, m, sums);
    hipLaunchKernelGGL(scan_top, dim3(1), dim3(1024), 0, s, sums, nb);
    hipLaunchKernelGGL(scan_down, dim3(nb), dim3(SC_BS), 0, s, in, out, m,
                       sums);
}

// ---- radix sort --------------------------------------------------------------
// Ranks a wavefront's IPT rows of 64 keys among its keys of equal digit, in
// row and lane order (stable), counting them in wc (the wavefront's own
// counters, zero at the start): a row's rank comes from eight ballots
// (match-any), the counter carries the rows before it.  The wavefront's LDS
// operations take effect in order, so no barrier is needed.
template <int IPT>
__device__ __forceinline__ void rank_rows(const uint32_t (&key)[IPT],
                                          uint32_t nrow, int shift,
                                          uint32_t* wc, uint32_t (&rank)[IPT])
{
    const uint32_t lane = lane_id();
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int k = 0; k < 4; k++) wc[k * 64 + lane] = 0;
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const bool valid = (uint32_t)it * 64u + lane < nrow;
        const uint32_t d = (key[it] >> shift) & 255u;
        const uint64_t peers = match_digit(d, __ballot(valid));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint32_t before = wc[d];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        rank[it] = before + (uint32_t)__popcll(peers & lt);
        if (valid && (peers & lt) == 0)
            wc[d] = before + (uint32_t)__popcll(peers);
    }
}

// keys of the calling wavefront's rows, of which the first `base` of the
// array belong to others
__device__ __forceinline__ uint32_t rows_left(uint32_t n, size_t base,
                                              uint32_t most)
{
    return base >= n ? 0u : (uint32_t)min((size_t)most, (size_t)n - base);
}

// counts: digit-major rows of ntiles (rs_rows), or tile-major (direct)
template <int IPT>
__global__ void __launch_bounds__(RS_BS)
    rs_hist(const uint32_t* __restrict__ keys, uint32_t n, int shift,
            uint32_t* __restrict__ counts, uint32_t ntiles, int direct)
{
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    const size_t base = (size_t)blockIdx.x * (RS_BS * IPT);
    const uint64_t lt = (1ull << lane_id()) - 1ull;
    uint32_t key[IPT];
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const size_t idx = base + (size_t)it * RS_BS + tid;
        key[it] = idx < n ? keys[idx] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const bool valid = base + (size_t)it * RS_BS + tid < n;
        const uint32_t d = (key[it] >> shift) & 255u;
        const uint64_t peers = match_digit(d, __ballot(valid));
        if (valid && (peers & lt) == 0)
            atomicAdd(&h[d], (uint32_t)__popcll(peers));
    }
    __syncthreads();
    counts[direct ? (size_t)blockIdx.x * 256 + tid
                  : (size_t)tid * ntiles + blockIdx.x] = h[tid];
}

// one workgroup per digit: exclusive scan of its row, total to totals[digit]
__global__ void __launch_bounds__(RS_BS)
    rs_rows(uint32_t* counts, uint32_t ntiles, uint32_t* __restrict__ totals)
{
    __shared__ uint32_t ws[RS_BS / 64];
    uint32_t* row = counts + (size_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (uint32_t b = 0; b < ntiles; b += RS_BS) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = i < ntiles ? row[i] : 0u;
        uint32_t tot;
        const uint32_t ex = block_excl_scan(v, ws, &tot);
        if (i < ntiles) row[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template <int IPT>
__global__ void __launch_bounds__(RS_BS)
    rs_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
               uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
               uint32_t* __restrict__ inv, uint32_t n, int shift,
               const uint32_t* __restrict__ counts,
               const uint32_t* __restrict__ totals, uint32_t ntiles,
               int direct)
{
    constexpr uint32_t TILE = RS_BS * IPT;
    __shared__ uint32_t wc[RS_BS / 64][256];
    __shared__ uint32_t dbase[256];
    __shared__ uint32_t ws[RS_BS / 64];
    __shared__ uint32_t sk[TILE], sv[TILE];
    const int tid = threadIdx.x;
    const uint32_t w = (uint32_t)tid >> 6, lane = lane_id();
    // a wavefront ranks a contiguous part of the tile
    const size_t tile = (size_t)blockIdx.x * TILE;
    const size_t wbase = tile + (size_t)w * (64 * IPT);
    const uint32_t nrow = rows_left(n, wbase, 64 * IPT);
    uint32_t key[IPT], val[IPT], rank[IPT];
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const uint32_t o = (uint32_t)it * 64u + lane;
        key[it] = o < nrow ? kin[wbase + o] : 0u;
        val[it] = (vin && o < nrow) ? vin[wbase + o] : (uint32_t)wbase + o;
    }
    // the digit's total, and its keys in the tiles before this one
    uint32_t tot = 0, pre = 0;
    if (direct) {
#pragma unroll 8
        for (uint32_t t = 0; t < ntiles; t++) {
            const uint32_t c = counts[(size_t)t * 256 + tid];
            tot += c;
            pre += t < blockIdx.x ? c : 0u;
        }
    } else {
        tot = totals[tid];
        pre = counts[(size_t)tid * ntiles + blockIdx.x];
    }
    rank_rows<IPT>(key, nrow, shift, wc[w], rank);
    uint32_t all;
    const uint32_t start = block_excl_scan(tot, ws, &all) + pre;
    uint32_t c[RS_BS / 64], cnt = 0;
#pragma unroll
    for (int k = 0; k < RS_BS / 64; k++) {
        c[k] = cnt;
        cnt += wc[k][tid];
    }
    const uint32_t ls = block_excl_scan(cnt, ws, &all);
#pragma unroll
    for (int k = 0; k < RS_BS / 64; k++) wc[k][tid] = ls + c[k];
    dbase[tid] = start - ls;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        if ((uint32_t)it * 64u + lane < nrow) {
            const uint32_t q = wc[w][(key[it] >> shift) & 255u] + rank[it];
            sk[q] = key[it];
            sv[q] = val[it];
        }
    }
    __syncthreads();
    const uint32_t nt = rows_left(n, tile, TILE);
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const uint32_t q = (uint32_t)it * RS_BS + tid;
        if (q < nt) {
            const uint32_t k = sk[q], v = sv[q];
            const uint32_t pos = dbase[(k >> shift) & 255u] + q;
            kout[pos] = k;
            vout[pos] = v;
            if (inv) inv[v] = pos;
        }
    }
}

// All passes over at most 1024 * IPT keys by one workgroup, the keys in
// registers and reordered through LDS.
constexpr int RS_SMALL_BS = 1024;
template <int IPT>
__global__ void __launch_bounds__(RS_SMALL_BS)
    rs_small(uint32_t* keys, uint32_t* __restrict__ perm,
             uint32_t* __restrict__ inv, uint32_t n, int passes)
{
    constexpr int NW = RS_SMALL_BS / 64;
    __shared__ uint32_t wc[NW][256];
    __shared__ uint32_t ws[NW];
    __shared__ uint32_t sk[RS_SMALL_BS * IPT], sv[RS_SMALL_BS * IPT];
    const int tid = threadIdx.x;
    const uint32_t w = (uint32_t)tid >> 6, lane = lane_id();
    const uint32_t wbase = w * (64 * IPT);
    const uint32_t nrow = rows_left(n, wbase, 64 * IPT);
    uint32_t key[IPT], val[IPT], rank[IPT];
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const uint32_t o = (uint32_t)it * 64u + lane;
        key[it] = o < nrow ? keys[wbase + o] : 0u;
        val[it] = wbase + o;
    }
    for (int p = 0; p < passes; p++) {
        const int shift = 8 * p;
        rank_rows<IPT>(key, nrow, shift, wc[w], rank);
        __syncthreads();
        uint32_t c[NW], cnt = 0;
        if (tid < 256) {
#pragma unroll
            for (int k = 0; k < NW; k++) {
                c[k] = cnt;
                cnt += wc[k][tid];
            }
        }
        uint32_t all;
        const uint32_t ls = block_excl_scan(cnt, ws, &all);
        if (tid < 256) {
#pragma unroll
            for (int k = 0; k < NW; k++) wc[k][tid] = ls + c[k];
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < IPT; it++) {
            if ((uint32_t)it * 64u + lane < nrow) {
                const uint32_t q = wc[w][(key[it] >> shift) & 255u] + rank[it];
                sk[q] = key[it];
                sv[q] = val[it];
            }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < IPT; it++) {
            const uint32_t o = (uint32_t)it * 64u + lane;
            if (o < nrow) {
                key[it] = sk[wbase + o];
                val[it] = sv[wbase + o];
            }
        }
    }
#pragma unroll
    for (int it = 0; it < IPT; it++) {
        const uint32_t o = (uint32_t)it * 64u + lane;
        if (o < nrow) {
            keys[wbase + o] = key[it];
            perm[wbase + o] = val[it];
            if (inv) inv[val[it]] = wbase + o;
        }
    }
}

// ---- permutations -----------------------------------------------------------
template <typename T>
__global__ void permute_k(const T* __restrict__ src, T* __restrict__ dst,
                          const uint32_t* __restrict__ perm, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[perm[i]];
}

// ---- driver -------------------------------------------------------------
static inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Largest array one workgroup sorts: launches bound the short sorts (two or
// three a pass).  A copy and a sort of uniform keys, us, one launch / passes
// of two: 500 keys of 8 bits 8.5 / 17.0, 2000 of 12 bits 9.5 / 23.4, 4000 of
// 16 bits 13.2 / 23.9, 8000 21.4 / 24.1.  (Tiles of 4096 keys ranked row by
// row between barriers and scattered unordered, three scan launches and an
// inverse permutation of its own took 20.2, 38.8, 49.0 and 54.9.)
constexpr uint32_t RS_SMALL = 8 * RS_SMALL_BS;
// Tiles up to which rs_scatter adds up the table of counts itself, a
// coalesced column walk that costs less than the launch of rs_rows: 65 k keys
// of 20 bits 34.5 / 36.4 us, 131 k 41.6 / 43.4.
constexpr uint32_t RS_DIRECT = 64;

// Keys per thread of a tile of n keys.  Short tiles keep every CU busy, long
// ones write longer runs and shorter tables.  Copy and sort, us, with 4 or 8
// keys per thread / with twice as many (with the earlier passes): 131 k keys
// of 20 bits 41.6 / 51.5 (112.7), 1 M 70.1 / 95.3 (127.4), 4 M 185.8 / 162.8
// (297.1), 4 M of 24 bits 199.0 / 169.8 (339.1).  A pass of 4 M keys moves
// 84 MB, 18 us at the rate of a large copy; beyond that it is the scattered
// runs, of 16 keys (64 B) for uniform digits.
constexpr uint32_t RS_IPT4 = 65536, RS_IPT8 = 2097152;
static inline int rs_ipt(uint32_t n)
{
    return n <= RS_IPT4 ? 4 : n <= RS_IPT8 ? 8 : 16;
}

// What a sort of exactly n keys uses
static size_t rs_bytes(uint32_t n)
{
    const size_t nt = blocks_for(n, RS_BS * rs_ipt(n));
    return align256((size_t)n * 4) * 2 + align256(nt * 256 * 4) +
           align256(256 * 4);
}

// The table of counts halves beyond each line of rs_ipt, so just above one a
// sort uses less than at it; a workspace holds every sort of up to n keys.
size_t radix_sort_workspace(uint32_t n)
{
    size_t b = rs_bytes(n);
    for (const uint32_t line : { RS_IPT4, RS_IPT8 })
        if (n > line) b = std::max(b, rs_bytes(line));
    return b;
}

void radix_sort(uint32_t* keys, uint32_t* perm, uint32_t* inv, uint32_t n,
                unsigned key_bits, void* workspace, hipStream_t s)
{
    if (n == 0) return;
    const int passes = key_bits == 0 ? 1 : (int)((key_bits + 7) / 8);
    if (n <= RS_SMALL) {
#define AQ_RS(IPT)                                                             \
    hipLaunchKernelGGL(rs_small<IPT>, dim3(1), dim3(RS_SMALL_BS), 0, s, keys,  \
                       perm, inv, n, passes)
        if (n <= 1 * RS_SMALL_BS) AQ_RS(1);
        else if (n <= 2 * RS_SMALL_BS) AQ_RS(2);
        else if (n <= 4 * RS_SMALL_BS) AQ_RS(4);
        else AQ_RS(8);
#undef AQ_RS
        return;
    }
    const int ipt = rs_ipt(n);
    const uint32_t nt = blocks_for(n, RS_BS * ipt);
    const int direct = nt <= RS_DIRECT;
    char* w = (char*)workspace;
    uint32_t* kb = (uint32_t*)w;
    w += align256((size_t)n * 4);
    uint32_t* vb = (uint32_t*)w;
    w += align256((size_t)n * 4);
    uint32_t* counts = (uint32_t*)w;
    w += align256((size_t)nt * 256 * 4);
    uint32_t* totals = (uint32_t*)w;
    // The keys alternate between kb and keys, ending in keys; of three passes
    // the first writes them into inv, which only the last pass fills.  The
    // values alternate between vb and perm, chosen so that the last pass
    // writes perm (the first pass reads no values).
    uint32_t *kin = keys, *vin = nullptr;
    for (int p = 0; p < passes; p++) {
        const int shift = 8 * p, left = passes - 1 - p;
        uint32_t* kout = left % 2 == 0 ? keys : kb;
        if (passes % 2 == 1) {
            if (passes == 3 && inv) kout = p == 0 ? inv : p == 1 ? kb : keys;
            else kout = p % 2 == 0 ? kb : keys;
        }
        uint32_t* vout = left % 2 == 0 ? perm : vb;
        uint32_t* iout = left == 0 ? inv : nullptr;
#define AQ_RS(IPT)                                                             \
    do {                                                                       \
        hipLaunchKernelGGL(rs_hist<IPT>, dim3(nt), dim3(RS_BS), 0, s, kin, n,  \
                           shift, counts, nt, direct);                         \
        if (!direct)                                                           \
            hipLaunchKernelGGL(rs_rows, dim3(256), dim3(RS_BS), 0, s, counts,  \
                               nt, totals);                                    \
        hipLaunchKernelGGL(rs_scatter<IPT>, dim3(nt), dim3(RS_BS), 0, s, kin,  \
                           vin, kout, vout, iout, n, shift, counts, totals,    \
                           nt, direct);                                        \
    } while (0)
        if (ipt == 4) AQ_RS(4);
        else if (ipt == 8) AQ_RS(8);
        else AQ_RS(16);
#undef AQ_RS
        kin = kout;
        vin = vout;
    }
    // one pass (or three without an inverse): the sorted keys are in kb
    if (kin != keys)
        AQ_HIP(hipMemcpyAsync(keys, kin, (size_t)n * 4,
                              hipMemcpyDeviceToDevice, s));
}

struct alignas(16) Words8 {
    uint4 a, b;
};

// Several gathers by one permutation in one pass (the perm entry read
// once): dst_f[i] = src_f[perm[i]] for the fields f < n, of 4, 8 or 16
// bytes per element.  Every field's loads are issued before its stores.
constexpr int PERM_BATCH = 8;
struct PermBatch {
    const void* src[PERM_BATCH];
    void* dst[PERM_BATCH];
    int esize[PERM_BATCH];
    int n;
};

__global__ void permute_batch_k(PermBatch b, const uint32_t* __restrict__ perm,
                                uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = perm[i];
    uint4 v[PERM_BATCH];
#pragma unroll
    for (int f = 0; f < PERM_BATCH; f++) {
        if (f >= b.n) break;
        const int es = b.esize[f];
        if (es == 16) {
            v[f] = ((const uint4*)b.src[f])[p];
        } else if (es == 8) {
            const uint2 t = ((const uint2*)b.src[f])[p];
            v[f] = make_uint4(t.x, t.y, 0u, 0u);
        } else {
            v[f] = make_uint4(((const uint32_t*)b.src[f])[p], 0u, 0u, 0u);
        }
    }
#pragma unroll
    for (int f = 0; f < PERM_BATCH; f++) {
        if (f >= b.n) break;
        const int es = b.esize[f];
        if (es == 16)
            ((uint4*)b.dst[f])[i] = v[f];
        else if (es == 8)
            ((uint2*)b.dst[f])[i] = make_uint2(v[f].x, v[f].y);
        else
            ((uint32_t*)b.dst[f])[i] = v[f].x;
    }
}

// Gathers (src[f] -> dst[f], esize[f] bytes per element) by one
// permutation.  Fields of 4, 8 or 16 bytes, none of whose destinations is
// another field's source, go through permute_batch_k, up to PERM_BATCH at
// a time; the others one by one, in order after them.
void permute(const void* src, void* dst, size_t esize, const uint32_t* perm,
             uint32_t n, hipStream_t s);
void permute_many(const void* const* src, void* const* dst,
                  const size_t* esize, int nf, const uint32_t* perm,
                  uint32_t n, hipStream_t s)
{
    if (n == 0 || nf <= 0) return;
    bool ok = true;
    for (int f = 0; f < nf && ok; f++) {
        ok = (esize[f] == 4 || esize[f] == 8 || esize[f] == 16) &&
             src[f] != dst[f];
        for (int g = 0; g < nf && ok; g++) ok = dst[f] != src[g];
    }
    if (!ok) {
        for (int f = 0; f < nf; f++) permute(src[f], dst[f], esize[f], perm, n, s);
        return;
    }
    for (int f0 = 0; f0 < nf; f0 += PERM_BATCH) {
        PermBatch b{};
        b.n = std::min(nf - f0, PERM_BATCH);
        for (int f = 0; f < b.n; f++) {
            b.src[f] = src[f0 + f];
            b.dst[f] = dst[f0 + f];
            b.esize[f] = (int)esize[f0 + f];
        }
        hipLaunchKernelGGL(permute_batch_k, dim3(blocks_for(n, 256)),
                           dim3(256), 0, s, b, perm, n);
    }
}

void permute(const void* src, void* dst, size_t esize, const uint32_t* perm,
             uint32_t n, hipStream_t s)
{
    const dim3 g(blocks_for(n, 256)), b(256);
    switch (esize) {
    case 1:
        hipLaunchKernelGGL(permute_k<uint8_t>, g, b, 0, s, (const uint8_t*)src,
                           (uint8_t*)dst, perm, n);
        break;
    case 2:
        hipLaunchKernelGGL(permute_k<uint16_t>, g, b, 0, s,
                           (const uint16_t*)src, (uint16_t*)dst, perm, n);
        break;
    case 4:
        hipLaunchKernelGGL(permute_k<uint32_t>, g, b, 0, s,
                           (const uint32_t*)src, (uint32_t*)dst, perm, n);
        break;
    case 8:
        hipLaunchKernelGGL(permute_k<uint2>, g, b, 0, s, (const uint2*)src,
                           (uint2*)dst, perm, n);
        break;
    case 16:
        hipLaunchKernelGGL(permute_k<uint4>, g, b, 0, s, (const uint4*)src,
                           (uint4*)dst, perm, n);
        break;
    case 32:
        hipLaunchKernelGGL(permute_k<Words8>, g, b, 0, s, (const Words8*)src,
                           (Words8*)dst, perm, n);
        break;
    default:
        throw Error(AQ_EINVAL, "aq_permute: element size must be 1,2,4,8,16");
    }
}

unsigned radix_key_bits(uint64_t max_val)
{
    uint64_t p = 1;
    while (p < max_val) p <<= 1;
    unsigned bits = 1;
    for (; (p & 1) == 0; p >>= 1, bits++)
        ;
    return (bits + 3u) / 4u * 4u;
}

}  // namespace aq

using namespace aq;

extern "C" {

AQ_API size_t aq_radix_sort_workspace(uint32_t n)
{
    return radix_sort_workspace(n);
}

AQ_API unsigned aq_radix_key_bits(uint64_t max_val)
{
    return radix_key_bits(max_val);
}

AQ_API int aq_radix_sort(uint32_t* keys, uint32_t* perm, uint32_t* inv_perm,
                         uint32_t n, unsigned key_bits, void* workspace,
                         void* stream)
{
    return guard([&] {
        AQ_REQUIRE(keys && perm && (workspace || n == 0),
                   "aq_radix_sort: null pointer");
        AQ_REQUIRE(key_bits <= 32, "aq_radix_sort: key_bits > 32");
        radix_sort(keys, perm, inv_perm, n, key_bits, workspace, S(stream));
    });
}

AQ_API int aq_permute(const void* src, void* dst, size_t esize,
                      const uint32_t* perm, uint32_t N, void* stream)
{
    return guard([&] {
        AQ_REQUIRE(src && dst && perm, "aq_permute: null pointer");
        AQ_REQUIRE(src != dst, "aq_permute: src and dst must differ");
        if (N) permute(src, dst, esize, perm, N, S(stream));
    });
}

}  // extern "C"
