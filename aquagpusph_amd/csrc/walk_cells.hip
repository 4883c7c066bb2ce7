// Cell-parallel neighbour walk with per-lane candidate bitsets.
//
// One wavefront owns one non-empty cell (64 of its particles at a time, one
// per lane); the candidates of the 27 (3D) / 9 (2D) neighbour cells are
// enumerated in the reference order (x offset outermost, then y, then z;
// sorted index inside a cell, types/3D.h:197-219), which is the same list
// for every particle of the cell.  The list is staged 64 candidates at a time
// and goes through a ring:
//
//   test     the lanes load 64 candidates (coalesced) into LDS, those out of
//            reach of the wave's box are dropped, and chunks of 64 survivors
//            are tested against the 64 particles by matrix instructions
//            (dist_tile), which leave each lane a word of accept bits per 32
//            candidates (q < 2 and the wanted particle type);
//   consume  every lane walks its own accepted candidates in increasing
//            order and evaluates the pair terms.  Lanes run ahead as far as
//            the ring has been tested; the oldest chunk is replaced once no
//            lane needs it.
//
// The fluid sums (grad p, lap u, div u, lap p, and the cfd Shepard sum) and
// the boundary-integral Shepard sum take their terms from disjoint candidate
// sets, so they are walked in two passes (the second only in wavefronts
// with a wall element in range), each keeping its terms and their order:
// every lane adds exactly what the reference kernels add, in the same
// order, and the results are bit-identical.  The pair arithmetic runs with
// the lanes that have work instead of under a mask of the lanes that
// accepted the current candidate.
#include <map>
#include <mutex>
#include <type_traits>

#include "aq_device.hpp"
#include "aq_internal.hpp"
#include "coop_device.hpp"
#include "walk_device.hpp"

namespace aq {

// Next cell (index into heads) for the calling wave, n_heads when all are
// taken.  `q` is the wave's current range (starts at its XCD's).
__device__ __forceinline__ uint32_t next_cell(const WalkArgs& w,
                                              uint32_t n_heads, int lane,
                                              uint32_t& q)
{
    uint32_t hk = n_heads;
    if (lane == 0) {
        const uint32_t nr = w.ranges;
        const uint32_t home = q;
        while (q < home + nr) {
            const uint32_t k = q % nr;
            const uint32_t lo = (uint32_t)(((uint64_t)n_heads * k) / nr);
            const uint32_t hi = (uint32_t)(((uint64_t)n_heads * (k + 1)) / nr);
            const uint32_t t = atomicAdd(w.next + k * RSTRIDE, 1u);
            if (t < hi - lo) {
                hk = lo + t;
                break;
            }
            q++;
        }
    }
    return uni(hk);
}

// Shared state of one wavefront of the fused walk: neighbour-cell table,
// staged candidates (two chunks of 64, see dist_tile) and the ring of tested
// chunks (SEGW words of accept bits per lane; positions and indices of their
// candidates, with one chunk more for the survivors staged ahead).
template <int SEGW, bool PER = false> struct RingLds {
    static constexpr uint32_t NCH = SEGW / 2 + 1;  // chunks of `ring`
    uint32_t start[27];
    uint32_t cum[28];
    float4 stage[2][80];
    float4 ring[NCH * 64];
    uint32_t bits[SEGW][64];
    // periodic box: the shift of each neighbour cell's particles, in the
    // gaps of the staged records
    __device__ __forceinline__ float4* shift_slot(uint32_t k)
    {
        return &stage[k >> 4][20u * ((k >> 2) & 3u) + 16u + (k & 3u)];
    }
    __device__ __forceinline__ void set_shift(int k, const float4& v)
    {
        *shift_slot((uint32_t)k) = v;
    }
    __device__ __forceinline__ float4 get_shift(int k)
    {
        return *shift_slot((uint32_t)k);
    }
};

// Walk the accepted candidates of one particle per lane.  `kind` selects
// the candidates (0: fluid particles, imove == 1; 1: wall elements,
// imove == -3); with kind 0 and `flag_el`, wall elements in range are also
// tested and reported through `el_near`.  pair(j, r_j) is called for the
// accepted candidates of each lane in increasing candidate order, r_j the
// candidate's position (at its nearest image in a periodic box).
//
// (A branch-free variant, calling pair() on every lane at every step with a
// dummy index on the idle lanes, measured 25% slower on the 3D dam break:
// the idle lanes' loads and the longer dependent chains cost more than the
// exec-mask changes they save.)
//
// Box prefilter: a candidate farther than the support from the bounding box
// of the active lanes' positions is accepted by no lane, so it is not
// staged.  The box distance is computed like the lanes' own test, one
// rounded subtraction, square and sum per axis in the same order, and
// rounding is monotone, so it never exceeds a lane's s: the prefilter
// drops only candidates every lane would reject.  The survivors are packed,
// in their order, into chunks of 64 across the cells' ends (a quarter of an
// interior 3D cell's candidates is dropped), and a chunk is refilled as soon
// as no lane reads from it.  The window of the ring sets the pace both ways:
// the lanes of a cell accept from different stretches of the list, so a
// narrow one leaves lanes idle, and a wide one scatters their gathers over
// more lines than the cache holds for 16 wavefronts.  3D dam break, 1.2 M /
// 4.5 M particles, walk in us by survivors in the ring: 128: 1867 / 6439,
// 192: 1816 / 6439, 256: 1789 / 6382, 384: 2099 / 7567, 512: 2359 / 8936
// (two slots of 256 list entries, refilled whole: 2014 / 6924).  The
// positions of the ring's candidates are kept in LDS beside their indices,
// which takes the widest of the five gathers of a pair off the cache: 1592 /
// 5534 with 256.  (39.8 KB per workgroup: four per CU, with 1 KB to spare.)
//
// Test: the squared distances of a chunk to the 64 particles by matrix
// instructions (dist_tile), on coordinates relative to the box centre c:
// s' = |r_i - c|^2 + |r_j - c|^2 - 2 (r_i - c).(r_j - c), within 64 ulp of
// R^2 (R bounds |r - c| for every owner and survivor: the half diagonal of
// the box plus the support radius) of the reference's s.  The test s' <=
// smax + 2^-14 R^2 accepts every candidate the exact test accepts, and a few
// within a relative 2^-14 R^2 / smax beyond; the consume repeats the exact
// test (s <= smax) before adding a pair, so the sums are unchanged.
template <int D, int SEGW, bool PER, class Pair>
__device__ __forceinline__ void
ring_walk_m(RingLds<SEGW, PER>& L, int lane, uint32_t total, const f3& r_i,
            bool act, const f3& bmin, const f3& bmax, float smax,
            const float* __restrict__ r, const int* __restrict__ imove,
            int kind, bool flag_el, bool& el_near, Pair pair,
            const float* __restrict__ per)
{
    constexpr uint32_t RING = SEGW;  // words of accept bits per lane
    f3 cen = { 0.f, 0.f, 0.f };
    float limit = smax;
    if (bmin.x <= bmax.x) {
        cen = f3{ uni_f(0.5f * (bmin.x + bmax.x)),
                  uni_f(0.5f * (bmin.y + bmax.y)),
                  D == 3 ? uni_f(0.5f * (bmin.z + bmax.z)) : 0.f };
        const f3 hd = sub<D>(bmax, cen);
        const float rb = sqrtf(dot<D>(hd, hd)) * 1.0001f + sqrtf(smax);
        limit = uni_f(smax + rb * rb * 0x1p-14f);
    }
    // lane (g, o): B and C of the particles o, 16 + o, 32 + o, 48 + o
    const int g = lane >> 4, o = lane & 15;
    float mB[4], mC[4];
    {
        const f3 rio = sub<D>(r_i, cen);
        const float ai = dot<D>(rio, rio);
#pragma unroll
        for (int n = 0; n < 4; n++) {
            const f3 v = { __shfl(rio.x, 16 * n + o),
                           __shfl(rio.y, 16 * n + o),
                           __shfl(rio.z, 16 * n + o) };
            const float av = __shfl(ai, 16 * n + o);
            mB[n] = dist_b(g, v, av);
            mC[n] = dist_c(av, limit);
        }
    }
    uint16_t* half = reinterpret_cast<uint16_t*>(&L.bits[0][0]);
    int kl = 0;        // per-lane cursor: neighbour cell of a candidate
    uint32_t nw = 0;   // next word to load (the current one is nw - 1)
    uint32_t bw = 0;   // remaining bits of the current word
    constexpr uint32_t NCH = RingLds<SEGW, PER>::NCH;
    uint32_t wb = NCH * 64 - 32;  // its first candidate's place in the ring
    uint32_t wt = 0;   // words tested
    uint32_t cb = 0;   // candidates read
    uint32_t ns = 0;   // survivors staged
    bool done = false; // every survivor is tested
    uint64_t elm[2] = { 0, 0 };  // wall elements of the staged chunks
    bool eln = false;
    auto advance = [&]() {
        const uint32_t tw = act ? wt : 0u;
        while (bw == 0 && nw < tw) {
            bw = L.bits[nw % RING][lane];
            nw++;
            wb = wb == NCH * 64 - 32 ? 0u : wb + 32;
        }
    };
    // consume while no chunk can be refilled (a lane still reads from the
    // oldest) and some lane has a candidate left
    auto go = [&]() {
        advance();
        if (!done && (wt < RING ||
                      __ballot(bw != 0 && nw <= wt - RING + 2) == 0))
            return false;
        return __ballot(bw != 0) != 0;
    };
    while (true) {
        // the test sits at the bottom of the consume loop, so the pair sums
        // leave it from where they are updated (no copies at the back edge)
        for (bool more = go(); more; more = go()) {
            if (bw != 0) {
                const uint32_t b = __builtin_clz(bw);
                bw ^= 0x80000000u >> b;
                const float4 c = L.ring[wb + b];
                pair(__float_as_uint(c.w), f3{ c.x, c.y, c.z });
            }
        }
        if (done) break;  // and no lane has a candidate left
        // stage survivors up to a whole chunk (or the candidates' end); the
        // ring has room for two (the oldest chunk and the one before it)
        const uint32_t k0 = wt >> 1;  // the chunk
        const uint32_t in0 = (k0 % NCH) * 64, in1 = ((k0 + 1) % NCH) * 64;
        while (ns < wt * 32 + 64 && cb < total) {
            const uint32_t t = cb + (uint32_t)lane;
            bool take = false, is_el = false;
            uint32_t j = 0;
            f3 rj = { 0.f, 0.f, 0.f };
            float4 st = make_float4(0.f, 0.f, 0.f, 0.f);
            if (t < total) {
                while (t >= L.cum[kl + 1]) kl++;
                j = L.start[kl] + (t - L.cum[kl]);
                rj = ldv_o<D>(r, j);
                const int im_j = ldi_o(imove, j);
                if constexpr (PER) {
                    const float4 sh = L.get_shift(kl);
                    rj = per_shift<D>(rj, f3{ sh.x, sh.y, sh.z }, per);
                }
                is_el = (im_j == -3);
                take = kind ? is_el : (im_j == 1 || (flag_el && is_el));
                if (take) {
                    const float dx =
                        fmaxf(fmaxf(bmin.x - rj.x, rj.x - bmax.x), 0.f);
                    const float dy =
                        fmaxf(fmaxf(bmin.y - rj.y, rj.y - bmax.y), 0.f);
                    float d2 = dx * dx;
                    d2 = d2 + dy * dy;
                    if constexpr (D == 3) {
                        const float dz =
                            fmaxf(fmaxf(bmin.z - rj.z, rj.z - bmax.z), 0.f);
                        d2 = d2 + dz * dz;
                    }
                    take = !(d2 > smax);
                }
                st = dist_stage<D>(sub<D>(rj, cen));
            }
            const uint64_t tm = __ballot(take);
            const uint32_t rank =
                ns + __builtin_amdgcn_mbcnt_hi(
                         (uint32_t)(tm >> 32),
                         __builtin_amdgcn_mbcnt_lo((uint32_t)tm, 0u));
            if (take) {
                L.stage[(rank >> 6) & 1][dist_slot(rank & 63u)] = st;
                L.ring[((rank >> 6) == k0 ? in0 : in1) + (rank & 63u)] =
                    make_float4(rj.x, rj.y, rj.z, __uint_as_float(j));
            }
            if (!kind) {
                uint64_t e = __ballot(take && is_el);
                while (e != 0) {
                    const int b = __builtin_ctzll(e);
                    const uint32_t k =
                        ns + (uint32_t)__popcll(tm & ((1ull << b) - 1ull));
                    if ((k >> 6) & 1) elm[1] |= 1ull << (k & 63u);
                    else elm[0] |= 1ull << (k & 63u);
                    e &= e - 1ull;
                }
            }
            ns += (uint32_t)__popcll(tm);
            cb += 64;
        }
        lds_order();
        const uint32_t have = min(ns - wt * 32, 64u);
        done = cb >= total && ns <= wt * 32 + 64;
        if (have != 0) {
            // the chunk's accept bits: candidates 16 g .. in the upper (g
            // even) or lower half of word wt + g / 2
            const uint32_t hf = (wt >> 1) & 1;
            const float* row = dist_row(L.stage[hf], lane);
            const float A[4] = { row[0], row[16], row[32], row[48] };
            const uint64_t valid =
                have < 64 ? (1ull << have) - 1ull : ~0ull;
            const uint32_t vb = dist_bits(valid, g);
            const uint32_t at =
                2u * (((wt + (uint32_t)(g >> 1)) % RING) * 64u +
                      (uint32_t)o) + ((g & 1) ? 0u : 1u);
#pragma unroll
            for (int n = 0; n < 4; n++) {
                half[at + 32u * (uint32_t)n] =
                    (uint16_t)(dist_tile(A, mB[n], mC[n]) & vb);
                // one tile's results live at a time (registers)
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_order();
            const uint64_t em = hf ? elm[1] : elm[0];
            if (!kind && em != 0) {
                // wall elements in range: flagged, then dropped
                const uint32_t el =
                    __builtin_bitreverse32((uint32_t)em);
                const uint32_t eh =
                    __builtin_bitreverse32((uint32_t)(em >> 32));
                const uint32_t lo = L.bits[wt % RING][lane];
                const uint32_t hi = L.bits[(wt + 1) % RING][lane];
                eln = eln || (act && ((lo & el) | (hi & eh)) != 0);
                L.bits[wt % RING][lane] = lo & ~el;
                L.bits[(wt + 1) % RING][lane] = hi & ~eh;
                if (hf) elm[1] = 0;
                else elm[0] = 0;
            }
            wt += 2;
        }
    }
    el_near = eln;
    lds_order();
}

// ---- one owner per lane over a ring of segments (cell_kernel_k) -------------
// Shared state of one wavefront: neighbour-cell table, the candidate chunk
// being tested and the two segment slots (candidate indices, accept bits;
// SEGW 32-bit words of bits per lane and slot).
template <int SEGW> struct WaveLds {
    uint32_t start[27];
    uint32_t cum[28];
    float4 stage[64];
    uint32_t cand[2][SEGW * 32];
    uint32_t bits[2][SEGW][64];
};

// ring_walk: as ring_walk_m with the exact distances on the vector ALU, for
// candidates of one kind (0 fluid, 1 wall elements).  Batched consume:
// `pair` has load(j), returning
// the candidate's fields, and use(j, fields); each step takes up to NB
// accepted candidates of the lane's current bit word, issues all their
// loads, then uses them in increasing candidate order.  A lane's pair
// terms form a chain of dependent loads (next accepted candidate, its
// fields, the terms), so a walk with few lanes busy (wall cells) is bound
// by the memory latency of that chain; batching takes one latency per NB
// candidates instead of one per candidate, with the same terms in the same
// order.
//
template <int D, int SEGW, int NB, class Pair>
__device__ __forceinline__ void ring_walk(WaveLds<SEGW>& L, int lane,
                                          uint32_t total, const f3& r_i,
                                          bool act, const f3& bmin,
                                          const f3& bmax, float smax,
                                          const float* __restrict__ r,
                                          const int* __restrict__ imove,
                                          int kind, Pair pair)
{
    constexpr uint32_t SEG = SEGW * 32;
    const uint32_t nsegs = (total + SEG - 1) / SEG;
    const uint32_t nwords = (total + 31) >> 5;
    // the two slots form a ring of 2 SEGW words: word w of the candidate
    // list sits at ring position w % (2 SEGW)
    constexpr uint32_t RING = 2 * SEGW;
    const uint32_t* bits = &L.bits[0][0][0];
    const uint32_t* cand = &L.cand[0][0];
    int kl = 0;          // per-lane cursor: neighbour cell of a staged candidate
    uint32_t nw = 0;     // next word to load (the current one is nw - 1)
    uint32_t bw = 0;     // remaining bits of the current word
    uint32_t tested = 0;
    auto advance = [&]() {
        const uint32_t tw = min(tested * SEGW, nwords);
        while (bw == 0 && nw < tw) {
            bw = bits[(nw % RING) * 64 + lane];
            nw++;
        }
    };
    // consume while no slot can be refilled (a lane still reads from the
    // oldest) and some lane has a candidate left
    auto go = [&]() {
        advance();
        if (tested < nsegs &&
            (tested < 2 ||
             __ballot(bw != 0 && nw <= (tested - 1) * SEGW) == 0))
            return false;
        return __ballot(bw != 0) != 0;
    };
    while (true) {
        // the test sits at the bottom of the consume loop, so the pair sums
        // leave it from where they are updated (no copies at the back edge)
        for (bool more = go(); more; more = go()) {
            uint32_t jb[NB];
            int nb = 0;
#pragma unroll
            for (int k = 0; k < NB; k++) {
                jb[k] = 0;
                if (bw != 0) {
                    const uint32_t b = __builtin_clz(bw);
                    bw ^= 0x80000000u >> b;
                    jb[k] = cand[((nw - 1) % RING) * 32 + b];
                    nb = k + 1;
                }
            }
            decltype(pair.load(0u)) cd[NB];
#pragma unroll
            for (int k = 0; k < NB; k++)
                if (k < nb) cd[k] = pair.load(jb[k]);
#pragma unroll
            for (int k = 0; k < NB; k++)
                if (k < nb) pair.use(jb[k], cd[k]);
        }
        if (tested >= nsegs) break;  // and no lane has a candidate left
        // refill the oldest slot: chunk(cb, ...) tests the candidates
        // cb .. cb + 63 of the segment (lane: candidate cb + lane, when
        // `have`, at j, rj, of kind im_j)
        const uint32_t seg = tested * SEG;
        const uint32_t nseg = min(SEG, total - seg);
        const int slot = tested & 1;
        auto chunk = [&](uint32_t cb, bool have, uint32_t j, f3 rj,
                         int im_j) {
            float4 st = make_float4(0.f, 0.f, 0.f, 0.f);
            bool take = false;
            if (have) {
                take = kind ? (im_j == -3) : (im_j == 1);
                if (take) {
                    const float dx =
                        fmaxf(fmaxf(bmin.x - rj.x, rj.x - bmax.x), 0.f);
                    const float dy =
                        fmaxf(fmaxf(bmin.y - rj.y, rj.y - bmax.y), 0.f);
                    float d2 = dx * dx;
                    d2 = d2 + dy * dy;
                    if constexpr (D == 3) {
                        const float dz =
                            fmaxf(fmaxf(bmin.z - rj.z, rj.z - bmax.z), 0.f);
                        d2 = d2 + dz * dz;
                    }
                    take = !(d2 > smax);
                }
                st = make_float4(rj.x, rj.y, rj.z, 0.f);
            }
            // the per-lane test of a staged candidate
            auto accept = [&](const float4& c) {
                const f3 r_ij = sub<D>(f3{ c.x, c.y, c.z }, r_i);
                const float s = dot<D>(r_ij, r_ij);
                return !(s > smax);
            };
            const uint64_t tm = __ballot(take);
            const uint32_t cnt = (uint32_t)__popcll(tm);
            uint32_t lo = 0, hi = 0;
            if (cnt != 0) {
                // compact the survivors into stage[0 .. cnt), in order
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(tm >> 32),
                    __builtin_amdgcn_mbcnt_lo((uint32_t)tm, 0u));
                if (take) {
                    L.stage[rank] = st;
                    L.cand[slot][cb + rank] = j;
                }
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_s_waitcnt(0);
                const uint32_t c1 = cnt < 32u ? cnt : 32u;
#pragma unroll 8
                for (uint32_t k = 0; k < c1; k++)
                    lo = (lo << 1) | (accept(L.stage[k]) ? 1u : 0u);
                if (c1 < 32u) lo <<= 32u - c1;
                if (cnt > 32u) {
#pragma unroll 8
                    for (uint32_t k = 32; k < cnt; k++)
                        hi = (hi << 1) | (accept(L.stage[k]) ? 1u : 0u);
                    if (cnt < 64u) hi <<= 64u - cnt;
                }
                if (!act) lo = hi = 0;
            }
            L.bits[slot][cb >> 5][lane] = lo;
            if (nseg - cb > 32) L.bits[slot][(cb >> 5) + 1][lane] = hi;
            __builtin_amdgcn_wave_barrier();
        };
        // the whole segment's candidate loads issued together
        constexpr uint32_t NCH = SEG / 64;
        uint32_t pj[NCH];
        f3 prj[NCH];
        int pim[NCH];
#pragma unroll
        for (uint32_t ch = 0; ch < NCH; ch++) {
            pj[ch] = 0;
            const uint32_t t = seg + ch * 64 + lane;
            if (ch * 64 + lane < nseg) {
                while (t >= L.cum[kl + 1]) kl++;
                pj[ch] = L.start[kl] + (t - L.cum[kl]);
            }
        }
#pragma unroll
        for (uint32_t ch = 0; ch < NCH; ch++) {
            prj[ch] = f3{ 0.f, 0.f, 0.f };
            pim[ch] = 0;
            if (ch * 64 + lane < nseg) {
                prj[ch] = ldv_o<D>(r, pj[ch]);
                pim[ch] = ldi_o(imove, pj[ch]);
            }
        }
#pragma unroll
        for (uint32_t ch = 0; ch < NCH; ch++) {
            if (ch * 64 >= nseg) break;
            chunk(ch * 64, ch * 64 + lane < nseg, pj[ch], prj[ch],
                  pim[ch]);
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_s_waitcnt(0);
        tested++;
    }
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// Fused fluid walk (same terms as fluid_pass_k in sph.hip).
//   MATH 0: IEEE-754 terms and sums, bit-identical to the oracle;
//   MATH 1: OpenCL relaxed-math terms (reciprocals, hardware sqrt, fma);
//   MATH 2: the IEEE terms with compensated (Neumaier) sums for the
//           momentum (grad_p, lap_u) and density (div_u, lap_p) rates.
// ---------------------------------------------------------------------------
__constant__ const uint32_t rec_init[NREC] = { 0x7F800000u, 0u, 0xFFFFFFFFu,
                                               0u, 0xFFFFFFFFu, 0u, 0u };

__device__ __forceinline__ uint32_t wave_min(uint32_t x)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
        x = min(x, (uint32_t)__shfl_xor((int)x, o));
    return x;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
        x = max(x, (uint32_t)__shfl_xor((int)x, o));
    return x;
}

template <int D>
__global__ void __launch_bounds__(256)
    fluid_ranges_k(const int* __restrict__ imove, const float* __restrict__ p,
                   const float* __restrict__ rho, const float* __restrict__ m,
                   const float* __restrict__ u, uint32_t N,
                   uint32_t* __restrict__ rec)
{
    uint32_t v[NREC];
#pragma unroll
    for (uint32_t k = 0; k < NREC; k++) v[k] = rec_init[k];
    // four particles per thread and pass, every load issued before the
    // fluid tests
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < N;
         i0 += 4 * stride) {
        int im[4];
        uint32_t pa[4], rb[4], mb[4];
        f3 uu[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t i = i0 + t * stride;
            im[t] = 0;
            if (i < N) {
                im[t] = imove[i];
                pa[t] = __float_as_uint(p[i]) & 0x7FFFFFFFu;
                rb[t] = __float_as_uint(rho[i]);
                mb[t] = __float_as_uint(m[i]);
                uu[t] = ldv<D>(u, i);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (im[t] != 1) continue;
            const uint32_t pa_ = pa[t], rb_ = rb[t], mb_ = mb[t];
            const f3 ui = uu[t];
            if (pa_) v[0] = min(v[0], pa_);
            v[1] = max(v[1], pa_);
            v[2] = min(v[2], rb_);
            v[3] = max(v[3], rb_);
            v[4] = min(v[4], mb_);
            v[5] = max(v[5], mb_);
            uint32_t ua = max(__float_as_uint(ui.x) & 0x7FFFFFFFu,
                              __float_as_uint(ui.y) & 0x7FFFFFFFu);
            if constexpr (D == 3) ua = max(ua, __float_as_uint(ui.z) & 0x7FFFFFFFu);
            v[6] = max(v[6], ua);
        }
    }
    __shared__ uint32_t part[4][NREC];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (uint32_t k = 0; k < NREC; k++) {
        const bool is_min = (k == 0 || k == 2 || k == 4);
        const uint32_t x = is_min ? wave_min(v[k]) : wave_max(v[k]);
        if (lane == 0) part[wv][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < NREC) {
        const uint32_t k = threadIdx.x;
        const bool is_min = (k == 0 || k == 2 || k == 4);
        uint32_t x = part[0][k];
        for (int w2 = 1; w2 < 4; w2++)
            x = is_min ? min(x, part[w2][k]) : max(x, part[w2][k]);
        if (is_min) atomicMin(rec + k * RSTRIDE, x);
        else atomicMax(rec + k * RSTRIDE, x);
    }
}

template <int D, int SHEP, bool LAPP, int SEGW, int LAPF, int MATH,
          bool PER = false>
__global__ void __launch_bounds__(64 * WC_WAVES)
    fluid_pass_cells_k(const int* __restrict__ imove,
                       const float* __restrict__ r,
                       const float* __restrict__ u,
                       const float* __restrict__ rho,
                       const float* __restrict__ m,
                       const float* __restrict__ p,
                       const float* __restrict__ normal,
                       const float* __restrict__ tangent,
                       const float* __restrict__ binormal,
                       float* __restrict__ shepard, float* __restrict__ grad_p,
                       float* __restrict__ lap_u, float* __restrict__ div_u,
                       float* __restrict__ lap_p, uint8_t* __restrict__ near,
                       WalkArgs w, float H, float CONW, float CONF, float DIMS,
                       float smax, float iH, const uint32_t* __restrict__ rec)
{
    constexpr float CLEARY = (D == 2) ? 8.f : 10.f;
    __shared__ RingLds<SEGW, PER> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    RingLds<SEGW, PER>& L = lds[wv];
    if (w.status && (*w.status & 1u)) return;
    const uint32_t n_heads = uni(*w.n_heads);
    const float eps = 1E-8f * H;
    // wall elements in range are needed for the boundary-integral Shepard
    // sum and for the near-wall flags
    const bool flag_el = (SHEP == 2) || (near != nullptr);
    // divisions and square roots without range scaling (div_nr, sqrt_nr)
    // when the range record allows them; IEEE sequences otherwise
    float fdT = 0.f;
    if constexpr (MATH != 1)
        if (rec) fdT = fast_threshold<D>(rec, H, CONF, smax, LAPF, LAPP);
    const bool fastdiv = fdT > 0.f;
    const Rcp RH = rcp_nr(H);

    uint32_t range = blockIdx.x % w.ranges;
    while (true) {
        // cells are handed out one at a time (a vector atomic from lane 0)
        const uint32_t hk = next_cell(w, n_heads, lane, range);
        if (hk >= n_heads) break;
        uint32_t cstart, c_i, ce;
        if (w.blist) {
            cstart = uni(w.blist[3 * hk]);
            c_i = uni(w.blist[3 * hk + 1]);
            ce = uni(w.blist[3 * hk + 2]);
        } else {
            cstart = uni(w.heads[hk]);
            c_i = uni(w.icell[cstart]);
            ce = uni(w.cell_end[c_i]);
        }
        const uint32_t cend = ce & AQ_CELL_END;
        if (w.flagged && !(ce & AQ_CELL_FLUID)) continue;  // no fluid here
        bool cell_near = false;  // some fluid particle of the cell is near
        for (uint32_t i0 = cstart; i0 < cend; i0 += 64) {
            const uint32_t i = i0 + lane;
            const bool act = (i < cend) && (imove[i] == 1);
            if (__ballot(act) == 0) continue;  // no fluid particle here
            const uint32_t total = neighbour_table<D, PER>(
                w, c_i, L, lane,
                AQ_CELL_FLUID | (flag_el ? AQ_CELL_ELEM : 0u));
            f3 r_i = { 0.f, 0.f, 0.f }, u_i = { 0.f, 0.f, 0.f };
            float p_i = 0.f, rho_i = 1.f;
            f3 gp = { 0.f, 0.f, 0.f }, lu = { 0.f, 0.f, 0.f };
            float dv = 0.f, lp = 0.f, sh = 0.f;
            // compensations (MATH 2)
            f3 cgp = { 0.f, 0.f, 0.f }, clu = { 0.f, 0.f, 0.f };
            float cdv = 0.f, clp = 0.f;
            if (act) {
                r_i = ldv<D>(r, i);
                u_i = ldv<D>(u, i);
                p_i = p[i];
                rho_i = rho[i];
                gp = ldv<D>(grad_p, i);
                lu = ldv<D>(lap_u, i);
                dv = div_u[i];
                if (LAPP) lp = lap_p[i];
                sh = (SHEP == 2) ? 1.f : (SHEP == 1 ? shepard[i] : 0.f);
            }
            constexpr bool FAST = MATH == 1;
            const float irho_i = FAST ? __builtin_amdgcn_rcpf(rho_i) : 0.f;
            // ---- fluid neighbours ------------------------------------------
            bool nearw = false;
            f3 bmin, bmax;
            wave_box<D>(r_i, act, bmin, bmax);
            // pair terms; FD selects div_nr for the divisions
            auto terms = [&](auto fd, const f3& r_ij, float q, float m_j,
                             float rho_j, float p_j, const f3& u_ij,
                             float udr) {
                constexpr bool FD = decltype(fd)::value;
                // The reference skips j == i here.  For i itself r_ij,
                // u_ij and p_j - p_i are exact zeros, so every term below
                // is +-0 and leaves the accumulators unchanged (they are
                // never -0: they start at +0 and an exact cancellation
                // rounds to +0); with finite fields the sums are
                // bit-identical without the test.
                const PairTerms pt = fluid_pair<D, SHEP, FD>(
                    LAPF, LAPP, q, m_j, rho_j, p_j, udr, p_i, rho_i, H, CONW,
                    CONF);
                if (SHEP == 1) sh += pt.sh;
                const float sg = pt.sg, sl = pt.sl, td = pt.td, tl = pt.tl;
                if constexpr (MATH == 2) {
                    naxpy<D>(gp, cgp, sg, r_ij);
                    naxpy<D>(lu, clu, sl,
                             LAPF == AQ_LAP_MONAGHAN ? r_ij : u_ij);
                    nsum(dv, cdv, td);
                    if (LAPP) nsum(lp, clp, tl);
                } else {
                    axpy<D>(gp, sg, r_ij);
                    axpy<D>(lu, sl, LAPF == AQ_LAP_MONAGHAN ? r_ij : u_ij);
                    dv += td;
                    if (LAPP) lp += tl;
                }
            };
            // div_nr / sqrt_nr where the per-pair bounds hold (s == 0 or
            // s >= 2^-96, udr == 0 or |udr| >= T), the IEEE sequences for
            // the other pairs
            // The relative-coordinate test accepts a thin shell beyond the
            // support.  Such a candidate is given zero mass here
            // (the reference's test, s <= smax, as a select rather than a
            // branch, so every load of the pair is issued at once): its
            // terms are then +-0 (finite fields), and adding +-0 leaves the
            // sums unchanged, since they are never -0 (they start at +0, or
            // 1, and an exact cancellation rounds to +0).  SKIP: it is
            // passed over, whatever its fields hold.
            constexpr bool SKIP = PER || FAST;
            auto pair_fd = [&](uint32_t j, const f3& r_j) {
                const f3 r_ij = sub<D>(r_j, r_i);
                const float s = dot<D>(r_ij, r_ij);
                if (SKIP && s > smax) return;
                const float qf = div_nr(sqrt_nr(s), RH);
                float m_j = ldf_o(m, j);
                m_j = (s > smax) ? 0.f : m_j;
                const float rho_j = ldf_o(rho, j);
                const float p_j = ldf_o(p, j);
                const f3 u_ij = sub<D>(ldv_o<D>(u, j), u_i);
                const float udr = dot<D>(u_ij, r_ij);
                const bool bad = ((s < 0x1p-96f) & (s != 0.f)) |
                                 ((udr != 0.f) & (fabsf(udr) < fdT));
                if (!bad)
                    terms(std::true_type{}, r_ij, qf, m_j, rho_j, p_j, u_ij,
                          udr);
                else
                    terms(std::false_type{}, r_ij, sqrtf(s) / H, m_j, rho_j,
                          p_j, u_ij, udr);
            };
            auto pair_ieee = [&](uint32_t j, const f3& r_j) {
                    if constexpr (FAST) {
                        // OpenCL C default accuracy: reciprocal-based
                        // division, hardware square root, contracted
                        // multiply-adds
                        const f3 r_ij = sub<D>(r_j, r_i);
                        const float s = fdot<D>(r_ij, r_ij);
                        if (SKIP && s > smax) return;
                        const float q = __builtin_amdgcn_sqrtf(s) * iH;
                        const float m_j = ldf_o(m, j);
                        const float irho_j =
                            __builtin_amdgcn_rcpf(ldf_o(rho, j));
                        if (SHEP == 1)
                            sh = fmaf(kernelW<D>(q) * CONW * m_j, irho_j, sh);
                        const float p_j = ldf_o(p, j);
                        const f3 u_ij = sub<D>(ldv_o<D>(u, j), u_i);
                        const float udr = fdot<D>(u_ij, r_ij);
                        const float f_ij = kernelF<D>(q) * CONF * m_j;
                        const float fr = f_ij * irho_i * irho_j;
                        faxpy<D>(gp, (p_i + p_j) * fr, r_ij);
                        if constexpr (LAPF == AQ_LAP_MONAGHAN) {
                            const float r2 = fmaf(q, q, 0.01f) * (H * H);
                            faxpy<D>(lu,
                                     CLEARY * udr * fr *
                                         __builtin_amdgcn_rcpf(r2),
                                     r_ij);
                        } else {
                            faxpy<D>(lu, 2.f * fr, u_ij);
                        }
                        dv = fmaf(udr * f_ij * rho_i, irho_j, dv);
                        if (LAPP) lp = fmaf(p_j - p_i, f_ij * irho_j, lp);
                        return;
                    }
                    const f3 r_ij = sub<D>(r_j, r_i);
                    const float s = dot<D>(r_ij, r_ij);
                    if (SKIP && s > smax) return;
                    const float q = sqrtf(s) / H;
                    float m_j = ldf_o(m, j);
                    m_j = (s > smax) ? 0.f : m_j;
                    const float rho_j = ldf_o(rho, j);
                    const float p_j = ldf_o(p, j);
                    const f3 u_ij = sub<D>(ldv_o<D>(u, j), u_i);
                    const float udr = dot<D>(u_ij, r_ij);
                    terms(std::false_type{}, r_ij, q, m_j, rho_j, p_j, u_ij,
                          udr);
            };
            if (MATH != 1 && fastdiv)
                ring_walk_m<D, SEGW, PER>(L, lane, total, r_i, act, bmin,
                                          bmax, smax, r, imove, 0, flag_el,
                                          nearw, pair_fd, w.per);
            else
                ring_walk_m<D, SEGW, PER>(L, lane, total, r_i, act, bmin,
                                          bmax, smax, r, imove, 0, flag_el,
                                          nearw, pair_ieee, w.per);
            // ---- wall elements (boundary-integral Shepard) ------------------
            if (SHEP == 2 && __ballot(nearw) != 0) {
                bool self_added = false;
                bool unused = false;
                const uint32_t total_el =
                    neighbour_table<D, PER>(w, c_i, L, lane, AQ_CELL_ELEM);
                ring_walk_m<D, SEGW, PER>(
                    L, lane, total_el, r_i, act && nearw, bmin, bmax, smax,
                    r, imove, 1, false, unused, [&](uint32_t j, const f3& r_j) {
                        const f3 r_ij = sub<D>(r_j, r_i);
                        const float s = dot<D>(r_ij, r_ij);
                        if (s > smax) return;
                        const float q = sqrtf(s) / H;
                        const f3 n_j = ldv_o<D>(normal, j);
                        const f3 t_j = ldv_o<D>(tangent, j);
                        const f3 b_j = ldv_o<D>(binormal, j);
                        const float r_n = dot<D>(r_ij, n_j);
                        const float area_j = ldf_o(m, j);
                        if ((r_n > -eps) && (r_n < eps)) {
                            if (!self_added) {
                                const float r_t = fabsf(dot<D>(r_ij, t_j));
                                const float r_b = fabsf(dot<D>(r_ij, b_j));
                                const float dr =
                                    0.55f * pow_cl(area_j, 1.f / (DIMS - 1.f));
                                if ((r_t <= dr) && (r_b <= dr)) {
                                    self_added = true;
                                    sh -= 0.5f;
                                }
                            }
                            return;
                        }
                        const float r_t = fabsf(dot<D>(r_ij, t_j));
                        const float r_b = fabsf(dot<D>(r_ij, b_j));
                        sh += r_n * CONW * kernelS_P<D>(q) * area_j +
                              kernelS_D<D>(fabsf(r_n), r_t, r_b, area_j);
                    },
                    w.per);
            }
            if (act) {
                if constexpr (MATH == 2) {
                    gp = { gp.x + cgp.x, gp.y + cgp.y, gp.z + cgp.z };
                    lu = { lu.x + clu.x, lu.y + clu.y, lu.z + clu.z };
                    dv += cdv;
                    lp += clp;
                }
                stxyz<D>(grad_p, i, gp);
                stxyz<D>(lap_u, i, lu);
                div_u[i] = dv;
                if (LAPP) lap_p[i] = lp;
                if (SHEP) shepard[i] = sh;
                if (near) near[i] = nearw ? 1 : 0;
            }
            if (w.nlist) cell_near = cell_near || __ballot(act && nearw) != 0;
            __builtin_amdgcn_wave_barrier();
        }
        if (w.nlist && cell_near && lane == 0) {
            uint32_t* cnt = const_cast<uint32_t*>(w.n_heads) + AQ_CL_NNCELLS;
            const uint32_t k = atomicAdd(cnt, 1u);
            w.nlist[3 * k] = cstart;
            w.nlist[3 * k + 1] = c_i;
            w.nlist[3 * k + 2] = ce;
        }
    }
}

// ---------------------------------------------------------------------------
// Generic cell-parallel pair kernel: one policy per reference kernel.
//   Pol::KIND           candidates walked (0 fluid, 1 wall elements)
//   pol.owner(i, im_i)  the particles that run the kernel (the reference
//                       kernel's early exits)
//   Pol::State          per-particle accumulators
//   pol.init(i, r_i, st), pol.finish(i, st)
//   pol.load(j)         a candidate's fields (Pol::Cand)
//   pol.use<NRQ>(i, j, cand, r_i, st)
//                       its terms added to the accumulators (NRQ: q by
//                       div_nr, see qof)
// use() is called for the accepted candidates of each particle in the
// reference walk order, so every sum is bit-identical to the per-particle
// kernel of sph.hip.
// ---------------------------------------------------------------------------
// q = sqrt(s) / H.  NRQ: the quotient by div_nr, which is the IEEE quotient
// for H in [2^-40, 2^40] and every accepted pair: sqrtf(s) is 0 or at
// least 2^-75, and at most about 2 H.
template <bool NRQ> __device__ __forceinline__ float qof(float s, float H)
{
    if constexpr (NRQ) return div_nr(sqrtf(s), rcp_nr(H));
    else return sqrtf(s) / H;
}

// A policy as ring_walk's batched pair: fields loaded ahead of their use.
template <class Pol, bool NRQ> struct BatchPair {
    const Pol& pol;
    uint32_t i;
    const f3& r_i;
    typename Pol::State& st;
    __device__ __forceinline__ typename Pol::Cand load(uint32_t j) const
    {
        return pol.load(j);
    }
    __device__ __forceinline__ void use(uint32_t j,
                                        const typename Pol::Cand& c) const
    {
        pol.template use<NRQ>(i, j, c, r_i, st);
    }
};

// Batched consume (ring_walk, NB candidates).  olist: walk the cells it lists
// ((first particle, cell, cell_end) triplets, counted in
// n_heads[count_word]) instead of every non-empty cell.
template <int D, int SEGW, class Pol, int NB>
__global__ void __launch_bounds__(64 * WC_WAVES)
    cell_kernel_k(Pol pol, const int* __restrict__ imove,
                  const float* __restrict__ r, WalkArgs w, float smax,
                  int nrq, const uint32_t* __restrict__ olist,
                  uint32_t count_word)
{
    __shared__ WaveLds<SEGW> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    WaveLds<SEGW>& L = lds[threadIdx.x >> 6];
    if (w.status && (*w.status & 1u)) return;
    const uint32_t n_heads =
        olist ? uni(w.n_heads[count_word]) : uni(*w.n_heads);
    // static hand-out: wavefront v takes the cells v, v + W, ...  (One
    // counter per XCD costs an atomic per cell on 8 cache lines, some 16 ns
    // each: 217 against 84 us for BI Interactions over the 66 k cells of 64
    // sloshing tanks.)
    const uint32_t nwv = gridDim.x * WC_WAVES;
    for (uint32_t hk = blockIdx.x * WC_WAVES + (threadIdx.x >> 6);
         hk < n_heads; hk += nwv) {
        uint32_t cstart, c_i, ce;
        if (olist) {
            // (first particle, cell, cell_end) triplets: one round trip
            cstart = uni(olist[3 * hk]);
            c_i = uni(olist[3 * hk + 1]);
            ce = uni(olist[3 * hk + 2]);
        } else {
            cstart = uni(w.heads[hk]);
            c_i = uni(w.icell[cstart]);
            ce = uni(w.cell_end[c_i]);
        }
        const uint32_t cend = ce & AQ_CELL_END;
        if (w.flagged && Pol::OWNERS && !(ce & Pol::OWNERS)) continue;
        bool table = false;
        uint32_t total = 0;
        for (uint32_t i0 = cstart; i0 < cend; i0 += 64) {
            const uint32_t i = i0 + lane;
            const bool act = (i < cend) && pol.owner(i, imove[i]);
            if (__ballot(act) == 0) continue;
            if (!table) {
                total = neighbour_table<D, false>(
                    w, c_i, L, lane,
                    Pol::KIND ? AQ_CELL_ELEM : AQ_CELL_FLUID);
                table = true;
            }
            typename Pol::State st{};
            f3 r_i = { 0.f, 0.f, 0.f };
            if (act) {
                r_i = ldv<D>(r, i);
                pol.init(i, r_i, st);
            }
            bool unused = false;
            f3 bmin, bmax;
            wave_box<D>(r_i, act, bmin, bmax);
            if (nrq)
                ring_walk<D, SEGW, NB>(
                    L, lane, total, r_i, act, bmin, bmax, smax, r, imove,
                    Pol::KIND, BatchPair<Pol, true>{ pol, i, r_i, st });
            else
                ring_walk<D, SEGW, NB>(
                    L, lane, total, r_i, act, bmin, bmax, smax, r, imove,
                    Pol::KIND, BatchPair<Pol, false>{ pol, i, r_i, st });
            if (act) pol.finish(i, st);
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// ---------------------------------------------------------------------------
// Group kernel: Q lanes per owner (coop_device.hpp).
//
// A wall cell holds few owners (the 16 elements of a 3D wall plane in a cell
// of side 2h at h = 2 dr), and a launch over the wall cells, or over the
// cells of a small case, has too few of them to hide the latency of each
// owner's chain of pair terms, so every owner gets Q lanes, and a listed
// cell is cut into S groups of 64 / Q owners handed out to different
// wavefronts: item k is group k % S of entry k / S, wavefront v takes the
// items v, v + W, ... (no atomic per item).  The policy splits its pair
// into load(j) (the candidate's fields), term<NRQ>(i, j, cand, r_i, st) (a
// pure function of the owner and the candidate) and add_group<Q>(st, term),
// which adds the terms of the group's lanes in lane order on all of them:
// every owner's sums take the terms of the one-lane walk in the same order.
// A lane without a candidate adds Pol::none(), which holds -0: x + -0 is x
// for every x.
// PER: the candidate's position is moved to its periodic image first.
// olist as in cell_kernel_k, its count in n_heads[count_word] (0: the cells).
// ---------------------------------------------------------------------------
template <int D, int Q, class Pol, bool PER>
__global__ void __launch_bounds__(64 * WC_WAVES)
    cell_group_k(Pol pol, const int* __restrict__ imove,
                 const float* __restrict__ r, WalkArgs w, float smax, int nrq,
                 const uint32_t* __restrict__ olist, uint32_t count_word,
                 uint32_t S)
{
    constexpr int OW = 64 / Q;
    using Term = typename Pol::Term;
    __shared__ CoopLds<Q, PER> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int q = lane & (Q - 1), o = lane / Q;
    CoopLds<Q, PER>& L = lds[wv];
    if (w.status && (*w.status & 1u)) return;
    const uint32_t n_heads =
        olist ? uni(w.n_heads[count_word]) : uni(*w.n_heads);
    if (count_word == 0) S = items_per_cell<Q>(S, n_heads, w.N);
    const uint32_t n_items = n_heads * S;
    const uint32_t nwv = gridDim.x * WC_WAVES;
    for (uint32_t item = blockIdx.x * WC_WAVES + (uint32_t)wv; item < n_items;
         item += nwv) {
        const uint32_t hk = item / S;
        uint32_t cstart, c_i, ce;
        if (olist) {
            cstart = uni(olist[3 * hk]);
            c_i = uni(olist[3 * hk + 1]);
            ce = uni(olist[3 * hk + 2]);
        } else {
            cstart = uni(w.heads[hk]);
            c_i = uni(w.icell[cstart]);
            ce = uni(w.cell_end[c_i]);
        }
        const uint32_t cend = ce & AQ_CELL_END;
        if (w.flagged && Pol::OWNERS && !(ce & Pol::OWNERS)) continue;
        for (uint32_t lo = (item % S) * OW;; lo += S * OW) {
            const uint32_t nf = group_owners<Q>(
                L, lane, cstart, cend, lo, imove,
                [&](uint32_t ii, int im) { return pol.owner(ii, im); });
            if (nf == 0) break;
            const uint32_t total = neighbour_table<D, PER>(
                w, c_i, L, lane, Pol::KIND ? AQ_CELL_ELEM : AQ_CELL_FLUID);
            const bool act = (uint32_t)o < nf;
            const uint32_t i = act ? L.owns[o] : cstart;
            typename Pol::State st{};
            f3 r_i = { 0.f, 0.f, 0.f };
            if (act) {
                r_i = ldv<D>(r, i);
                pol.init(i, r_i, st);
            }
            f3 bmin, bmax;
            wave_box<D>(r_i, act, bmin, bmax);
            auto round = [&](uint32_t n, uint32_t cw) {
                Term t = Pol::none();
                if ((uint32_t)q < n) {
                    const uint32_t j = PER ? cw & PER_J_MASK : cw;
                    auto c = pol.load(j);
                    if constexpr (PER) {
                        const float4 sh =
                            L.get_shift((int)(cw >> PER_KL_SHIFT));
                        c.r = per_shift<D>(c.r, f3{ sh.x, sh.y, sh.z },
                                           w.per);
                    }
                    // the walk's test accepts a thin shell beyond: such a
                    // candidate adds nothing, whatever its fields hold (the
                    // term is selected, so that every load of the pair is
                    // issued at once)
                    const f3 r_ij = sub<D>(c.r, r_i);
                    const bool out = (dot<D>(r_ij, r_ij) > smax) |
                                     (Pol::NO_SELF && j == i);
                    t = nrq ? pol.template term<true>(i, j, c, r_i, st)
                            : pol.template term<false>(i, j, c, r_i, st);
                    if (out) t = Pol::none();
                }
                pol.template add_group<Q>(st, t);
            };
            bool unused = false;
            coop_list_walk<D, Q, PER>(
                L, lane, total, r_i, act, bmin, bmax, smax, r, imove,
                Pol::KIND, false, unused, w.per, round);
            if (act && q == 0) pol.finish(i, st);
            lds_order();
            if (nf < (uint32_t)OW) break;
        }
    }
}

// One owner per lane through the fused walk's ring (ring_walk_m), for fluid
// owners once their cells fill the chip.  Policies as in cell_group_k, with
// add(st, term) for one term; hand-out as in cell_kernel_k.
template <int D, class Pol, bool PER>
__global__ void __launch_bounds__(64 * WC_WAVES)
    cell_lane_k(Pol pol, const int* __restrict__ imove,
                const float* __restrict__ r, WalkArgs w, float smax, int nrq,
                const uint32_t* __restrict__ olist, uint32_t count_word)
{
    __shared__ RingLds<8, PER> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    RingLds<8, PER>& L = lds[threadIdx.x >> 6];
    if (w.status && (*w.status & 1u)) return;
    const uint32_t n_heads =
        olist ? uni(w.n_heads[count_word]) : uni(*w.n_heads);
    const uint32_t nwv = gridDim.x * WC_WAVES;
    for (uint32_t hk = blockIdx.x * WC_WAVES + (threadIdx.x >> 6);
         hk < n_heads; hk += nwv) {
        uint32_t cstart, c_i, ce;
        if (olist) {
            cstart = uni(olist[3 * hk]);
            c_i = uni(olist[3 * hk + 1]);
            ce = uni(olist[3 * hk + 2]);
        } else {
            cstart = uni(w.heads[hk]);
            c_i = uni(w.icell[cstart]);
            ce = uni(w.cell_end[c_i]);
        }
        const uint32_t cend = ce & AQ_CELL_END;
        if (w.flagged && Pol::OWNERS && !(ce & Pol::OWNERS)) continue;
        for (uint32_t i0 = cstart; i0 < cend; i0 += 64) {
            const uint32_t i = i0 + lane;
            const bool act = (i < cend) && pol.owner(i, imove[i]);
            if (__ballot(act) == 0) continue;
            const uint32_t total = neighbour_table<D, PER>(
                w, c_i, L, lane, Pol::KIND ? AQ_CELL_ELEM : AQ_CELL_FLUID);
            typename Pol::State st{};
            f3 r_i = { 0.f, 0.f, 0.f };
            if (act) {
                r_i = ldv<D>(r, i);
                pol.init(i, r_i, st);
            }
            f3 bmin, bmax;
            wave_box<D>(r_i, act, bmin, bmax);
            auto walk = [&](auto fd) {
                constexpr bool NRQ = decltype(fd)::value;
                auto pair = [&](uint32_t j, const f3& r_j) {
                    auto c = pol.load(j);
                    c.r = r_j;
                    const f3 r_ij = sub<D>(r_j, r_i);
                    const bool out = (dot<D>(r_ij, r_ij) > smax) |
                                     (Pol::NO_SELF && j == i);
                    auto t = pol.template term<NRQ>(i, j, c, r_i, st);
                    if (out) t = Pol::none();
                    pol.add(st, t);
                };
                bool unused = false;
                ring_walk_m<D, 8, PER>(L, lane, total, r_i, act, bmin, bmax,
                                       smax, r, imove, Pol::KIND, false,
                                       unused, pair, w.per);
            };
            if (nrq) walk(std::true_type{});
            else walk(std::false_type{});
            if (act) pol.finish(i, st);
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// a += the values v of the group's lanes, in lane order
template <int Q> __device__ __forceinline__ void add_lanes(float& a, float v)
{
    each_lane<Q>(v, [&](float x) { a += x; });
}

// The element-owner policies below split each pair into load(j) (the
// candidate's fields), term<NRQ>(i, j, cand, r_i, st) (a pure function of
// the owner's state and the candidate) and add(st, term); use applies them
// in that order, so every walk form adds the same terms.
#define AQ_POL_USE_FROM_TERM                                                  \
    template <bool NRQ>                                                        \
    __device__ void use(uint32_t i, uint32_t j, const Cand& c,                 \
                        const f3& r_i, State& st) const                        \
    {                                                                          \
        add(st, term<NRQ>(i, j, c, r_i, st));                                  \
    }

// cfd/Boundary/BI/Shepard.cl:61-150 (compute) for the non-fluid particles
// (skip_fluid) or all of them
template <int D> struct PolBiShepard {
    static constexpr int BATCH = 4;  // candidates loaded together
    static constexpr int KIND = 1;
    static constexpr bool NO_SELF = false;  // its own element counts (term)
    static constexpr uint32_t OWNERS = 0;  // elements, sensors, ...
    const int* imove;
    const float *normal, *tangent, *binormal, *m;
    float* shepard;
    float H, CONW, DIMS;
    int skip_fluid;
    struct State {
        float acc;
        bool self_added;
    };
    struct Cand {
        f3 r, n, t, b;
        float area;
    };
    // kind 0: add v; 1: the particle's own element (i itself, or a
    // coplanar element within half a spacing), which takes 1/2 once;
    // 2: nothing
    struct Term {
        float v;
        uint32_t kind;
    };
    __device__ bool owner(uint32_t, int im) const
    {
        return !((im < -3) || (im > 1)) && !(skip_fluid && im == 1);
    }
    __device__ void init(uint32_t, const f3&, State& st) const
    {
        st.acc = 1.f;
        st.self_added = false;
    }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldv_o<D>(normal, j),
                     ldv_o<D>(tangent, j), ldv_o<D>(binormal, j),
                     ldf_o(m, j) };
    }
    template <bool NRQ>
    __device__ Term term(uint32_t i, uint32_t j, const Cand& c,
                         const f3& r_i, const State&) const
    {
        if (i == j) return Term{ 0.f, 1u };
        const float eps = 1E-8f * H;
        const f3 r_ij = sub<D>(c.r, r_i);
        const float r_n = dot<D>(r_ij, c.n);
        const float r_t = fabsf(dot<D>(r_ij, c.t));
        const float r_b = fabsf(dot<D>(r_ij, c.b));
        if ((r_n > -eps) && (r_n < eps)) {
            // a coplanar element (most candidates on a flat wall): no q
            const float dr = 0.55f * pow_cl(c.area, 1.f / (DIMS - 1.f));
            return Term{ 0.f, ((r_t <= dr) && (r_b <= dr)) ? 1u : 2u };
        }
        const float q = qof<NRQ>(dot<D>(r_ij, r_ij), H);
        return Term{ r_n * CONW * kernelS_P<D>(q) * c.area +
                         kernelS_D<D>(fabsf(r_n), r_t, r_b, c.area),
                     0u };
    }
    __device__ void add(State& st, const Term& t) const
    {
        if (t.kind == 0u) {
            st.acc += t.v;
        } else if (t.kind == 1u && !st.self_added) {
            st.self_added = true;
            st.acc -= 0.5f;
        }
    }
    __device__ static Term none() { return Term{ 0.f, 2u }; }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        // (v is 0 where kind != 0, and acc is never -0)
        if (__ballot(t.kind == 1u) == 0) {
            add_lanes<Q>(st.acc, t.v);
            return;
        }
        // the half angle in its place in the order
        float v[Q], k[Q];
        int e = 0;
        each_lane<Q>(t.v, [&](float x) { v[e++] = x; });
        e = 0;
        each_lane<Q>((float)t.kind, [&](float x) { k[e++] = x; });
#pragma unroll
        for (int l = 0; l < Q; l++) add(st, Term{ v[l], (uint32_t)k[l] });
    }
    AQ_POL_USE_FROM_TERM
    __device__ void finish(uint32_t i, const State& st) const
    {
        shepard[i] = st.acc;
    }
    const float* r_;
};

// cfd/Boundary/BI/LapU.cl:58-123 (freeslip)
template <int D> struct PolBiLapU {
    static constexpr int BATCH = 4;  // candidates loaded together
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = false;  // never its own candidate
    static constexpr uint32_t OWNERS = AQ_CELL_ELEM;
    const float *r_, *u, *rho, *m;
    float* lap_u;
    float H, CONF;
    int lap;
    struct State {
        f3 u_i, lu;
    };
    struct Cand {
        f3 r, u;
        float rho, m;
    };
    struct Term {
        f3 v;  // the rounded products of the axpy
        uint32_t use;
    };
    __device__ bool owner(uint32_t, int im) const { return im == -3; }
    __device__ void init(uint32_t i, const f3&, State& st) const
    {
        st.u_i = ldv<D>(u, i);
        st.lu = ldv<D>(lap_u, i);
    }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldv_o<D>(u, j), ldf_o(rho, j),
                     ldf_o(m, j) };
    }
    template <bool NRQ>
    __device__ Term term(uint32_t i, uint32_t j, const Cand& c,
                         const f3& r_i, const State& st) const
    {
        constexpr float CLEARY = (D == 2) ? 8.f : 10.f;
        if (i == j) return Term{ f3{ 0.f, 0.f, 0.f }, 0u };
        const f3 r_ij = sub<D>(c.r, r_i);
        const float s = dot<D>(r_ij, r_ij);
        const float q = qof<NRQ>(s, H);
        const float rho_j = c.rho;
        const float f_ij = kernelF<D>(q) * CONF * c.m;
        const f3 u_ij = sub<D>(c.u, st.u_i);
        float sc;
        f3 v;
        if (lap == AQ_LAP_MONAGHAN) {
            const float udr = dot<D>(u_ij, r_ij);
            const float r2 = (q * q + 0.01f) * H * H;
            sc = f_ij * CLEARY * udr / (r2 * rho_j);
            v = r_ij;
        } else {
            sc = f_ij * 2.f / rho_j;
            v = u_ij;
        }
        return Term{ f3{ sc * v.x, sc * v.y, sc * v.z }, 1u };
    }
    __device__ void add(State& st, const Term& t) const
    {
        if (!t.use) return;
        st.lu.x += t.v.x;
        st.lu.y += t.v.y;
        if constexpr (D == 3) st.lu.z += t.v.z;
    }
    __device__ static Term none()
    {
        return Term{ f3{ -0.f, -0.f, -0.f }, 0u };
    }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.lu.x, t.v.x);
        add_lanes<Q>(st.lu.y, t.v.y);
        if constexpr (D == 3) add_lanes<Q>(st.lu.z, t.v.z);
    }
    AQ_POL_USE_FROM_TERM
    __device__ void finish(uint32_t i, const State& st) const
    {
        stxyz<D>(lap_u, i, st.lu);
    }
};

// cfd/Boundary/BI/Interpolation.cl:54-107
template <int D> struct PolBiInterp {
    static constexpr int BATCH = 4;  // candidates loaded together
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = false;  // never its own candidate
    static constexpr uint32_t OWNERS = AQ_CELL_ELEM;
    const float *r_, *m, *rho, *grad_p;
    float* p;
    float H, CONW;
    struct State {
        f3 gp_i;
        float acc;
    };
    struct Cand {
        f3 r;
        float m, rho, p;
    };
    using Term = float;
    __device__ bool owner(uint32_t, int im) const { return im == -3; }
    __device__ void init(uint32_t i, const f3&, State& st) const
    {
        const float rho_i = rho[i];
        st.gp_i = ldv<D>(grad_p, i);
        st.gp_i.x = rho_i * st.gp_i.x;
        st.gp_i.y = rho_i * st.gp_i.y;
        st.gp_i.z = rho_i * st.gp_i.z;
        st.acc = 0.f;
    }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldf_o(m, j), ldf_o(rho, j),
                     ldf_o(p, j) };
    }
    template <bool NRQ>
    __device__ Term term(uint32_t, uint32_t, const Cand& c, const f3& r_i,
                         const State& st) const
    {
        const f3 r_ij = sub<D>(c.r, r_i);
        const float s = dot<D>(r_ij, r_ij);
        const float q = qof<NRQ>(s, H);
        const float w_ij = kernelW<D>(q) * CONW * c.m / c.rho;
        return (c.p - dot<D>(st.gp_i, r_ij)) * w_ij;
    }
    __device__ void add(State& st, const Term& t) const { st.acc += t; }
    __device__ static Term none() { return -0.f; }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.acc, t);
    }
    AQ_POL_USE_FROM_TERM
    __device__ void finish(uint32_t i, const State& st) const
    {
        p[i] = st.acc;
    }
};

// cfd/Boundary/BI/Interactions.cl:51-133, for the fluid particles with an
// element inside the support (near flags of the fused walk) or all of them
template <int D> struct PolBiInteractions {
    static constexpr int BATCH = 4;  // candidates loaded together
    static constexpr int KIND = 1;
    static constexpr bool NO_SELF = false;  // never its own candidate
    static constexpr uint32_t OWNERS = AQ_CELL_FLUID;
    const float *r_, *normal, *u, *rho, *m, *p;
    float *grad_p, *div_u;
    const uint8_t* near;
    float H, CONW;
    struct State {
        f3 u_i, gp;
        float p_i, rho_i, dv;
    };
    __device__ bool owner(uint32_t i, int im) const
    {
        return im == 1 && (!near || near[i]);
    }
    __device__ void init(uint32_t i, const f3&, State& st) const
    {
        st.u_i = ldv<D>(u, i);
        st.p_i = p[i];
        st.rho_i = rho[i];
        st.gp = ldv<D>(grad_p, i);
        st.dv = div_u[i];
    }
    struct Cand {
        f3 r, n, u;
        float area, p;
    };
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldv_o<D>(normal, j), ldv_o<D>(u, j),
                     ldf_o(m, j), ldf_o(p, j) };
    }
    struct Term {
        f3 g;  // the rounded products of the axpy
        float d;
    };
    template <bool NRQ>
    __device__ Term term(uint32_t, uint32_t, const Cand& c, const f3& r_i,
                         const State& st) const
    {
        const f3 r_ij = sub<D>(c.r, r_i);
        const float s = dot<D>(r_ij, r_ij);
        const float q = qof<NRQ>(s, H);
        const f3 du = sub<D>(c.u, st.u_i);
        const float w_ij = kernelW<D>(q) * CONW * c.area;
        return Term{ scl<D>((st.p_i + c.p) / st.rho_i * w_ij, c.n),
                     st.rho_i * dot<D>(du, c.n) * w_ij };
    }
    __device__ void add(State& st, const Term& t) const
    {
        st.gp = add3<D>(st.gp, t.g);
        st.dv += t.d;
    }
    __device__ static Term none()
    {
        return Term{ f3{ -0.f, -0.f, -0.f }, -0.f };
    }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.gp.x, t.g.x);
        add_lanes<Q>(st.gp.y, t.g.y);
        if constexpr (D == 3) add_lanes<Q>(st.gp.z, t.g.z);
        add_lanes<Q>(st.dv, t.d);
    }
    AQ_POL_USE_FROM_TERM
    __device__ void finish(uint32_t i, const State& st) const
    {
        stxyz<D>(grad_p, i, st.gp);
        div_u[i] = st.dv;
    }
};

#undef AQ_POL_USE_FROM_TERM

// ---- LES closure pair kernels (cfd/LES/GradU.cl, cfd/LES/Interactions.cl
// of Presets/cfd/LES.xml; no counterpart in the reference) -------------------
// The SPH velocity gradient of the fluid particles,
//   G_i = sum_j m_j / rho_j (u_j - u_i) (x) F_ij r_ij,
// grad_u[a n + b] = du_a / dx_b (row stride n = 2 in 2D, 4 in 3D), summed
// in the walk order.  The non-fluid particles' rows are cleared by the
// launcher.
template <int D> struct PolLesGradU {
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = true;
    static constexpr uint32_t OWNERS = AQ_CELL_FLUID;
    static constexpr int NR = (D == 2) ? 2 : 4;
    const float *r_, *u, *rho, *m;
    float* grad_u;
    float H, CONF;
    struct State {
        f3 u_i;
        float G[D * D];
    };
    __device__ bool owner(uint32_t, int im) const { return im == 1; }
    __device__ void init(uint32_t i, const f3&, State& st) const
    {
        st.u_i = ldv<D>(u, i);
#pragma unroll
        for (int k = 0; k < D * D; k++) st.G[k] = 0.f;
    }
    struct Cand {
        f3 r, u;
        float m, rho;
    };
    struct Term {
        float g[D * D];
    };
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldv_o<D>(u, j), ldf_o(m, j),
                     ldf_o(rho, j) };
    }
    template <bool NRQ>
    __device__ Term term(uint32_t, uint32_t, const Cand& c, const f3& r_i,
                         const State& st) const
    {
        Term t;
        const f3 r_ij = sub<D>(c.r, r_i);
        const float q = qof<NRQ>(dot<D>(r_ij, r_ij), H);
        const float w = kernelF<D>(q) * CONF * c.m / c.rho;
        const f3 du = sub<D>(c.u, st.u_i);
        const float dv[3] = { du.x, du.y, du.z };
        const float rv[3] = { r_ij.x, r_ij.y, r_ij.z };
#pragma unroll
        for (int a = 0; a < D; a++)
#pragma unroll
            for (int b = 0; b < D; b++) t.g[a * D + b] = dv[a] * (w * rv[b]);
        return t;
    }
    __device__ static Term none()
    {
        Term t;
#pragma unroll
        for (int k = 0; k < D * D; k++) t.g[k] = -0.f;
        return t;
    }
    __device__ void add(State& st, const Term& t) const
    {
#pragma unroll
        for (int k = 0; k < D * D; k++) st.G[k] += t.g[k];
    }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
#pragma unroll
        for (int k = 0; k < D * D; k++) add_lanes<Q>(st.G[k], t.g[k]);
    }
    __device__ void finish(uint32_t i, const State& st) const
    {
        constexpr int S = (D == 2) ? 4 : 16;
        float o[S];
#pragma unroll
        for (int k = 0; k < S; k++) o[k] = 0.f;
#pragma unroll
        for (int a = 0; a < D; a++)
#pragma unroll
            for (int b = 0; b < D; b++) o[a * NR + b] = st.G[a * D + b];
#pragma unroll
        for (int k = 0; k < S; k++) grad_u[(size_t)i * S + k] = o[k];
    }
};

// The eddy-viscosity term in the variable-viscosity Morris form,
//   dudt_i += sum_j F_ij m_j (rho_i nu_i + rho_j nu_j) / (rho_i rho_j)
//             (u_j - u_i),
// summed in the walk order and added to dudt at the end.
template <int D> struct PolLesInteractions {
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = true;
    static constexpr uint32_t OWNERS = AQ_CELL_FLUID;
    const float *r_, *u, *rho, *m, *nu_t;
    float* dudt;
    float H, CONF;
    struct State {
        f3 u_i, acc;
        float rho_i, mu_i;
    };
    __device__ bool owner(uint32_t, int im) const { return im == 1; }
    __device__ void init(uint32_t i, const f3&, State& st) const
    {
        st.u_i = ldv<D>(u, i);
        st.rho_i = rho[i];
        st.mu_i = st.rho_i * nu_t[i];
        st.acc = f3{ 0.f, 0.f, 0.f };
    }
    struct Cand {
        f3 r, u;
        float m, rho, nu;
    };
    using Term = f3;
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r_, j), ldv_o<D>(u, j), ldf_o(m, j),
                     ldf_o(rho, j), ldf_o(nu_t, j) };
    }
    template <bool NRQ>
    __device__ Term term(uint32_t, uint32_t, const Cand& c, const f3& r_i,
                         const State& st) const
    {
        const f3 r_ij = sub<D>(c.r, r_i);
        const float q = qof<NRQ>(dot<D>(r_ij, r_ij), H);
        const float f = kernelF<D>(q) * CONF * c.m;
        const float sc =
            f * (st.mu_i + c.rho * c.nu) / (st.rho_i * c.rho);
        return scl<D>(sc, sub<D>(c.u, st.u_i));
    }
    __device__ static Term none() { return f3{ -0.f, -0.f, -0.f }; }
    __device__ void add(State& st, const Term& t) const
    {
        st.acc = add3<D>(st.acc, t);
    }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.acc.x, t.x);
        add_lanes<Q>(st.acc.y, t.y);
        if constexpr (D == 3) add_lanes<Q>(st.acc.z, t.z);
    }
    __device__ void finish(uint32_t i, const State& st) const
    {
        const f3 d = ldv<D>(dudt, i);
        stxyz<D>(dudt, i, f3{ d.x + st.acc.x, d.y + st.acc.y,
                              d.z + st.acc.z });
    }
};

// grad_u of the particles that are not fluid: zero (the per-particle
// kernel writes zeros for them)
template <int D>
__global__ void les_gradu_clear_k(const int* __restrict__ imove,
                                  float* __restrict__ grad_u, uint32_t N)
{
    constexpr int S = (D == 2) ? 4 : 16;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N || imove[i] == 1) return;
#pragma unroll
    for (int k = 0; k < S; k++) grad_u[(size_t)i * S + k] = 0.f;
}

// Clears the NRANGE range counters.
__global__ void zero_u32_k(uint32_t* p, uint32_t* rec,
                           uint32_t* extra = nullptr)
{
    if (threadIdx.x < NRANGE) p[threadIdx.x * RSTRIDE] = 0u;
    if (rec && threadIdx.x < NREC)
        rec[threadIdx.x * RSTRIDE] = rec_init[threadIdx.x];
    if (extra && threadIdx.x == 0) *extra = 0u;
}

// Cell hand-out ranges: NRANGE (one per XCD) unless AQ_WALK_RANGES=1.
static uint32_t walk_ranges()
{
    static const uint32_t nr = [] {
        const char* e = getenv("AQ_WALK_RANGES");
        return (e && atoi(e) == 1) ? 1u : NRANGE;
    }();
    return nr;
}

// Workgroups of `ker` that fit on the device at once (all CUs), cached per
// kernel: the grid of the walks, which hand out their cells to the wavefronts
// there are (the one-lane fused walk by counters, the others by stride).
unsigned resident_blocks(const void* ker, int block)
{
    static std::mutex mu;
    static std::map<std::pair<int, const void*>, unsigned> cache;
    int dev = 0;
    AQ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> g(mu);
    auto key = std::make_pair(dev, ker);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int per_cu = 0, ncu = 0;
    AQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ker, block,
                                                        0));
    AQ_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                                 dev));
    const unsigned nb = (unsigned)std::max(1, per_cu) * (unsigned)std::max(1, ncu);
    cache[key] = nb;
    return nb;
}

// Compute units of the current device (cached).
static unsigned cu_count()
{
    static std::mutex mu;
    static std::map<int, unsigned> cache;
    int dev = 0;
    AQ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> g(mu);
    auto it = cache.find(dev);
    if (it != cache.end()) return it->second;
    int ncu = 0;
    AQ_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                                 dev));
    return cache[dev] = (unsigned)std::max(1, ncu);
}

// Workgroups per compute unit the walks of the side stream take
// (AQ_SIDE_WGS, default 1); the fused walk beside them leaves them that
// room, so both stay resident together.
unsigned side_wgs_per_cu()
{
    static const unsigned n = [] {
        const char* e = getenv("AQ_SIDE_WGS");
        const int v = e ? atoi(e) : 1;
        return (unsigned)std::min(4, std::max(0, v));
    }();
    return n;
}

// A resident grid less `reserve` workgroups per compute unit (one per
// compute unit at least).
static unsigned reserved_grid(unsigned resident, unsigned reserve)
{
    const unsigned ncu = cu_count();
    const unsigned cut = reserve * ncu;
    return resident > cut + ncu ? resident - cut : std::min(resident, ncu);
}

// Grid of a walk: the resident grid, or the side stream's share.
static unsigned walk_grid(const void* ker, const CellArgs& c)
{
    const unsigned res = resident_blocks(ker, 64 * WC_WAVES);
    if (!c.side) return res;
    return std::min(res, std::max(1u, side_wgs_per_cu()) * cu_count());
}

int fluid_coop_lanes(int dims, uint32_t N, int math, bool per);
void launch_fluid_coop(int dims, int shep, bool lapp, int q,
                       const int32_t* imove, const float* r, const float* u,
                       const float* rho, const float* m, const float* p,
                       const float* normal, const float* tangent,
                       const float* binormal, float* shepard, float* grad_p,
                       float* lap_u, float* div_u, float* lap_p,
                       uint8_t* near, const WalkArgs& w, aq_defs d,
                       float smax, int math, const uint32_t* rec,
                       hipStream_t s);

void launch_fluid_pass_cells(int dims, int shep, bool lapp,
                             const int32_t* imove, const float* r,
                             const float* u, const float* rho, const float* m,
                             const float* p, const float* normal,
                             const float* tangent, const float* binormal,
                             float* shepard, float* grad_p, float* lap_u,
                             float* div_u, float* lap_p, uint8_t* near,
                             uint32_t N, const uint32_t* icell,
                             const uint32_t* ihoc, const uint32_t* n_cells,
                             const uint32_t* cell_end, const uint32_t* heads,
                             const uint32_t* n_heads, const uint32_t* status,
                             aq_defs d, float smax, unsigned nblocks, int segw,
                             int flagged, int math, unsigned ranges,
                             int fast_div, hipStream_t s, const float* per,
                             unsigned reserve_per_cu, uint32_t* nlist,
                             const uint32_t* blist)
{
    // a periodic box has no walls: the boundary-integral Shepard pass is
    // not built for it
    AQ_REQUIRE(!per || shep != 2,
               "periodic box: boundary-integral walls are not supported");
    // candidate loads use 32-bit byte offsets (16 B per particle at most)
    AQ_REQUIRE(N < (1u << 28), "cell-parallel walk: more than 2^28 particles");
    // the hand-out counters live after the non-empty cell count
    uint32_t* next = const_cast<uint32_t*>(n_heads) + RSTRIDE;
    // the range record (relaxed arithmetic has no use for it)
    uint32_t* rec =
        (fast_div && math != 1) ? const_cast<uint32_t*>(n_heads) + RREC
                                : nullptr;
    // the near-cell list is filled from the walk's near flags
    if (!near || shep != 2) nlist = nullptr;
    hipLaunchKernelGGL(zero_u32_k, dim3(1), dim3(64), 0, s, next, rec,
                       nlist ? const_cast<uint32_t*>(n_heads) + AQ_CL_NNCELLS
                             : nullptr);
    if (rec && N) {
        const unsigned nb = std::min(512u, (N + 1023u) / 1024u);
        if (dims == 2)
            hipLaunchKernelGGL(fluid_ranges_k<2>, dim3(nb), dim3(256), 0, s,
                               imove, p, rho, m, u, N, rec);
        else
            hipLaunchKernelGGL(fluid_ranges_k<3>, dim3(nb), dim3(256), 0, s,
                               imove, p, rho, m, u, N, rec);
    }
    WalkArgs w{ icell,  ihoc,   n_cells, cell_end, heads,
                n_heads, next, status, N,       (uint32_t)flagged,
                ranges ? std::min<unsigned>(ranges, NRANGE) : walk_ranges(),
                per, nlist, flagged ? blist : nullptr };
    // few particles: several lanes each (the default launch configuration
    // only: an explicit segment width or grid asks for the one-lane walk)
    if (const int q = segw == 8 && !nblocks && ranges != 1 && !reserve_per_cu
                              && math != 1
                          ? fluid_coop_lanes(dims, N, math, per != nullptr)
                          : 0) {
        launch_fluid_coop(dims, shep, lapp, q, imove, r, u, rho, m, p, normal,
                          tangent, binormal, shepard, grad_p, lap_u, div_u,
                          lap_p, near, w, d, smax, math, rec, s);
        return;
    }
#define AQ_FC3(DD, SH, LP, SW, LF, PR)                                         \
    do {                                                                       \
        auto* ker = math == 1                                                  \
                        ? fluid_pass_cells_k<DD, SH, LP, SW, LF, 1, PR>        \
                    : math == 2 ? fluid_pass_cells_k<DD, SH, LP, 8, LF, 2, PR> \
                                : fluid_pass_cells_k<DD, SH, LP, SW, LF, 0, PR>; \
        const unsigned nb =                                                    \
            nblocks ? nblocks                                                  \
                    : reserved_grid(resident_blocks((const void*)ker,          \
                                                    64 * WC_WAVES),            \
                                    reserve_per_cu);                           \
        hipLaunchKernelGGL(ker, dim3(nb), dim3(64 * WC_WAVES), 0, s, imove, r, \
                           u, rho, m, p, normal, tangent, binormal, shepard,   \
                           grad_p, lap_u, div_u, lap_p, near, w, d.H, d.CONW,  \
                           d.CONF, d.DIMS, smax, 1.f / d.H, rec);              \
    } while (0)
#define AQ_FC2(DD, SH, LP, SW, LF)                                             \
    do {                                                                       \
        if (per && SH != 2) AQ_FC3(DD, SH, LP, SW, LF, (SH != 2));             \
        else AQ_FC3(DD, SH, LP, SW, LF, false);                                \
    } while (0)
#define AQ_FC(DD, SH, LP, SW)                                                  \
    do {                                                                       \
        if (d.lap_formulation == AQ_LAP_MONAGHAN)                              \
            AQ_FC2(DD, SH, LP, SW, AQ_LAP_MONAGHAN);                           \
        else                                                                   \
            AQ_FC2(DD, SH, LP, SW, AQ_LAP_MORRIS);                             \
    } while (0)
#define AQ_FC_D(SH, LP)                                                        \
    do {                                                                       \
        if (dims == 2 && segw == 8) AQ_FC(2, SH, LP, 8);                       \
        else if (dims == 2) AQ_FC(2, SH, LP, 16);                              \
        else if (segw == 8) AQ_FC(3, SH, LP, 8);                               \
        else AQ_FC(3, SH, LP, 16);                                             \
    } while (0)
    if (shep == 0 && !lapp) AQ_FC_D(0, false);
    else if (shep == 0 && lapp) AQ_FC_D(0, true);
    else if (shep == 1 && !lapp) AQ_FC_D(1, false);
    else if (shep == 1 && lapp) AQ_FC_D(1, true);
    else if (shep == 2 && !lapp) AQ_FC_D(2, false);
    else AQ_FC_D(2, true);
#undef AQ_FC_D
#undef AQ_FC
#undef AQ_FC2
#undef AQ_FC3
}


// ---- launchers of the generic cell kernels ---------------------------------
// One owner per lane over `olist` (its count in n_heads[count_word]; nullptr:
// every non-empty cell, in blocked order when the link-list built it),
// batched loads.
template <int D, class Pol>
static void launch_bi_cells(const Pol& pol, const int32_t* imove,
                            const float* r, const CellArgs& c, float smax,
                            hipStream_t s, const uint32_t* olist = nullptr,
                            uint32_t count_word = 0)
{
    AQ_REQUIRE(c.N < (1u << 28), "cell-parallel walk: more than 2^28 particles");
    WalkArgs w{ c.icell,   c.ihoc,   c.n_cells, c.cell_end, c.heads,
                c.n_heads, nullptr,  c.status,  c.N,        c.flagged,
                walk_ranges() };
    auto* ker = cell_kernel_k<D, 8, Pol, Pol::BATCH>;
    const unsigned nb = walk_grid((const void*)ker, c);
    const int nrq = (pol.H >= 0x1p-40f && pol.H <= 0x1p40f) ? 1 : 0;
    if (!olist) {
        olist = c.blist;
        count_word = 0;
    }
    hipLaunchKernelGGL(ker, dim3(nb), dim3(64 * WC_WAVES), 0, s, pol, imove,
                       r, w, smax, nrq, olist, count_word);
}

// The group kernel with `wide` ? 16 : 4 lanes per owner over `olist`
// (nullptr: every non-empty cell, in blocked order when there is one);
// `per_cell`: owners of a full entry.  Measured in us, 4 / 16 lanes:
//   BI LapU          3D  29 k particles 46 / 25   394 k 52 / 34
//                        1.2 M 57 / 62   4.5 M 113 / 126
//                    2D  21 k 13 / 11   1.2 M (64 tanks) 23 / 28
//   BI Interactions  3D  29 k 26 / 34
// The elements are few and hold a fifth of their neighbours' particles each,
// so 16 lanes pay as long as latency rules; fluid owners fill the chip much
// earlier (les_lanes; launch_bi_interactions_cells).  (Before, in us at 4.5 M
// / 1.2 M / 29 k: 4 lanes with the terms through LDS and a full wait per
// segment, LapU 240 / 134 / 127, Interpolation 200 / 119 / 113; one lane per
// owner, Interactions at 29 k 65.)
template <int D, class Pol, bool PER = false>
static void launch_groups(const Pol& pol, const int32_t* imove,
                          const float* r, const CellArgs& c, float smax,
                          hipStream_t s, bool wide, const uint32_t* olist,
                          uint32_t count_word, uint32_t per_cell,
                          const float* per = nullptr)
{
    AQ_REQUIRE(c.N < (1u << 28), "cell-parallel walk: more than 2^28 particles");
    AQ_REQUIRE(!PER || c.N <= PER_GROUP_MAX_N,
               "periodic box: more than 2^27 particles in a group walk");
    WalkArgs w{ c.icell,   c.ihoc,   c.n_cells, c.cell_end, c.heads,
                c.n_heads, nullptr,  c.status,  c.N,        c.flagged,
                walk_ranges(), per };
    if (!olist && c.blist) {
        olist = c.blist;
        count_word = 0;
    }
    const int nrq = (pol.H >= 0x1p-40f && pol.H <= 0x1p40f) ? 1 : 0;
    auto launch = [&](auto* ker, unsigned q) {
        const unsigned nb = std::min(walk_grid((const void*)ker, c),
                                     blocks_for((size_t)c.N * q * 2,
                                                64 * WC_WAVES));
        hipLaunchKernelGGL(ker, dim3(nb), dim3(64 * WC_WAVES), 0, s, pol,
                           imove, r, w, smax, nrq, olist, count_word,
                           std::max(1u, per_cell * q / 64u));
    };
    if (wide) launch(cell_group_k<D, 16, Pol, PER>, 16);
    else launch(cell_group_k<D, 4, Pol, PER>, 4);
}

// Lanes per wall element or sensor of the owner-list walks (launch_groups)
static int elem_lanes(int dims, uint32_t N)
{
    return N <= (dims == 2 ? 100000u : 600000u) ? 16 : 4;
}

// list: 0 every non-empty cell (one owner per lane), 1 the owner cells,
// 2 the wet owner cells (group kernel)
template <int D, class Pol>
static void launch_bi_coop(const Pol& pol, const int32_t* imove,
                           const float* r, const CellArgs& c, float smax,
                           hipStream_t s, int list)
{
    const uint32_t* ol = !c.flagged ? nullptr
                         : list == 1 ? c.ocells
                         : list == 2 ? c.wcells
                                     : nullptr;
    if (!ol)
        launch_bi_cells<D>(pol, imove, r, c, smax, s);
    else
        launch_groups<D>(pol, imove, r, c, smax, s,
                         elem_lanes(D, c.N) == 16, ol,
                         list == 1 ? AQ_CL_NOCELLS : AQ_CL_NWCELLS,
                         AQ_OWNER_CHUNK);
}

// p = 0 for the wall elements (imove == -3): the value BI Interpolation
// gives the elements without fluid in range, which the walk over the wet
// owner cells does not visit
__global__ void elem_zero_k(const int* __restrict__ imove,
                            float* __restrict__ p, uint32_t N)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N && imove[i] == -3) p[i] = 0.f;
}

void launch_bi_shepard_compute_cells(int dims, const int32_t* imove,
                                     const float* r, const float* normal,
                                     const float* tangent,
                                     const float* binormal, const float* m,
                                     float* shepard, const CellArgs& c,
                                     aq_defs d, float smax, int skip_fluid,
                                     hipStream_t s)
{
    // with the fluid among the owners (skip_fluid == 0) every cell owns
    if (dims == 2) {
        PolBiShepard<2> p{ imove, normal, tangent, binormal, m, shepard,
                           d.H,   d.CONW, d.DIMS,  skip_fluid, r };
        launch_bi_coop<2>(p, imove, r, c, smax, s, skip_fluid ? 1 : 0);
    } else {
        PolBiShepard<3> p{ imove, normal, tangent, binormal, m, shepard,
                           d.H,   d.CONW, d.DIMS,  skip_fluid, r };
        launch_bi_coop<3>(p, imove, r, c, smax, s, skip_fluid ? 1 : 0);
    }
}

void launch_bi_lapu_cells(int dims, const int32_t* imove, const float* r,
                          const float* u, const float* rho, const float* m,
                          float* lap_u, const CellArgs& c, aq_defs d,
                          float smax, hipStream_t s)
{
    if (dims == 2) {
        PolBiLapU<2> p{ r, u, rho, m, lap_u, d.H, d.CONF, d.lap_formulation };
        launch_bi_coop<2>(p, imove, r, c, smax, s, 2);
    } else {
        PolBiLapU<3> p{ r, u, rho, m, lap_u, d.H, d.CONF, d.lap_formulation };
        launch_bi_coop<3>(p, imove, r, c, smax, s, 2);
    }
}

void launch_bi_interp_cells(int dims, const int32_t* imove, const float* r,
                            const float* m, const float* rho,
                            const float* grad_p, float* p, const CellArgs& c,
                            aq_defs d, float smax, hipStream_t s)
{
    if (c.flagged && c.wcells)
        hipLaunchKernelGGL(elem_zero_k, dim3(blocks_for(c.N, 256)), dim3(256),
                           0, s, imove, p, c.N);
    if (dims == 2) {
        PolBiInterp<2> q{ r, m, rho, grad_p, p, d.H, d.CONW };
        launch_bi_coop<2>(q, imove, r, c, smax, s, 2);
    } else {
        PolBiInterp<3> q{ r, m, rho, grad_p, p, d.H, d.CONW };
        launch_bi_coop<3>(q, imove, r, c, smax, s, 2);
    }
}

void launch_bi_interactions_cells(int dims, const int32_t* imove,
                                  const float* r, const float* normal,
                                  const float* u, const float* rho,
                                  const float* m, const float* p,
                                  float* grad_p, float* div_u,
                                  const uint8_t* near, const CellArgs& c,
                                  aq_defs d, float smax, hipStream_t s)
{
    // with the near flags, only the cells the fused walk listed as near
    const uint32_t* ol = (near && c.flagged) ? c.nlist : nullptr;
    // A near cell holds few near particles, but above a million particles in
    // 3D there are cells enough for one lane each.  4 lanes / one, us, on the
    // lattice and displaced by up to 0.4 of the spacing: 29 k 26 / 56, 27 /
    // 58; 394 k 49 / 67, 50 / 71; 1.2 M 84 / 78, 89 / 83; 4.5 M 159 / 136,
    // 166 / 148; 11 M 328 / 303, 355 / 336; 2D 507 k 11 / 13.
    const bool one = dims == 3 && c.N > 1000000u;
    auto go = [&](const auto& pol, auto dim) {
        constexpr int D = decltype(dim)::value;
        if (ol && one)
            launch_bi_cells<D>(pol, imove, r, c, smax, s, ol, AQ_CL_NNCELLS);
        else if (ol)
            launch_groups<D>(pol, imove, r, c, smax, s, false, ol,
                             AQ_CL_NNCELLS, D == 2 ? 16 : 64);
        else
            launch_bi_cells<D>(pol, imove, r, c, smax, s);
    };
    if (dims == 2)
        go(PolBiInteractions<2>{ r, normal, u, rho, m, p, grad_p, div_u, near,
                                 d.H, d.CONW },
           std::integral_constant<int, 2>{});
    else
        go(PolBiInteractions<3>{ r, normal, u, rho, m, p, grad_p, div_u, near,
                                 d.H, d.CONW },
           std::integral_constant<int, 3>{});
}

// Lanes per particle of the LES kernels for N particles; 0: one lane each
// (cell_lane_k).  Both kernels of a step in us, 16 / 4 / one, on the lattice
// and with the particles displaced by up to 0.4 of their spacing:
//   3D   22 k  230 /  302 /  889     242 /  344 / 1094
//        47 k  279 /  200 /  445     322 /  242 /  570
//       195 k 1507 /  997 / 1101    1848 / 1083 / 1259
//       262 k 1360 /  843 /  645    1502 /  956 /  835
//       373 k 2001 / 1190 / 1111    2103 / 1277 / 1347
//       512 k 2740 / 1740 / 1325    2879 / 1799 / 1622
//       2.1 M  11610 / 7078 / 5148  12289 / 7330 / 6157
//   2D   16 k   40 /   54 /   64      45 /   57 /   74
//        40 k   54 /   42 /   74      59 /   48 /   88
//       1.0 M 1006 /  620 / 1123    1422 /  848 / 1227
// One lane each wins, as in the fused walk, once the 3D cells fill the chip
// (4096 wavefronts, 262 k particles).
// A periodic box of more particles than the group walk can name: one lane.
static int les_lanes(int dims, uint32_t N, bool per)
{
    if (per && N > PER_GROUP_MAX_N) return 0;
    if (N <= (dims == 2 ? 16000u : 24000u)) return 16;
    return dims == 3 && N > 250000u ? 0 : 4;
}

// LES kernels over every cell
template <int D, class Pol, bool PER>
static void launch_les_form(const Pol& pol, const int32_t* imove,
                            const float* r, const CellArgs& c, float smax,
                            const float* per, hipStream_t s)
{
    const int q = les_lanes(D, c.N, PER);
    if (q) {
        launch_groups<D, Pol, PER>(pol, imove, r, c, smax, s, q == 16,
                                   nullptr, 0, D == 2 ? 16 : 64, per);
        return;
    }
    AQ_REQUIRE(c.N < (1u << 28), "cell-parallel walk: more than 2^28 particles");
    WalkArgs w{ c.icell,   c.ihoc,   c.n_cells, c.cell_end, c.heads,
                c.n_heads, nullptr,  c.status,  c.N,        c.flagged,
                walk_ranges(), per };
    auto* ker = cell_lane_k<D, Pol, PER>;
    const int nrq = (pol.H >= 0x1p-40f && pol.H <= 0x1p40f) ? 1 : 0;
    hipLaunchKernelGGL(ker, dim3(walk_grid((const void*)ker, c)),
                       dim3(64 * WC_WAVES), 0, s, pol, imove, r, w, smax, nrq,
                       c.blist, 0u);
}

template <int D, class Pol>
static void launch_les(const Pol& pol, const int32_t* imove, const float* r,
                       const CellArgs& c, float smax, const float* per,
                       hipStream_t s)
{
    if (per) launch_les_form<D, Pol, true>(pol, imove, r, c, smax, per, s);
    else launch_les_form<D, Pol, false>(pol, imove, r, c, smax, nullptr, s);
}

void launch_les_gradu_cells(int dims, const int32_t* imove, const float* r,
                            const float* u, const float* rho, const float* m,
                            float* grad_u, const CellArgs& c, aq_defs d,
                            float smax, const float* per, hipStream_t s)
{
    const dim3 g(blocks_for(c.N, 256)), b(256);
    if (dims == 2) {
        hipLaunchKernelGGL(les_gradu_clear_k<2>, g, b, 0, s, imove, grad_u,
                           c.N);
        PolLesGradU<2> p{ r, u, rho, m, grad_u, d.H, d.CONF };
        launch_les<2>(p, imove, r, c, smax, per, s);
    } else {
        hipLaunchKernelGGL(les_gradu_clear_k<3>, g, b, 0, s, imove, grad_u,
                           c.N);
        PolLesGradU<3> p{ r, u, rho, m, grad_u, d.H, d.CONF };
        launch_les<3>(p, imove, r, c, smax, per, s);
    }
}

void launch_les_interactions_cells(int dims, const int32_t* imove,
                                   const float* r, const float* u,
                                   const float* rho, const float* m,
                                   const float* nu_t, float* dudt,
                                   const CellArgs& c, aq_defs d, float smax,
                                   const float* per, hipStream_t s)
{
    if (dims == 2) {
        PolLesInteractions<2> p{ r, u, rho, m, nu_t, dudt, d.H, d.CONF };
        launch_les<2>(p, imove, r, c, smax, per, s);
    } else {
        PolLesInteractions<3> p{ r, u, rho, m, nu_t, dudt, d.H, d.CONF };
        launch_les<3>(p, imove, r, c, smax, per, s);
    }
}

}  // namespace aq

using namespace aq;

extern "C" AQ_API int aq_walk_lanes(int kernel, int dims, uint32_t N,
                                    int periodic)
{
    if ((dims != 2 && dims != 3) || N >= (1u << 28)) return AQ_EINVAL;
    const bool per = periodic != 0;
    switch (kernel) {
    case AQ_WALK_FLUID:
        return std::max(1, fluid_coop_lanes(dims, N, 0, per));
    case AQ_WALK_COMPENSATED:
        return std::max(1, fluid_coop_lanes(dims, N, 2, per));
    case AQ_WALK_ELEMENTS: return per ? AQ_EINVAL : elem_lanes(dims, N);
    case AQ_WALK_LES: return std::max(1, les_lanes(dims, N, per));
    default: return AQ_EINVAL;
    }
}
