// Neighbour walk with a group of Q lanes per particle, for kernels whose
// cells hold few owners or whose launches have few cells:
//   test     a chunk of 64 candidates is staged through LDS as in
//            ring_walk (box prefilter, survivors compacted in order), each
//            survivor is tested against each particle, and the accepted
//            ones are appended, in candidate order, to the particles' lists
//            in LDS.  Q == 4: the distances to the 16 particles by matrix
//            instructions (dist_tile); Q == 16: lane q tests the survivors
//            q, q + 16, ..., their places in the list from ballots.
//   consume  when a list has no room for another chunk (and at the end),
//            the lanes of every particle with Q listed take its next Q,
//            evaluate their terms, and all Q lanes add the terms in list
//            order, each term broadcast from its lane by a DPP modifier of
//            the addition: the Q copies of the sums stay equal, and every
//            sum takes the terms of the one-lane walk in the same order.
//            (The particles of a cell accept from different stretches of
//            the candidate list; consuming only when a list fills up lets
//            them work side by side.)
#pragma once
#include "aq_device.hpp"
#include "walk_device.hpp"

namespace aq {

// Orders the LDS accesses of one wavefront (its LDS operations complete in
// program order; nothing in flight from memory is waited for).
__device__ __forceinline__ void lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of lane K of the caller's group of Q lanes: DPP quad_perm
// (Q == 4) or row_newbcast (Q == 16).
template <int Q, int K> __device__ __forceinline__ float lane_of(float v)
{
    static_assert(Q == 4 || Q == 16, "lanes per particle");
    constexpr int ctrl = Q == 4 ? K * 0x55 : 0x150 + K;
    return __int_as_float(__builtin_amdgcn_update_dpp(
        0, __float_as_int(v), ctrl, 0xf, 0xf, true));
}
// f(lane 0's v), f(lane 1's v), ... of the caller's group, in that order
template <int Q, int K = 0, class F>
__device__ __forceinline__ void each_lane(float v, F f)
{
    if constexpr (K < Q) {
        f(lane_of<Q, K>(v));
        each_lane<Q, K + 1>(v, f);
    }
}

template <int Q, bool PER> struct CoopLds {
    uint32_t start[27];
    uint32_t cum[28];
    // Q == 4: see dist_tile; the gap after each 16 records holds their
    // candidate words (four workgroups then fit a CU's LDS, periodic too)
    float4 stage[80];
    // ring of accepted candidates of each particle
    static constexpr uint32_t CAP = Q == 4 ? 128 : 256;
    uint32_t list[64 / Q][CAP];
    uint32_t owns[64 / Q];
    float4 shift[PER ? 27 : 1];
    __device__ __forceinline__ void set_shift(int k, const float4& v)
    {
        shift[k] = v;
    }
    __device__ __forceinline__ float4 get_shift(int k) { return shift[k]; }
};

// Relative squared distances by v_mfma_f32_16x16x4_f32: with a point
// relative to a centre, s' = |r_j|^2 - 2 r_i . r_j + |r_i|^2 is a product
// over K = 4, candidates (x, y, z, |r_j|^2) by particles (-2x, -2y, -2z, 1),
// plus |r_i|^2.  One instruction gives the 256 values of 16 candidates and
// 16 particles, where the vector ALU takes four multiply-adds per 64 of
// them, an LDS broadcast and its wait for each.
// Lane 16 g + o holds row (candidate) o and component g of A, column
// (particle) o and component g of B, and D's rows 4 g .. 4 g + 3 of column o.
// Row 4 a + i of product m is candidate 16 a + 4 m + i, so that the four
// products leave lane (g, o) with the candidates 16 g .. 16 g + 15, in
// order, against particle o.  Candidate c is staged in float4 slot
// c + 4 (c / 16): the 64 words of one A operand then lie in 64 banks.
typedef float dist4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t dist_slot(uint32_t c)
{
    return c + 4u * (c >> 4);
}
__device__ __forceinline__ const float* dist_row(const float4* stage,
                                                 int lane)
{
    const int a = (lane >> 2) & 3, i = lane & 3, k = lane >> 4;
    return reinterpret_cast<const float*>(stage) + 4 * (20 * a + i) + k;
}
// The candidate word of record c, in the gap after its 16 records; Q == 16
// (unpadded records): after all of them.
template <int Q>
__device__ __forceinline__ uint32_t* dist_word(float4* stage, uint32_t c)
{
    uint32_t* w = reinterpret_cast<uint32_t*>(stage);
    return Q == 4 ? w + 80u * (c >> 4) + 64u + (c & 15u) : w + 256u + c;
}
// Accept bits of the candidates 16 g .. 16 g + 15 (the first in bit 15)
// against the particle of column o: the signs of s' - limit (C is |r_i|^2 -
// limit in every row, so that a bit costs one v_alignbit).
__device__ __forceinline__ uint32_t dist_tile(const float (&A)[4], float B,
                                              float C)
{
    dist4 d[4];
#pragma unroll
    for (int m = 0; m < 4; m++)
        d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[m], B,
                                                    dist4{ C, C, C, C }, 0, 0,
                                                    0);
    uint32_t w = 0;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            w = __builtin_amdgcn_alignbit(w, __float_as_uint(d[m][i]), 31);
    return w;
}
// The staged record of a candidate at rjo from the centre.  One that is not
// finite is accepted by every particle, as s > smax is false for it.
template <int D> __device__ __forceinline__ float4 dist_stage(const f3& rjo)
{
    float bj = rjo.x * rjo.x;
    bj = __builtin_fmaf(rjo.y, rjo.y, bj);
    if constexpr (D == 3) bj = __builtin_fmaf(rjo.z, rjo.z, bj);
    return bj < 3e38f ? make_float4(rjo.x, rjo.y, rjo.z, bj)
                      : make_float4(0.f, 0.f, 0.f, -3e38f);
}
// B and C of a particle (its position from the centre and |r_i|^2) for lane
// group g; likewise a particle that is not finite accepts every candidate
__device__ __forceinline__ float dist_b(int g, const f3& rio, float ai)
{
    const float b = g == 0   ? -2.f * rio.x
                    : g == 1 ? -2.f * rio.y
                    : g == 2 ? -2.f * rio.z
                             : 1.f;
    return ai < 3e38f ? b : 0.f;
}
__device__ __forceinline__ float dist_c(float ai, float limit)
{
    return ai < 3e38f ? ai - limit : -1.f;
}
// The 16 bits of candidates 16 g .. (the first in bit 15) of a mask over a
// chunk's survivors (the first in bit 0)
__device__ __forceinline__ uint32_t dist_bits(uint64_t m, int g)
{
    return __builtin_bitreverse32((uint32_t)(m >> (16 * g)) & 0xFFFFu) >> 16;
}

// Walk the accepted candidates of one particle per group of Q lanes.  kind,
// flag_el and el_near: as in ring_walk (kind 2: candidates with imove < 3).
// The test runs on coordinates relative to the box centre with the margin of
// ring_walk's LOOSE form, so it accepts a thin shell beyond the support:
// the callers repeat the exact test (s <= smax) on every pair.
// round(n, cw): one round, in which lane q of the group takes the list entry
// q < n (cw); called by every lane.
template <int D, int Q, bool PER, class Round>
__device__ __forceinline__ void
coop_list_walk(CoopLds<Q, PER>& L, int lane, uint32_t total,
               const f3& r_i, bool act, const f3& bmin, const f3& bmax,
               float smax, const float* __restrict__ r,
               const int* __restrict__ imove, int kind, bool flag_el,
               bool& el_near, const float* __restrict__ per, Round round)
{
    const int q = lane & (Q - 1), o = lane / Q;
    uint32_t* list = L.list[o];
    f3 cen = { 0.f, 0.f, 0.f };
    float smaxl = smax;
    if (bmin.x <= bmax.x) {
        cen = f3{ uni_f(0.5f * (bmin.x + bmax.x)),
                  uni_f(0.5f * (bmin.y + bmax.y)),
                  D == 3 ? uni_f(0.5f * (bmin.z + bmax.z)) : 0.f };
        const f3 hd = sub<D>(bmax, cen);
        const float rb = sqrtf(dot<D>(hd, hd)) * 1.0001f + sqrtf(smax);
        smaxl = uni_f(smax + rb * rb * 0x1p-14f);
    }
    const f3 rio = sub<D>(r_i, cen);
    const float ai = dot<D>(rio, rio);
    int kl = 0;         // neighbour cell of the lane's next candidate
    uint32_t head = 0, pend = 0;  // the particle's ring: first entry, entries
    constexpr uint32_t CAP = CoopLds<Q, PER>::CAP;
    bool eln = false;
    // Q == 4, lane (g, o16): the B operand and threshold of particle o16
    // and the entries its list has taken
    const int g = lane >> 4, o16 = lane & 15;
    float mB = 0.f, mC = 0.f;
    uint32_t tail = 0;
    if constexpr (Q == 4) {
        const f3 v = { __shfl(rio.x, 4 * o16), __shfl(rio.y, 4 * o16),
                       __shfl(rio.z, 4 * o16) };
        const float av = __shfl(ai, 4 * o16);
        mB = dist_b(g, v, av);
        mC = dist_c(av, smaxl);
    }
    const uint64_t actm = __ballot(act);
    const bool act16 = ((actm >> (4 * o16)) & 1ull) != 0;
    const float* row = dist_row(L.stage, lane);
    // the loads of the next chunk are issued before a chunk is tested
    uint32_t j = 0;
    int klj = 0, im_j = 0;
    f3 rj = { 0.f, 0.f, 0.f };
    auto fetch = [&](uint32_t cb) {
        const uint32_t t = cb + (uint32_t)lane;
        im_j = 0;
        if (t < total) {
            while (t >= L.cum[kl + 1]) kl++;
            j = L.start[kl] + (t - L.cum[kl]);
            klj = kl;
            rj = ldv_o<D>(r, j);
            im_j = ldi_o(imove, j);
        }
    };
    // rounds while some particle has `most` or more listed; those with a
    // whole round's worth (any, at the end) take part
    // (the test at the bottom: the sums are updated in place)
    auto consume = [&](uint32_t most, uint32_t least) {
        if (__ballot(pend >= most) == 0) return;
        do {
            const uint32_t n = pend >= least ? min(pend, (uint32_t)Q) : 0u;
            round(n, list[(head + (uint32_t)q) & (CAP - 1)]);
            head += n;
            pend -= n;
        } while (__ballot(pend >= most) != 0);
    };
    fetch(0);
    for (uint32_t cb = 0; cb < total; cb += 64) {
        // stage the chunk
        bool take = false, is_el = false;
        float4 st = make_float4(0.f, 0.f, 0.f, 0.f);
        const uint32_t word =
            PER ? (j | ((uint32_t)klj << PER_KL_SHIFT)) : j;
        if (cb + (uint32_t)lane < total) {
            if constexpr (PER) {
                const float4 sh = L.get_shift(klj);
                rj = per_shift<D>(rj, f3{ sh.x, sh.y, sh.z }, per);
            }
            is_el = (im_j == -3);
            take = kind == 1   ? is_el
                   : kind == 2 ? im_j < 3
                               : (im_j == 1 || (flag_el && is_el));
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
        const uint32_t cnt = (uint32_t)__popcll(tm);
        if (cnt != 0) {
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                (uint32_t)(tm >> 32),
                __builtin_amdgcn_mbcnt_lo((uint32_t)tm, 0u));
            if (take) {
                L.stage[Q == 4 ? dist_slot(rank) : rank] = st;
                *dist_word<Q>(L.stage, rank) = word;
            }
        }
        // wall elements among the survivors (flagged, then dropped): bit c
        // for the c-th survivor
        uint64_t elm = 0;
        if (kind == 0) {
            uint64_t e = __ballot(take && is_el);
            while (e != 0) {
                const int b = __builtin_ctzll(e);
                elm |= 1ull << __popcll(tm & ((1ull << b) - 1ull));
                e &= e - 1ull;
            }
        }
        if (cb + 64 < total) fetch(cb + 64);
        if (cnt == 0) continue;
        lds_order();
        if constexpr (Q == 4) {
            const float A[4] = { row[0], row[16], row[32], row[48] };
            uint32_t w = dist_tile(A, mB, mC);
            const uint64_t valid = cnt < 64 ? (1ull << cnt) - 1ull : ~0ull;
            w &= dist_bits(valid, g);
            if (!act16) w = 0;
            if (elm != 0) {
                const uint32_t ew = dist_bits(elm, g);
                eln = eln || (w & ew) != 0;
                w &= ~ew;
            }
            // places in the lists: the lanes (0, o) .. (3, o) in turn
            const uint32_t c = (uint32_t)__popc(w);
            const uint32_t c16 = __shfl_xor(c, 16);
            const uint32_t c32 = __shfl_xor(c + c16, 32);
            uint32_t pa = tail + ((g & 1) ? c16 : 0u) + ((g & 2) ? c32 : 0u);
            uint32_t pb = pa + c - 1u;
            uint32_t* lst = L.list[o16];
            const uint32_t* cj = dist_word<Q>(L.stage, 16u * (uint32_t)g);
            // from both ends of the piece: two entries per LDS round trip
            while (w != 0) {
                const uint32_t a = 31u - (uint32_t)__builtin_clz(w);
                const uint32_t b = (uint32_t)__builtin_ctz(w);
                const uint32_t ja = cj[15u - a], jb = cj[15u - b];
                w &= ~((1u << a) | (1u << b));
                lst[pa & (CAP - 1)] = ja;
                lst[pb & (CAP - 1)] = jb;
                pa++;
                pb--;
            }
            const uint32_t tot = c + c16 + c32;
            tail += tot;
            pend += (uint32_t)__shfl(tot, o);
        } else {
            // survivors q, q + Q, ...: the bits of the group's lanes are
            // the accept flags of Q successive survivors
            const uint32_t sh = ((uint32_t)(o * Q)) & 31u;
            const bool upper = o * Q >= 32;
            const uint32_t below = (1u << q) - 1u;
            for (uint32_t t = 0; t < cnt; t += Q) {
                const uint32_t k = t + (uint32_t)q;
                const float4 c = L.stage[k & 63u];
                float d = rio.x * c.x;
                d = __builtin_fmaf(rio.y, c.y, d);
                if constexpr (D == 3) d = __builtin_fmaf(rio.z, c.z, d);
                const float s = __builtin_fmaf(-2.f, d, ai + c.w);
                bool acc = !(s > smaxl) && act && k < cnt;
                if (elm != 0) {
                    const bool e = ((elm >> (k & 63u)) & 1ull) != 0;
                    eln = eln || (acc && e);
                    acc = acc && !e;
                }
                const uint64_t bm = __ballot(acc);
                const uint32_t half =
                    upper ? (uint32_t)(bm >> 32) : (uint32_t)bm;
                const uint32_t mine = (half >> sh) & 0xFFFFu;
                if (acc)
                    list[(head + pend + (uint32_t)__popc(mine & below)) &
                         (CAP - 1)] = *dist_word<Q>(L.stage, k & 63u);
                pend += (uint32_t)__popc(mine);
            }
        }
        lds_order();
        consume(CAP - 63, Q);  // room for the next chunk
    }
    consume(1, 1);
    // every lane of the group learns what one of its lanes saw
    const uint64_t em = __ballot(eln);
    if constexpr (Q == 4)
        el_near = ((em >> o | em >> (o + 16) | em >> (o + 32) |
                    em >> (o + 48)) & 1ull) != 0;
    else
        el_near = ((em >> (o * Q)) & 0xFFFFull) != 0;
    lds_order();
}

// Items (groups of 64 / Q particles) a cell is handed out as, S in a full one.
// Sparse cells, under 16 of the N particles each on average (a spray): items
// for half as many particles again, since the others would find none.
template <int Q>
__device__ __forceinline__ uint32_t items_per_cell(uint32_t S,
                                                   uint32_t n_heads,
                                                   uint32_t N)
{
    if ((uint64_t)n_heads * 16 <= N) return S;
    return min(S, (N + N / 2) / n_heads / (64 / Q) + 1u);
}

// Owners of one group: the owner(i, imove)s of the particles [cstart, cend)
// with ranks lo .. lo + 64 / Q - 1 into L.owns; returns their number.
template <int Q, class Lds, class Owner>
__device__ __forceinline__ uint32_t
group_owners(Lds& L, int lane, uint32_t cstart, uint32_t cend, uint32_t lo,
             const int* __restrict__ imove, Owner owner)
{
    constexpr uint32_t OW = 64 / Q;
    uint32_t seen = 0, nf = 0;
    for (uint32_t pos = cstart; pos < cend && nf < OW; pos += 64) {
        const uint32_t ii = pos + (uint32_t)lane;
        const bool own = ii < cend && owner(ii, imove[ii]);
        const uint64_t bm = __ballot(own);
        const uint32_t rank =
            seen +
            __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                      __builtin_amdgcn_mbcnt_lo((uint32_t)bm,
                                                                0u));
        if (own && rank >= lo && rank < lo + OW) L.owns[rank - lo] = ii;
        seen += (uint32_t)__popcll(bm);
        nf = seen > lo ? min(seen - lo, OW) : 0u;
    }
    return nf;
}

}  // namespace aq
