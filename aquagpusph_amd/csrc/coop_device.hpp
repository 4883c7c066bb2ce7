// Neighbour walk with a group of Q lanes per particle, for kernels whose
// cells hold few owners or whose launches have few cells:
//   test     a chunk of 64 candidates is staged through LDS as in
//            ring_walk (box prefilter, survivors compacted in order); lane
//            q of a particle tests the survivors q, q + Q, ..., and every
//            accepted one is appended, in candidate order, to the
//            particle's list in LDS (its place from the ballots);
//   consume  when a list has no room for another chunk (and at the end),
//            the lanes of every particle with Q B listed take its next Q B,
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

template <int Q, int B, bool PER> struct CoopLds {
    uint32_t start[27];
    uint32_t cum[28];
    float4 stage[64];
    uint32_t candj[64];
    // ring of accepted candidates of each particle
    static constexpr uint32_t CAP = Q == 4 ? 128 : 256;
    uint32_t list[64 / Q][CAP];
    uint32_t owns[64 / Q];
    float4 shift[PER ? 27 : 1];
};

// Walk the accepted candidates of one particle per group of Q lanes.  kind,
// flag_el, el_near and the relative test (LOOSE): as in ring_walk (kind 2:
// candidates with imove < 3).
// round(n, cw): one round, in which lane q of the group takes the list
// entries q + Q b < n (cw[b]); called by every lane.
template <int D, int Q, int B, bool LOOSE, bool PER, class Round>
__device__ __forceinline__ void
coop_list_walk(CoopLds<Q, B, PER>& L, int lane, uint32_t total,
               const f3& r_i, bool act, const f3& bmin, const f3& bmax,
               float smax, const float* __restrict__ r,
               const int* __restrict__ imove, int kind, bool flag_el,
               bool& el_near, const float* __restrict__ per, Round round)
{
    static_assert(!(LOOSE && PER), "relative test: not for periodic walks");
    const int q = lane & (Q - 1), o = lane / Q;
    uint32_t* list = L.list[o];
    f3 cen = { 0.f, 0.f, 0.f }, rio = r_i;
    float ai = 0.f, smaxl = smax;
    if constexpr (LOOSE) {
        if (bmin.x <= bmax.x) {
            cen = f3{ uni_f(0.5f * (bmin.x + bmax.x)),
                      uni_f(0.5f * (bmin.y + bmax.y)),
                      D == 3 ? uni_f(0.5f * (bmin.z + bmax.z)) : 0.f };
            const f3 hd = sub<D>(bmax, cen);
            const float rb = sqrtf(dot<D>(hd, hd)) * 1.0001f + sqrtf(smax);
            smaxl = uni_f(smax + rb * rb * 0x1p-14f);
        }
        rio = sub<D>(r_i, cen);
        ai = dot<D>(rio, rio);
    }
    int kl = 0;         // neighbour cell of the lane's next candidate
    uint32_t head = 0, pend = 0;  // the particle's ring: first entry, entries
    constexpr uint32_t CAP = CoopLds<Q, B, PER>::CAP;
    bool eln = false;
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
    auto consume = [&](uint32_t most, uint32_t least) {
        while (__ballot(pend >= most) != 0) {
            const uint32_t n =
                pend >= least ? min(pend, (uint32_t)(Q * B)) : 0u;
            uint32_t cw[B];
#pragma unroll
            for (int b = 0; b < B; b++)
                cw[b] = list[(head + (uint32_t)(q + Q * b)) & (CAP - 1)];
            round(n, cw);
            head += n;
            pend -= n;
        }
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
                const float4 sh = L.shift[klj];
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
            if constexpr (LOOSE) {
                const f3 rjo = sub<D>(rj, cen);
                float bj = rjo.x * rjo.x;
                bj = __builtin_fmaf(rjo.y, rjo.y, bj);
                if constexpr (D == 3) bj = __builtin_fmaf(rjo.z, rjo.z, bj);
                st = make_float4(rjo.x, rjo.y, rjo.z, is_el ? -bj : bj);
            } else {
                st = make_float4(rj.x, rj.y, rj.z, is_el ? -1.f : 1.f);
            }
        }
        const uint64_t tm = __ballot(take);
        const uint32_t cnt = (uint32_t)__popcll(tm);
        if (cnt != 0) {
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                (uint32_t)(tm >> 32),
                __builtin_amdgcn_mbcnt_lo((uint32_t)tm, 0u));
            if (take) {
                L.stage[rank] = st;
                L.candj[rank] = word;
            }
        }
        if (cb + 64 < total) fetch(cb + 64);
        if (cnt == 0) continue;
        lds_order();
        const bool els = kind == 0 && __ballot(take && is_el) != 0;
        // survivors q, q + Q, ...: the bits of the group's lanes are the
        // accept flags of Q successive survivors
        const uint32_t sh = ((uint32_t)(o * Q)) & 31u;
        const bool upper = o * Q >= 32;
        const uint32_t below = (1u << q) - 1u;
        for (uint32_t t = 0; t < cnt; t += Q) {
            const uint32_t k = t + (uint32_t)q;
            const float4 c = L.stage[k & 63u];
            bool acc;
            if constexpr (LOOSE) {
                float d = rio.x * c.x;
                d = __builtin_fmaf(rio.y, c.y, d);
                if constexpr (D == 3) d = __builtin_fmaf(rio.z, c.z, d);
                const float s = __builtin_fmaf(-2.f, d, ai + fabsf(c.w));
                acc = !(s > smaxl);
            } else {
                const f3 r_ij = sub<D>(f3{ c.x, c.y, c.z }, r_i);
                const float s = dot<D>(r_ij, r_ij);
                acc = !(s > smax);
            }
            acc = acc && act && k < cnt;
            if (els) {
                // wall elements in range: flagged, then dropped
                const bool e = (__float_as_uint(c.w) >> 31) != 0u;
                eln = eln || (acc && e);
                acc = acc && !e;
            }
            const uint64_t bm = __ballot(acc);
            const uint32_t half =
                upper ? (uint32_t)(bm >> 32) : (uint32_t)bm;
            const uint32_t mine =
                Q == 4 ? (half >> sh) & 15u : (half >> sh) & 0xFFFFu;
            if (acc)
                list[(head + pend + (uint32_t)__popc(mine & below)) &
                     (CAP - 1)] = L.candj[k];
            pend += (uint32_t)__popc(mine);
        }
        lds_order();
        consume(CAP - 63, Q * B);  // room for the next chunk
    }
    consume(1, 1);
    // every lane of the group learns what one of them saw
    const uint64_t em = __ballot(eln);
    constexpr uint64_t grp = Q == 4 ? 15ull : 0xFFFFull;
    el_near = ((em >> (o * Q)) & grp) != 0;
    lds_order();
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
