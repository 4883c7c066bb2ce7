// Fused fluid walk with several lanes per particle (the same terms and sums
// as fluid_pass_cells_k of walk_cells.hip, bit for bit).
//
// One lane per particle leaves a launch short of work when there are few
// particles: a 2D cell holds some 16 of them for 64 lanes, and below a few
// hundred thousand particles there are fewer cells than wavefronts the chip
// holds, while each particle's pairs (50 in 2D, 250 in 3D) form a serial
// chain.  Here Q lanes serve one particle: a wavefront takes 64 / Q fluid
// particles of a cell, and a cell is cut into such groups, handed out to
// different wavefronts.
// The group walk itself is coop_list_walk (coop_device.hpp).
#include "aq_device.hpp"
#include "aq_internal.hpp"
#include "coop_device.hpp"
#include "walk_device.hpp"

namespace aq {

namespace {

// See fluid_pass_cells_k.  Item k of the launch is group k % S of the fluid
// particles of the k / S-th cell: its particles (S t + k % S) OW + 0 .. OW -
// 1 for t = 0, 1, ..., OW = 64 / Q.  nlist gets one entry per item with a
// near particle: the runs of particles of different items do not overlap,
// so BI Interactions meets every near particle once.
template <int D, int SHEP, int MATH, bool PER, int Q>
__global__ void __launch_bounds__(64 * WC_WAVES)
    fluid_coop_k(const int* __restrict__ imove, const float* __restrict__ r,
                 const float* __restrict__ u, const float* __restrict__ rho,
                 const float* __restrict__ m, const float* __restrict__ p,
                 const float* __restrict__ normal,
                 const float* __restrict__ tangent,
                 const float* __restrict__ binormal,
                 float* __restrict__ shepard, float* __restrict__ grad_p,
                 float* __restrict__ lap_u, float* __restrict__ div_u,
                 float* __restrict__ lap_p, uint8_t* __restrict__ near,
                 WalkArgs w, float H, float CONW, float CONF, float DIMS,
                 float smax, const uint32_t* __restrict__ rec, int lapf,
                 int lapp_, uint32_t S)
{
    constexpr int OW = 64 / Q;
    const bool lapp = lapp_ != 0;
    __shared__ CoopLds<Q, PER> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int q = lane & (Q - 1), o = lane / Q;
    CoopLds<Q, PER>& L = lds[wv];
    if (w.status && (*w.status & 1u)) return;
    // 3D walk in us with S items per cell / with items_per_cell's (one lane per
    // particle), at 64, 8 and 1 particles per cell of the fluid:
    //    8 k (16 lanes)  139 / 138 ( 912)   91 /  51 (268)  109 /  44 (194)
    //   29 k (4 lanes)   252 / 253 ( 914)  157 / 118 (261)  200 / 113 (219)
    //  177 k (4 lanes)   786 / 796 (1015)  478 / 234 (397)  701 / 294 (456)
    const uint32_t n_heads = uni(*w.n_heads);
    S = items_per_cell<Q>(S, n_heads, w.N);
    const uint32_t n_items = n_heads * S;
    const float eps = 1E-8f * H;
    const bool flag_el = (SHEP == 2) || (near != nullptr);
    const uint32_t nwv = gridDim.x * WC_WAVES;
    uint32_t item = blockIdx.x * WC_WAVES + (uint32_t)wv;
    if (item >= n_items) return;
    float fdT = 0.f;
    if (rec) fdT = fast_threshold<D>(rec, H, CONF, smax, lapf, lapp);
    const bool fastdiv = fdT > 0.f;
    const Rcp RH = rcp_nr(H);
    auto rjof = [&](uint32_t j, uint32_t kl) {
        f3 v = ldv_o<D>(r, j);
        if constexpr (PER) {
            const float4 s = L.get_shift((int)kl);
            v = per_shift<D>(v, f3{ s.x, s.y, s.z }, w.per);
        }
        return v;
    };
    for (; item < n_items; item += nwv) {
        const uint32_t hk = item / S, sub_i = item % S;
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
        for (uint32_t lo = sub_i * OW;; lo += S * OW) {
            // fluid particles lo .. lo + OW - 1 of the cell
            const uint32_t nf = group_owners<Q>(
                L, lane, cstart, cend, lo, imove,
                [](uint32_t, int im) { return im == 1; });
            if (nf == 0) break;
            const uint32_t total = neighbour_table<D, PER>(
                w, c_i, L, lane,
                AQ_CELL_FLUID | (flag_el ? AQ_CELL_ELEM : 0u));
            const bool act = (uint32_t)o < nf;
            const uint32_t i = act ? L.owns[o] : cstart;
            f3 r_i = { 0.f, 0.f, 0.f }, u_i = { 0.f, 0.f, 0.f };
            float p_i = 0.f, rho_i = 1.f;
            f3 gp = { 0.f, 0.f, 0.f }, lu = { 0.f, 0.f, 0.f };
            float dv = 0.f, lp = 0.f, sh = 0.f;
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
                if (lapp) lp = lap_p[i];
                sh = (SHEP == 2) ? 1.f : (SHEP == 1 ? shepard[i] : 0.f);
            }
            bool nearw = false;
            f3 bmin, bmax;
            wave_box<D>(r_i, act, bmin, bmax);
            auto acc1 = [&](float& s, float& c, float v) {
                each_lane<Q>(v, [&](float x) {
                    if constexpr (MATH == 2) nsum(s, c, x);
                    else s += x;
                });
            };
            // ---- fluid neighbours ------------------------------------------
            // A lane without a candidate adds zeros, and so does a candidate
            // of the relative test's shell beyond the support (zero mass):
            // the sums are never -0 (they start at +0, or 1, and an exact
            // cancellation rounds to +0), so +-0 leaves them unchanged.
            auto round = [&](uint32_t n, uint32_t cw) {
                PairTerms t{ 0.f, 0.f, 0.f, 0.f, 0.f };
                f3 g = { 0.f, 0.f, 0.f }, l = { 0.f, 0.f, 0.f };
                if ((uint32_t)q < n) {
                    const uint32_t j = PER ? cw & PER_J_MASK : cw;
                    const f3 r_ij =
                        sub<D>(rjof(j, PER ? cw >> PER_KL_SHIFT : 0u), r_i);
                    const float s = dot<D>(r_ij, r_ij);
                    float m_j = ldf_o(m, j);
                    const float rho_j = ldf_o(rho, j);
                    const float p_j = ldf_o(p, j);
                    const f3 u_j = ldv_o<D>(u, j);
                    m_j = (s > smax) ? 0.f : m_j;
                    const f3 u_ij = sub<D>(u_j, u_i);
                    const float udr = dot<D>(u_ij, r_ij);
                    const bool fd =
                        fastdiv && !(((s < 0x1p-96f) & (s != 0.f)) |
                                     ((udr != 0.f) & (fabsf(udr) < fdT)));
                    if (fd)
                        t = fluid_pair<D, SHEP, true>(
                            lapf, lapp, div_nr(sqrt_nr(s), RH), m_j, rho_j,
                            p_j, udr, p_i, rho_i, H, CONW, CONF);
                    else
                        t = fluid_pair<D, SHEP, false>(
                            lapf, lapp, sqrtf(s) / H, m_j, rho_j, p_j, udr,
                            p_i, rho_i, H, CONW, CONF);
                    const f3 v = lapf == AQ_LAP_MONAGHAN ? r_ij : u_ij;
                    g = scl<D>(t.sg, r_ij);
                    l = scl<D>(t.sl, v);
                    if (PER && s > smax) {
                        t = PairTerms{ 0.f, 0.f, 0.f, 0.f, 0.f };
                        g = l = f3{ 0.f, 0.f, 0.f };
                    }
                }
                if constexpr (SHEP == 1)
                    each_lane<Q>(t.sh, [&](float x) { sh += x; });
                acc1(gp.x, cgp.x, g.x);
                acc1(gp.y, cgp.y, g.y);
                if constexpr (D == 3) acc1(gp.z, cgp.z, g.z);
                acc1(lu.x, clu.x, l.x);
                acc1(lu.y, clu.y, l.y);
                if constexpr (D == 3) acc1(lu.z, clu.z, l.z);
                acc1(dv, cdv, t.td);
                acc1(lp, clp, t.tl);  // zeros without lap p
            };
            coop_list_walk<D, Q, PER>(
                L, lane, total, r_i, act, bmin, bmax, smax, r, imove, 0,
                flag_el, nearw, w.per, round);
            // ---- wall elements (boundary-integral Shepard) ------------------
            if constexpr (SHEP == 2) {
                if (__ballot(nearw) != 0) {
                    bool self_added = false, unused = false;
                    const uint32_t total_el =
                        neighbour_table<D, PER>(w, c_i, L, lane, AQ_CELL_ELEM);
                    auto round_el = [&](uint32_t n, uint32_t j) {
                        // v: the element's part; on: the particle lies on
                        // the element (1/2, once)
                        float v = 0.f;
                        bool on = false;
                        if ((uint32_t)q < n) {
                            const f3 r_ij = sub<D>(ldv_o<D>(r, j), r_i);
                            const float s = dot<D>(r_ij, r_ij);
                            const f3 n_j = ldv_o<D>(normal, j);
                            const f3 t_j = ldv_o<D>(tangent, j);
                            const f3 b_j = ldv_o<D>(binormal, j);
                            const float area_j = ldf_o(m, j);
                            const float qq = sqrtf(s) / H;
                            const float r_n = dot<D>(r_ij, n_j);
                            const float r_t = fabsf(dot<D>(r_ij, t_j));
                            const float r_b = fabsf(dot<D>(r_ij, b_j));
                            if (s > smax) {
                            } else if ((r_n > -eps) && (r_n < eps)) {
                                const float dr =
                                    0.55f * pow_cl(area_j, 1.f / (DIMS - 1.f));
                                on = (r_t <= dr) && (r_b <= dr);
                            } else {
                                v = r_n * CONW * kernelS_P<D>(qq) * area_j +
                                    kernelS_D<D>(fabsf(r_n), r_t, r_b,
                                                 area_j);
                            }
                        }
                        if (__ballot(on) == 0) {
                            each_lane<Q>(v, [&](float x) { sh += x; });
                        } else {
                            // the half angle in its place in the order
                            const float f = on ? 1.f : 0.f;
                            float xs[Q], fs[Q];
                            int k = 0;
                            each_lane<Q>(v, [&](float x) { xs[k++] = x; });
                            k = 0;
                            each_lane<Q>(f, [&](float x) { fs[k++] = x; });
#pragma unroll
                            for (int e = 0; e < Q; e++) {
                                if (fs[e] != 0.f) {
                                    if (!self_added) {
                                        self_added = true;
                                        sh -= 0.5f;
                                    }
                                } else {
                                    sh += xs[e];
                                }
                            }
                        }
                    };
                    coop_list_walk<D, Q, PER>(
                        L, lane, total_el, r_i, act && nearw, bmin, bmax,
                        smax, r, imove, 1, false, unused, w.per, round_el);
                }
            }
            if (act && q == 0) {
                if constexpr (MATH == 2) {
                    gp = { gp.x + cgp.x, gp.y + cgp.y, gp.z + cgp.z };
                    lu = { lu.x + clu.x, lu.y + clu.y, lu.z + clu.z };
                    dv += cdv;
                    lp += clp;
                }
                stxyz<D>(grad_p, i, gp);
                stxyz<D>(lap_u, i, lu);
                div_u[i] = dv;
                if (lapp) lap_p[i] = lp;
                if (SHEP) shepard[i] = sh;
                if (near) near[i] = nearw ? 1 : 0;
            }
            if (w.nlist && __ballot(act && nearw) != 0 && lane == 0) {
                uint32_t* cnt =
                    const_cast<uint32_t*>(w.n_heads) + AQ_CL_NNCELLS;
                const uint32_t k = atomicAdd(cnt, 1u);
                w.nlist[3 * k] = L.owns[0];
                w.nlist[3 * k + 1] = c_i;
                w.nlist[3 * k + 2] =
                    (L.owns[nf - 1] + 1u) | (ce & ~AQ_CELL_END);
            }
            lds_order();
            if (nf < (uint32_t)OW) break;
        }
    }
}

}  // namespace

// Lanes per particle of the fused walk for N particles (the host knows no
// other count); 0: the one-lane walk of walk_cells.hip.  Walk times in us,
// one lane / 4 lanes / 16 lanes, on dam breaks with their walls:
//   2D      2 k 107 / 34 / 27     8 k 104 / 35 / 28    31 k 101 / 38 / 45
//         184 k 185 / 92 / 159   1.1 M 820 / 435 / 869
//   3D     11 k - / 114 / 72     23 k - / 128 / 122     40 k - / 139 / 158
//         135 k 487 / 301 / -    240 k 502 / 497 / -    314 k 534 / 635 / -
//         394 k 705 / 747 / -    764 k 1109 / 1381 / -
// A 2D cell has 16 particles, so four lanes each fill a wavefront at any
// size; a 3D cell has 64, and one lane each wins once the cells fill the
// chip: 4096 wavefronts, 262 k fluid particles (periodic cube of 262 k on the
// lattice 467 / 583, out of lattice order 846 / 943; of 195 k 778 / 663 and
// 873 / 729).  The compensated sums (math == 2) take their six operations per
// term on every lane of the group, which moves that line down (135 k on the
// lattice 503 / 503, out of it 888 / 819; 193 k 502 / 782 and 902 / 1186); 16
// lanes pay it 16 times (2D 8 k 109 / 39 / 37, 31 k 107 / 44 / 72; 3D 11 k
// - / 147 / 111, 23 k - / 171 / 242).
// A periodic box of more particles than the group walk can name: one lane.
int fluid_coop_lanes(int dims, uint32_t N, int math, bool per)
{
    const bool comp = math == 2;
    if (per && N > PER_GROUP_MAX_N) return 0;
    if (dims == 2) return N <= (comp ? 8000u : 16000u) ? 16 : 4;
    if (N <= (comp ? 12000u : 24000u)) return 16;
    return N <= (comp ? 150000u : 250000u) ? 4 : 0;
}

void launch_fluid_coop(int dims, int shep, bool lapp, int q,
                       const int32_t* imove, const float* r, const float* u,
                       const float* rho, const float* m, const float* p,
                       const float* normal, const float* tangent,
                       const float* binormal, float* shepard, float* grad_p,
                       float* lap_u, float* div_u, float* lap_p,
                       uint8_t* near, const WalkArgs& w, aq_defs d,
                       float smax, int math, const uint32_t* rec,
                       hipStream_t s)
{
    AQ_REQUIRE(!w.per || w.N <= PER_GROUP_MAX_N,
               "periodic box: more than 2^27 particles in a group walk");
    // a 2D cell holds one group of 16 particles, a 3D cell four
    const uint32_t S = q == 16 ? (dims == 2 ? 4u : 16u)
                               : (dims == 2 ? 1u : 4u);
#define AQ_CO4(DD, SH, MM, PR, QQ)                                             \
    do {                                                                       \
        auto* ker = fluid_coop_k<DD, SH, MM, PR, QQ>;                          \
        const unsigned nb =                                                    \
            std::min(resident_blocks((const void*)ker, 64 * WC_WAVES),         \
                     std::max(1u, blocks_for((size_t)w.N * QQ * 2,             \
                                             64 * WC_WAVES)));                 \
        hipLaunchKernelGGL(ker, dim3(nb), dim3(64 * WC_WAVES), 0, s, imove, r, \
                           u, rho, m, p, normal, tangent, binormal, shepard,   \
                           grad_p, lap_u, div_u, lap_p, near, w, d.H, d.CONW,  \
                           d.CONF, d.DIMS, smax, rec, d.lap_formulation,       \
                           lapp ? 1 : 0, S);                                   \
    } while (0)
#define AQ_CO3(DD, SH, MM, PR)                                                 \
    do {                                                                       \
        if (q == 16) AQ_CO4(DD, SH, MM, PR, 16);                               \
        else AQ_CO4(DD, SH, MM, PR, 4);                                        \
    } while (0)
#define AQ_CO2(DD, SH, MM)                                                     \
    do {                                                                       \
        if (w.per && SH != 2) AQ_CO3(DD, SH, MM, (SH != 2));                   \
        else AQ_CO3(DD, SH, MM, false);                                        \
    } while (0)
#define AQ_CO1(DD, SH)                                                         \
    do {                                                                       \
        if (math == 2) AQ_CO2(DD, SH, 2);                                      \
        else AQ_CO2(DD, SH, 0);                                                \
    } while (0)
    if (dims == 2) {
        if (shep == 0) AQ_CO1(2, 0);
        else if (shep == 1) AQ_CO1(2, 1);
        else AQ_CO1(2, 2);
    } else {
        if (shep == 0) AQ_CO1(3, 0);
        else if (shep == 1) AQ_CO1(3, 1);
        else AQ_CO1(3, 2);
    }
#undef AQ_CO1
#undef AQ_CO2
#undef AQ_CO3
#undef AQ_CO4
}

}  // namespace aq
