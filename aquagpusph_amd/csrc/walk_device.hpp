// Device-side pieces shared by the fused fluid walks (walk_cells.hip: one
// lane per particle; fluid_coop.hip: several lanes per particle) and the
// generic cell kernels.
#pragma once
#include "aq_device.hpp"
#include "aq_internal.hpp"

namespace aq {

constexpr int WC_WAVES = 4;  // wavefronts per workgroup

template <int D> struct NCell {
    static constexpr int n = (D == 2) ? 9 : 27;
};

__device__ __forceinline__ uint32_t uni(uint32_t x)
{
    return __builtin_amdgcn_readfirstlane(x);
}
// a wave-uniform float, moved to a scalar register
__device__ __forceinline__ float uni_f(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// Cells are handed out in NRANGE contiguous ranges of the non-empty cell
// list, one per XCD: workgroups are dispatched to the XCDs round-robin, so
// workgroup b runs on XCD b % NRANGE and takes the cells of range b % NRANGE
// first; the neighbourhoods in flight on one XCD then lie in one slab of
// the domain and share that XCD's L2.  A workgroup whose range is done
// helps with the next ones.  Each range has its own counter, RSTRIDE words
// apart (one cache line each).
constexpr uint32_t NRANGE = 8;
constexpr uint32_t RSTRIDE = 32;

struct WalkArgs {
    const uint32_t* icell;
    const uint32_t* ihoc;
    const uint32_t* n_cells;
    const uint32_t* cell_end;
    const uint32_t* heads;
    const uint32_t* n_heads;
    uint32_t* next;  // range counters (zero at launch), RSTRIDE words apart
    const uint32_t* status;
    uint32_t N;
    uint32_t flagged;  // cell_end carries AQ_CELL_FLUID / AQ_CELL_ELEM flags
    uint32_t ranges;   // 1: one global counter; NRANGE: per-XCD ranges
    // periodic_L of a periodic box (the walks instantiated with PER wrap
    // their neighbour cells), nullptr otherwise
    const float* per = nullptr;
    // near-cell list the fused walk fills: (first, cell, cell_end)
    // triplets of the cells with a fluid particle near a wall element,
    // counted in n_heads[AQ_CL_NNCELLS]; nullptr: not built
    uint32_t* nlist = nullptr;
    // the non-empty cells in blocked order, as (first, cell, cell_end)
    // triplets (n_heads[0] of them), for the fused walk's hand-out;
    // nullptr: the row-major heads list
    const uint32_t* blist = nullptr;
};
// Candidate words of the periodic walks: the particle index in the low
// bits and the neighbour-table entry (0..26) in the top 5.
constexpr uint32_t PER_KL_SHIFT = 27;
constexpr uint32_t PER_J_MASK = (1u << PER_KL_SHIFT) - 1u;
// Particles such a word can name (the group walks; the one-lane walks keep
// the index alone)
constexpr uint32_t PER_GROUP_MAX_N = 1u << PER_KL_SHIFT;

// Candidate table of cell c_i: start and prefix count of each neighbour
// cell in walk order.  Cells known to hold none of the `want` kinds
// (AQ_CELL_FLUID / AQ_CELL_ELEM) count as empty: they have no candidate the
// caller accepts, so the sums are unchanged.
template <int D, bool PER = false, class Lds>
__device__ __forceinline__ uint32_t neighbour_table(const WalkArgs& w,
                                                    uint32_t c_i, Lds& L,
                                                    int lane, uint32_t want)
{
    // lane k < NC fills entry k; the prefix sums by a scan over those lanes
    // (a serial loop over LDS on one lane took about 1.5 us per cell)
    constexpr int NC = NCell<D>::n;
    const uint32_t nx = w.n_cells[0], ny = w.n_cells[1];
    uint32_t n = 0;
    if (lane < NC) {
        int ci, cj, ck;
        if (D == 2) {
            ci = lane / 3 - 1;
            cj = lane % 3 - 1;
            ck = 0;
        } else {
            ci = lane / 9 - 1;
            cj = (lane / 3) % 3 - 1;
            ck = lane % 3 - 1;
        }
        uint32_t c;
        if constexpr (PER) {
            f3 sh;
            c = per_neighbour<D>(c_i, ci, cj, ck, w.n_cells, w.per, sh);
            L.set_shift(lane, make_float4(sh.x, sh.y, sh.z, 0.f));
        } else {
            c = c_i + (uint32_t)ci + (uint32_t)cj * nx +
                (uint32_t)ck * nx * ny;
        }
        const uint32_t s = w.ihoc[c];
        if (s < w.N) {
            const uint32_t ce = w.cell_end[c];
            if (!w.flagged || (ce & want)) n = (ce & AQ_CELL_END) - s;
        }
        L.start[lane] = s;
    }
    uint32_t x = n;  // inclusive sums (NC <= 27 lanes)
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 0) L.cum[0] = 0;
    if (lane < NC) L.cum[lane + 1] = x;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0);
    return __builtin_amdgcn_readlane(x, NC - 1);
}

// Bounding box of the active lanes' positions (uniform; +-inf if none)
template <int D>
__device__ __forceinline__ void wave_box(const f3& r_i, bool act, f3& bmin,
                                         f3& bmax)
{
    const float inf = __builtin_huge_valf();
    float lo[3] = { act ? r_i.x : inf, act ? r_i.y : inf,
                    act ? r_i.z : inf };
    float hi[3] = { act ? r_i.x : -inf, act ? r_i.y : -inf,
                    act ? r_i.z : -inf };
#pragma unroll
    for (int k = 0; k < D; k++) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], o));
        }
    }
    // uniform: held in scalar registers
    bmin = f3{ uni_f(lo[0]), uni_f(lo[1]), D == 3 ? uni_f(lo[2]) : 0.f };
    bmax = f3{ uni_f(hi[0]), uni_f(hi[1]), D == 3 ? uni_f(hi[2]) : 0.f };
}
// s + x with the rounding error of every addition collected in c (Kahan-
// Babuska / Neumaier: the larger operand's low bits are the ones lost)
__device__ __forceinline__ void nsum(float& s, float& c, float x)
{
    const float t = s + x;
    const bool big = fabsf(s) >= fabsf(x);
    const float lo = big ? ((s - t) + x) : ((x - t) + s);
    c += lo;
    s = t;
}

template <int D>
__device__ __forceinline__ void naxpy(f3& acc, f3& c, float s, const f3& v)
{
    nsum(acc.x, c.x, s * v.x);
    nsum(acc.y, c.y, s * v.y);
    if (D == 3) nsum(acc.z, c.z, s * v.z);
}

// ---------------------------------------------------------------------------
// Range record of the fluid fields, for the division and square root path
// without range scaling (div_nr, sqrt_nr): 7 words from RREC words after
// the non-empty cell count on, RSTRIDE words apart (one cache line each, so
// that the workgroups' atomics on different words proceed in parallel), bit
// patterns of non-negative floats compared as
// integers (a negative rho or m, an infinity or a NaN lands above every
// finite positive pattern): min |p| over p != 0, max |p|, min and max rho,
// min and max m, max |u| component over the fluid particles.
// ---------------------------------------------------------------------------
constexpr uint32_t RREC = 288;
// the cell list's count buffer holds 512 words (runtime/tools.cpp)
static_assert(RREC + 6 * RSTRIDE < 512, "range record beyond the count buffer");
constexpr uint32_t NREC = 7;
// The threshold T (a power of two, 0 when the path is not usable) such
// that every division of the fused walk's pair terms meets div_nr's
// conditions (b in [2^-100, 2^100]; a == 0 or |a| >= 2^-100 and a / b in
// [2^-120, 2^90]) for all fluid pairs with s == 0 or s >= 2^-96 and
// udr == 0 or |udr| >= T (both tested per pair), from the range record.
// Each operand's bounds follow its expression with a factor 2 of margin
// for the roundings:
//   sqrt(s) / H          sqrt(s) in {0} U [2^-48, sqrt(smax)]
//   f_ij = kF(q) CONF m_j, kF = wcon a^3, a = 2 - q: a == 0 or
//                        |a| in [2^-23, 2] (a nonzero difference of 2 and
//                        a float in [0, 4) is a multiple of 2^-23)
//   (p_i + p_j) / (rho_i rho_j)   a nonzero sum of two floats of magnitude
//                                 >= Pmin is >= Pmin 2^-24
//   f_ij CLEARY udr / (r2 rho_i rho_j), r2 = (q^2 + 0.01) H^2   (Monaghan)
//   2 f_ij / (rho_i rho_j)                                     (Morris)
//   udr f_ij rho_i / rho_j,  f_ij / rho_j,  |udr| <= 3 (2 Umax) sqrt(smax)
// A zero numerator (f_ij == 0 at q == 2, udr == 0, p_i + p_j == 0) needs
// no bound.
template <int D>
__device__ __forceinline__ float fast_threshold(
    const uint32_t* __restrict__ rec, float H, float CONF, float smax,
    int lapf, bool lapp)
{
    uint32_t b[NREC];
#pragma unroll
    for (uint32_t k = 0; k < NREC; k++) b[k] = uni(rec[k * RSTRIDE]);
    if (b[1] >= 0x7F800000u || b[3] >= 0x7F800000u ||
        b[5] >= 0x7F800000u || b[6] >= 0x7F800000u)
        return 0.f;  // an infinity, a NaN, a negative rho or m
    if (b[2] > b[3] || b[4] > b[5]) return 0.f;  // no fluid particle
    const double Pmin = __uint_as_float(b[0]), Pmax = __uint_as_float(b[1]);
    const double Rmin = __uint_as_float(b[2]), Rmax = __uint_as_float(b[3]);
    const double Mmin = __uint_as_float(b[4]), Mmax = __uint_as_float(b[5]);
    const double Umax = __uint_as_float(b[6]);
    const double h = H, conf = CONF;
    if (!(h > 0.0) || !(conf > 0.0) || !(smax > 0.f) || !(Mmin > 0.0) ||
        !(Rmin > 0.0))
        return 0.f;
    auto win = [](double nlo, double nhi, double dlo, double dhi) {
        return dlo >= 0x1p-100 && dhi <= 0x1p100 && nlo >= 0x1p-100 &&
               nhi <= 0x1p100 && nlo / dhi >= 0x1p-120 &&
               nhi / dlo <= 0x1p90;
    };
    constexpr double CLEARY = (D == 2) ? 8.0 : 10.0;
    const double wcon = ((D == 2) ? 1.09375 : 0.8203125) * 0.318309886;
    const double rs = 2.0 * sqrt((double)smax);
    const double flo = wcon * 0x1p-69 * conf * Mmin * 0.5;
    const double fhi = wcon * 8.0 * conf * Mmax * 2.0;
    const double ud = 12.0 * Umax * rs;
    const double rrlo = Rmin * Rmin * 0.5, rrhi = Rmax * Rmax * 2.0;
    // q <= sqrt(smax) / H, about 2: r2 <= 4.2 H^2
    const double slo = 0.01 * h * h * 0.5 * rrlo, shi = 4.2 * h * h * 2.0 * rrhi;
    // smallest T for the two terms with udr in the numerator
    double need = fmax(0x1p-100 / (flo * Rmin * 0.5),
                       0x1p-120 * Rmax * 2.0 / (flo * Rmin * 0.5));
    if (lapf == AQ_LAP_MONAGHAN)
        need = fmax(need, fmax(0x1p-100 / (flo * CLEARY * 0.5),
                               0x1p-120 * shi / (flo * CLEARY * 0.5)));
    if (!(need <= 0x1p-20)) return 0.f;  // not worth the per-pair fall-backs
    int e = 0;
    frexp(need, &e);
    const double T = ldexp(1.0, e);  // a power of two >= need
    bool ok = win(0x1p-49, rs, h, h);
    if (b[0] != 0x7F800000u)  // some p != 0
        ok = ok && win(Pmin * 0x1p-25, 4.0 * Pmax, rrlo, rrhi);
    if (lapf == AQ_LAP_MONAGHAN)
        ok = ok && win(flo * CLEARY * T * 0.5, fhi * CLEARY * ud * 2.0, slo,
                       shi);
    else
        ok = ok && win(flo, 4.0 * fhi, rrlo, rrhi);
    ok = ok && win(T * flo * Rmin * 0.5, ud * fhi * Rmax * 2.0, Rmin * 0.5,
                   Rmax * 2.0);
    if (lapp) ok = ok && win(flo, fhi, Rmin * 0.5, Rmax * 2.0);
    return ok ? (float)T : 0.f;
}
// The fluid terms of one pair (cfd/Interactions.cl:60-145, basic/deltaSPH.cl
// :191-242, cfd/Shepard.cl), as the factors the sums take: grad p += sg
// r_ij, lap u += sl (r_ij or u_ij), div u += td, lap p += tl, and with SHEP
// == 1 the Shepard sum += sh.  FD: the divisions by div_nr.
struct PairTerms {
    float sg, sl, td, tl, sh;
};
template <int D, int SHEP, bool FD>
__device__ __forceinline__ PairTerms
fluid_pair(int lapf, bool lapp, float q, float m_j, float rho_j, float p_j,
           float udr, float p_i, float rho_i, float H, float CONW, float CONF)
{
    constexpr float CLEARY = (D == 2) ? 8.f : 10.f;
    PairTerms t;
    t.sh = (SHEP == 1) ? kernelW<D>(q) * CONW * m_j / rho_j : 0.f;
    const float fk = kernelF<D>(q) * CONF;
    const float f_ij = fk * m_j;
    t.tl = 0.f;
    if constexpr (FD) {
        const Rcp Rr = rcp_nr(rho_i * rho_j);
        const Rcp Rj = rcp_nr(rho_j);
        t.sg = div_nr(p_i + p_j, Rr) * f_ij;
        if (lapf == AQ_LAP_MONAGHAN) {
            const float r2 = (q * q + 0.01f) * H * H;
            t.sl = div_nr(f_ij * CLEARY * udr, rcp_nr(r2 * rho_i * rho_j));
        } else {
            t.sl = div_nr(f_ij * 2.f, Rr);
        }
        t.td = div_nr(udr * f_ij * rho_i, Rj);
        if (lapp) t.tl = (p_j - p_i) * div_nr(f_ij, Rj);
    } else {
        t.sg = (p_i + p_j) / (rho_i * rho_j) * f_ij;
        if (lapf == AQ_LAP_MONAGHAN) {
            const float r2 = (q * q + 0.01f) * H * H;
            t.sl = f_ij * CLEARY * udr / (r2 * rho_i * rho_j);
        } else {
            t.sl = f_ij * 2.f / (rho_i * rho_j);
        }
        t.td = udr * f_ij * rho_i / rho_j;
        if (lapp) t.tl = (p_j - p_i) * (f_ij / rho_j);
    }
    return t;
}

}  // namespace aq
