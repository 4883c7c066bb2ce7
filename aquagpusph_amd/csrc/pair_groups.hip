// The fluid pair kernels of the per-kernel C ABI (aq_shepard,
// aq_interactions, aq_lapp) with a group of Q lanes per particle
// (coop_device.hpp).
//
// A caller of the C ABI brings the link-list (icell, ihoc, n_cells) and no
// cell list, so a wavefront takes OW = 64 / Q consecutive particles of the
// sorted arrays and walks the cells among them one after the other; the ends
// of the neighbour cells come from icell itself, 64 of its entries per cell
// read together.  Every sum takes the terms of the per-particle kernels of
// sph.hip in the same order, bit for bit.
//
// The per-particle kernels are bound by latency and divergence: each lane
// reads its own candidates one at a time (256 accepted of 1728 in 3D).  At
// 150 k particles in 3D: Shepard 841 -> 380 us, interactions 1278 ->
// 510 us, lap p 935 -> 386 us.  A wavefront pays some 2 us per cell among its
// particles, though, so where they are scattered over many cells, or where
// the per-particle form fills the chip, that form is the faster one: a large
// launch comes in both, and the device takes one (pair_groups_edges).
#include "aq_device.hpp"
#include "aq_internal.hpp"
#include "coop_device.hpp"
#include "walk_device.hpp"

namespace aq {

namespace {

// Largest launch with 16 lanes per particle, 4 above.  Shepard /
// interactions in us, 16 and 4 lanes:
//   2D, 16 per cell   20 k  19 /  25  34 /  45    48 k  33 /  46   38 /  51
//                     64 k  40 /  57  53 /  67   150 k  77 / 113   87 / 117
//   3D, 64 per cell   20 k  79 / 127 138 / 181    48 k 137 / 213  168 / 224
//                     64 k 163 / 263 183 / 252   150 k 320 / 548  386 / 513
constexpr uint32_t GROUPS_16 = 50000;
// Largest launch by groups whatever the cells hold: the per-particle form
// gains 5 us at most there (20 k particles, 0.3 per cell, 19 against 14 us),
// about what its launch takes.
constexpr uint32_t GROUPS_ALL = 16384;

// Link-list of the caller
struct RunArgs {
    const uint32_t* icell;
    const uint32_t* ihoc;
    const uint32_t* n_cells;
    uint32_t N;
    uint32_t edges;  // pair_groups_edges
};

// neighbour_table without a cell list: a cell's particles are the run of
// equal icell from its head on.
template <int D, class Lds>
__device__ __forceinline__ uint32_t run_table(const RunArgs& w, uint32_t c_i,
                                              Lds& L, int lane)
{
    constexpr int NC = NCell<D>::n;
    const uint32_t nx = w.n_cells[0], ny = w.n_cells[1];
    uint32_t c = 0, s = w.N;
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
        c = c_i + (uint32_t)ci + (uint32_t)cj * nx + (uint32_t)ck * nx * ny;
        s = w.ihoc[c];
    }
    // the first 64 entries of every cell, all reads issued together
    uint32_t v[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const uint32_t sk = __builtin_amdgcn_readlane(s, k);
        const uint32_t ck = __builtin_amdgcn_readlane(c, k);
        v[k] = ck + 1u;
        if (sk < w.N && sk + (uint32_t)lane < w.N) v[k] = w.icell[sk + lane];
    }
    uint32_t n = 0;
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const uint32_t sk = __builtin_amdgcn_readlane(s, k);
        const uint32_t ck = __builtin_amdgcn_readlane(c, k);
        uint64_t out = __ballot(v[k] != ck);
        uint32_t m = out ? (uint32_t)__builtin_ctzll(out) : 64u;
        while (!out) {  // more than 64 particles
            const uint32_t j = sk + m + (uint32_t)lane;
            const uint32_t x = j < w.N ? w.icell[j] : ck + 1u;
            out = __ballot(x != ck);
            m += out ? (uint32_t)__builtin_ctzll(out) : 64u;
        }
        if (lane == k) n = m;
    }
    uint32_t x = n;  // inclusive sums (NC <= 27 lanes)
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 0) L.cum[0] = 0;
    if (lane < NC) {
        L.start[lane] = s;
        L.cum[lane + 1] = x;
    }
    lds_order();
    return __builtin_amdgcn_readlane(x, NC - 1);
}

// Policies: KIND of the candidates (coop_list_walk), owner(im), State,
// init(i, st), load(j) (Cand: position r, ...), term(cand, r_ij, s, st),
// add_group<Q>(st, term), finish(i, st); none(): the term of a lane without
// a candidate, -0 (x + -0 is x for every x); NO_SELF: a particle is not its
// own candidate.
template <int D, int Q, class Pol>
__global__ void __launch_bounds__(64 * WC_WAVES)
    run_group_k(Pol pol, const int* __restrict__ imove,
                const float* __restrict__ r, RunArgs w, float smax,
                uint32_t nblocks)
{
    constexpr uint32_t OW = 64 / Q;
    __shared__ CoopLds<Q, false> lds[WC_WAVES];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int q = lane & (Q - 1), o = lane / Q;
    CoopLds<Q, false>& L = lds[wv];
    // one contiguous stretch of the particles per XCD (workgroup b runs on
    // XCD b % 8), so that the neighbourhoods in flight share its L2
    const uint32_t b = (blockIdx.x % NRANGE) * (gridDim.x / NRANGE) +
                       blockIdx.x / NRANGE;
    if (b >= nblocks) return;
    if (w.edges && sampled_cells(w.icell, w.N) > w.edges) return;  // sparse
    const uint32_t i = (b * WC_WAVES + (uint32_t)wv) * OW + (uint32_t)o;
    uint32_t c = 0;
    bool own = false;
    if (i < w.N) {
        c = w.icell[i];
        own = pol.owner(imove[i]);
    }
    uint64_t left = __ballot(own);
    while (left) {
        const uint32_t c_i =
            __builtin_amdgcn_readlane(c, __builtin_ctzll(left));
        const bool act = own && c == c_i;
        left &= ~__ballot(act);
        const uint32_t total = run_table<D>(w, c_i, L, lane);
        typename Pol::State st{};
        f3 r_i = { 0.f, 0.f, 0.f };
        if (act) {
            r_i = ldv<D>(r, i);
            pol.init(i, st);
        }
        f3 bmin, bmax;
        wave_box<D>(r_i, act, bmin, bmax);
        auto round = [&](uint32_t n, uint32_t j) {
            typename Pol::Term t = Pol::none();
            if ((uint32_t)q < n) {
                const typename Pol::Cand cd = pol.load(j);
                const f3 r_ij = sub<D>(cd.r, r_i);
                const float s = dot<D>(r_ij, r_ij);
                // the walk's test accepts a thin shell beyond: such a
                // candidate adds nothing, whatever its fields hold (the term
                // is selected, so that every load of the pair is issued at
                // once)
                const bool out =
                    (s > smax) | (Pol::NO_SELF && j == i);
                t = pol.term(cd, r_ij, s, st);
                if (out) t = Pol::none();
            }
            pol.template add_group<Q>(st, t);
        };
        bool unused = false;
        coop_list_walk<D, Q, false>(
            L, lane, total, r_i, act, bmin, bmax, smax, r, imove, Pol::KIND,
            false, unused, nullptr, round);
        if (act && q == 0) pol.finish(i, st);
        lds_order();
    }
}

template <int Q> __device__ __forceinline__ void add_lanes(float& a, float v)
{
    each_lane<Q>(v, [&](float x) { a += x; });
}

// basic/Shepard.cl:76-125; KIND 0: cfd/Shepard.cl (fluid candidates and no
// other positive imove among the owners), KIND 2: imove < 3
template <int D, int K> struct PolShepard {
    static constexpr int KIND = K;
    static constexpr bool NO_SELF = false;
    const float *r, *rho, *m;
    float* shepard;
    float H, CONW;
    struct State {
        float acc;
    };
    struct Cand {
        f3 r;
        float rho, m;
    };
    using Term = float;
    __device__ bool owner(int im) const
    {
        return im >= -3 && (im <= 0 || (K == 0 ? im == 1 : im < 3));
    }
    __device__ void init(uint32_t i, State& st) const { st.acc = shepard[i]; }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r, j), ldf_o(rho, j), ldf_o(m, j) };
    }
    __device__ Term term(const Cand& c, const f3&, float s,
                         const State&) const
    {
        return kernelW<D>(sqrtf(s) / H) * CONW * c.m / c.rho;
    }
    __device__ static Term none() { return -0.f; }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.acc, t);
    }
    __device__ void finish(uint32_t i, const State& st) const
    {
        shepard[i] = st.acc;
    }
};

// cfd/Interactions.cl:60-145
template <int D> struct PolInteractions {
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = true;
    const float *r, *u, *rho, *m, *p;
    float *grad_p, *lap_u, *div_u;
    float H, CONF;
    int lap;
    struct State {
        f3 u_i, gp, lu;
        float p_i, rho_i, dv;
    };
    struct Cand {
        f3 r, u;
        float rho, m, p;
    };
    struct Term {
        f3 g, l;  // the rounded products of the axpys
        float d;
    };
    __device__ bool owner(int im) const { return im == 1; }
    __device__ void init(uint32_t i, State& st) const
    {
        st.u_i = ldv<D>(u, i);
        st.p_i = p[i];
        st.rho_i = rho[i];
        st.gp = ldv<D>(grad_p, i);
        st.lu = ldv<D>(lap_u, i);
        st.dv = div_u[i];
    }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r, j), ldv_o<D>(u, j), ldf_o(rho, j),
                     ldf_o(m, j), ldf_o(p, j) };
    }
    __device__ Term term(const Cand& c, const f3& r_ij, float s,
                         const State& st) const
    {
        const f3 u_ij = sub<D>(c.u, st.u_i);
        const float udr = dot<D>(u_ij, r_ij);
        const PairTerms t = fluid_pair<D, 0, false>(
            lap, false, sqrtf(s) / H, c.m, c.rho, c.p, udr, st.p_i, st.rho_i,
            H, 0.f, CONF);
        return Term{ scl<D>(t.sg, r_ij),
                     scl<D>(t.sl, lap == AQ_LAP_MONAGHAN ? r_ij : u_ij),
                     t.td };
    }
    __device__ static Term none()
    {
        return Term{ f3{ -0.f, -0.f, -0.f }, f3{ -0.f, -0.f, -0.f }, -0.f };
    }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.gp.x, t.g.x);
        add_lanes<Q>(st.gp.y, t.g.y);
        if constexpr (D == 3) add_lanes<Q>(st.gp.z, t.g.z);
        add_lanes<Q>(st.lu.x, t.l.x);
        add_lanes<Q>(st.lu.y, t.l.y);
        if constexpr (D == 3) add_lanes<Q>(st.lu.z, t.l.z);
        add_lanes<Q>(st.dv, t.d);
    }
    __device__ void finish(uint32_t i, const State& st) const
    {
        stxyz<D>(grad_p, i, st.gp);
        stxyz<D>(lap_u, i, st.lu);
        div_u[i] = st.dv;
    }
};

// basic/deltaSPH.cl:191-242 (lapp), fluid only
template <int D> struct PolLapP {
    static constexpr int KIND = 0;
    static constexpr bool NO_SELF = true;
    const float *r, *rho, *m, *p;
    float* lap_p;
    float H, CONF;
    struct State {
        float p_i, acc;
    };
    struct Cand {
        f3 r;
        float rho, m, p;
    };
    using Term = float;
    __device__ bool owner(int im) const { return im == 1; }
    __device__ void init(uint32_t i, State& st) const
    {
        st.p_i = p[i];
        st.acc = lap_p[i];
    }
    __device__ Cand load(uint32_t j) const
    {
        return Cand{ ldv_o<D>(r, j), ldf_o(rho, j), ldf_o(m, j),
                     ldf_o(p, j) };
    }
    __device__ Term term(const Cand& c, const f3&, float s,
                         const State& st) const
    {
        const float f_ij = kernelF<D>(sqrtf(s) / H) * CONF * c.m / c.rho;
        return (c.p - st.p_i) * f_ij;
    }
    __device__ static Term none() { return -0.f; }
    template <int Q>
    __device__ void add_group(State& st, const Term& t) const
    {
        add_lanes<Q>(st.acc, t);
    }
    __device__ void finish(uint32_t i, const State& st) const
    {
        lap_p[i] = st.acc;
    }
};

template <int D, class Pol>
void launch_runs(const Pol& pol, const int32_t* imove, const float* r,
                 const RunArgs& w, aq_defs d, hipStream_t s)
{
    auto go = [&](auto* ker, unsigned q) {
        const unsigned nb = blocks_for(w.N, 64 / q * WC_WAVES);
        hipLaunchKernelGGL(ker, dim3((nb + NRANGE - 1) / NRANGE * NRANGE),
                           dim3(64 * WC_WAVES), 0, s, pol, imove, r, w,
                           support_threshold(d.H), nb);
    };
    if (w.N <= GROUPS_16) go(run_group_k<D, 16, Pol>, 16);
    else go(run_group_k<D, 4, Pol>, 4);
}

}  // namespace

// Sampled cell boundaries (sampled_cells) up to which the groups take the
// launch and above which the per-particle kernels do; 0: always the groups.
// The line lies at `few` particles per cell.  aq_shepard in us by the groups
// (4 lanes; 48 k: 16) / per particle, by particles per cell:
//   2D          0.3       2          6          10         16         30
//      48 k   36 / 14   32 / 29    28 / 49    29 / 73    33 / 94   43 / 142
//      64 k   67 / 14   55 / 29    52 / 49    40 / 68    53 / 94   59 / 142
//     150 k  159 / 19  123 / 35   111 / 65    90 / 82    89 / 115 112 / 171
//     300 k  279 / 35  213 / 48   143 / 81   161 / 107  151 / 139 194 / 223
//     1.0 M  853 / 74  629 / 139  425 / 246  433 / 312  437 / 370 576 / 689
//   3D          0.3       2          5           8         12         64
//      48 k   64 / 34   59 / 67    56 / 108   60 / 146   57 / 190 147 / 685
//      64 k  111 / 35  102 / 69    98 / 114   75 / 156   87 / 193 183 / 709
//     100 k                      156 / 120  146 / 159  145 / 210 293 / 736
//     150 k  269 / 40  227 / 89   209 / 168  156 / 213  182 / 248 384 / 780
//     300 k  472 / 80  371 / 172  315 / 280  277 / 370  298 / 392 674 / 1440
//     1.0 M 1459 / 180 1089 / 362 875 / 582  787 / 776  798 / 988 2088 / 3357
// The form not taken adds 3 to 5 us (13 us for the 62 k idle wavefronts of
// 1 M scattered particles).
uint32_t pair_groups_edges(int dims, uint32_t N)
{
    if (N <= GROUPS_ALL) return 0;
    const uint32_t few = dims == 2 ? std::min(22u, N / 16000u + 1u)
                                   : std::min(8u, N / 20000u + 1u);
    return CELL_SAMPLE / few;
}

// Each returns false, launching nothing, beyond the 32-bit byte offsets of
// the candidate loads.
bool shepard_groups(int dims, const int32_t* imove, const float* r,
                    const float* rho, const float* m, float* shepard,
                    uint32_t N, const uint32_t* icell, const uint32_t* ihoc,
                    const uint32_t* n_cells, aq_defs d, int cfd,
                    hipStream_t s)
{
    if (N >= (1u << 28)) return false;
    const RunArgs w{ icell, ihoc, n_cells, N, pair_groups_edges(dims, N) };
#define AQ_SH(DD, KK)                                                          \
    launch_runs<DD>(PolShepard<DD, KK>{ r, rho, m, shepard, d.H, d.CONW },     \
                    imove, r, w, d, s)
    if (dims == 2) {
        if (cfd) AQ_SH(2, 0);
        else AQ_SH(2, 2);
    } else {
        if (cfd) AQ_SH(3, 0);
        else AQ_SH(3, 2);
    }
#undef AQ_SH
    return true;
}

bool interactions_groups(int dims, const int32_t* imove, const float* r,
                         const float* u, const float* rho, const float* m,
                         const float* p, float* grad_p, float* lap_u,
                         float* div_u, uint32_t N, const uint32_t* icell,
                         const uint32_t* ihoc, const uint32_t* n_cells,
                         aq_defs d, hipStream_t s)
{
    if (N >= (1u << 28)) return false;
    const RunArgs w{ icell, ihoc, n_cells, N, pair_groups_edges(dims, N) };
    if (dims == 2)
        launch_runs<2>(PolInteractions<2>{ r, u, rho, m, p, grad_p, lap_u,
                                           div_u, d.H, d.CONF,
                                           d.lap_formulation },
                       imove, r, w, d, s);
    else
        launch_runs<3>(PolInteractions<3>{ r, u, rho, m, p, grad_p, lap_u,
                                           div_u, d.H, d.CONF,
                                           d.lap_formulation },
                       imove, r, w, d, s);
    return true;
}

bool lapp_groups(int dims, const int32_t* imove, const float* r,
                 const float* rho, const float* m, const float* p,
                 float* lap_p, uint32_t N, const uint32_t* icell,
                 const uint32_t* ihoc, const uint32_t* n_cells, aq_defs d,
                 hipStream_t s)
{
    if (N >= (1u << 28)) return false;
    const RunArgs w{ icell, ihoc, n_cells, N, pair_groups_edges(dims, N) };
    if (dims == 2)
        launch_runs<2>(PolLapP<2>{ r, rho, m, p, lap_p, d.H, d.CONF }, imove,
                       r, w, d, s);
    else
        launch_runs<3>(PolLapP<3>{ r, rho, m, p, lap_p, d.H, d.CONF }, imove,
                       r, w, d, s);
    return true;
}

}  // namespace aq
