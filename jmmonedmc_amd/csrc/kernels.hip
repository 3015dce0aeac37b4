// kernels.hip -- gfx950 kernels of the Metropolis engine.
//
// Compiled with -ffp-contract=off: the FP64 paths round once per operation in
// the oracle's order, which makes positions and per-trial energy changes
// reproducible bit for bit (only sums over lanes differ in their order).
//
//   k_sweep_batched  persistent, work-queue driven: one workgroup takes a
//                    bundle of chains, keeps their sorted positions in LDS,
//                    one lane per block of particles, phases separated by
//                    workgroup barriers.  FP64 or FP32 pair arithmetic.
//   k_sweep_plain    one wavefront per chain; trials one at a time, the
//                    energy change a wavefront reduction over the neighbour
//                    window (lanes 0-31 left partners, 32-63 right).
//   k_observables    U, virial, dU/dtheta, dW/dtheta and dU/dx per
//                    configuration (the differentiation path), one workgroup
//                    per tile of a configuration; k_obs_sum adds the tiles.
//   k_begin          resets a work queue and advances the sample row.
#include "kernels.h"

namespace jmm {

__device__ __forceinline__ bool nbpos(const double *X, int64_t j, int64_t N, bool per, double L,
                                      double &xj)
{
    if (j >= 0 && j < N) {
        xj = X[j];
        return true;
    }
    if (!per) return false;
    xj = (j < 0) ? X[j + N] - L : X[j - N] + L;
    return true;
}

// A partner's contribution to the pair-term counter: 1 for each of the old
// and new separations inside the cutoff (the counter is n_old + n_new).
template <int KIND>
__device__ __forceinline__ uint32_t n_inside(const Pot &q, double o, double n)
{
    return (inside64<KIND>(q, o) ? 1u : 0u) + (inside64<KIND>(q, n) ? 1u : 0u);
}

// The same from the flags a walk step has: `in` (the partner is walked),
// io and inn (inside at the old / new position).  For LJ and Yukawa a
// walked partner is inside at one position at least (the walk's test is
// io || inn), so two selects suffice; with a strict cutoff a partner at
// exactly rc is walked but inside at neither.
template <int KIND>
__device__ __forceinline__ uint32_t n_walked(bool in, bool io, bool inn)
{
    if (KIND == POT_LJ || KIND == POT_YUKAWA) return in ? ((io && inn) ? 2u : 1u) : 0u;
    return in ? (io ? 1u : 0u) + (inn ? 1u : 0u) : 0u;
}

// Energy change for moving the particle at xi (index i) to xn.  Partners:
// left side nearest first and right side nearest first, each stopping at the
// first partner beyond the cutoff from both positions or at index distance
// w; the two side sums are added at the end.  Restates the
// partner sums of qad2 (src/jmmMCState.cpp:1213-1348), whose far pairs
// contribute exactly zero.
template <int KIND>
__device__ __forceinline__ double delta_e64(const Pot &q, const double *X, int64_t i, int64_t N,
                                            bool per, double L, uint32_t w, double xi, double xn,
                                            uint32_t &terms)
{
    double dEL = 0.0, dER = 0.0;
    for (uint32_t k = 1; k <= w; ++k) {
        double xj;
        if (!nbpos(X, i - (int64_t)k, N, per, L, xj)) break;
        const double dold = xi - xj, dnew = xn - xj;
        if (dold > q.rc && dnew > q.rc) break;
        dEL += phi64<KIND>(q, dnew) - phi64<KIND>(q, dold);
        terms += n_inside<KIND>(q, dold, dnew);
    }
    for (uint32_t k = 1; k <= w; ++k) {
        double xj;
        if (!nbpos(X, i + (int64_t)k, N, per, L, xj)) break;
        const double dold = xj - xi, dnew = xj - xn;
        if (dold > q.rc && dnew > q.rc) break;
        dER += phi64<KIND>(q, dnew) - phi64<KIND>(q, dold);
        terms += n_inside<KIND>(q, dold, dnew);
    }
    return dEL + dER;
}

// FP32 form: separations formed in FP64 (positions are FP64), cutoff decided
// in FP64, pair energies in FP32, each side's terms summed in FP64 (exact
// sums of the FP32 terms; an FP64 add issues at the FP32 rate on gfx950).
template <int KIND>
__device__ __forceinline__ double delta_e32(const Pot &q, const double *X, int64_t i, int64_t N,
                                            bool per, double L, uint32_t w, double xi, double xn,
                                            uint32_t &terms)
{
    double left = 0.0, right = 0.0;
    for (uint32_t k = 1; k <= w; ++k) {
        double xj;
        if (!nbpos(X, i - (int64_t)k, N, per, L, xj)) break;
        const double dold = xi - xj, dnew = xn - xj;
        if (dold > q.rc && dnew > q.rc) break;
        const bool io = inside64<KIND>(q, dold), in = inside64<KIND>(q, dnew);
        left += (double)(phi32<KIND>(q, (float)dnew, in) - phi32<KIND>(q, (float)dold, io));
        terms += (io ? 1u : 0u) + (in ? 1u : 0u);
    }
    for (uint32_t k = 1; k <= w; ++k) {
        double xj;
        if (!nbpos(X, i + (int64_t)k, N, per, L, xj)) break;
        const double dold = xj - xi, dnew = xj - xn;
        if (dold > q.rc && dnew > q.rc) break;
        const bool io = inside64<KIND>(q, dold), in = inside64<KIND>(q, dnew);
        right += (double)(phi32<KIND>(q, (float)dnew, in) - phi32<KIND>(q, (float)dold, io));
        terms += (io ? 1u : 0u) + (in ? 1u : 0u);
    }
    return left + right;
}

__device__ __forceinline__ uint32_t half_of(uint32_t size)
{
    return size >= HALF_MIN ? (size + 1) / 2 : size;
}

// Box-length trial energy over the pairs whose left member is in [p0, p1),
// for a scaling of every coordinate by sc.  Sets bad when a scaled nearest
// pair falls inside the hard core.  The energy change pair by pair,
// restating fav's trial energy (src/jmmMCState.cpp:2175-2235) as a
// difference per pair, each partner walk ending at the first partner beyond
// the cutoff at both separations: FP64 form phi64(s d) - phi64(d); FP32 form
// box_term32 of the two separations (summed in FP64).  FP32 form: u0
// receives the same pairs' energy at the unscaled separations (FP32 pair
// energies summed in FP64); for the square well the return value is the
// scaled configuration's energy instead (-eps times its pairs inside the
// well, each walk ending at the first scaled partner outside), from which
// the caller subtracts the running energy (exact, as in vol_lane).
template <typename Real, int KIND>
__device__ __forceinline__ double scaled_delta(const Pot &q, const BoxK &bk, double gmin, const double *X,
                                               int64_t N, bool per, double L, double Lp, double sc,
                                               uint32_t w, uint32_t p0, uint32_t p1, uint32_t stride,
                                               uint32_t &bad, double &u0)
{
    double part = 0.0;
    int wc = 0;
    u0 = 0.0;
    for (uint32_t p = p0; p < p1 && !bad; p += stride) {
        const double xi = X[p], xis = xi * sc;
        for (uint32_t k = 1; k <= w; ++k) {
            const int64_t j = (int64_t)p + k;
            double xj, xjs;
            if (j < N) {
                xj = X[j];
                xjs = xj * sc;
            } else if (per) {
                xj = X[j - N] + L;
                xjs = X[j - N] * sc + Lp;
            } else {
                break;
            }
            const double d0 = xj - xi, d1 = xjs - xis;
            if (k == 1 && d1 < gmin) {
                bad = 1;
                break;
            }
            if (sizeof(Real) == 8) {
                if (d0 > q.rc && d1 > q.rc) break;
                part += phi64<KIND>(q, d1) - phi64<KIND>(q, d0);
            } else {
                const bool in0 = inside64<KIND>(q, d0), in1 = inside64<KIND>(q, d1);
                if (!(in0 || in1)) break;
                if (KIND == POT_HRSW) {
                    if (!in1) break;
                    ++wc;
                    continue;
                }
                float e0;
                part += (double)box_term32<KIND>(q, bk, (float)d0, (float)d1, in0, in1, e0);
                u0 += (double)e0;
            }
        }
    }
    if (sizeof(Real) == 8 || KIND != POT_HRSW) return part;
    return -q.p1 * (double)wc;
}

// FP64 full energy of the pairs whose left member is in [p0, p1) (ECheck's
// recompute, src/jmmMCState.cpp:1973-1993).
template <int KIND>
__device__ __forceinline__ double energy_part(const Pot &q, const double *X, int64_t N, bool per,
                                              double L, uint32_t w, uint32_t p0, uint32_t p1,
                                              uint32_t stride)
{
    double U = 0.0;
    for (uint32_t p = p0; p < p1; p += stride) {
        const double xi = X[p];
        for (uint32_t k = 1; k <= w; ++k) {
            const int64_t j = (int64_t)p + k;
            double xj;
            if (j < N) xj = X[j];
            else if (per) xj = X[j - N] + L;
            else break;
            const double d = xj - xi;
            if (d > q.rc) break;
            U += phi64<KIND>(q, d);
        }
    }
    return U;
}

// Virial and hypervirial (FP64) of the pairs whose left member is in
// [p0, p1) (the reference's Vir and HV totals, src/jmmMCState.cpp:86-96).
template <int KIND>
__device__ __forceinline__ void virial_part(const Pot &q, const double *X, int64_t N, bool per, double L,
                                            uint32_t w, uint32_t p0, uint32_t p1, uint32_t stride,
                                            double &W, double &H)
{
    W = 0.0;
    H = 0.0;
    for (uint32_t p = p0; p < p1; p += stride) {
        const double xi = X[p];
        for (uint32_t k = 1; k <= w; ++k) {
            const int64_t j = (int64_t)p + k;
            double xj;
            if (j < N) xj = X[j];
            else if (per) xj = X[j - N] + L;
            else break;
            const double d = xj - xi;
            if (d > q.rc) break;
            if (!inside64<KIND>(q, d)) continue;
            double wp, hp;
            virial64<KIND>(q, d, wp, hp);
            W += wp;
            H += hp;
        }
    }
}

// Acceptance of a box-length trial (src/jmmMCState.cpp:2249-2255).
__device__ __forceinline__ bool vol_accept(double dU, double dL, double lns, double P, double beta,
                                           double jac, double u)
{
    const double bf = exp(-beta * (dU + P * dL) + jac * lns);
    return bf >= 1.0 || bf > u;
}

struct VolProp {
    double sc, Lp, lns, jac, dL, u;
    BoxK bk;  // FP32 form: the scaling constants of the pair differences
    bool valid;
};

// Out of line: its FP64 log/exp/division temporaries would otherwise raise
// the register count of the whole sweep loop.  BOXK: with the scaling constants
// of the LJ pair differences (two expm1), which only the FP32 LJ form reads.
template <bool BOXK>
__device__ __noinline__ VolProp vol_propose(const DevChain &ch, double L, uint64_t sweep)
{
    uint32_t r[4];
    philox4x32_10(0xFFFFFFFFu, (uint32_t)sweep, ch.chain_id, 0u, (uint32_t)ch.seed,
                  (uint32_t)(ch.seed >> 32), r);
    const double a = u53(r[0], r[1]);
    VolProp v;
    v.u = u53(r[2], r[3]);
    const double dv = ((a - 0.5) * 2.0) * ch.max_dv;
    if (!(ch.flags & F_VOLLOG)) {
        v.Lp = L + dv;
        v.sc = v.Lp / L;
        v.lns = log(v.sc);
        v.jac = (double)ch.N;
        v.dL = dv;
    } else {
        v.sc = det_exp(dv);
        v.Lp = L * v.sc;
        v.lns = dv;
        v.jac = (double)ch.N + 1.0;
        v.dL = v.Lp - L;
    }
    v.valid = v.Lp > 0.0 && (!(ch.flags & F_PERIODIC) || v.Lp > ch.Lmin);
    v.bk.c12 = v.bk.c6 = 0.0f;
    if (BOXK) {
        // s^-12 - 1 and s^-6 - 1 from expm1 of ln s: no cancellation
        const double a6 = ch.pot.e4 * ch.pot.sig6;
        v.bk.c12 = (float)(a6 * ch.pot.sig6 * expm1(-12.0 * v.lns));
        v.bk.c6 = (float)(a6 * expm1(-6.0 * v.lns));
    }
    return v;
}


// v + the value of the lane whose index differs in bit OFF, for values that
// are equal within aligned groups of OFF lanes (the levels of a butterfly sum):
// there a mirrored lane of the other half holds the partner's value, so the
// levels inside a row are one data-parallel move and the two across rows a
// swap, without the LDS round trip of a general shuffle.
template <int OFF>
__device__ __forceinline__ uint32_t xor_add(uint32_t v)
{
    if constexpr (OFF == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return r[0] + r[1];
    } else if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return r[0] + r[1];
    } else {
        // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror
        constexpr int ctrl = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x140;
        return v + (uint32_t)__builtin_amdgcn_mov_dpp((int)v, ctrl, 0xf, 0xf, true);
    }
}

template <int OFF>
__device__ __forceinline__ double xor_add(double v)
{
    const uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
    if constexpr (OFF == 16) {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else if constexpr (OFF == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else {
        constexpr int ctrl = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x140;
        return v + __hiloint2double(__builtin_amdgcn_mov_dpp((int)hi, ctrl, 0xf, 0xf, true),
                                    __builtin_amdgcn_mov_dpp((int)lo, ctrl, 0xf, 0xf, true));
    }
}

// One level of the sums below: lanes whose segment is longer than OFF add.
template <int OFF, int ND, int NI>
__device__ __forceinline__ void seg_level(double (&v)[ND], uint32_t (&k)[NI], uint32_t seg)
{
    const bool on = seg > (uint32_t)OFF;
#pragma unroll
    for (int m = 0; m < ND; ++m) {
        const double s = xor_add<OFF>(v[m]);
        v[m] = on ? s : v[m];
    }
#pragma unroll
    for (int m = 0; m < NI; ++m) {
        const uint32_t s = xor_add<OFF>(k[m]);
        k[m] = on ? s : k[m];
    }
}

// Sum over lane segments of size seg (seg <= T) whose first lane is base:
// a power of two up to 64 with base a multiple of seg, or a multiple of 64
// with base a multiple of 64 (whole waves).  Every lane of a segment
// receives the same bits: the butterfly is symmetric in its operands, and
// the cross-wave stage reads the segment's wave totals in a fixed order.
// rd/ri: flat LDS scratch of (T/64)*ND doubles and (T/64)*NI words.  TRAIL:
// a barrier at the end, after which the scratch may be used again; without it
// the caller has a barrier before the scratch's next use.
template <int T, int ND, int NI, bool TRAIL = true>
__device__ __forceinline__ void seg_allreduce(double (&v)[ND], uint32_t (&k)[NI], uint32_t seg,
                                              uint32_t base, double *rd, uint32_t *ri)
{
    seg_level<1>(v, k, seg);
    seg_level<2>(v, k, seg);
    seg_level<4>(v, k, seg);
    seg_level<8>(v, k, seg);
    seg_level<16>(v, k, seg);
    seg_level<32>(v, k, seg);
    if (T > 64) {
        const uint32_t tid = threadIdx.x, wv = tid >> 6;
        if ((tid & 63) == 0) {
#pragma unroll
            for (int m = 0; m < ND; ++m) rd[wv * ND + m] = v[m];
#pragma unroll
            for (int m = 0; m < NI; ++m) ri[wv * NI + m] = k[m];
        }
        __syncthreads();
        if (seg > 64) {
            const uint32_t w0 = base >> 6, nw = seg >> 6;
#pragma unroll
            for (int m = 0; m < ND; ++m) {
                double acc = 0.0;
                for (uint32_t q = 0; q < nw; ++q) acc += rd[(w0 + q) * ND + m];
                v[m] = acc;
            }
#pragma unroll
            for (int m = 0; m < NI; ++m) {
                uint32_t acc = 0;
                for (uint32_t q = 0; q < nw; ++q) acc += ri[(w0 + q) * NI + m];
                k[m] = acc;
            }
        }
        if (TRAIL) __syncthreads();
    }
}

// Full 64-lane sum, identical in every lane.
template <typename V>
__device__ __forceinline__ V wave_sum(V v)
{
    v = xor_add<1>(v);
    v = xor_add<2>(v);
    v = xor_add<4>(v);
    v = xor_add<8>(v);
    v = xor_add<16>(v);
    return xor_add<32>(v);
}

// ------------------------------------------------------------ batched form

template <int T>
struct BatchedScratch {
    // no larger than before the proposals were shared: the image of a chain
    // may leave 512 bytes of the LDS
    static constexpr int NVP = T >= 1024 ? 1 : 2;
    double rd[(T / 64) * 3];
    VolProp vp[NVP];  // box-length proposals of chains of at least T / NVP blocks
    uint32_t ri[(T / 64) * 4];
    uint32_t item;
    uint8_t need[T / 64];
};
static_assert(sizeof(BatchedScratch<256>) <= 512 && sizeof(BatchedScratch<512>) <= 512, "LDS left to a chain's image");

template <typename Real, int KIND, int T>
__device__ __forceinline__ void run_bundle_gx(const SweepArgs &a, const DevBundle &bd, BatchedScratch<T> &sc,
                              uint32_t soff)
{
    const uint32_t tid = threadIdx.x;
    // lane -> slot: the largest slot whose first lane is <= tid
    uint32_t lo = 0, hi = bd.nslots - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (a.slots[bd.slot0 + mid].lane_off <= tid) lo = mid;
        else hi = mid - 1;
    }
    const DevSlot me = a.slots[bd.slot0 + lo];
    const bool act = tid >= me.lane_off && tid < me.lane_off + me.B;
    const uint32_t ic = me.chain;

    double *X = a.x + bd.x_off;
    __syncthreads();

    const DevChain &ch = a.chains[ic];
    const Pot q = ch.pot;
    const int64_t N = ch.N;
    const uint32_t w = ch.w;
    const bool per = (ch.flags & F_PERIODIC) != 0;
    const bool npt = (ch.flags & F_NPT) != 0;  // uniform within a bundle
    const double beta = ch.beta, gmin = ch.gmin, max_step = ch.max_step;
    const float betaf = ch.betaf;
    const uint32_t key0 = (uint32_t)ch.seed, key1 = (uint32_t)(ch.seed >> 32);
    const uint64_t log_off = ch.log_off;
    const uint32_t eci = ch.eci;
    const uint32_t chain_id = ch.chain_id;
    const double P = ch.P;

    const DevState st = a.states[ic];
    double L = st.L, U = st.U, mdrift = st.max_drift;
    uint64_t sweep = st.sweep;

    const uint32_t B = me.B;
    const uint32_t r = tid - me.lane_off;
    const uint32_t qb = (uint32_t)N / B, rem = (uint32_t)N % B;
    const uint32_t size = act ? qb + (r < rem ? 1u : 0u) : 0u;
    const uint32_t start = act ? r * qb + (r < rem ? r : rem) : 0u;
    const uint32_t seg = act ? B : 1u;
    const bool leader = act && r == 0;

    uint32_t n_tr = 0, n_wall = 0, n_core = 0, n_terms = 0;
    uint32_t acc_total = 0, n_vt = 0, n_av = 0, n_rc = 0;

    for (uint32_t sw = 0; sw < a.n_sweeps; ++sw, ++sweep) {
        double dUs = 0.0;
        uint32_t acc = 0;
        uint32_t w_md = 0, w_u = 0, w_next_md = 0, w_next_u = 0;
        for (uint32_t t = 0; t < bd.smax; ++t) {
            if (t < size) {
                const uint32_t i = start + t;
                // one Philox block per pair of block positions (t, t+1):
                // computed at even t, its second half kept for odd t (t is
                // the same on every lane, so the branch is uniform)
                if ((t & 1u) == 0) {
                    uint32_t rr[4];
                    philox4x32_10(i, (uint32_t)sweep, chain_id, 0u, key0, key1, rr);
                    w_md = rr[0];
                    w_u = rr[1];
                    w_next_md = rr[2];
                    w_next_u = rr[3];
                } else {
                    w_md = w_next_md;
                    w_u = w_next_u;
                }
                const double a1 = u32o(w_md);
                const double u = u32o(w_u);
                const double md = ((a1 - 0.5) * 2.0) * max_step;
                const double xi = X[i];
                const double xn = xi + md;
                ++n_tr;
                bool ok = true;
                if (!per && fabs(xn) > L / 2.0) {
                    ok = false;
                    ++n_wall;
                } else if (N >= 2) {
                    double xl, xr;
                    if ((nbpos(X, (int64_t)i - 1, N, per, L, xl) && (xn - xl) < gmin) ||
                        (nbpos(X, (int64_t)i + 1, N, per, L, xr) && (xr - xn) < gmin)) {
                        ok = false;
                        ++n_core;
                    }
                }
                bool accd = false;
                if (ok) {
                    double dE;
                    if (sizeof(Real) == 8)
                        dE = delta_e64<KIND>(q, X, i, N, per, L, w, xi, xn, n_terms);
                    else
                        dE = delta_e32<KIND>(q, X, i, N, per, L, w, xi, xn, n_terms);
                    if (dE <= 0.0) accd = true;
                    else if (sizeof(Real) == 8) accd = exp(-dE * beta) > u;
                    else accd = (double)fexp(-betaf * (float)dE) > u;
                    if (accd) {
                        X[i] = xn;
                        dUs += dE;
                        ++acc;
                    }
                }
                if (a.acclog) a.acclog[log_off + (uint64_t)(soff + sw) * N + i] = accd ? 1 : 0;
            }
            __syncthreads();
        }

        // box-length trial (fav, src/jmmMCState.cpp:2161-2293)
        VolProp vp{};
        uint32_t bad = 0;
        double vpart = 0.0, upart = 0.0;
        if (npt) {
            vp = vol_propose<sizeof(Real) == 4 && KIND == POT_LJ>(ch, L, sweep);
            // long blocks in two halves, as the other placements (half_of)
            uint32_t p0 = start, p1 = start + half_of(size);
#pragma unroll 1
            for (int part = 0; part < 2; ++part) {
                double u = 0.0;
                if (vp.valid && p0 < p1)
                    vpart += scaled_delta<Real, KIND>(q, vp.bk, gmin, X, N, per, L, vp.Lp, vp.sc, w, p0, p1, 1, bad, u);
                upart += u;
                p0 = p1;
                p1 = start + size;
            }
        }
        {
            double v[3] = {dUs, vpart, upart};
            uint32_t k2[2] = {acc, bad};
            seg_allreduce<T, 3, 2>(v, k2, seg, me.lane_off, sc.rd, sc.ri);
            U = U + v[0];
            vpart = v[1];
            acc = k2[0];
            bad = k2[1];
            // FP32 form: the box-length pass summed the configuration's FP32
            // energy over every pair; it replaces the running sum, so FP32
            // trial errors do not accumulate between recomputes.  Square
            // well: the pass gave the scaled energy, the running energy is
            // exact
            if (sizeof(Real) == 4 && KIND == POT_HRSW) vpart = vpart - U;
            else if (sizeof(Real) == 4 && npt && vp.valid && !bad) U = v[2];
        }
        acc_total += acc;
        uint32_t accv = 0;
        if (npt) {
            ++n_vt;
            if (vp.valid && !bad && vol_accept(vpart, vp.dL, vp.lns, P, beta, vp.jac, vp.u)) {
                for (uint32_t p = start; p < start + size; ++p) X[p] = X[p] * vp.sc;
                L = vp.Lp;
                U = U + vpart;
                accv = 1;
                ++n_av;
            }
            __syncthreads();
        }

        // drift guard (ECheck, src/jmmMCState.cpp:1965-2095), always FP64
        const int need = act && eci && ((sweep + 1) % eci == 0);
        if (__syncthreads_or(need)) {
            double v[1] = {need ? energy_part<KIND>(q, X, N, per, L, w, start, start + size, 1)
                                : 0.0};
            uint32_t k1[1] = {0};
            seg_allreduce<T, 1, 1>(v, k1, seg, me.lane_off, sc.rd, sc.ri);
            if (need) {
                const double dr = fabs(v[0] - U);
                if (dr > mdrift) mdrift = dr;
                U = v[0];
                ++n_rc;
            }
        }

        double Ws = 0.0, Hs = 0.0;
        if (a.sW) {
            double v[2] = {0.0, 0.0};
            if (act) virial_part<KIND>(q, X, N, per, L, w, start, start + size, 1, v[0], v[1]);
            uint32_t k1[1] = {0};
            seg_allreduce<T, 2, 1>(v, k1, seg, me.lane_off, sc.rd, sc.ri);
            Ws = v[0];
            Hs = v[1];
        }
        if (leader) {
            const uint64_t row = (uint64_t)(soff + sw) * a.n_chains + ic;
            a.sU[row] = U;
            a.sL[row] = L;
            a.sA[row] = make_uint2(acc, accv);
            if (a.sW) {
                a.sW[row] = Ws;
                a.sH[row] = Hs;
            }
        }
    }

    {
        double vz[1] = {0.0};
        uint32_t k4[4] = {n_tr, n_wall, n_core, n_terms};
        seg_allreduce<T, 1, 4>(vz, k4, seg, me.lane_off, sc.rd, sc.ri);
        if (leader) {
            DevState &o = a.states[ic];
            o.L = L;
            o.U = U;
            o.sweep = sweep;
            o.cnt[0] += k4[0];
            o.cnt[1] += acc_total;
            o.cnt[2] += k4[1];
            o.cnt[3] += k4[2];
            o.cnt[4] += k4[3];
            o.cnt[5] += n_vt;
            o.cnt[6] += n_av;
            o.cnt[7] += n_rc;
            o.max_drift = mdrift;
        }
    }
    __syncthreads();
}

// Per-lane view of a chain held in LDS.  Region layout:
//   [ghost-left: wg][block 0 .. block B-1 at stride Sp][ghost-right: wg]
// Sp is odd and at least the longest block, so the lanes of one chain, which
// touch the same offset of consecutive blocks in a phase, hit distinct LDS
// banks.  Periodic chains keep images of the particles near the ends:
// ghost-left[m] = x_{N-wg+m} - L, ghost-right[m] = x_m + L (the same FP64
// operation the oracle applies on the fly), so a neighbour walk never
// branches on the wrap.  wg = max(w, 1).
struct LdsChain {
    double *R;
    uint32_t N, B, w, wg, Sp, qb, rem;
    bool per;
};

// Images of the first and last wg particles, lanes r = 0 .. n - 1 sharing the
// work.  They lie in the first and the last block (a block holds at least
// M_min >= wg particles, or all of them).
__device__ __forceinline__ void fill_ghosts(const LdsChain &c, uint32_t r, uint32_t n, double L)
{
    if (!c.per) return;
    const uint32_t tail = c.wg + (c.B - 1) * c.Sp + (c.qb + (c.B - 1 < c.rem ? 1u : 0u)) - c.wg;
    for (uint32_t m = r; m < c.wg; m += n) {
        c.R[c.wg + c.B * c.Sp + m] = c.R[c.wg + m] + L;
        c.R[m] = c.R[tail + m] - L;
    }
}

// The periodic images of particle i at its new position x.
__device__ __forceinline__ void put_images(const LdsChain &c, uint32_t i, double x, double L)
{
    if (i < c.wg) c.R[c.wg + c.B * c.Sp + i] = x + L;
    if (i + c.wg >= c.N) c.R[i + c.wg - c.N] = x - L;
}

// The FP32 walks' keep-going test for one partner: inside the cutoff at the
// old or the new position (the FP64 flags).  For LJ and Yukawa (inside is
// d <= rc) this is the FP64 form's rule, not beyond the cutoff from both
// positions.  For the strict cutoffs of the square well and the spring the
// two differ only for a partner at exactly rc: it adds nothing to the sums
// or the pair-term count, and the FP64 walk's next partner lies beyond rc
// and adds nothing either, so both walks give the same result.
template <int KIND>
__device__ __forceinline__ bool walk_in(const Pot &, double, double, bool io, bool in)
{
    return io || in;
}

// Energy change of one side's partners, FP32 form, for two lanes per block:
// the lane walks the partners at my - k (left) or my + k (right), four per
// loop iteration, and returns the sum of their FP32 terms in FP64, added in
// the order k = 1, 2, ... as the one-lane walk adds that side's.  The
// positions are sorted, so the separations grow with k and a partner outside
// the cutoff at both positions is followed by none inside: the FP64
// inside-the-cutoff flags alone make the later terms zero, and the walk needs
// no liveness or per-lane limit beyond them (w, the same on every lane, ends
// the loop; a chain with walls holds NaN where it has no partner, which is
// inside nothing).  |x| replaces the side's orientation of a separation
// (xj - xi is -(xi - xj) exactly; a trial that goes on keeps the sign of the
// new separation by the hard-core test).  A lane whose trial is already
// rejected walks with the others and its result is dropped.
//
// Bound by vector issue: per partner 2 quarter-rate instructions per pair
// energy for Yukawa (exponential, reciprocal) and about 30 others.  Eight
// independent pair energies per iteration keep one wave issuing; the walk of
// one partner per iteration, with liveness, was latency-bound.  With it and
// the shared box-length pass two lanes per block (two waves per SIMD, VALU
// busy 74 %) run 50 sweeps of 64 chains of 65,536 in 16.9 ms, one lane per
// block (one wave, 56 %) in 20.1.
template <int KIND>
__device__ __forceinline__ double walk_side32(const double *X, const Pot &q, uint32_t w, bool go, bool left,
                                              uint32_t t, uint32_t size, uint32_t my, uint32_t gapL, uint32_t gapR,
                                              double xi, double xn, uint32_t &terms)
{
    const uint32_t m = left ? t : size - 1 - t;           // partners of the own block on this side
    const uint32_t gap = (left ? 0u - gapL : gapR) * 8u;  // bytes to the next block's, modulo 2^32
    const uint32_t dir = left ? 0u - 8u : 8u;
    const uint32_t at = my * 8u;
    const char *XB = (const char *)X;
    double sum = 0.0;
    int well = 0;
    uint32_t cnt = 0;
    bool more = go;
    auto step = [&](uint32_t k, double &o, double &n) {
        const double xj = *(const double *)(XB + (at + dir * k + (k > m ? gap : 0u)));
        o = fabs(xi - xj);
        n = fabs(xn - xj);
    };
    auto term = [&](double o, double n, bool io, bool in) -> float {
        return phi32<KIND>(q, (float)n, in) - phi32<KIND>(q, (float)o, io);
    };
    uint32_t k = 1;
    while (k + 3 <= w && __any(more)) {
        double o[4], n[4];
        bool io[4], in[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            step(k + u, o[u], n[u]);
            io[u] = inside64<KIND>(q, o[u]);
            in[u] = inside64<KIND>(q, n[u]);
            cnt += (io[u] ? 1u : 0u) + (in[u] ? 1u : 0u);
        }
        if (KIND == POT_HRSW) {
#pragma unroll
            for (int u = 0; u < 4; ++u) well += (int)in[u] - (int)io[u];
        } else {
            float e[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) e[u] = term(o[u], n[u], io[u], in[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) sum += (double)e[u];
        }
        more = go && (io[3] || in[3]);
        k += 4;
    }
    while (k <= w && __any(more)) {
        double o, n;
        step(k, o, n);
        const bool io = inside64<KIND>(q, o), in = inside64<KIND>(q, n);
        cnt += (io ? 1u : 0u) + (in ? 1u : 0u);
        if (KIND == POT_HRSW) well += (int)in - (int)io;
        else sum += (double)term(o, n, io, in);
        more = go && (io || in);
        ++k;
    }
    terms += go ? cnt : 0u;
    return KIND == POT_HRSW ? -q.p1 * (double)well : sum;
}

// One displacement trial of particle i (block position t of a block of
// length size, LDS address my) by md.  Same decisions as orc_trial_with: wall
// test, hard core against the nearest partners (FP64), then the partner sums
// of qad2 (src/jmmMCState.cpp:1213-1348) walked outward on both sides at once
// in a wave-uniform loop; each side stops at its first partner beyond the
// cutoff from both positions.  FP64 form: the oracle's operations exactly.
// FP32 form: separations formed in FP64, cutoff decided in FP64 (the FP64
// set-up and recompute energies count the same pairs), pair energies in FP32
// without branches, each side's FP32 terms summed in FP64 (on gfx950 an FP64
// add issues at the FP32 rate: exact sums of the FP32 terms for fewer
// instructions than a compensated FP32 sum with its freeze selects); the
// loop-exit test runs on the separations in FP64 as in the FP64 form.  Partner k's address is read
// on every lane of the wave, live or not: for k <= w it lies in the chain's
// image (ghosts or halos are wg >= w wide, blocks longer than w), and a lane
// that is not live drops the value.  Returns the decision; dE receives the
// energy change.
//
// PAIR = false: one lane walks both sides.  PAIR = true: two adjacent lanes
// share the trial, side 0 (even lane) walking the left partners and side 1
// the right; each forms its side's sum exactly as the one-lane walk does
// (same terms, same order; once a side's walk ends its terms are zero and
// adding them is exact), then the two sums are exchanged and added.  Addition commutes, so
// both lanes hold the one-lane result bit for bit.  Both lanes of a pair
// must be active together.
//
// W2 (FP32, one lane): two partners per side per loop iteration, four
// independent pair evaluations in flight instead of two and half the
// loop-exit tests; the terms are added in the same order, so the result is
// the one-step walk's bit for bit.
template <typename Real, int KIND, bool PAIR = false, bool W2 = false>
__device__ __forceinline__ bool trial_lds(const LdsChain &c, const Pot &q, double gmin,
                                          double beta, float betaf, uint32_t i, uint32_t t,
                                          uint32_t size, uint32_t my, uint32_t gapL,
                                          uint32_t gapR, double L, double xi, double xn, double md,
                                          double u, double &dE, uint32_t &terms, uint32_t &n_wall,
                                          uint32_t &n_core, uint32_t side = 0)
{
    const double *X = c.R;
    // rejections by the walls and the hard core are flags, not early exits:
    // the wavefront walks the window anyway for its other lanes
    const bool wall = !c.per && fabs(xn) > L / 2.0;
    const bool hasL = c.N >= 2 && (c.per || i > 0);
    const bool hasR = c.N >= 2 && (c.per || i + 1 < c.N);
    // the nearest slots on both sides (ghost or halo slots at a chain's
    // ends: in the image; their values count only where hasL / hasR)
    const double xl = X[my - 1 - (t == 0 ? gapL : 0)];
    const double xr = X[my + 1 + (t + 1 >= size ? gapR : 0)];
    const bool core = !wall && ((hasL && (xn - xl) < gmin) || (hasR && (xr - xn) < gmin));
    n_wall += wall ? 1u : 0u;
    n_core += core ? 1u : 0u;
    const bool go = !wall && !core;
    const uint32_t kL = c.per ? c.w : min(c.w, i);
    const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - i);
    if (PAIR) {
        // one side per lane: partner k at my - k (left) or my + k (right),
        // separations oriented as in the two-sided walk
        const bool left = side == 0;
        const uint32_t kS = left ? kL : kR;
        bool live = go && kS >= 1;
        if (sizeof(Real) == 8) {
            double dS = 0.0;
            uint32_t k = 1;
            if (__any(live)) {
#pragma unroll 1
            do {
                const uint32_t jl = my - k - (k > t ? gapL : 0), jr = my + k + (t + k >= size ? gapR : 0);
                const double xj = X[left ? jl : jr];
                const double o = left ? xi - xj : xj - xi, nn = left ? xn - xj : xj - xn;
                const bool in = live && !(o > q.rc && nn > q.rc);
                const double tt = phi64<KIND>(q, nn) - phi64<KIND>(q, o);
                dS += in ? tt : 0.0;
                terms += in ? n_inside<KIND>(q, o, nn) : 0u;
                live = in && k < kS;
                ++k;
            } while (__any(live));
            }
            dE = dS + __shfl_xor(dS, 1);
            const double bf = exp(-dE * beta);
            return go && (dE <= 0.0 || bf > u);
        }
        const double mine = walk_side32<KIND>(X, q, c.w, go, left, t, size, my, gapL, gapR, xi, xn, terms);
        dE = mine + __shfl_xor(mine, 1);
        const float bf = fexp(-betaf * (float)dE);
        return go && (dE <= 0.0 || (double)bf > u);
    }
    bool liveL = go && kL >= 1, liveR = go && kR >= 1;
    if (sizeof(Real) == 8) {
        double dEL = 0.0, dER = 0.0;
        uint32_t k = 1;
        if (__any(liveL || liveR)) {
#pragma unroll 1
        do {
            const double xjL = X[my - k - (k > t ? gapL : 0)];
            const double xjR = X[my + k + (t + k >= size ? gapR : 0)];
            const double oL = xi - xjL, nL = xn - xjL;
            const double oR = xjR - xi, nR = xjR - xn;
            const bool inL = liveL && !(oL > q.rc && nL > q.rc);
            const bool inR = liveR && !(oR > q.rc && nR > q.rc);
            const double tL = phi64<KIND>(q, nL) - phi64<KIND>(q, oL);
            const double tR = phi64<KIND>(q, nR) - phi64<KIND>(q, oR);
            dEL += inL ? tL : 0.0;
            dER += inR ? tR : 0.0;
            terms += n_walked<KIND>(inL, inside64<KIND>(q, oL), inside64<KIND>(q, nL)) +
                     n_walked<KIND>(inR, inside64<KIND>(q, oR), inside64<KIND>(q, nR));
            liveL = inL && k < kL;
            liveR = inR && k < kR;
            ++k;
        } while (__any(liveL || liveR));
        }
        dE = dEL + dER;
        const double bf = exp(-dE * beta);
        return go && (dE <= 0.0 || bf > u);
    }
    // each side's FP32 pair terms summed in FP64 (exact; the terms of
    // partners off a side's walk are zero, exact no-op adds)
    double sL = 0.0, sR = 0.0;
    // hard rod + square well: every pair term is -eps or 0, so each side's
    // change is -eps times the change in the number of partners inside the
    // well, counted exactly
    int wL = 0, wR = 0;
    uint32_t k = 1;
    if (W2) {
    if (__any(liveL || liveR)) {
#pragma unroll 1
    do {
        // partners k and k + 1 on both sides: a side still walking after
        // step k has k < its limit <= w, so partner k + 1 is in the image;
        // the clamp keeps the other lanes' reads there too
        const uint32_t k2 = min(k + 1, c.w);
        const double xjL = X[my - k - (k > t ? gapL : 0)];
        const double xjR = X[my + k + (t + k >= size ? gapR : 0)];
        const double xjL2 = X[my - k2 - (k2 > t ? gapL : 0)];
        const double xjR2 = X[my + k2 + (t + k2 >= size ? gapR : 0)];
        const double oL = xi - xjL, nL = xn - xjL;
        const double oR = xjR - xi, nR = xjR - xn;
        const bool ioL = inside64<KIND>(q, oL), inL64 = inside64<KIND>(q, nL);
        const bool ioR = inside64<KIND>(q, oR), inR64 = inside64<KIND>(q, nR);
        const bool inL = liveL && walk_in<KIND>(q, oL, nL, ioL, inL64);
        const bool inR = liveR && walk_in<KIND>(q, oR, nR, ioR, inR64);
        const float tL = phi32<KIND>(q, (float)nL, inL && inL64) - phi32<KIND>(q, (float)oL, inL && ioL);
        const float tR = phi32<KIND>(q, (float)nR, inR && inR64) - phi32<KIND>(q, (float)oR, inR && ioR);
        const bool liveL2 = inL && k < kL, liveR2 = inR && k < kR;
        const double oL2 = xi - xjL2, nL2 = xn - xjL2;
        const double oR2 = xjR2 - xi, nR2 = xjR2 - xn;
        const bool ioL2 = inside64<KIND>(q, oL2), inL642 = inside64<KIND>(q, nL2);
        const bool ioR2 = inside64<KIND>(q, oR2), inR642 = inside64<KIND>(q, nR2);
        const bool inL2 = liveL2 && walk_in<KIND>(q, oL2, nL2, ioL2, inL642);
        const bool inR2 = liveR2 && walk_in<KIND>(q, oR2, nR2, ioR2, inR642);
        const float tL2 = phi32<KIND>(q, (float)nL2, inL2 && inL642) - phi32<KIND>(q, (float)oL2, inL2 && ioL2);
        const float tR2 = phi32<KIND>(q, (float)nR2, inR2 && inR642) - phi32<KIND>(q, (float)oR2, inR2 && ioR2);
        if (KIND == POT_HRSW) {
            wL += (inL ? (int)inL64 - (int)ioL : 0) + (inL2 ? (int)inL642 - (int)ioL2 : 0);
            wR += (inR ? (int)inR64 - (int)ioR : 0) + (inR2 ? (int)inR642 - (int)ioR2 : 0);
        } else {
            sL += (double)tL;
            sR += (double)tR;
            sL += (double)tL2;
            sR += (double)tR2;
        }
        terms += n_walked<KIND>(inL, ioL, inL64) + n_walked<KIND>(inR, ioR, inR64) +
                 n_walked<KIND>(inL2, ioL2, inL642) + n_walked<KIND>(inR2, ioR2, inR642);
        liveL = inL2 && k + 1 < kL;
        liveR = inR2 && k + 1 < kR;
        k += 2;
    } while (__any(liveL || liveR));
    }
    } else {
    if (__any(liveL || liveR)) {
#pragma unroll 1
    do {
        const double xjL = X[my - k - (k > t ? gapL : 0)];
        const double xjR = X[my + k + (t + k >= size ? gapR : 0)];
        // separations are FP64 differences; the cutoff decisions are made on
        // them (the FP64 energies of set-up and recompute count the same
        // pairs, and the walk ends where the FP64 form's does), the pair
        // energies on their FP32 roundings
        const double oL = xi - xjL, nL = xn - xjL;
        const double oR = xjR - xi, nR = xjR - xn;
        const bool ioL = inside64<KIND>(q, oL), inL64 = inside64<KIND>(q, nL);
        const bool ioR = inside64<KIND>(q, oR), inR64 = inside64<KIND>(q, nR);
        const bool inL = liveL && walk_in<KIND>(q, oL, nL, ioL, inL64);
        const bool inR = liveR && walk_in<KIND>(q, oR, nR, ioR, inR64);
        const float tL = phi32<KIND>(q, (float)nL, inL && inL64) - phi32<KIND>(q, (float)oL, inL && ioL);
        const float tR = phi32<KIND>(q, (float)nR, inR && inR64) - phi32<KIND>(q, (float)oR, inR && ioR);
        if (KIND == POT_HRSW) {
            wL += inL ? (int)inL64 - (int)ioL : 0;
            wR += inR ? (int)inR64 - (int)ioR : 0;
        } else {
            sL += (double)tL;
            sR += (double)tR;
        }
        terms += n_walked<KIND>(inL, ioL, inL64) + n_walked<KIND>(inR, ioR, inR64);
        liveL = inL && k < kL;
        liveR = inR && k < kR;
        ++k;
    } while (__any(liveL || liveR));
    }
    }
    dE = KIND == POT_HRSW ? -q.p1 * (double)wL + -q.p1 * (double)wR : sL + sR;
    const float bf = fexp(-betaf * (float)dE);
    return go && (dE <= 0.0 || (double)bf > u);
}

// Box-length trial (fav, src/jmmMCState.cpp:2161-2293), one lane's share
// over the pairs (i, i+k) whose left member is at the block positions [t0, t1)
// of the lane's block, in the
// order t = t0.., k = 1.. : the energy change of scaling the configuration by
// vp.sc pair by pair, FP64 form phi64(s d) - phi64(d), FP32 form box_term32
// (one reciprocal per LJ pair through the scaling identity) summed in FP64;
// each particle's walk ends at its first partner beyond
// the cutoff at both the unscaled and the scaled separation (the FP64
// inside-the-cutoff flags decide in both forms, so both sum the same pairs).
// The walk over (particle, partner) is one
// flat loop with per-lane state, so lanes at different particles advance
// together without nested divergent loops; it adds the same terms in the
// same order as the nested walk (particle t's walk ends at its first partner
// beyond the cutoff from both scaled and unscaled positions, at k = kR, or
// at an overlap of nearest neighbours, which ends the lane's walk and sets
// `bad`).  The partner at k = 1 is the next particle, so its position and
// scaled position are kept rather than read again.  `last`: the lane holds
// the chain's last block of a periodic chain, whose partners past the end
// are the first particles shifted by L; wrap(m) returns particle m's
// unshifted position (scaled and shifted by Lp here).  Hard rod + square
// well, FP32 form: the lane returns the scaled configuration's energy, -eps
// times the number of its scaled pairs inside the well (each walk ends at
// the first scaled partner outside), and the caller subtracts the running
// energy, which is -eps times the unscaled count exactly (every trial and
// recompute changes it by whole pairs), so the energy change is the one the
// pairwise sum gives.  W2: two partners of
// a particle per iteration (for the common walk of one partner inside and
// the next beyond the cutoff, one iteration per particle), same terms in
// the same order (four for the long windows of split chains: 4 % more
// instructions, the walk's bookkeeping grew with them, and no time saved).
template <typename Real, int KIND, bool W2 = false, typename Wrap>
__device__ __forceinline__ double vol_lane(const LdsChain &c, const Pot &q, double gmin,
                                           const VolProp &vp, bool on, uint32_t start,
                                           uint32_t size, uint32_t t0, uint32_t t1, uint32_t a0,
                                           uint32_t gapR, bool last, Wrap wrap, uint32_t &bad, double &u0)
{
    constexpr bool WELL = sizeof(Real) == 4 && KIND == POT_HRSW;
    const double *X = c.R;
    double part = 0.0;  // FP64 terms, or the FP32 form's FP32 terms summed in FP64
    int wc = 0;  // hard rod + square well, FP32: scaled pairs inside the well
    u0 = 0.0;    // FP32 form: the pairs' FP32 energy at the unscaled separations
    bool run = on && t0 < t1;
    uint32_t t = t0, k = 1;
    double xi = X[run ? a0 + t0 : 0u];
    double xis = xi * vp.sc;
    double x1 = 0.0, x1s = 0.0;
    if (W2) {
    if (__any(run)) {
#pragma unroll 1
    do {
        // partners k and k + 1 of particle t; the second counts only where
        // the first continued the walk (then k < kR <= w, so the clamp to w
        // changes no address that counts and keeps the others in the image)
        const uint32_t i = start + t;
        const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - i);
        const bool valid = run && k <= kR;
        const uint32_t k2 = min(k + 1, c.w);
        const bool cross = t + k >= size, cross2 = t + k2 >= size;
        const double xj = X[valid ? a0 + t + k + (cross ? gapR : 0u) : 0u];
        const double xj2 = X[valid ? a0 + t + k2 + (cross2 ? gapR : 0u) : 0u];
        double xjs = xj * vp.sc, xjs2 = xj2 * vp.sc;
        if (valid && cross && last) xjs = wrap(t + k - size) * vp.sc + vp.Lp;
        if (valid && cross2 && last) xjs2 = wrap(t + k2 - size) * vp.sc + vp.Lp;
        const double d0 = xj - xi, d1 = xjs - xis;
        const double e0 = xj2 - xi, e1 = xjs2 - xis;
        const bool in0 = inside64<KIND>(q, d0), in1 = inside64<KIND>(q, d1);
        const bool jn0 = inside64<KIND>(q, e0), jn1 = inside64<KIND>(q, e1);
        const bool isbad = valid && k == 1 && d1 < gmin;
        const bool stop = valid && (sizeof(Real) == 8 ? d0 > q.rc && d1 > q.rc : WELL ? !in1 : !(in0 || in1));
        const bool add = valid && !isbad && !stop;
        const bool valid2 = add && k < kR;
        const bool stop2 = valid2 && (sizeof(Real) == 8 ? e0 > q.rc && e1 > q.rc : WELL ? !jn1 : !(jn0 || jn1));
        const bool add2 = valid2 && !stop2;
        if (sizeof(Real) == 8) {
            const double tt = phi64<KIND>(q, d1) - phi64<KIND>(q, d0);
            const double tt2 = phi64<KIND>(q, e1) - phi64<KIND>(q, e0);
            part = add ? part + tt : part;
            part = add2 ? part + tt2 : part;
        } else if (WELL) {
            wc += (add && in1 ? 1 : 0) + (add2 && jn1 ? 1 : 0);
        } else {
            // flags masked by add / add2: pairs off the walk give zeros
            float g0, g1;
            const float tt = box_term32<KIND>(q, vp.bk, (float)d0, (float)d1, add && in0, add && in1, g0);
            const float tt2 = box_term32<KIND>(q, vp.bk, (float)e0, (float)e1, add2 && jn0, add2 && jn1, g1);
            part += (double)tt;
            part += (double)tt2;
            u0 += (double)g0;
            u0 += (double)g1;
        }
        bad |= isbad ? 1u : 0u;
        x1 = k == 1 ? xj : x1;
        x1s = k == 1 ? xjs : x1s;
        // the same particle goes on at k + 2 only if partner k + 1 was
        // inside and more partners remain
        const bool nextp = !(add2 && k + 1 < kR);
        const uint32_t tn = nextp ? t + 1 : t;
        run = run && !isbad && tn < t1;
        xi = nextp ? x1 : xi;
        xis = nextp ? x1s : xis;
        k = nextp ? 1u : k + 2;
        t = tn;
    } while (__any(run));
    }
    } else {
    if (__any(run)) {
#pragma unroll 1
    do {
        const uint32_t i = start + t;
        const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - i);
        const bool valid = run && k <= kR;
        const bool cross = t + k >= size;
        const double xj = X[valid ? a0 + t + k + (cross ? gapR : 0u) : 0u];
        double xjs = xj * vp.sc;
        if (valid && cross && last) xjs = wrap(t + k - size) * vp.sc + vp.Lp;
        const double d0 = xj - xi, d1 = xjs - xis;
        const bool in0 = inside64<KIND>(q, d0), in1 = inside64<KIND>(q, d1);
        const bool isbad = valid && k == 1 && d1 < gmin;
        const bool stop = valid && (sizeof(Real) == 8 ? d0 > q.rc && d1 > q.rc : WELL ? !in1 : !(in0 || in1));
        const bool add = valid && !isbad && !stop;
        if (sizeof(Real) == 8) {
            const double tt = phi64<KIND>(q, d1) - phi64<KIND>(q, d0);
            part = add ? part + tt : part;
        } else if (WELL) {
            wc += add && in1 ? 1 : 0;
        } else {
            float g0;
            part += (double)box_term32<KIND>(q, vp.bk, (float)d0, (float)d1, add && in0, add && in1, g0);
            u0 += (double)g0;
        }
        bad |= isbad ? 1u : 0u;
        x1 = k == 1 ? xj : x1;
        x1s = k == 1 ? xjs : x1s;
        // next partner, or the next particle (lanes no longer running keep
        // stepping t; their reads are redirected and their terms dropped)
        const bool nextp = !valid || stop || k == kR;
        const uint32_t tn = nextp ? t + 1 : t;
        run = run && !isbad && tn < t1;
        xi = nextp ? x1 : xi;
        xis = nextp ? x1s : xis;
        k = nextp ? 1u : k + 1;
        t = tn;
    } while (__any(run));
    }
    }
    return WELL ? -q.p1 * (double)wc : part;
}

// Virial and hypervirial (FP64) of the pairs whose left member is in the
// lane's block, read from the LDS image (the recompute's walk).
template <int KIND>
__device__ __forceinline__ void virial_lane(const LdsChain &c, const Pot &q, uint32_t start, uint32_t size,
                                            uint32_t a0, uint32_t gapR, double &W, double &H)
{
    for (uint32_t t = 0; t < size; ++t) {
        const uint32_t i = start + t;
        const double xi = c.R[a0 + t];
        const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - i);
        for (uint32_t k = 1; k <= kR; ++k) {
            const double d = c.R[a0 + t + k + (t + k >= size ? gapR : 0)] - xi;
            if (d > q.rc) break;
            if (!inside64<KIND>(q, d)) continue;
            double wp, hp;
            virial64<KIND>(q, d, wp, hp);
            W += wp;
            H += hp;
        }
    }
}

template <typename Real, int KIND, int T>
__device__ __forceinline__ void run_bundle_lds(const SweepArgs &a, const DevBundle &bd, double *smem,
                                            BatchedScratch<T> &sc, uint32_t soff)
{
    const uint32_t tid = threadIdx.x;
    uint32_t lo = 0, hi = bd.nslots - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (a.slots[bd.slot0 + mid].lane_off <= tid) lo = mid;
        else hi = mid - 1;
    }
    const DevSlot me = a.slots[bd.slot0 + lo];
    const bool act = tid >= me.lane_off && tid < me.lane_off + me.B;
    const uint32_t ic = me.chain;
    const DevChain &ch = a.chains[ic];
    // Chains of a bundle share their shape (potential and its parameters,
    // boundary, ensemble, step sizes, window): read it once per bundle.
    const DevChain &sh = a.chains[__builtin_amdgcn_readfirstlane(a.slots[bd.slot0].chain)];
    const Pot q = sh.pot;
    const double gmin = sh.gmin;
    // per chain: step adaptation may change it (2^-32: see the displacement)
    const double step32 = ch.max_step * (1.0 / 4294967296.0);
    // per-chain fields as values: read once, not reloaded after every store
    // of the loops below (the compiler cannot rule out aliasing)
    const double beta = ch.beta;
    const float betaf = ch.betaf;
    const uint32_t key0 = (uint32_t)ch.seed, key1 = (uint32_t)(ch.seed >> 32);
    const uint32_t chain_id = ch.chain_id;
    const uint64_t log_off = ch.log_off;
    const double P = ch.P;
    const uint32_t eci = sh.eci;

    LdsChain c;
    c.R = smem + me.lds_off;
    c.N = ch.N;
    c.B = me.B;
    c.w = sh.w;
    c.wg = sh.wg;
    c.Sp = ch.Sp;
    c.qb = ch.N / me.B;
    c.rem = ch.N % me.B;
    c.per = (sh.flags & F_PERIODIC) != 0;
    const bool npt = (sh.flags & F_NPT) != 0;
    // FP32: walks of one partner per step where the window is one partner
    const bool one = sizeof(Real) == 4 && c.w == 1;

    const uint32_t r = tid - me.lane_off;
    const uint32_t size = act ? c.qb + (r < c.rem ? 1u : 0u) : 0u;
    const uint32_t start = act ? r * c.qb + (r < c.rem ? r : c.rem) : 0u;
    const uint32_t a0 = c.wg + r * c.Sp;
    const uint32_t gapR = c.Sp - size;
    const uint32_t gapL = r == 0 ? 0u : c.Sp - (c.qb + (r - 1 < c.rem ? 1u : 0u));
    const uint32_t seg = act ? c.B : 1u;
    const bool leader = act && r == 0;
    // waves none of whose particles has an image skip the image stores
    const bool edges = c.per && __any(act && (start < c.wg || start + size + c.wg > c.N));
    // a chain of several waves has its box-length proposal made by the first
    // (some 200 to 400 instructions the others need not issue)
    constexpr uint32_t WV = T / BatchedScratch<T>::NVP;
    const bool waves = me.B >= WV;

    const double *xg = a.x + ch.x_off;
    for (uint32_t t = 0; t < size; ++t) c.R[a0 + t] = xg[start + t];
    const DevState st = a.states[ic];
    double L = st.L, U = st.U, mdrift = st.max_drift;
    uint64_t sweep = st.sweep;
    __syncthreads();
    if (act) fill_ghosts(c, r, c.B, L);
    __syncthreads();

    uint32_t n_wall = 0, n_core = 0, n_terms = 0;
    uint32_t acc_total = 0, n_vt = 0, n_av = 0, n_rc = 0;
    // sweeps to the next recompute
    uint32_t to_eci = eci ? eci - (uint32_t)(sweep % eci) : 0u;

#pragma unroll 1
    for (uint32_t sw = 0; sw < a.n_sweeps; ++sw, ++sweep) {
        double dUs = 0.0;
        uint32_t acc = 0;
        uint32_t w_md = 0, w_u = 0, w_next_md = 0, w_next_u = 0;
        constexpr bool BOXK = sizeof(Real) == 4 && KIND == POT_LJ;
        if (npt && waves && r < 64) {
            const VolProp v = vol_propose<BOXK>(ch, L, sweep);
            if (r == 0) sc.vp[me.lane_off / WV] = v;
        }
#pragma unroll 1
        for (uint32_t t = 0; t < bd.smax; ++t) {
            if (t < size) {
                const uint32_t i = start + t;
                const uint32_t my = a0 + t;
                // one Philox block per pair of block positions (t, t+1):
                // computed at even t, its second half kept for odd t (t is
                // the same on every lane, so the branch is uniform)
                if ((t & 1u) == 0) {
                    uint32_t rr[4];
                    philox4x32_10(i, (uint32_t)sweep, chain_id, 0u, key0, key1, rr);
                    w_md = rr[0];
                    w_u = rr[1];
                    w_next_md = rr[2];
                    w_next_u = rr[3];
                } else {
                    w_md = w_next_md;
                    w_u = w_next_u;
                }
                // ((u1 - 1/2) 2) max_step with u1 = (w + 1/2) 2^-32: the odd
                // integer 2 (w - 2^31) + 1 times max_step 2^-32, the same
                // product rounded once
                const double u = u32o(w_u);
                const double md = fma((double)(int32_t)(w_md ^ 0x80000000u), 2.0, 1.0) * step32;
                const double xi = c.R[my];
                const double xn = xi + md;
                double dE = 0.0;
                // a window of one partner per side (the hard core keeps the
                // second beyond the cutoff): the one-partner walk, which
                // evaluates no clamped duplicate (wave-uniform: a bundle
                // shares its window)
                const bool accd =
                    one ? trial_lds<Real, KIND, false, false>(c, q, gmin, beta, betaf, i, t, size, my, gapL, gapR,
                                                              L, xi, xn, md, u, dE, n_terms, n_wall, n_core)
                        : trial_lds<Real, KIND, false, true>(c, q, gmin, beta, betaf, i, t, size, my, gapL, gapR,
                                                             L, xi, xn, md, u, dE, n_terms, n_wall, n_core);
                const double xs = accd ? xn : xi;
                c.R[my] = xs;
                if (edges) put_images(c, i, xs, L);
                dUs += accd ? dE : 0.0;
                acc += accd ? 1u : 0u;
                if (a.acclog) a.acclog[log_off + (uint64_t)(soff + sw) * c.N + i] = accd ? 1 : 0;
            }
            __syncthreads();
        }

        // box-length trial (fav, src/jmmMCState.cpp:2161-2293): energy change
        // pair by pair over the pairs whose left member is in this block
        VolProp vp{};
        uint32_t bad = 0;
        double vpart = 0.0, upart = 0.0;
        if (npt) {
            if (waves) vp = sc.vp[me.lane_off / WV];
            else vp = vol_propose<BOXK>(ch, L, sweep);
            auto wrap = [&](uint32_t m) { return c.R[c.wg + m]; };
            const bool last = c.per && r + 1 == c.B, von = vp.valid && act;
            // long blocks in two halves (half_of; a bundle's longest decides)
            const int parts = bd.smax >= HALF_MIN ? 2 : 1;
            uint32_t t0 = 0, t1 = half_of(size);
#pragma unroll 1
            for (int part = 0; part < parts; ++part) {
                double u = 0.0;
                vpart += one ? vol_lane<Real, KIND, false>(c, q, gmin, vp, von, start, size, t0, t1, a0, gapR, last,
                                                           wrap, bad, u)
                             : vol_lane<Real, KIND, sizeof(Real) == 4>(c, q, gmin, vp, von, start, size, t0, t1, a0,
                                                                       gapR, last, wrap, bad, u);
                upart += u;
                t0 = t1;
                t1 = size;
            }
        }
        {
            double v[3] = {dUs, vpart, upart};
            uint32_t k2[2] = {acc, bad};
            if (eci) {
                --to_eci;
                const bool any = __any(act && to_eci == 0);
                if ((tid & 63) == 0) sc.need[tid >> 6] = any ? 1 : 0;
            }
            seg_allreduce<T, 3, 2, false>(v, k2, seg, me.lane_off, sc.rd, sc.ri);
            U = U + v[0];
            vpart = v[1];
            acc = k2[0];
            bad = k2[1];
            // FP32 form: the box-length pass summed the configuration's FP32
            // energy over every pair; it replaces the running sum, so FP32
            // trial errors do not accumulate between recomputes.  Square
            // well: the pass gave the scaled energy, the running energy is
            // exact
            if (sizeof(Real) == 4 && KIND == POT_HRSW) vpart = vpart - U;
            else if (sizeof(Real) == 4 && npt && vp.valid && !bad) U = v[2];
        }
        acc_total += acc;
        uint32_t accv = 0;
        if (npt) {
            ++n_vt;
            if (vp.valid && !bad && vol_accept(vpart, vp.dL, vp.lns, P, beta, vp.jac, vp.u)) {
                L = vp.Lp;
                // (idle lanes of the workgroup have size 0)
                for (uint32_t t = 0; t < size; ++t) {
                    const double xs = c.R[a0 + t] * vp.sc;
                    c.R[a0 + t] = xs;
                    if (edges) put_images(c, start + t, xs, L);
                }
                U = U + vpart;
                accv = 1;
                ++n_av;
            }
            __syncthreads();
        }

        // (constant length: the sums' scratch is read until here)
        if (!npt && (eci || a.sW)) __syncthreads();

        // drift guard (ECheck, src/jmmMCState.cpp:1965-2095), always FP64
        const bool need = act && eci && to_eci == 0;
        uint32_t some = 0;
        if (eci)
            for (uint32_t m = 0; m < T / 64; ++m) some |= sc.need[m];
        if (__builtin_amdgcn_readfirstlane(some)) {
            double Up = 0.0;
            if (need) {
                for (uint32_t t = 0; t < size; ++t) {
                    const uint32_t i = start + t;
                    const uint32_t my = a0 + t;
                    const double xi = c.R[my];
                    const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - i);
                    for (uint32_t k = 1; k <= kR; ++k) {
                        const double d = c.R[my + k + (t + k >= size ? gapR : 0)] - xi;
                        if (d > q.rc) break;
                        Up += phi64<KIND>(q, d);
                    }
                }
            }
            double v[1] = {Up};
            uint32_t k1[1] = {0};
            seg_allreduce<T, 1, 1>(v, k1, seg, me.lane_off, sc.rd, sc.ri);
            if (eci && to_eci == 0) to_eci = eci;
            if (need) {
                const double dr = fabs(v[0] - U);
                if (dr > mdrift) mdrift = dr;
                U = v[0];
                ++n_rc;
            }
        }

        double Ws = 0.0, Hs = 0.0;
        if (a.sW) {
            double v[2] = {0.0, 0.0};
            if (act) virial_lane<KIND>(c, q, start, size, a0, gapR, v[0], v[1]);
            uint32_t k1[1] = {0};
            seg_allreduce<T, 2, 1>(v, k1, seg, me.lane_off, sc.rd, sc.ri);
            Ws = v[0];
            Hs = v[1];
        }
        if (leader) {
            const uint64_t row = (uint64_t)(soff + sw) * a.n_chains + ic;
            a.sU[row] = U;
            a.sL[row] = L;
            a.sA[row] = make_uint2(acc, accv);
            if (a.sW) {
                a.sW[row] = Ws;
                a.sH[row] = Hs;
            }
        }
    }

    __syncthreads();
    {
        double vz[1] = {0.0};
        uint32_t k4[4] = {size * a.n_sweeps, n_wall, n_core, n_terms};
        seg_allreduce<T, 1, 4>(vz, k4, seg, me.lane_off, sc.rd, sc.ri);
        if (leader) {
            DevState &o = a.states[ic];
            o.L = L;
            o.U = U;
            o.sweep = sweep;
            o.cnt[0] += k4[0];
            o.cnt[1] += acc_total;
            o.cnt[2] += k4[1];
            o.cnt[3] += k4[2];
            o.cnt[4] += k4[3];
            o.cnt[5] += n_vt;
            o.cnt[6] += n_av;
            o.cnt[7] += n_rc;
            o.max_drift = mdrift;
        }
    }
    double *xw = a.x + ch.x_off;
    for (uint32_t t = 0; t < size; ++t) xw[start + t] = c.R[a0 + t];
    __syncthreads();
}

// Persistent kernel, one instantiation per (precision, workgroup size,
// memory mode, waves per SIMD): every workgroup pulls bundles from one queue
// (all potentials together, longest first) until it is empty; all waves of a
// workgroup leave together when the queue is drained.  The potential is
// uniform per bundle.  W waves per SIMD bound the registers: 2 (256, 193 used),
// or 3 for 256 lanes (168; 9 spilled in FP32, 1 in FP64, outside the phases), which hides more of
// the phases' latency where there are bundles for it: 4096 mixed chains of 32 to
// 4000, FP32, 55.0 us a sweep with 2, 44.6 with 3 (4: 128 registers, 269
// spilled, 59.5); bundles that fit at 2 lose 1 to 2 % to the spills.
template <typename Real, int T, bool GX, int W>
__global__ void __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(W)))
k_sweep_batched(SweepArgs a)
{
    extern __shared__ double smem[];
    __shared__ BatchedScratch<T> sc;
    const uint32_t soff = a.ctrl->sample_off;
    for (;;) {
        if (threadIdx.x == 0) sc.item = atomicAdd(&a.ctrl->queue, 1u);
        __syncthreads();
        // the same value in every lane: keep the bundle in scalar registers
        const uint32_t item = __builtin_amdgcn_readfirstlane(sc.item);
        __syncthreads();
        if (item >= a.n_items) break;
        const DevBundle bd = a.bundles[item];
        if (GX) {
            switch (bd.kind) {
            case POT_LJ: run_bundle_gx<Real, POT_LJ, T>(a, bd, sc, soff); break;
            case POT_HARMONIC: run_bundle_gx<Real, POT_HARMONIC, T>(a, bd, sc, soff); break;
            case POT_HRSW: run_bundle_gx<Real, POT_HRSW, T>(a, bd, sc, soff); break;
            default: run_bundle_gx<Real, POT_YUKAWA, T>(a, bd, sc, soff); break;
            }
        } else {
            switch (bd.kind) {
            case POT_LJ: run_bundle_lds<Real, POT_LJ, T>(a, bd, smem, sc, soff); break;
            case POT_HARMONIC: run_bundle_lds<Real, POT_HARMONIC, T>(a, bd, smem, sc, soff); break;
            case POT_HRSW: run_bundle_lds<Real, POT_HRSW, T>(a, bd, smem, sc, soff); break;
            default: run_bundle_lds<Real, POT_YUKAWA, T>(a, bd, smem, sc, soff); break;
            }
        }
        __syncthreads();
    }
}

// --------------------------------------------------------- cooperative form

// Data-parallel control that gives every lane of a group of G lanes lane I's
// value: row_newbcast:I, quad_perm:[I,I,I,I], quad_perm:[I,I,2+I,2+I].
template <int G, int I>
constexpr int lane_ctrl()
{
    return G == 16 ? 0x150 + I : G == 4 ? I * 0x55 : 0xA0 + I * 0x55;
}

// The value of lane I of the caller's group of G lanes (16: a row; 4: a
// quad; 2), through the data-parallel primitives: no LDS round trip.
template <int G, int I>
__device__ __forceinline__ double from_lane(double v)
{
    constexpr int ctrl = lane_ctrl<G, I>();
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

template <int G, int I>
__device__ __forceinline__ int from_lane_i(int v)
{
    return __builtin_amdgcn_mov_dpp(v, lane_ctrl<G, I>(), 0xf, 0xf, true);
}

// exp out of line: its constants would otherwise sit in registers through the
// phases, where it is almost never needed.
__device__ __noinline__ double exp_apart(double x) { return exp(x); }

// phi64 of a separation whose cutoff test has been made, without branches
// (hard cores are handled before any pair is evaluated).
template <int KIND>
__device__ __forceinline__ double phi64_in(const Pot &q, double d, bool in)
{
    double v;
    if (KIND == POT_LJ) {
        const double d3 = d * d * d;
        const double i6 = (1.0 / (d3 * d3)) * q.sig6;
        const double i12 = i6 * i6;
        v = (q.e4 * i12 - q.e4 * i6) - q.shift;
    } else if (KIND == POT_HARMONIC) {
        const double m = d - 1.0;
        v = d <= 0.0 ? 10e10 : m * m;
    } else if (KIND == POT_HRSW) {
        v = -q.p1;
    } else {
        v = (q.p0 * (exp(-q.p1 * d) / d)) - q.shift;
    }
    return in ? v : 0.0;
}

// acc plus the group's lanes I0, I0 + 1, ... I1 - 1, each lane's KP terms in
// turn.
template <int G, int I0, int I1, uint32_t KP>
__device__ __forceinline__ double add_lanes(double acc, const double (&v)[KP])
{
    if constexpr (I0 < I1) {
#pragma unroll
        for (uint32_t u = 0; u < KP; ++u) acc += from_lane<G, I0>(v[u]);
        return add_lanes<G, I0 + 1, I1, KP>(acc, v);
    } else {
        return acc;
    }
}

// One side's ordered sum of a trial's terms (the group's lanes I0 .. I0 +
// G/2 - 1), the far lanes only where some trial of the wave reaches them:
// some lane's h of at least 1, 2, 4 holds a partner inside the cutoff
// (uniform); the terms left out are zeros.
template <int G, int I0, uint32_t KP>
__device__ __forceinline__ double add_side(double acc, const double (&v)[KP], bool far1, bool far2, bool far4)
{
    constexpr int H = G / 2;
    acc = add_lanes<G, I0, I0 + 1, KP>(acc, v);
    if constexpr (H > 1) {
        if (far1) {
            acc = add_lanes<G, I0 + 1, I0 + 2, KP>(acc, v);
            if constexpr (H > 2) {
                if (far2) {
                    acc = add_lanes<G, I0 + 2, I0 + 4, KP>(acc, v);
                    if (far4) acc = add_lanes<G, I0 + 4, I0 + H, KP>(acc, v);
                }
            }
        }
    }
    return acc;
}

// What the waves of a workgroup share: the sweep's box-length proposal, its
// integer totals (two slots, by sweep parity: one is cleared while the other
// is read) and the 64-block sums, and the launch's counters.
struct CoopScratch {
    VolProp vp;
    double grp[COOP_B / 64][3];
    uint32_t acc[2], bad[2];
    uint32_t wall, core, terms;
};

// Sum of a block's pair terms in the order of the one-lane walks (particle by
// particle, each particle's partners outwards): the G lanes of the block take
// a particle each, put their terms into LDS and all add them in sequence, so
// every lane holds the one-lane sum bit for bit.  pair(k, t, xi, xj, v) sets
// a pair's NF terms and returns whether the particle's walk goes on; a partner
// after the last has zero terms, whose addition is exact.
template <int G, int NF, typename Pair>
__device__ __forceinline__ void block_sum(const LdsChain &c, uint32_t start, uint32_t size, uint32_t t0, uint32_t t1,
                                          uint32_t a0, uint32_t gapR, uint32_t g, double *terms, double (&acc)[NF],
                                          Pair pair)
{
    for (uint32_t tb = t0; __any(tb < t1); tb += G) {
        const uint32_t t = tb + g;
        bool run = t < t1;
        const double xi = c.R[run ? a0 + t : 0u];
        const uint32_t kR = c.per ? c.w : min(c.w, c.N - 1 - (start + t));
        double v[NF][COOP_W];
        uint32_t kmax = 0;
        // two partners at a time: their reads and pair energies overlap
#pragma unroll
        for (uint32_t k = 1; k <= COOP_W; k += 2) {
#pragma unroll
            for (int f = 0; f < NF; ++f) v[f][k - 1] = v[f][k] = 0.0;
            if (k <= c.w) {
                run = run & (k <= kR);
                if (__any(run)) {
                    const bool run2 = run & (k + 1 <= kR);
                    const double xj = c.R[run ? a0 + t + k + (t + k >= size ? gapR : 0u) : 0u];
                    const double xj2 = c.R[run2 ? a0 + t + k + 1 + (t + k + 1 >= size ? gapR : 0u) : 0u];
                    double q[NF], q2[NF];
                    const bool on = pair(k, t, xi, xj, run, q) & run;
                    const bool on2 = pair(k + 1, t, xi, xj2, run2, q2) & run2 & on;
#pragma unroll
                    for (int f = 0; f < NF; ++f) {
                        v[f][k - 1] = on ? q[f] : 0.0;
                        v[f][k] = on2 ? q2[f] : 0.0;
                    }
                    kmax = min(k + 1, c.w);
                    run = on2;
                }
            }
        }
        // the group's terms, lane-major; a wave's own lanes only: LDS keeps a
        // wave's order, the fences keep the compiler's
        const uint32_t M = G * kmax;
        double *mine = terms + (threadIdx.x / G) * (G * c.w * NF);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t k = 0; k < COOP_W; ++k)
            if (k < kmax)
#pragma unroll
                for (int f = 0; f < NF; ++f) mine[f * M + g * kmax + k] = v[f][k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        constexpr int E = G < 4 ? G : 4;
        for (uint32_t m = 0; m < M; m += E) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                double e[E];
#pragma unroll
                for (int u = 0; u < E; ++u) e[u] = mine[f * M + m + u];
#pragma unroll
                for (int u = 0; u < E; ++u) acc[f] += e[u];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// Sums over the chain's blocks in the order of seg_allreduce (pairwise trees
// over 64 blocks, then the trees in sequence), from per-block values in LDS:
// one wave per 64 blocks, a block per lane; every lane of the workgroup
// receives the same bits.  Contains a workgroup barrier.
template <int ND>
__device__ __forceinline__ void chain_sum(const double *blk, uint32_t B, CoopScratch &sc, double (&v)[ND])
{
    const uint32_t l = threadIdx.x & 63u, q = threadIdx.x >> 6, top = B < 64 ? B : 64u;
    if (q * 64 < B) {
        double p[ND];
#pragma unroll
        for (int m = 0; m < ND; ++m) p[m] = l < top ? blk[m * B + q * 64 + l] : 0.0;
        uint32_t none[1] = {0};
        if (top > 1) seg_level<1>(p, none, 64);
        if (top > 2) seg_level<2>(p, none, 64);
        if (top > 4) seg_level<4>(p, none, 64);
        if (top > 8) seg_level<8>(p, none, 64);
        if (top > 16) seg_level<16>(p, none, 64);
        if (top > 32) seg_level<32>(p, none, 64);
        if (l == 0)
#pragma unroll
            for (int m = 0; m < ND; ++m) sc.grp[q][m] = p[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < ND; ++m) {
        double acc = sc.grp[0][m];
        for (uint32_t k = 1; k * 64 < B; ++k) acc += sc.grp[k][m];
        v[m] = acc;
    }
}

// One chain per workgroup, G lanes per block, for engines with too few
// chains to fill the GPU: a phase's time is then the latency of one trial,
// and the batched kernel's lane walks its partners, its random numbers and
// (box-length move, recompute, virial) its block's pairs one after another.
// Here the partners of a trial are G/2 lanes a side at once, the random
// numbers of the next 2 G block positions are drawn G lanes at once before
// them (with ln u in the FP64 form, so that the Metropolis exponential is
// evaluated only where |ln u + beta dE| < 1e-4: outside, the comparison of the
// logarithms decides the same, |ln u| < 23 from the hardware's FP32 logarithm
// being good to 1e-5), and the sums over a block's pairs take a
// particle per lane.  Trials, random numbers and the order of every sum are
// run_bundle_lds's, so a chain has the same bits in both.
//
// Bound by the latency of a phase: about 120 vector and 65 scalar
// instructions of one wave (some 5 cycles each), two dependent LDS reads and a
// barrier.  One LJ chain of 64, FP64: 0.56 us a phase where the batched
// kernel takes 1.9 (100 sweeps and their read: 1494 -> 593 us); 64 chains of
// 32 to 256, both potentials, FP32 NPT: 3154 -> 1158 us; one chain of 2000
// with two partners a side, virials, FP64: 10 sweeps 294 -> 254 us.
template <typename Real, int KIND, int G, uint32_t KP>
__device__ __forceinline__ void run_coop(const SweepArgs &a, uint32_t ic, double *smem, CoopScratch &sc, uint32_t soff)
{
    constexpr uint32_t H = G / 2;  // lanes a side
    constexpr bool WELL = sizeof(Real) == 4 && KIND == POT_HRSW;
    constexpr uint32_t GM = (1u << G) - 1;
    const uint32_t tid = threadIdx.x, T = blockDim.x, lane = tid & 63u;
    const DevChain &ch = a.chains[ic];
    const Pot q = ch.pot;
    const double gmin = ch.gmin, beta = ch.beta, P = ch.P;
    const double step32 = ch.max_step * (1.0 / 4294967296.0);
    const float betaf = ch.betaf;
    const uint32_t key0 = (uint32_t)ch.seed, key1 = (uint32_t)(ch.seed >> 32);
    const uint32_t chain_id = ch.chain_id, eci = ch.eci;
    const uint64_t log_off = ch.log_off;
    const bool npt = (ch.flags & F_NPT) != 0;
    const uint32_t smax = ch.smax;

    LdsChain c;
    c.R = smem;
    c.N = ch.N;
    c.B = ch.B;
    c.w = ch.w;
    c.wg = ch.wg;
    c.Sp = ch.Sp;
    c.qb = ch.N / ch.B;
    c.rem = ch.N % ch.B;
    c.per = (ch.flags & F_PERIODIC) != 0;
    double *blk = smem + ch.lds_len;   // [3][B]: per-block sums
    double *work = blk + 3 * c.B;      // random numbers, or pair terms
    double2 *rnd = (double2 *)(work + ((ch.lds_len + 3 * c.B) & 1u));
    uint32_t *rndw = (uint32_t *)(rnd + (size_t)c.B * 2 * G);

    const uint32_t b = tid / G, g = tid % G;
    const bool act = b < c.B;
    const uint32_t size = act ? c.qb + (b < c.rem ? 1u : 0u) : 0u;
    const uint32_t start = act ? b * c.qb + (b < c.rem ? b : c.rem) : 0u;
    const uint32_t a0 = c.wg + b * c.Sp;
    const uint32_t gapR = c.Sp - size;
    const uint32_t gapL = b == 0 ? 0u : c.Sp - (c.qb + (b - 1 < c.rem ? 1u : 0u));
    const bool left = g < H;
    const uint32_t h = left ? g : g - H;
    const uint32_t gl = lane & ~(uint32_t)(G - 1);  // the group's first lane in its wave
    const uint32_t dir = left ? ~0u : 1u, gap = left ? 0u - gapL : gapR;
    // what the lane stores after a trial: the particle (lane 0), its image in
    // the right (lane 1) or left (lane 2) ghosts; putb + t for the block
    // positions t of [put0, put0 + putn)
    uint32_t putb = a0, put0 = 0, putn = g == 0 ? size : 0u;
    double puts = 0.0;
    if (c.per && g == 1 && start < c.wg) {
        putb = c.wg + c.B * c.Sp + start;
        putn = c.wg - start;
        puts = 1.0;
    }
    // (two lanes per block: chains of many blocks, the last not the first)
    if (c.per && g == (G == 2 ? 1 : 2) && size && start + size + c.wg > c.N) {
        put0 = start + c.wg < c.N ? c.N - c.wg - start : 0u;
        putb = start + c.wg - c.N;  // modulo 2^32 below put0
        putn = size - put0;
        puts = -1.0;
    }

    const double *xg = a.x + ch.x_off;
    for (uint32_t t = g; t < size; t += G) c.R[a0 + t] = xg[start + t];
    const DevState st = a.states[ic];
    double L = st.L, U = st.U, mdrift = st.max_drift;
    uint64_t sweep = st.sweep;
    if (tid == 0) {
        sc.acc[0] = sc.acc[1] = sc.bad[0] = sc.bad[1] = 0;
        sc.wall = sc.core = sc.terms = 0;
    }
    __syncthreads();
    fill_ghosts(c, tid, T, L);
    __syncthreads();

    uint32_t to_eci = eci ? eci - (uint32_t)(sweep % eci) : 0u;  // sweeps to the next recompute
    // rejections per block, pair terms per lane
    uint32_t n_wall = 0, n_core = 0, n_terms = 0;
    uint32_t acc_total = 0, n_vt = 0, n_av = 0, n_rc = 0;

#pragma unroll 1
    for (uint32_t sw = 0; sw < a.n_sweeps; ++sw, ++sweep) {
        double dUs = 0.0;
        uint32_t acc = 0;
        const double putL = puts * L;
        // the sweep's box-length proposal depends on L alone: the last wave
        // (the shortest blocks) prepares it
        if (npt && tid >= T - 64) {
            const VolProp v = vol_propose<sizeof(Real) == 4 && KIND == POT_LJ>(ch, L, sweep);
            if (lane == 0) sc.vp = v;
        }
#pragma unroll 1
        for (uint32_t t = 0; t < smax; ++t) {
            const uint32_t tr = t & (2 * G - 1);
            if (tr == 0) {
                // random numbers of the block positions t .. t + 2 G - 1
                const uint32_t j = t + 2 * g;
                if (j < size) {
                    uint32_t rr[4];
                    philox4x32_10(start + j, (uint32_t)sweep, chain_id, 0u, key0, key1, rr);
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        const double u = u32o(rr[2 * m + 1]);
                        const uint32_t at = b * 2 * G + 2 * g + m;
                        rnd[at] = make_double2(fma((double)(int32_t)(rr[2 * m] ^ 0x80000000u), 2.0, 1.0) * step32,
                                               sizeof(Real) == 8 ? (double)__logf((float)u) : u);
                        if (sizeof(Real) == 8) rndw[at] = rr[2 * m + 1];
                    }
                }
                __syncthreads();
            }
            if (t < size) {
                const uint32_t i = start + t, my = a0 + t;
                const uint32_t ri = b * 2 * G + tr;
                // partner k0 + h + 1 on the lane's side (clamped to the image)
                const uint32_t side_n = c.per ? UINT32_MAX : left ? i : c.N - 1 - i;
                const uint32_t own_n = left ? t : size - 1 - t;  // partners in the own block
                auto partner = [&](uint32_t k) {
                    const uint32_t kk = min(k, c.wg);
                    return c.R[my + dir * kk + (kk > own_n ? gap : 0u)];
                };
                double xj[KP];
#pragma unroll
                for (uint32_t u = 0; u < KP; ++u) xj[u] = partner(h * KP + u + 1);
                const double2 rn = rnd[ri];
                const double xi = c.R[my];
                const double xn = xi + rn.x;
                const bool wall = !c.per && fabs(xn) > L / 2.0;
                const double s0 = xn - xj[0], sn = left ? s0 : -s0;
                // the nearest partners' hard-core test, on one lane a side
                const int hit = (int)((h == 0) & (c.N >= 2) & (side_n >= 1) & (sn < gmin));
                const bool core = (from_lane_i<G, 0>(hit) | from_lane_i<G, H>(hit)) != 0;
                const bool go = !wall & !core;
                n_wall += wall ? 1u : 0u;
                n_core += !wall & core ? 1u : 0u;
                double dEL = 0.0, dER = 0.0, side = 0.0;
                int wL = 0, wR = 0;
                uint32_t k0 = 0;
                for (;;) {
                    // all evaluated on every lane, side by side: a branch
                    // each would run them one after the other
                    double term[KP];
                    uint64_t any = 0, last_in = 0;
#pragma unroll
                    for (uint32_t u = 0; u < KP; ++u) {
                        const uint32_t k = k0 + h * KP + u + 1;
                        const double o = fabs(xi - xj[u]), n = fabs(xn - xj[u]);
                        const bool valid = go & (k <= c.w) & (k <= side_n);
                        const bool io = valid & inside64<KIND>(q, o), in = valid & inside64<KIND>(q, n);
                        n_terms += (io ? 1u : 0u) + (in ? 1u : 0u);
                        const uint64_t bo = __ballot(io), bn = __ballot(in);
                        last_in = bo | bn;
                        any |= last_in;
                        if (WELL) {
                            const uint32_t mo = (uint32_t)(bo >> gl) & GM, mn = (uint32_t)(bn >> gl) & GM;
                            constexpr uint32_t LM = (1u << H) - 1;
                            wL += (int)__popc(mn & LM) - (int)__popc(mo & LM);
                            wR += (int)__popc(mn & ~LM) - (int)__popc(mo & ~LM);
                        } else if (sizeof(Real) == 8) {
                            const double en = phi64_in<KIND>(q, n, in), eo = phi64_in<KIND>(q, o, io);
                            term[u] = en - eo;
                        } else {
                            term[u] = (double)(phi32<KIND>(q, (float)n, in) - phi32<KIND>(q, (float)o, io));
                        }
                    }
                    if (!WELL) {
                        if (H == 1) {
#pragma unroll
                            for (uint32_t u = 0; u < KP; ++u) side += term[u];
                        } else {
                            // lanes whose h is at least 1, 2, 4
                            constexpr uint64_t F1 = G == 16 ? 0xfefefefefefefefeull : 0xaaaaaaaaaaaaaaaaull;
                            constexpr uint64_t F2 = 0xfcfcfcfcfcfcfcfcull, F4 = 0xf0f0f0f0f0f0f0f0ull;
                            const bool far1 = (any & F1) != 0, far2 = (any & F2) != 0, far4 = (any & F4) != 0;
                            dEL = add_side<G, 0, KP>(dEL, term, far1, far2, far4);
                            dER = add_side<G, H, KP>(dER, term, far1, far2, far4);
                        }
                    }
                    if (H * KP >= COOP_W) break;
                    k0 += H * KP;
                    // the last partner of a side inside somewhere: the next ones
                    constexpr uint64_t LAST = G == 16 ? 0x8080808080808080ull : G == 4 ? 0xaaaaaaaaaaaaaaaaull : ~0ull;
                    if (k0 >= c.w || (last_in & LAST) == 0) break;
#pragma unroll
                    for (uint32_t u = 0; u < KP; ++u) xj[u] = partner(k0 + h * KP + u + 1);
                }
                if (H == 1 && !WELL) {
                    dEL = from_lane<G, 0>(side);
                    dER = from_lane<G, H>(side);
                }
                const double dE = WELL ? -q.p1 * (double)wL + -q.p1 * (double)wR : dEL + dER;
                bool accd;
                if (sizeof(Real) == 8) {
                    const double e = -dE * beta;
                    accd = go & ((dE <= 0.0) | (e > rn.y + 1e-4));
                    const bool unsure = go & !accd & !(e < rn.y - 1e-4);
                    if (__any(unsure)) accd = accd || (unsure && exp_apart(e) > u32o(rndw[ri]));
                } else {
                    accd = go & ((dE <= 0.0) | ((double)fexp(-betaf * (float)dE) > rn.y));
                }
                // the position and its periodic images: one lane each
                const double xs = accd ? xn : xi;
                if (t - put0 < putn) c.R[putb + t] = xs + putL;
                if (a.acclog && g == 0) a.acclog[log_off + (uint64_t)(soff + sw) * c.N + i] = accd ? 1 : 0;
                dUs += accd ? dE : 0.0;
                acc += accd ? 1u : 0u;
            }
            __syncthreads();
        }

        // box-length trial (fav, src/jmmMCState.cpp:2161-2293)
        VolProp vp{};
        bool bad = false;
        double vpart = 0.0, upart = 0.0;
        if (npt) {
            vp = sc.vp;
            const bool last = c.per && b + 1 == c.B, von = vp.valid && act;
            uint32_t t0 = 0, t1 = von ? half_of(size) : 0u;
            const uint32_t tend = von ? size : 0u;
            const int parts = smax >= HALF_MIN ? 2 : 1;
#pragma unroll 1
            for (int part = 0; part < parts; ++part) {
                constexpr int NF = sizeof(Real) == 4 && !WELL ? 2 : 1;
                double s[NF] = {};
                block_sum<G, NF>(c, start, size, t0, t1, a0, gapR, g, work, s,
                                 [&](uint32_t k, uint32_t t, double xi, double xj, bool run, double (&v)[NF]) {
                                     const double xis = xi * vp.sc;
                                     double xjs = xj * vp.sc;
                                     if (run && last && t + k >= size) xjs = c.R[c.wg + t + k - size] * vp.sc + vp.Lp;
                                     const double d0 = xj - xi, d1 = xjs - xis;
                                     const bool hit = (k == 1) & run & (d1 < gmin);
                                     bad = bad | hit;
                                     const bool in0 = inside64<KIND>(q, d0), in1 = inside64<KIND>(q, d1);
                                     if constexpr (sizeof(Real) == 8) {
                                         v[0] = phi64_in<KIND>(q, d1, in1) - phi64_in<KIND>(q, d0, in0);
                                         return !(hit | ((d0 > q.rc) & (d1 > q.rc)));
                                     } else if constexpr (WELL) {
                                         v[0] = in1 ? 1.0 : 0.0;
                                         return in1 & !hit;
                                     } else {
                                         float e0;
                                         v[0] = (double)box_term32<KIND>(q, vp.bk, (float)d0, (float)d1, in0, in1, e0);
                                         v[1] = (double)e0;
                                         return (in0 | in1) & !hit;
                                     }
                                 });
                vpart += WELL ? -q.p1 * s[0] : s[0];
                if constexpr (NF == 2) upart += s[1];
                t0 = t1;
                t1 = tend;
            }
        }
        {
            if (act && g == 0) {
                blk[b] = dUs;
                if (npt) {
                    blk[c.B + b] = vpart;
                    blk[2 * c.B + b] = upart;
                }
            }
            const uint32_t par = (uint32_t)sweep & 1u;
            // the wave's accepted trials, a bit of the blocks' counts at a time
            uint32_t wacc = 0;
            for (uint32_t m = 0; m < 32; ++m) {
                const uint32_t rest = act && g == 0 ? acc >> m : 0u;
                if (!__any(rest != 0)) break;
                wacc += (uint32_t)__popcll(__ballot(rest & 1u)) << m;
            }
            if (lane == 0 && wacc) atomicAdd(&sc.acc[par], wacc);
            if (__any(bad) && lane == 0) sc.bad[par] = 1u;
            __syncthreads();
            double v[3] = {0.0, 0.0, 0.0};
            if (npt) {
                chain_sum<3>(blk, c.B, sc, v);
            } else {
                double v1[1];
                chain_sum<1>(blk, c.B, sc, v1);
                v[0] = v1[0];
            }
            acc = sc.acc[par];
            bad = sc.bad[par] != 0;
            if (tid == 0) sc.acc[par ^ 1u] = sc.bad[par ^ 1u] = 0;
            U = U + v[0];
            vpart = v[1];
            if (WELL) vpart = vpart - U;
            else if (sizeof(Real) == 4 && npt && vp.valid && !bad) U = v[2];
        }
        acc_total += acc;
        uint32_t accv = 0;
        if (npt) {
            ++n_vt;
            if (vp.valid && !bad && vol_accept(vpart, vp.dL, vp.lns, P, beta, vp.jac, vp.u)) {
                for (uint32_t t = g; t < size; t += G) c.R[a0 + t] = c.R[a0 + t] * vp.sc;
                L = vp.Lp;
                U = U + vpart;
                accv = 1;
                ++n_av;
                __syncthreads();
                fill_ghosts(c, tid, T, L);
            }
        }
        __syncthreads();

        // drift guard (ECheck, src/jmmMCState.cpp:1965-2095), always FP64
        if (eci && --to_eci == 0) {
            to_eci = eci;
            double s[1] = {0.0};
            block_sum<G, 1>(c, start, size, 0u, size, a0, gapR, g, work, s,
                            [&](uint32_t, uint32_t, double xi, double xj, bool, double (&v)[1]) {
                                const double d = xj - xi;
                                v[0] = phi64<KIND>(q, d);
                                return !(d > q.rc);
                            });
            if (act && g == 0) blk[b] = s[0];
            __syncthreads();
            double v[1];
            chain_sum<1>(blk, c.B, sc, v);
            const double dr = fabs(v[0] - U);
            if (dr > mdrift) mdrift = dr;
            U = v[0];
            ++n_rc;
            __syncthreads();
        }

        double Ws = 0.0, Hs = 0.0;
        if (a.sW) {
            double s[2] = {0.0, 0.0};
            block_sum<G, 2>(c, start, size, 0u, size, a0, gapR, g, work, s,
                            [&](uint32_t, uint32_t, double xi, double xj, bool, double (&v)[2]) {
                                const double d = xj - xi;
                                virial64<KIND>(q, d, v[0], v[1]);
                                // inside nothing adds nothing (strict cutoffs)
                                const bool in = inside64<KIND>(q, d);
                                v[0] = in ? v[0] : 0.0;
                                v[1] = in ? v[1] : 0.0;
                                return !(d > q.rc);
                            });
            if (act && g == 0) {
                blk[b] = s[0];
                blk[c.B + b] = s[1];
            }
            __syncthreads();
            double v[2];
            chain_sum<2>(blk, c.B, sc, v);
            Ws = v[0];
            Hs = v[1];
            __syncthreads();
        }
        if (tid == 0) {
            const uint64_t row = (uint64_t)(soff + sw) * a.n_chains + ic;
            a.sU[row] = U;
            a.sL[row] = L;
            a.sA[row] = make_uint2(acc, accv);
            if (a.sW) {
                a.sW[row] = Ws;
                a.sH[row] = Hs;
            }
        }
    }

    if (act && g == 0) {
        atomicAdd(&sc.wall, n_wall);
        atomicAdd(&sc.core, n_core);
    }
    atomicAdd(&sc.terms, n_terms);
    __syncthreads();
    if (tid == 0) {
        DevState &o = a.states[ic];
        o.L = L;
        o.U = U;
        o.sweep = sweep;
        o.cnt[0] += (uint64_t)a.n_sweeps * c.N;
        o.cnt[1] += acc_total;
        o.cnt[2] += sc.wall;
        o.cnt[3] += sc.core;
        o.cnt[4] += sc.terms;
        o.cnt[5] += n_vt;
        o.cnt[6] += n_av;
        o.cnt[7] += n_rc;
        o.max_drift = mdrift;
    }
    double *xw = a.x + ch.x_off;
    for (uint32_t t = g; t < size; t += G) xw[start + t] = c.R[a0 + t];
}

// The layout of a chain: lanes per block by the block count (coop_lanes), and
// with few of them two partners per lane at once, so that one pass over the
// partners is the usual case.
template <typename Real, int KIND>
__device__ __forceinline__ void run_coop_kind(const SweepArgs &a, uint32_t ic, double *smem, CoopScratch &sc,
                                              uint32_t soff, uint32_t lanes, uint32_t w)
{
    if (lanes == 16) run_coop<Real, KIND, 16, 1>(a, ic, smem, sc, soff);
    else if (KIND != POT_HRSW && w > 2 && lanes == 4) run_coop<Real, KIND, 4, 2>(a, ic, smem, sc, soff);
    else if (lanes == 4) run_coop<Real, KIND, 4, 1>(a, ic, smem, sc, soff);
    else run_coop<Real, KIND, 2, 2>(a, ic, smem, sc, soff);
}

template <typename Real>
__global__ void __launch_bounds__(COOP_T) k_sweep_coop(SweepArgs a)
{
    extern __shared__ __align__(16) double smem[];
    __shared__ CoopScratch sc;
    const uint32_t soff = a.ctrl->sample_off;
    const uint32_t ic = a.plain_list[blockIdx.x];
    const DevChain &ch = a.chains[ic];
    const uint32_t lanes = coop_lanes(ch.B);
    switch (ch.kind) {
    case POT_LJ:
        run_coop_kind<Real, POT_LJ>(a, ic, smem, sc, soff, lanes, ch.w);
        break;
    case POT_HARMONIC:
        run_coop_kind<Real, POT_HARMONIC>(a, ic, smem, sc, soff, lanes, ch.w);
        break;
    case POT_HRSW:
        run_coop_kind<Real, POT_HRSW>(a, ic, smem, sc, soff, lanes, ch.w);
        break;
    default:
        run_coop_kind<Real, POT_YUKAWA>(a, ic, smem, sc, soff, lanes, ch.w);
        break;
    }
}

// ---------------------------------------------------------- segmented chains

// Synchronisation between the workgroups (segments) of one chain.  A
// workgroup barrier brings every wave's boundary stores to the CU's L2;
// thread 0 then fences at agent scope (one write-back of that L2 per
// workgroup, where a fence in every wave cost one per wave) and advances the
// segment's counter.  A waiter polls its partners' counters with agent-scope
// loads and, once all have arrived, fences once before the workgroup reads
// what they published.  Every wait is bounded: after 2^22
// polls the error flag is set and all later waits return at once, so the
// grid drains in bounded time and the host reports the error.
__device__ __forceinline__ void seg_signal(unsigned long long *ctr, unsigned long long v)
{
    __threadfence();
    __hip_atomic_store(ctr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __noinline__ void seg_wait(const unsigned long long *ctr, unsigned long long target,
                                      uint32_t *err)
{
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    for (uint32_t it = 0; it < (1u << 22); ++it) {
        if (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= target) return;
        __builtin_amdgcn_s_sleep(2);
    }
    __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double seg_load(const double *p)
{
    const unsigned long long v =
        __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __longlong_as_double((long long)v);
}

// Slot of a segment's partial sum: [segment][sweep parity][field][wave].
__device__ __forceinline__ uint64_t seg_pidx(uint32_t j, uint32_t par, uint32_t f, uint32_t wv)
{
    return (((uint64_t)j * 2 + par) * SEG_FIELDS + f) * SEG_WAVES + wv;
}

// The sums' scratch of a segment's workgroup.  The image of a segment leaves
// 512 bytes of the LDS (the splitting threshold); one for the four potentials.
template <int TW>
struct SegScratch {
    double rd[(TW / 64) * 3];
    double tot[SEG_FIELDS];
    uint32_t ri[(TW / 64) * 4];
};
static_assert(sizeof(SegScratch<256>) <= 512 && sizeof(SegScratch<512>) <= 512, "LDS left to a segment's image");

// One segment of a chain: blocks s*Bs .. s*Bs+Bs-1, one lane each, in LDS
// with halos of wg positions on either side that hold the neighbouring
// segments' boundary particles (periodic images at the chain's ends, as the
// single-workgroup layout's ghosts).  The trials, the random numbers, the
// per-lane sums and the order in which the sums are combined are those of
// run_bundle_lds, so a split chain produces the same bits as a whole one.
//
// Neighbour syncs every K = qb - wg phases (qb the smaller block size): in
// phase t the last block of a segment reads the right neighbour's first-block
// particles m <= t + wg - size, updated in phases before the previous sync,
// and the first block reads the left neighbour's last-block particles
// p >= size - wg + t, which the neighbour (at most K phases ahead) has not
// updated yet in this sweep.  So between two syncs every halo value read is
// the one the sequential schedule reads.
//
// LPB = 2 gives every block two lanes (adjacent; the even lane owns the
// block's state): they share each displacement trial, one walking the left
// partners and one the right (trial_lds with PAIR), which halves the walk a
// lane does and doubles the waves per CU when LDS limits the workgroups.
// The box-length sums of a block are cut in two halves (half_of), one lane
// each.  Everything else (loads, stores, the recompute sums) is the
// even lane's, and the sums are combined per 64 blocks as with one lane per
// block, so LPB changes no result bit.  Sync points, the same in every
// segment of a chain: the initial publication (neighbours); phases
// K-1, 2K-1, ... and the last phase (neighbours); every sweep's partial sums
// (all segments); a box-length acceptance (neighbours); a recompute (all);
// the final counters (all).  Partial sums are double-buffered by sweep
// parity: a segment is at most one all-segment point ahead of another.
template <typename Real, int KIND, int TW, int LPB>
__device__ __forceinline__ void run_segment(const SegArgs &g, const DevSeg &sg, double *smem,
                            SegScratch<TW> &sc, uint32_t soff)
{
    const SweepArgs &a = g.a;
    const uint32_t tid = threadIdx.x;
    const uint32_t ic = sg.chain, S = sg.S, s = sg.s, Bs = sg.Bs;
    const uint32_t me = sg.first + s;
    const DevChain &ch = a.chains[ic];
    const Pot q = ch.pot;
    const double gmin = ch.gmin, max_step = ch.max_step;
    const double beta = ch.beta, P = ch.P;
    const float betaf = ch.betaf;
    const uint32_t key0 = (uint32_t)ch.seed, key1 = (uint32_t)(ch.seed >> 32);
    const uint32_t chain_id = ch.chain_id, eci = ch.eci;
    const uint64_t log_off = ch.log_off;
    const bool per = (ch.flags & F_PERIODIC) != 0, npt = (ch.flags & F_NPT) != 0;
    const uint32_t N = ch.N, w = ch.w, wg = ch.wg, Sp = ch.Sp, smax = ch.smax;
    const uint32_t qb = N / ch.B, rem = N % ch.B;
    const bool hasLn = per || s > 0, hasRn = per || s + 1 < S;
    const uint32_t ln = sg.first + (s + S - 1) % S, rn = sg.first + (s + 1) % S;
    const uint32_t W = g.wgmax;
    const uint32_t K = qb > wg ? qb - wg : 1u;
    const uint32_t nwv = Bs >= 64 ? Bs / 64 : 1u;  // 64-block totals per segment and field

    LdsChain c;
    c.R = smem;
    c.N = N;
    c.B = Bs;
    c.w = w;
    c.wg = wg;
    c.Sp = Sp;
    c.qb = qb;
    c.rem = rem;
    c.per = per;

    const uint32_t r = LPB == 2 ? tid >> 1 : tid;
    const uint32_t side = LPB == 2 ? (tid & 1u) : 0u;
    const bool own = side == 0;  // the lane that owns the block's state
    const bool act = r < Bs;
    const uint32_t b = s * Bs + r;
    const uint32_t size = act ? qb + (b < rem ? 1u : 0u) : 0u;
    const uint32_t start = act ? b * qb + (b < rem ? b : rem) : 0u;
    const uint32_t a0 = wg + r * Sp;
    const uint32_t gapR = Sp - size;
    const uint32_t gapL = (r == 0 || !act) ? 0u : Sp - (qb + (b - 1 < rem ? 1u : 0u));
    const uint32_t seg = act ? Bs * LPB : 1u;
    // the segment's last block
    const uint32_t bl = s * Bs + Bs - 1;
    const uint32_t size_last = qb + (bl < rem ? 1u : 0u);
    const uint32_t a0_last = wg + (Bs - 1) * Sp;

    const double *xg = a.x + ch.x_off;
    if (own)
        for (uint32_t t = 0; t < size; ++t) c.R[a0 + t] = xg[start + t];
    const DevState st = a.states[ic];
    double L = st.L, U = st.U, mdrift = st.max_drift;
    uint64_t sweep = st.sweep;
    unsigned long long sp = __hip_atomic_load(&g.ctr[me], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();

    auto publish_all = [&]() {
        for (uint32_t m = tid; m < wg; m += TW) {
            g.pub_head[(uint64_t)me * W + m] = c.R[wg + m];
            g.pub_tail[(uint64_t)me * W + m] = c.R[a0_last + size_last - wg + m];
        }
    };
    auto refresh = [&]() {
        for (uint32_t m = tid; m < wg; m += TW) {
            if (hasLn) {
                const double v = seg_load(&g.pub_tail[(uint64_t)ln * W + m]);
                c.R[m] = (per && s == 0) ? v - L : v;
            }
            if (hasRn) {
                const double v = seg_load(&g.pub_head[(uint64_t)rn * W + m]);
                c.R[wg + Bs * Sp + m] = (per && s + 1 == S) ? v + L : v;
            }
        }
        __syncthreads();
    };
    auto sync_nb = [&]() {
        ++sp;
        __syncthreads();
        if (tid == 0) {
            seg_signal(&g.ctr[me], sp);
            if (hasLn) seg_wait(&g.ctr[ln], sp, g.err);
            if (hasRn) seg_wait(&g.ctr[rn], sp, g.err);
            __threadfence();
        }
        __syncthreads();
    };
    auto sync_all = [&]() {
        ++sp;
        __syncthreads();
        if (tid == 0) {
            seg_signal(&g.ctr[me], sp);
            for (uint32_t j = 0; j < S; ++j)
                if (j != s) seg_wait(&g.ctr[sg.first + j], sp, g.err);
            __threadfence();
        }
        __syncthreads();
    };
    // this segment's totals per 64 blocks of slot m of the last nd-wide
    // seg_allreduce (thread 0): wave totals, or pairs of them with two lanes
    // per block (the top level of the 64-block tree)
    auto put = [&](uint32_t par, uint32_t f, uint32_t m, uint32_t nd) {
        for (uint32_t wv = 0; wv < nwv; ++wv)
            g.part[seg_pidx(me, par, f, wv)] =
                (LPB == 2 && Bs >= 64) ? sc.rd[(2 * wv) * nd + m] + sc.rd[(2 * wv + 1) * nd + m]
                                       : sc.rd[wv * nd + m];
    };
    // Field f summed over the chain's blocks in the order of seg_allreduce
    // over B = S*Bs lanes: pairwise trees within 64-lane groups, the group
    // totals then added in sequence from zero (no sequence when B <= 64).
    // Every segment reads the same values in the same order: the same bits.
    double *tot = sc.tot;
    auto gather = [&](uint32_t par, uint32_t f) {
        if (tid < 64) {
            double acc = 0.0;
            if (Bs >= 64) {
                if (tid == 0)
                    for (uint32_t j = 0; j < S; ++j)
                        for (uint32_t wv = 0; wv < nwv; ++wv)
                            acc += seg_load(&g.part[seg_pidx(sg.first + j, par, f, wv)]);
            } else {
                const uint32_t Bt = S * Bs;
                const uint32_t gs = Bt <= 64 ? S : 64u / Bs;  // segment totals per group
                const uint32_t ng = Bt <= 64 ? 1u : Bt / 64u;
                for (uint32_t k = 0; k < ng; ++k) {
                    double v = tid < gs ? seg_load(&g.part[seg_pidx(sg.first + k * gs + tid, par, f, 0)]) : 0.0;
#pragma unroll
                    for (uint32_t off = 1; off < 64; off <<= 1) {
                        const double p = __shfl_xor(v, (int)off);
                        if (off < gs) v += p;
                    }
                    acc = Bt <= 64 ? v : acc + v;
                }
            }
            if (tid == 0) tot[f] = acc;
        }
        __syncthreads();
    };
    // integer totals (exact in double), any order
    auto gather_int = [&](uint32_t par, uint32_t f, uint32_t wv) {
        if (tid == 0) {
            double v = 0.0;
            for (uint32_t j = 0; j < S; ++j) v += seg_load(&g.part[seg_pidx(sg.first + j, par, f, wv)]);
            tot[f] = v;
        }
        __syncthreads();
    };

    // no partner beyond a wall: NaN is inside no cutoff (walk_side32)
    for (uint32_t m = tid; m < wg; m += TW) {
        if (!hasLn) c.R[m] = __longlong_as_double(0x7ff8000000000000ll);
        if (!hasRn) c.R[wg + Bs * Sp + m] = __longlong_as_double(0x7ff8000000000000ll);
    }
    publish_all();
    sync_nb();
    refresh();

    uint32_t n_tr = 0, n_wall = 0, n_core = 0, n_terms = 0;
    uint32_t acc_total = 0, n_vt = 0, n_av = 0, n_rc = 0;

#pragma unroll 1
    for (uint32_t sw = 0; sw < a.n_sweeps; ++sw, ++sweep) {
        double dUs = 0.0;
        uint32_t acc = 0;
        uint32_t w_md = 0, w_u = 0, w_next_md = 0, w_next_u = 0;
#pragma unroll 1
        for (uint32_t t = 0; t < smax; ++t) {
            if (t < size) {
                const uint32_t i = start + t;
                const uint32_t my = a0 + t;
                if ((t & 1u) == 0) {
                    uint32_t rr[4];
                    philox4x32_10(i, (uint32_t)sweep, chain_id, 0u, key0, key1, rr);
                    w_md = rr[0];
                    w_u = rr[1];
                    w_next_md = rr[2];
                    w_next_u = rr[3];
                } else {
                    w_md = w_next_md;
                    w_u = w_next_u;
                }
                const double a1 = u32o(w_md);
                const double u = u32o(w_u);
                const double md = ((a1 - 0.5) * 2.0) * max_step;
                const double xi = c.R[my];
                const double xn = xi + md;
                ++n_tr;
                double dE = 0.0;
                // one lane per block, FP32: two partners per side per walk
                // step, as the whole-chain kernel (the same sums, bit for bit)
                const bool accd = trial_lds<Real, KIND, LPB == 2, LPB == 1 && sizeof(Real) == 4>(
                    c, q, gmin, beta, betaf, i, t, size, my, gapL, gapR, L, xi, xn, md, u, dE, n_terms, n_wall,
                    n_core, side);
                if (own) {
                    const double xs = accd ? xn : xi;
                    c.R[my] = xs;
                    dUs += accd ? dE : 0.0;
                    acc += accd ? 1u : 0u;
                    if (a.acclog) a.acclog[log_off + (uint64_t)(soff + sw) * N + i] = accd ? 1 : 0;
                    // boundary particles the neighbouring segments read
                    if (r == 0 && t < wg) g.pub_head[(uint64_t)me * W + t] = xs;
                    if (r + 1 == Bs && t + wg >= size) g.pub_tail[(uint64_t)me * W + (t + wg - size)] = xs;
                }
            }
            if ((t + 1) % K == 0 || t + 1 == smax) {
                sync_nb();
                refresh();
            } else {
                __syncthreads();
            }
        }

        // box-length trial: per-lane sums over the pairs whose left member
        // is in the lane's block, across segment boundaries through the halo
        VolProp vp{};
        uint32_t bad = 0;
        double vpart = 0.0, upart = 0.0;
        if (npt) {
            vp = vol_propose<sizeof(Real) == 4 && KIND == POT_LJ>(ch, L, sweep);
            const bool last = per && r + 1 == Bs && s + 1 == S, von = vp.valid && act;
            auto wrap = [&](uint32_t m) { return seg_load(&g.pub_head[(uint64_t)sg.first * W + m]); };
            const uint32_t h = half_of(size);
            uint32_t t0 = own ? 0u : h, t1 = own ? h : size;
            const bool two = LPB == 1 && __any(h < size);
#pragma unroll 1
            for (int part = 0; part < (two ? 2 : 1); ++part) {
                double u = 0.0;
                vpart += vol_lane<Real, KIND, sizeof(Real) == 4>(c, q, gmin, vp, von, start, size, t0, t1, a0, gapR,
                                                                 last, wrap, bad, u);
                upart += u;
                t0 = t1;
                t1 = size;
            }
            if (LPB == 2) {
                // the two lanes' halves, on the lane that owns the block
                const double v2 = __shfl_xor(vpart, 1), u2 = __shfl_xor(upart, 1);
                vpart = own ? vpart + v2 : 0.0;
                upart = own ? upart + u2 : 0.0;
            }
        }
        const uint32_t par = (uint32_t)(sweep & 1u);
        {
            double v[3] = {dUs, vpart, upart};
            uint32_t k2[2] = {acc, bad};
            seg_allreduce<TW, 3, 2>(v, k2, seg, 0u, sc.rd, sc.ri);
            if (tid == 0) {
                put(par, 0, 0, 3);
                put(par, 1, 1, 3);
                put(par, 8, 2, 3);
                g.part[seg_pidx(me, par, 2, 0)] = (double)k2[0];
                g.part[seg_pidx(me, par, 3, 0)] = (double)k2[1];
            }
        }
        sync_all();
        gather(par, 0);
        gather(par, 1);
        gather(par, 8);
        gather_int(par, 2, 0);
        gather_int(par, 3, 0);
        U = U + tot[0];
        // FP32 form: the configuration's FP32 energy from the box-length
        // pass replaces the running sum (as in the whole-chain kernel);
        // square well: the pass gave the scaled energy
        if (sizeof(Real) == 4 && KIND != POT_HRSW && npt && vp.valid && tot[3] == 0.0) U = tot[8];
        acc = (uint32_t)tot[2];
        acc_total += acc;
        uint32_t accv = 0;
        if (npt) {
            ++n_vt;
            const double dUv = (sizeof(Real) == 4 && KIND == POT_HRSW) ? tot[1] - U : tot[1];
            if (vp.valid && tot[3] == 0.0 && vol_accept(dUv, vp.dL, vp.lns, P, beta, vp.jac, vp.u)) {
                // the blocks' image as one array (its pads hold nothing)
                for (uint32_t m = tid; m < Bs * Sp; m += TW) c.R[wg + m] = c.R[wg + m] * vp.sc;
                L = vp.Lp;
                U = U + dUv;
                accv = 1;
                ++n_av;
                __syncthreads();
                publish_all();
                sync_nb();
                refresh();
            }
        }

        // drift guard (ECheck, src/jmmMCState.cpp:1965-2095), always FP64
        if (eci && ((sweep + 1) % eci == 0)) {
            double Up = 0.0;
            if (act && own) {
                for (uint32_t t = 0; t < size; ++t) {
                    const uint32_t i = start + t;
                    const uint32_t my = a0 + t;
                    const double xi = c.R[my];
                    const uint32_t kR = per ? w : min(w, N - 1 - i);
                    for (uint32_t k = 1; k <= kR; ++k) {
                        const double d = c.R[my + k + (t + k >= size ? gapR : 0)] - xi;
                        if (d > q.rc) break;
                        Up += phi64<KIND>(q, d);
                    }
                }
            }
            double v[1] = {Up};
            uint32_t k1[1] = {0};
            seg_allreduce<TW, 1, 1>(v, k1, seg, 0u, sc.rd, sc.ri);
            if (tid == 0) put(par, 4, 0, 1);
            sync_all();
            gather(par, 4);
            const double dr = fabs(tot[4] - U);
            if (dr > mdrift) mdrift = dr;
            U = tot[4];
            ++n_rc;
        }

        double Ws = 0.0, Hs = 0.0;
        if (a.sW) {
            double v[2] = {0.0, 0.0};
            if (act && own) virial_lane<KIND>(c, q, start, size, a0, gapR, v[0], v[1]);
            uint32_t k1[1] = {0};
            seg_allreduce<TW, 2, 1>(v, k1, seg, 0u, sc.rd, sc.ri);
            if (tid == 0) {
                put(par, 6, 0, 2);
                put(par, 7, 1, 2);
            }
            sync_all();
            gather(par, 6);
            gather(par, 7);
            Ws = tot[6];
            Hs = tot[7];
        }
        if (s == 0 && tid == 0) {
            const uint64_t row = (uint64_t)(soff + sw) * a.n_chains + ic;
            a.sU[row] = U;
            a.sL[row] = L;
            a.sA[row] = make_uint2(acc, accv);
            if (a.sW) {
                a.sW[row] = Ws;
                a.sH[row] = Hs;
            }
        }
    }

    // counters: segment totals, summed by segment 0, which alone writes the
    // chain's state
    {
        double vz[1] = {0.0};
        uint32_t k4[4] = {own ? n_tr : 0u, own ? n_wall : 0u, own ? n_core : 0u, n_terms};
        seg_allreduce<TW, 1, 4>(vz, k4, seg, 0u, sc.rd, sc.ri);
        const uint32_t par = (uint32_t)(sweep & 1u);
        if (tid == 0)
            for (uint32_t m = 0; m < 4; ++m) g.part[seg_pidx(me, par, 5, m)] = (double)k4[m];
        sync_all();
        if (s == 0 && tid == 0) {
            uint64_t tt[4];
            for (uint32_t m = 0; m < 4; ++m) {
                double v = 0.0;
                for (uint32_t j = 0; j < S; ++j) v += seg_load(&g.part[seg_pidx(sg.first + j, par, 5, m)]);
                tt[m] = (uint64_t)v;
            }
            DevState &o = a.states[ic];
            o.L = L;
            o.U = U;
            o.sweep = sweep;
            o.cnt[0] += tt[0];
            o.cnt[1] += acc_total;
            o.cnt[2] += tt[1];
            o.cnt[3] += tt[2];
            o.cnt[4] += tt[3];
            o.cnt[5] += n_vt;
            o.cnt[6] += n_av;
            o.cnt[7] += n_rc;
            o.max_drift = mdrift;
        }
    }
    double *xw = a.x + ch.x_off;
    if (own)
        for (uint32_t t = 0; t < size; ++t) xw[start + t] = c.R[a0 + t];
}

template <typename Real, int TW, int LPB>
__global__ void __launch_bounds__(TW) __attribute__((amdgpu_waves_per_eu(1)))
k_sweep_seg(SegArgs g)
{
    extern __shared__ double smem[];
    __shared__ SegScratch<TW> sc;
    const uint32_t soff = g.a.ctrl->sample_off;
    const DevSeg sg = g.segs[blockIdx.x];
    switch (g.a.chains[sg.chain].kind) {
    case POT_LJ: run_segment<Real, POT_LJ, TW, LPB>(g, sg, smem, sc, soff); break;
    case POT_HARMONIC: run_segment<Real, POT_HARMONIC, TW, LPB>(g, sg, smem, sc, soff); break;
    case POT_HRSW: run_segment<Real, POT_HRSW, TW, LPB>(g, sg, smem, sc, soff); break;
    default: run_segment<Real, POT_YUKAWA, TW, LPB>(g, sg, smem, sc, soff); break;
    }
}

// --------------------------------------------------------------- plain form

template <int KIND, bool GX>
__device__ void run_plain(const SweepArgs &a, uint32_t ic, double *smem, uint32_t soff)
{
    const uint32_t lane = threadIdx.x;
    const DevChain &ch = a.chains[ic];
    const Pot q = ch.pot;
    const int64_t N = ch.N;
    const uint32_t w = ch.w, B = ch.B, smax = ch.smax;
    const bool per = (ch.flags & F_PERIODIC) != 0;
    const bool npt = (ch.flags & F_NPT) != 0;
    const double beta = ch.beta, gmin = ch.gmin, max_step = ch.max_step;
    const uint32_t key0 = (uint32_t)ch.seed, key1 = (uint32_t)(ch.seed >> 32);
    const uint64_t log_off = ch.log_off;
    const double P = ch.P;
    const uint32_t eci = ch.eci;
    const uint32_t chain_id = ch.chain_id;
    double *X;
    if (GX) {
        X = a.x + ch.x_off;
    } else {
        for (uint32_t k = lane; k < (uint32_t)N; k += 64) smem[k] = a.x[ch.x_off + k];
        X = smem;
    }
    __syncthreads();
    const DevState st = a.states[ic];
    double L = st.L, U = st.U, mdrift = st.max_drift;
    uint64_t sweep = st.sweep;
    const uint32_t qb = (uint32_t)N / B, rem = (uint32_t)N % B;
    const uint32_t side = lane >> 5, kk = (lane & 31) + 1;
    uint64_t n_tr = 0, n_wall = 0, n_core = 0, n_terms = 0, acc_total = 0;
    uint32_t n_vt = 0, n_av = 0, n_rc = 0;

    for (uint32_t sw = 0; sw < a.n_sweeps; ++sw, ++sweep) {
        double dUs = 0.0;
        uint32_t acc = 0;
        for (uint32_t t = 0; t < smax; ++t) {
            for (uint32_t b = 0; b < B; ++b) {
                const uint32_t size = qb + (b < rem ? 1u : 0u);
                if (t >= size) continue;
                const uint32_t i = b * qb + (b < rem ? b : rem) + t;
                uint32_t rr[4];
                philox4x32_10(i - (t & 1u), (uint32_t)sweep, chain_id, 0u, key0, key1, rr);
                const double a1 = u32o((t & 1u) ? rr[2] : rr[0]);
                const double u = u32o((t & 1u) ? rr[3] : rr[1]);
                const double md = ((a1 - 0.5) * 2.0) * max_step;
                const double xi = X[i];
                const double xn = xi + md;
                ++n_tr;
                bool ok = true;
                if (!per && fabs(xn) > L / 2.0) {
                    ok = false;
                    ++n_wall;
                } else if (N >= 2) {
                    double xl, xr;
                    if ((nbpos(X, (int64_t)i - 1, N, per, L, xl) && (xn - xl) < gmin) ||
                        (nbpos(X, (int64_t)i + 1, N, per, L, xr) && (xr - xn) < gmin)) {
                        ok = false;
                        ++n_core;
                    }
                }
                bool accd = false;
                if (ok) {
                    double term = 0.0;
                    uint32_t tm = 0;
                    for (uint32_t base = 0; base < w; base += 32) {
                        const uint32_t k = base + kk;
                        if (k <= w) {
                            const int64_t j = side ? (int64_t)i + k : (int64_t)i - k;
                            double xj;
                            if (nbpos(X, j, N, per, L, xj)) {
                                const double dold = side ? xj - xi : xi - xj;
                                const double dnew = side ? xj - xn : xn - xj;
                                if (!(dold > q.rc && dnew > q.rc)) {
                                    term += phi64<KIND>(q, dnew) - phi64<KIND>(q, dold);
                                    tm += n_inside<KIND>(q, dold, dnew);
                                }
                            }
                        }
                    }
                    const double dE = wave_sum(term);
                    n_terms += wave_sum(tm);
                    accd = dE <= 0.0 || exp(-dE * beta) > u;
                    if (accd) {
                        if (lane == 0) X[i] = xn;
                        dUs += dE;
                        ++acc;
                    }
                    __syncthreads();
                }
                if (a.acclog && lane == 0)
                    a.acclog[log_off + (uint64_t)(soff + sw) * N + i] = accd ? 1 : 0;
            }
        }
        U = U + dUs;
        acc_total += acc;

        uint32_t accv = 0;
        if (npt) {
            ++n_vt;
            const VolProp vp = vol_propose<false>(ch, L, sweep);
            if (vp.valid) {
                uint32_t bad = 0;
                double u0;
                double part = scaled_delta<double, KIND>(q, vp.bk, gmin, X, N, per, L, vp.Lp, vp.sc, w,
                                                         lane, (uint32_t)N, 64, bad, u0);
                part = wave_sum(part);
                bad = wave_sum(bad);
                if (!bad && vol_accept(part, vp.dL, vp.lns, P, beta, vp.jac, vp.u)) {
                    __syncthreads();
                    for (uint32_t p = lane; p < (uint32_t)N; p += 64) X[p] = X[p] * vp.sc;
                    L = vp.Lp;
                    U = U + part;
                    accv = 1;
                    ++n_av;
                }
                __syncthreads();
            }
        }
        if (eci && ((sweep + 1) % eci == 0)) {
            const double Uf = wave_sum(energy_part<KIND>(q, X, N, per, L, w, lane, (uint32_t)N, 64));
            const double dr = fabs(Uf - U);
            if (dr > mdrift) mdrift = dr;
            U = Uf;
            ++n_rc;
        }
        double Ws = 0.0, Hs = 0.0;
        if (a.sW) {
            virial_part<KIND>(q, X, N, per, L, w, lane, (uint32_t)N, 64, Ws, Hs);
            Ws = wave_sum(Ws);
            Hs = wave_sum(Hs);
        }
        if (lane == 0) {
            const uint64_t row = (uint64_t)(soff + sw) * a.n_chains + ic;
            a.sU[row] = U;
            a.sL[row] = L;
            a.sA[row] = make_uint2(acc, accv);
            if (a.sW) {
                a.sW[row] = Ws;
                a.sH[row] = Hs;
            }
        }
    }
    if (lane == 0) {
        DevState &o = a.states[ic];
        o.L = L;
        o.U = U;
        o.sweep = sweep;
        o.cnt[0] += n_tr;
        o.cnt[1] += acc_total;
        o.cnt[2] += n_wall;
        o.cnt[3] += n_core;
        o.cnt[4] += n_terms;
        o.cnt[5] += n_vt;
        o.cnt[6] += n_av;
        o.cnt[7] += n_rc;
        o.max_drift = mdrift;
    }
    __syncthreads();
    if (!GX)
        for (uint32_t k = lane; k < (uint32_t)N; k += 64) a.x[ch.x_off + k] = smem[k];
}

template <bool GX>
__global__ void __launch_bounds__(64) k_sweep_plain(SweepArgs a)
{
    extern __shared__ double smem[];
    const uint32_t soff = a.ctrl->sample_off;
    const uint32_t ic = a.plain_list[blockIdx.x];
    switch (a.chains[ic].kind) {
    case POT_LJ: run_plain<POT_LJ, GX>(a, ic, smem, soff); break;
    case POT_HARMONIC: run_plain<POT_HARMONIC, GX>(a, ic, smem, soff); break;
    case POT_HRSW: run_plain<POT_HRSW, GX>(a, ic, smem, soff); break;
    default: run_plain<POT_YUKAWA, GX>(a, ic, smem, soff); break;
    }
}

__global__ void k_begin(Ctrl *c, uint32_t n)
{
    c->queue = 0;
    c->sample_off = c->next_off;
    c->next_off = c->next_off + n;
}

// ------------------------------------------------------- differentiation

// pair_obs and the force over distance f = o[1] / d of one pair.  rsig = 1 / p1
// (LJ's sigma, as the FP32 form rounds it).  The FP32 LJ and Yukawa pairs hold
// four and two divisions, half of their instructions.  A quotient of two FP32
// numbers lies at least 2^-49 of itself from the middle of two neighbours, so
// a product in FP64 with a reciprocal good to a few 2^-53 rounds to the same
// FP32 number as the division: FP32 estimates, each with two Newton steps in
// FP64, give the same bits.  Two more steps from 1 / (float)d lead to 1 / d to
// the last bits of FP64.  Outside (1e-4, 1e4), where d^6 or its reciprocal
// could leave the estimate's range, for the other potentials and for FP64: the
// divisions.
template <int KIND, typename R>
__device__ __forceinline__ void pair_obs_f(const Pot &q, double rsig, double d, const R sh[3], R o[6], double &f)
{
    if constexpr (sizeof(R) == 4 && (KIND == POT_LJ || KIND == POT_YUKAWA)) {
        if (d > 1e-4 && d < 1e4) {
            const float x = (float)d;
            double r = (double)frcp(x);
            if constexpr (KIND == POT_LJ) {
                const float d3 = x * x * x, d6 = d3 * d3;
                double r6 = (double)frcp(d6);
                r6 = fma(fma(-(double)d6, r6, 1.0), r6, r6);
                r6 = fma(fma(-(double)d6, r6, 1.0), r6, r6);
                const float i6 = (float)r6 * q.sig6f, i12 = i6 * i6;
                const float a12 = q.e4f * i12, a6 = q.e4f * i6;
                o[0] = (a12 - a6) - sh[0];
                o[1] = 12.0f * a12 - 6.0f * a6;
                o[2] = (4.0f * i12 - 4.0f * i6) - sh[1];
                o[3] = (float)((double)o[1] * rsig) - sh[2];
                o[4] = 12.0f * (4.0f * i12) - 6.0f * (4.0f * i6);
                o[5] = (float)((double)(144.0f * a12 - 36.0f * a6) * rsig);
            } else {
                r = fma(fma(-(double)x, r, 1.0), r, r);
                r = fma(fma(-(double)x, r, 1.0), r, r);
                const float e = expf(-q.p1f * x);
                const float ed = (float)((double)e * r);
                const float E = q.p0f * ed;
                o[0] = E - sh[0];
                o[1] = E * (q.p1f * x + 1.0f);
                o[2] = ed - sh[1];
                o[3] = -q.p0f * e - sh[2];
                o[4] = ed * (q.p1f * x + 1.0f);
                o[5] = -q.p1f * x * x * E;
            }
            r = fma(fma(-d, r, 1.0), r, r);
            r = fma(fma(-d, r, 1.0), r, r);
            f = (double)o[1] * r;
            return;
        }
    }
    pair_obs<KIND, R>(q, R(d), sh, o);
    f = (double)o[1] / d;
}

// Waves of a tile.
constexpr uint32_t OBS_WAVES = OBS_TILE / 64;
static_assert(OBS_ONE <= 2 * OBS_TILE, "k_obs_sum adds two tiles as v0 + v1");

// LDS of the observables kernel: the waves' sums, forces handed to the next
// wave, and the edge's forces by wave.
struct ObsScratch {
    double red[16 * 6], next[16 * 64], edge[16 * 64];
};

// U, W and their parameter derivatives of one tile of a configuration
// (particles [p0, p1): the pairs whose left member is in the tile) and dU/dx
// of the tile's particles.  Pair arithmetic in Real, sums in FP64.
// out = (U, W, dU/dtheta0, dU/dtheta1, dW/dtheta0, dW/dtheta1) of the tile.
//
// Bound by vector issue (every SIMD's issue slots are taken on the 20 sigma
// Yukawa chains at density 0.8): about 16 pairs a side, each some 90
// instructions, against 16 bytes of memory per particle.  Two things matter:
// that every SIMD has waves to issue from (a particle per lane and tiles of
// OBS_TILE over the chip: one workgroup each left 64 configurations of 65,536
// on 64 of the 256 CUs with one wave per SIMD, 3.67 ms), and that each pair is
// evaluated once.  A lane walks its right-hand partners; the partner at index
// distance k gets the pair's force by a shift of the wave's lanes by k (in the
// wave, or its next one by an LDS row at the end: no barrier in the walk).
// Only pairs that cross the tile's left edge, or reach beyond 64 partners, are
// evaluated again from the right; the edge's are spread over the waves by
// index distance (left to the first wave they cost as much as both walks did:
// it sits on the same SIMD in every workgroup).  The walk is uniform over the
// wave with the next position loaded ahead.
// A configuration's sums and gradients are the same bits whatever the workgroup
// (engines take it from the longest chain): waves are added up per OBS_TILE
// particles, then the tiles as k_obs_sum does; a workgroup of two tiles
// evaluates the pairs across their boundary again as two workgroups do; and an
// edge's partners are summed in as many strides as the tile's particles have
// waves, whatever the workgroup has.
// The kernel, FP32: 64 Yukawa configurations of 65,536 314 us with both sides
// walked, 244 with each pair once, 225 with the divisions of pair_obs_f and
// tiles of 512 (back to back and with k_obs_sum 212); 1024 LJ chains of 1024 28
// and 22 us.
template <typename Real, int KIND>
__device__ __forceinline__ void run_obs(const DevChain &ch, const double *X, double L, double sc, uint32_t p0,
                                        uint32_t p1, double *out, double *grad, ObsScratch &sm)
{
    double *red = sm.red, *next = sm.next, *edge = sm.edge;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, waves = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Pot q = ch.pot;
    const uint32_t N = ch.N;
    // a compressed configuration (sc < 1) may hold gaps below the hard core:
    // walk to the cutoff (or the NBN limit) without the window limit
    const uint32_t w = sc < 1.0 ? min(ch.nbn_lim, N > 0 ? N - 1 : 0u) : ch.w;
    const bool per = (ch.flags & F_PERIODIC) != 0;
    const Real sh[3] = {Real(ch.sh[0]), Real(ch.sh[1]), Real(ch.sh[2])};
    const double rsig = 1.0 / (double)q.p1f;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t t0 = p0; t0 < p1; t0 += blockDim.x) {
        const uint32_t i = t0 + tid;
        // positions of the configuration scaled by sc to length L: x_j sc,
        // periodic images x_j sc -+ L.  Lanes past the end stay on the last
        // particle (j < 2N) and are never active.
        const uint32_t ic = min(i, p1 - 1);
        const double xi = X[ic] * sc;
        bool active = i < p1;
        double g = 0.0, gl = 0.0, gn = 0.0;
        uint32_t j = ic + 1;
        double off = 0.0;
        if (j == N) {
            j = 0;
            off = L;
            active = active && per;
        }
        double xn = X[j] * sc + off;
        for (uint32_t k = 1; k <= w; ++k) {
            const double d = xn - xi;
            active = active && !(d > q.rc);
            if (!__ballot(active)) break;
            const bool in = active && inside64<KIND>(q, d);
            // a caller's rods may be longer than the well is wide
            if (KIND == POT_HRSW && active && !in && d < q.p0) acc[0] += INFINITY;
            if (++j == N) {
                j = 0;
                off = L;
                active = active && per;
            }
            xn = X[j] * sc + off;
            double f = 0.0;
            if (in) {
                Real o[6];
                pair_obs_f<KIND, Real>(q, rsig, d, sh, o, f);
                // a rescaled configuration can overlap hard cores: infinite energy
                if ((KIND == POT_HRSW && d < q.p0) || (KIND == POT_YUKAWA && d < q.p2)) {
                    acc[0] += INFINITY;
                } else {
#pragma unroll
                    for (int m = 0; m < 6; ++m) acc[m] += (double)o[m];
                    g += f;
                }
            }
            if (grad && k <= 64) {
                const int from = (int)((lane - k) & 63u) << 2;
                const double fl = __hiloint2double(__builtin_amdgcn_ds_bpermute(from, __double2hiint(f)),
                                                   __builtin_amdgcn_ds_bpermute(from, __double2loint(f)));
                if (lane >= k) gl += fl;
                else gn += fl;
            }
        }
        if (!grad) continue;
        // pairs evaluated again: the force of the left-hand partners of
        // particle m at index distances k0, k0 + step, ...
        const auto left = [&](uint32_t m, uint32_t k0, uint32_t step) {
            const double xm = X[m] * sc;
            double s = 0.0;
            for (uint32_t k = k0; k <= w; k += step) {
                double xj;
                if (k <= m) xj = X[m - k] * sc;
                else if (per) xj = X[m + N - k] * sc - L;
                else break;
                const double d = xm - xj;
                if (d > q.rc) break;
                if (!inside64<KIND>(q, d)) continue;
                Real o[6];
                double f;
                pair_obs_f<KIND, Real>(q, rsig, d, sh, o, f);
                s += f;
            }
            return s;
        };
        next[tid] = gn;
        const uint32_t first = wave / OBS_WAVES * OBS_WAVES, m = t0 + first * 64 + lane;
        // waves of the tile that hold particles (no more than the workgroup's)
        const uint32_t strides = min(OBS_WAVES, (p1 - min(p1, t0 + first * 64) + 63) / 64);
        edge[tid] = wave - first < strides && m < p1 ? left(m, lane + 1 + wave - first, strides) : 0.0;
        __syncthreads();
        if (wave != first) {
            gl += next[tid - 64];
            if (i < p1) gl += left(i, 65, 1);
        } else {
            for (uint32_t v = 0; v < strides; ++v) gl += edge[tid + v * 64];
        }
        if (i < p1) grad[i] = g - gl;
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < 6; ++m) acc[m] = wave_sum(acc[m]);
    if ((tid & 63) == 0)
        for (int m = 0; m < 6; ++m) red[(tid >> 6) * 6 + m] = acc[m];
    __syncthreads();
    // a tile's waves in order, then the tiles: a lane per field and tile
    if (tid < 12) {
        const uint32_t half = tid / 6, field = tid - half * 6;
        double v = 0.0;
#pragma unroll
        for (uint32_t wv = 0; wv < OBS_WAVES; ++wv) {
            const uint32_t from = half * OBS_WAVES + wv;
            v += from < waves ? red[from * 6 + field] : 0.0;
        }
        const double second = __shfl(v, (int)tid + 6);
        if (tid < 6) out[tid] = v + second;
    }
}

// One workgroup per tile: a.tile particles of a configuration, or the whole
// configuration (a.tiles = nullptr), whose observables then go straight to
// the caller's row; with tiles they go to a.part, and k_obs_sum adds them.
// FP32: 64 registers, so that two workgroups of 1024 share a CU (27 -> 22 us
// for 1024 chains of 1024).
template <typename Real>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(sizeof(Real) == 4 ? 8 : 4)))
k_observables(ObsArgs a)
{
    __shared__ ObsScratch sm;  // one for the four potentials
    const uint32_t group = a.group0 + blockIdx.x;
    uint32_t c, p0 = 0, part = 0;
    if (a.standalone) {
        c = group / a.parts;
        part = group % a.parts;
    } else if (a.tiles) {
        c = a.tiles[group].chain;
        part = a.tiles[group].part;
    } else {
        c = group;
    }
    const DevChain &ch = a.standalone ? a.one : a.chains[c];
    const uint32_t N = ch.N;
    p0 = part * a.tile;
    const uint32_t p1 = min(N, p0 + a.tile);
    const double *X;
    double L, *grad, *out;
    double sc = 1.0;
    if (a.standalone) {
        X = a.x + (uint64_t)c * N;
        L = a.L[c];
        grad = a.grad ? a.grad + (uint64_t)c * N : nullptr;
    } else {
        X = a.x + ch.x_off;
        L = a.states[c].L;
        if (a.Lnew) {
            sc = a.Lnew[c] / L;
            L = a.Lnew[c];
        }
        grad = a.grad ? a.grad + (a.goff ? a.goff[c] : ch.x_off) : nullptr;
    }
    if (a.part) out = a.part + (uint64_t)group * 6;
    else out = a.obs + (uint64_t)(a.row ? a.row[c] : c) * 6;
    switch (ch.kind) {
    case POT_LJ: run_obs<Real, POT_LJ>(ch, X, L, sc, p0, p1, out, grad, sm); break;
    case POT_HARMONIC: run_obs<Real, POT_HARMONIC>(ch, X, L, sc, p0, p1, out, grad, sm); break;
    case POT_HRSW: run_obs<Real, POT_HRSW>(ch, X, L, sc, p0, p1, out, grad, sm); break;
    default: run_obs<Real, POT_YUKAWA>(ch, X, L, sc, p0, p1, out, grad, sm); break;
    }
}

// Sums each configuration's tiles: lanes stride over the tiles, then a wave
// sum per field (a fixed order, the same on every call).
__global__ void __launch_bounds__(64) k_obs_sum(ObsArgs a)
{
    const uint32_t c = blockIdx.x, lane = threadIdx.x;
    const uint32_t first = a.standalone ? c * a.parts : a.first[c];
    const uint32_t n = a.standalone ? a.parts : a.first[c + 1] - first;
    double v[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t p = lane; p < n; p += 64)
        for (int m = 0; m < 6; ++m) v[m] += a.part[(uint64_t)(first + p) * 6 + m];
#pragma unroll
    for (int m = 0; m < 6; ++m) v[m] = wave_sum(v[m]);
    double *o = a.obs + (uint64_t)(a.row ? a.row[c] : c) * 6;
    if (lane == 0)
        for (int m = 0; m < 6; ++m) o[m] = v[m];
}

// Sample rows [sweep][chain] (internal chain order) to the caller's layout
// [chain][sweep] (external order), through 32 x 32 tiles in LDS so that the
// reads (along chains) and the writes (along sweeps) are both contiguous.
// Grid-stride over tiles.  Also empties the sample buffer (n_ctrl <= 256
// queues).
__global__ void __launch_bounds__(256) k_pack_samples(const double *sU, const double *sL, const uint2 *sA,
                                                      const uint32_t *ext, uint32_t nc, uint32_t ns,
                                                      SampleRec *out, Ctrl *ctrl, uint32_t n_ctrl)
{
    // the read empties the sample buffer: the queues' rows start over
    if (blockIdx.x == 0 && threadIdx.x < n_ctrl) ctrl[threadIdx.x].next_off = 0;
    __shared__ double tU[32][33], tL[32][33];
    __shared__ uint2 tA[32][33];
    const uint32_t tx = threadIdx.x & 31u, ty = threadIdx.x >> 5;
    const uint32_t tk = (nc + 31u) / 32u, ts = (ns + 31u) / 32u;
    const uint64_t tiles = (uint64_t)tk * ts;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t k0 = (uint32_t)(tile % tk) * 32u, s0 = (uint32_t)(tile / tk) * 32u;
        for (uint32_t j = ty; j < 32u; j += 8u) {
            const uint32_t sw = s0 + j, k = k0 + tx;
            if (sw < ns && k < nc) {
                const uint64_t r = (uint64_t)sw * nc + k;
                tU[j][tx] = sU[r];
                tL[j][tx] = sL[r];
                tA[j][tx] = sA[r];
            }
        }
        __syncthreads();
        for (uint32_t j = ty; j < 32u; j += 8u) {
            const uint32_t k = k0 + j, sw = s0 + tx;
            if (k < nc && sw < ns) {
                SampleRec o;
                o.U = tU[tx][j];
                o.L = tL[tx][j];
                o.acc_d = tA[tx][j].x;
                o.acc_v = tA[tx][j].y;
                out[(uint64_t)ext[k] * ns + sw] = o;
            }
        }
        __syncthreads();
    }
}

// Virial rows [sweep][chain] to out[(ext * ns + sweep) * 2 + {0, 1}], through
// 32 x 32 LDS tiles as k_pack_samples.
__global__ void __launch_bounds__(256) k_pack_virials(const double *sW, const double *sH, const uint32_t *ext,
                                                      uint32_t nc, uint32_t ns, double *out)
{
    __shared__ double tW[32][33], tH[32][33];
    const uint32_t tx = threadIdx.x & 31u, ty = threadIdx.x >> 5;
    const uint32_t tk = (nc + 31u) / 32u, ts = (ns + 31u) / 32u;
    const uint64_t tiles = (uint64_t)tk * ts;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t k0 = (uint32_t)(tile % tk) * 32u, s0 = (uint32_t)(tile / tk) * 32u;
        for (uint32_t j = ty; j < 32u; j += 8u) {
            const uint32_t sw = s0 + j, k = k0 + tx;
            if (sw < ns && k < nc) {
                const uint64_t r = (uint64_t)sw * nc + k;
                tW[j][tx] = sW[r];
                tH[j][tx] = sH[r];
            }
        }
        __syncthreads();
        for (uint32_t j = ty; j < 32u; j += 8u) {
            const uint32_t k = k0 + j, sw = s0 + tx;
            if (k < nc && sw < ns) {
                const uint64_t o = ((uint64_t)ext[k] * ns + sw) * 2;
                out[o] = tW[tx][j];
                out[o + 1] = tH[tx][j];
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ histograms

// Position folded into [-L/2, L/2) on a periodic line; unchanged with walls.
__device__ __forceinline__ double fold(double x, double L, bool per)
{
    return per ? x - L * floor((x + L / 2.0) / L) : x;
}

__device__ __forceinline__ int64_t bin_of(double x, double width, uint32_t nb)
{
    return (int64_t)floor(x / width + nb / 2.0);
}

// One sample of the reference's density and pair-separation histograms
// (fgrho, src/jmmMCState.cpp:1069-1128): rho bin floor(x/rbw + rhonb/2) of
// every particle; for every pair closer than gnb*gbw, separation bin
// floor(d/gbw) counted once in the segment floor(x/gsw + gns/2) of each
// member.  Periodic chains: positions folded into [-L/2, L/2), each pair
// once at its shorter separation (below L/2).
//
// Bound by its counting: one 64-bit atomic to memory per pair and member
// (about 48 partners within 100 sigma at density 0.48), and, with a lane
// walking all of a particle's partners, one wave per SIMD.  A workgroup takes
// a tile of up to 256 particles with 4 lanes or more on each one's partners
// (every fourth of them: sorted positions, so each lane stops by itself), and
// counts in LDS: positions are sorted, so a tile and its partners lie in a
// few neighbouring segments, and a window of segments from the tile's first
// one on holds nearly every count; the others (a folded periodic end, windows
// cut by HIST_WORDS) go to memory one by one.  Both members in one segment
// are one addition of 2.  Counters in LDS have 32 bits, which a tile cannot
// exceed for N <= HIST_N_LDS;
// larger chains count in memory.
// 32 chains of 2000, 10 segments of 1000 bins: 95 us a sample with a particle
// per lane and atomics to memory, 15.5 us so.
// Grid: a workgroup per tile of every chain (workgroups for each chain's share
// of the longest one's tiles, most of them empty, cost more than the counting:
// 512 chains of 32 beside 4 of 60,000, rho alone 7.1 us against 94).
__global__ void __launch_bounds__(HIST_T) k_hist(HistArgs a)
{
    extern __shared__ uint32_t hw[];
    const Tile at = a.tiles[a.group0 + blockIdx.x];
    const uint32_t c = at.chain, tid = threadIdx.x;
    const DevChain &ch = a.chains[c];
    const uint32_t N = ch.N;
    const uint32_t P = hist_tile(N), K = blockDim.x / P;
    const bool per = (ch.flags & F_PERIODIC) != 0;
    const double L = a.states[c].L;
    const double *X = a.x + ch.x_off;
    const double gmax = a.gnb * a.gbw;
    unsigned long long *rho = a.rho + (uint64_t)c * a.rhonb;
    unsigned long long *g = a.g + (uint64_t)c * a.gns * a.gnb;
    const uint32_t kl = tid / P;
    const uint32_t p0 = at.part * P, i = p0 + tid % P;
    // window of segments counted in LDS: from the first particle's to the
    // last one's farthest partner's, where they lie in that order
    uint32_t s0 = 0, W = 0;
    if (N <= HIST_N_LDS && a.gns && a.gnb && a.gnb <= HIST_WORDS) {
        const double f0 = fold(X[p0], L, per), f1 = fold(X[min(p0 + P, N) - 1], L, per) + gmax;
        const int64_t top = (int64_t)a.gns - 1;
        const int64_t b0 = max((int64_t)0, min(top, bin_of(f0, a.gsw, a.gns)));
        const int64_t b1 = max(b0, min(top, bin_of(f1, a.gsw, a.gns)));
        s0 = (uint32_t)b0;
        W = (uint32_t)min((int64_t)(HIST_WORDS / a.gnb), (f1 < f0 ? top : b1) - b0 + 1);
    }
    const uint32_t words = W * a.gnb;
    for (uint32_t m = tid; m < words; m += blockDim.x) hw[m] = 0;
    __syncthreads();
    if (i < N) {
        const double xi = X[i];
        const double fi = fold(xi, L, per);
        if (kl == 0) {
            const int64_t rb = bin_of(fi, a.rbw, a.rhonb);
            if (rb >= 0 && rb < (int64_t)a.rhonb) atomicAdd(&rho[rb], 1ull);
        }
        const int64_t si = bin_of(fi, a.gsw, a.gns);
        const uint32_t kmax = a.gns && a.gnb ? N : 0;
        for (uint32_t k = 1 + kl; k < kmax; k += K) {
            const uint32_t j0 = i + k;
            double d, xj;
            if (j0 < N) {
                xj = X[j0];
                d = xj - xi;
            } else {
                if (!per) break;
                xj = X[j0 - N];
                d = (xj + L) - xi;
            }
            if (!(d < gmax) || (per && !(d < L / 2.0))) break;
            const int64_t gb = (int64_t)floor(d / a.gbw);
            if (gb < 0 || gb >= (int64_t)a.gnb) continue;
            const int64_t sj = bin_of(fold(xj, L, per), a.gsw, a.gns);
            const uint64_t ri = (uint64_t)(si - (int64_t)s0), rj = (uint64_t)(sj - (int64_t)s0);
            if (ri < W) atomicAdd(&hw[(uint32_t)ri * a.gnb + (uint32_t)gb], si == sj ? 2u : 1u);
            else if (si >= 0 && si < (int64_t)a.gns)
                atomicAdd(&g[(uint64_t)si * a.gnb + gb], si == sj ? 2ull : 1ull);
            if (si == sj) continue;
            if (rj < W) atomicAdd(&hw[(uint32_t)rj * a.gnb + (uint32_t)gb], 1u);
            else if (sj >= 0 && sj < (int64_t)a.gns) atomicAdd(&g[(uint64_t)sj * a.gnb + gb], 1ull);
        }
    }
    __syncthreads();
    for (uint32_t m = tid; m < words; m += blockDim.x)
        if (const uint32_t v = hw[m]) atomicAdd(&g[(uint64_t)s0 * a.gnb + m], (unsigned long long)v);
}

// Positions of every chain scaled to a new length: x -> x Lnew/L (moveVolume,
// src/jmmMCState.cpp:2831-2916).  The length itself is set by the host.
__global__ void __launch_bounds__(256) k_rescale(const DevChain *chains, const DevState *st,
                                                 double *x, const double *Lnew, uint32_t parts)
{
    const uint32_t c = blockIdx.x / parts, part = blockIdx.x % parts;
    const DevChain &ch = chains[c];
    const double sc = Lnew[c] / st[c].L;
    double *X = x + ch.x_off;
    for (uint32_t i = part * 256 + threadIdx.x; i < ch.N; i += 256 * parts) X[i] = X[i] * sc;
}

// ------------------------------------------------------------ launchers

hipError_t launch_begin(Ctrl *c, uint32_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_begin, dim3(1), dim3(1), 0, s, c, n);
    return hipGetLastError();
}

template <typename Real>
static const void *pick_shape(int T, int gx, int waves)
{
    if (T == 1024) return gx ? (const void *)k_sweep_batched<Real, 1024, true, 2>
                             : (const void *)k_sweep_batched<Real, 1024, false, 2>;
    if (T == 512) return gx ? (const void *)k_sweep_batched<Real, 512, true, 2>
                            : (const void *)k_sweep_batched<Real, 512, false, 2>;
    if (gx) return (const void *)k_sweep_batched<Real, 256, true, 2>;
    return waves == 3 ? (const void *)k_sweep_batched<Real, 256, false, 3>
                      : (const void *)k_sweep_batched<Real, 256, false, 2>;
}

const void *batched_kernel(int fp32, int T, int gx, int waves)
{
    return fp32 ? pick_shape<float>(T, gx, waves) : pick_shape<double>(T, gx, waves);
}

hipError_t launch_batched(const SweepArgs &a, int fp32, int T, int gx, int waves, uint32_t grid, size_t lds,
                          hipStream_t s)
{
    const void *fn = batched_kernel(fp32, T, gx, waves);
    void *args[] = {(void *)&a};
    return hipLaunchKernel(fn, dim3(grid), dim3(T), args, lds, s);
}

size_t coop_lds(const DevChain &c)
{
    const size_t G = coop_lanes(c.B), T = (c.B * G + 63) / 64 * 64;
    // the image and the block sums, then the random numbers (20 bytes for each
    // of two positions a lane) or the pair terms (two fields a lane and partner)
    const size_t rnd = T * 2 * 20 + 8, terms = T * c.w * 2 * sizeof(double);
    return sizeof(double) * ((size_t)c.lds_len + 3 * c.B) + std::max(rnd, terms);
}

uint32_t coop_threads(const DevChain &c)
{
    return (c.B * coop_lanes(c.B) + 63) / 64 * 64;
}

const void *coop_kernel(int fp32)
{
    return fp32 ? (const void *)k_sweep_coop<float> : (const void *)k_sweep_coop<double>;
}

hipError_t launch_coop(const SweepArgs &a, int fp32, uint32_t grid, uint32_t threads, size_t lds, hipStream_t s)
{
    void *args[] = {(void *)&a};
    return hipLaunchKernel(coop_kernel(fp32), dim3(grid), dim3(threads), args, lds, s);
}

const void *plain_kernel(int gx)
{
    return gx ? (const void *)k_sweep_plain<true> : (const void *)k_sweep_plain<false>;
}

hipError_t launch_plain(const SweepArgs &a, int gx, uint32_t grid, size_t lds, hipStream_t s)
{
    if (gx) hipLaunchKernelGGL(k_sweep_plain<true>, dim3(grid), dim3(64), lds, s, a);
    else hipLaunchKernelGGL(k_sweep_plain<false>, dim3(grid), dim3(64), lds, s, a);
    return hipGetLastError();
}

// Launches n_groups workgroups in parts that stay below a launch's 2^32 lanes.
template <typename Args>
static void launch_groups(void (*kernel)(Args), Args a, uint32_t n_groups, uint32_t lanes, size_t lds, hipStream_t s)
{
    const uint32_t most = 0xffffffffu / lanes;
    for (a.group0 = 0; a.group0 < n_groups;) {
        const uint32_t n = std::min(n_groups - a.group0, most);
        hipLaunchKernelGGL(kernel, dim3(n), dim3(lanes), lds, s, a);
        a.group0 += n;
    }
}

hipError_t launch_observables(const ObsArgs &a, int fp32, uint32_t n_tiles, uint32_t n_configs, int threads,
                              hipStream_t s)
{
    launch_groups(fp32 ? k_observables<float> : k_observables<double>, a, n_tiles, (uint32_t)threads, 0, s);
    if (a.part) hipLaunchKernelGGL(k_obs_sum, dim3(n_configs), dim3(64), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_rescale(const DevChain *chains, const DevState *st, double *x, const double *Lnew,
                          uint32_t n_chains, uint32_t parts, hipStream_t s)
{
    hipLaunchKernelGGL(k_rescale, dim3(n_chains * parts), dim3(256), 0, s, chains, st, x, Lnew, parts);
    return hipGetLastError();
}

const void *segmented_kernel(int fp32, int tw, int lpb)
{
    if (lpb == 2 && tw == 512)
        return fp32 ? (const void *)k_sweep_seg<float, 512, 2> : (const void *)k_sweep_seg<double, 512, 2>;
    if (lpb == 2)
        return fp32 ? (const void *)k_sweep_seg<float, 256, 2> : (const void *)k_sweep_seg<double, 256, 2>;
    return fp32 ? (const void *)k_sweep_seg<float, 256, 1> : (const void *)k_sweep_seg<double, 256, 1>;
}

// An ordinary launch: the segments' synchronisation needs every workgroup
// resident at once, which jmm_create checks against the occupancy of the
// whole device (the launch follows the stream's previous work, so the
// device is free when it starts), and a wait that never completes ends
// after its bounded polls with the error flag set.  A cooperative launch
// would add only a runtime check of the same residency, and a rocprofv3
// kernel trace of a program using one ended in a segmentation fault with
// no results written.
hipError_t launch_segmented(const SegArgs &a, int fp32, int tw, int lpb, size_t lds, hipStream_t s)
{
    void *args[] = {(void *)&a};
    return hipLaunchKernel(segmented_kernel(fp32, tw, lpb), dim3(a.n_segs), dim3(tw), args, lds, s);
}

hipError_t launch_hist(const HistArgs &a, hipStream_t s)
{
    const size_t words = a.gnb <= HIST_WORDS ? std::min<uint64_t>((uint64_t)a.gns * a.gnb, HIST_WORDS) : 0;
    launch_groups(k_hist, a, a.n_tiles, a.gns && a.gnb ? HIST_T : HIST_TILE, words * sizeof(uint32_t), s);
    return hipGetLastError();
}

hipError_t launch_pack_virials(const double *sW, const double *sH, const uint32_t *ext, uint32_t n_chains,
                               uint32_t n_sweeps, double *out, hipStream_t s)
{
    const uint64_t tiles = (uint64_t)((n_chains + 31u) / 32u) * ((n_sweeps + 31u) / 32u);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(tiles, 1u << 16);
    if (!grid) return hipSuccess;
    hipLaunchKernelGGL(k_pack_virials, dim3(grid), dim3(256), 0, s, sW, sH, ext, n_chains, n_sweeps, out);
    return hipGetLastError();
}

hipError_t launch_pack_samples(const double *sU, const double *sL, const uint2 *sA, const uint32_t *ext,
                               uint32_t n_chains, uint32_t n_sweeps, SampleRec *out, Ctrl *ctrl, uint32_t n_ctrl,
                               hipStream_t s)
{
    const uint64_t tiles = (uint64_t)((n_chains + 31u) / 32u) * ((n_sweeps + 31u) / 32u);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(tiles, 1u << 16);
    if (!grid) return hipSuccess;
    hipLaunchKernelGGL(k_pack_samples, dim3(grid), dim3(256), 0, s, sU, sL, sA, ext, n_chains, n_sweeps, out, ctrl,
                       n_ctrl);
    return hipGetLastError();
}

}  // namespace jmm
