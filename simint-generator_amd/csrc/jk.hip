// Coulomb and exchange digestion of shell-quartet integrals (the consumer a
// Fock build puts after the integral kernels; the reference returns the
// integrals only).
//
// A unique shell quartet (AB|CD) stands for its images under the eight
// index permutations.  Its stabiliser has s = s_AB s_CD s_(AB)(CD) elements
// (each factor 2 when the two sides are the same shell / pair), so summing
// all eight images with weight f = 1/s counts every ordered quartet of
// functions once.  For a symmetric density the eight images collapse to
//     J'_ab += 4 f v D_cd      J'_cd += 4 f v D_ab
//     K'_ac += 2 f v D_bd      K'_ad += 2 f v D_bc
//     K'_bc += 2 f v D_ad      K'_bd += 2 f v D_ac
// and J = (J' + J'^T)/2, K = (K' + K'^T)/2 (jk_symmetrize).
//
// One wavefront digests one work item of the class launch (a bra pair
// against up to 64 kets of a tile, the same items the class kernel ran):
// each lane reads its quartet's integrals where the kernel wrote them.  The
// bra-side J sums are reduced across the wave before one atomic add per
// element; the ket-side J and the four exchange blocks are added per lane.
// The exchange blocks whose row is a bra function (K_ac, K_ad) are summed
// over b (and K_bc, K_bd over a) in registers before their atomic adds, and
// where the bra's rows fit the local data share one block takes all of a
// bra's items and sums those rows over all its kets there first
// (jk_digest_rows).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "simint/simint_eri.h"
#include "simint/simint_hip.h"
#include "device_types.h"
#include "runtime_internal.h"

namespace {

__device__ inline double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

struct JkDev {
    int nbf, same;
    const int *bra_fun, *ket_fun;
    const double *D;
    double *J, *K;
};

__global__ void __launch_bounds__(256) jk_digest(const WorkItem *items, long long nitems, const long long *col,
                                                 const double *ints, int na, int nb, int nc, int nd, JkDev jk)
{
    const long long w = (long long)blockIdx.x * 4 + threadIdx.x / 64;
    if (w >= nitems) return;   // uniform over the wave
    const int lane = threadIdx.x & 63;
    const WorkItem it = items[w];
    const int n = jk.nbf;
    const int fa = jk.bra_fun[2 * it.bra], fb = jk.bra_fun[2 * it.bra + 1];
    if (fa < 0 || fb < 0 || fa + na > n || fb + nb > n) return;
    bool act = lane >= it.lane_lo && lane < it.lane_hi;
    const long long k = act ? col[(long long)it.tile * 64 + lane] : -1;
    act = act && k >= 0;
    int fc = 0, fd = 0;
    if (act) {
        fc = jk.ket_fun[2 * k];
        fd = jk.ket_fun[2 * k + 1];
        act = fc >= 0 && fd >= 0 && fc + nc <= n && fd + nd <= n;
    }
    const int ncd = nc * nd;
    const long long stride = (long long)na * nb * ncd;
    const double *q = ints + it.obase + (act ? k : 0) * stride;
    double f = act ? 1.0 : 0.0;
    if (fa == fb) f *= 0.5;
    if (fc == fd) f *= 0.5;
    if (jk.same && k == it.bra) f *= 0.5;
    const double *D = jk.D;
    if (jk.J) {
        for (int a = 0; a < na; a++)
            for (int b = 0; b < nb; b++) {
                double s = 0.0;
                if (act) {
                    const double *r = q + (a * nb + b) * ncd;
                    for (int c = 0; c < nc; c++)
                        for (int d = 0; d < nd; d++) s += r[c * nd + d] * D[(long long)(fc + c) * n + fd + d];
                }
                s = wave_sum(f * s);
                if (lane == 0) unsafeAtomicAdd(jk.J + (long long)(fa + a) * n + fb + b, 4.0 * s);
            }
        if (act)
            for (int c = 0; c < nc; c++)
                for (int d = 0; d < nd; d++) {
                    double t = 0.0;
                    for (int a = 0; a < na; a++)
                        for (int b = 0; b < nb; b++)
                            t += q[(a * nb + b) * ncd + c * nd + d] * D[(long long)(fa + a) * n + fb + b];
                    unsafeAtomicAdd(jk.J + (long long)(fc + c) * n + fd + d, 4.0 * f * t);
                }
    }
    if (jk.K && act) {
        const double g = 2.0 * f;
        for (int a = 0; a < na; a++)
            for (int c = 0; c < nc; c++) {   // K_ac += v D_bd
                double t = 0.0;
                for (int b = 0; b < nb; b++)
                    for (int d = 0; d < nd; d++)
                        t += q[(a * nb + b) * ncd + c * nd + d] * D[(long long)(fb + b) * n + fd + d];
                unsafeAtomicAdd(jk.K + (long long)(fa + a) * n + fc + c, g * t);
            }
        for (int a = 0; a < na; a++)
            for (int d = 0; d < nd; d++) {   // K_ad += v D_bc
                double t = 0.0;
                for (int b = 0; b < nb; b++)
                    for (int c = 0; c < nc; c++)
                        t += q[(a * nb + b) * ncd + c * nd + d] * D[(long long)(fb + b) * n + fc + c];
                unsafeAtomicAdd(jk.K + (long long)(fa + a) * n + fd + d, g * t);
            }
        for (int b = 0; b < nb; b++)
            for (int c = 0; c < nc; c++) {   // K_bc += v D_ad
                double t = 0.0;
                for (int a = 0; a < na; a++)
                    for (int d = 0; d < nd; d++)
                        t += q[(a * nb + b) * ncd + c * nd + d] * D[(long long)(fa + a) * n + fd + d];
                unsafeAtomicAdd(jk.K + (long long)(fb + b) * n + fc + c, g * t);
            }
        for (int b = 0; b < nb; b++)
            for (int d = 0; d < nd; d++) {   // K_bd += v D_ac
                double t = 0.0;
                for (int a = 0; a < na; a++)
                    for (int c = 0; c < nc; c++)
                        t += q[(a * nb + b) * ncd + c * nd + d] * D[(long long)(fa + a) * n + fc + c];
                unsafeAtomicAdd(jk.K + (long long)(fb + b) * n + fd + d, g * t);
            }
    }
}

// The same digestion with the ket shells' and the second bra shell's
// component counts fixed at compile time: each lane reads every row
// (a, b, :, :) of its quartet once and applies all six updates from
// registers (the density values it needs are loaded once per item, per a or
// per row), instead of one pass over the quartet per update.  The second
// ket shell's components are taken DC at a time (DC divides ND, chosen so
// the accumulators stay in registers), each chunk reading its columns of
// every row.  K_b. is summed over a before it goes to global memory.
template <int NB, int NC, int ND, int DC>
__device__ __forceinline__ void digest_item(const WorkItem &it, int lane, const long long *col, const double *ints,
                                            int na, const JkDev &jk)
{
    static_assert(ND % DC == 0, "chunks of the second ket shell divide it");
    constexpr int NCD = NC * ND;
    const int n = jk.nbf;
    const int fa = jk.bra_fun[2 * it.bra], fb = jk.bra_fun[2 * it.bra + 1];
    if (fa < 0 || fb < 0 || fa + na > n || fb + NB > n) return;
    bool act = lane >= it.lane_lo && lane < it.lane_hi;
    const long long k = act ? col[(long long)it.tile * 64 + lane] : -1;
    act = act && k >= 0;
    int fc = 0, fd = 0;
    if (act) {
        fc = jk.ket_fun[2 * k];
        fd = jk.ket_fun[2 * k + 1];
        act = fc >= 0 && fd >= 0 && fc + NC <= n && fd + ND <= n;
    }
    // idle lanes read a quartet of the item (its first lane's, which the
    // class kernel wrote) and density element 0, and add nothing (weight 0)
    const long long kq = act ? k : col[(long long)it.tile * 64 + it.lane_lo];
    const double *q = ints + it.obase + kq * (long long)(na * NB * NCD);
    const double *__restrict__ D = jk.D;
    auto Dl = [&](long long idx) { return D[act ? idx : 0]; };
    // exchange update: row r of the bra's (na + NB) rows, column c
    auto addK = [&](int r, int c, double v) {
        unsafeAtomicAdd(jk.K + (long long)(r < na ? fa + r : fb + r - na) * n + c, v);
    };
    double f = act ? 1.0 : 0.0;
    if (fa == fb) f *= 0.5;
    if (fc == fd) f *= 0.5;
    if (jk.same && k == it.bra) f *= 0.5;
    const double g = 2.0 * f;
    for (int d0 = 0; d0 < ND; d0 += DC) {
        double dcd[NC * DC], jcd[NC * DC], kbc[NB][NC], kbd[NB][DC];
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int d = 0; d < DC; d++) {
                dcd[c * DC + d] = Dl((long long)(fc + c) * n + fd + d0 + d);
                jcd[c * DC + d] = 0.0;
            }
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int c = 0; c < NC; c++) kbc[b][c] = 0.0;
#pragma unroll
            for (int d = 0; d < DC; d++) kbd[b][d] = 0.0;
        }
        for (int a = 0; a < na; a++) {
            double dad[DC], dac[NC], kac[NC], kad[DC];
#pragma unroll
            for (int d = 0; d < DC; d++) {
                dad[d] = Dl((long long)(fa + a) * n + fd + d0 + d);
                kad[d] = 0.0;
            }
#pragma unroll
            for (int c = 0; c < NC; c++) {
                dac[c] = Dl((long long)(fa + a) * n + fc + c);
                kac[c] = 0.0;
            }
            // one row (a, b, :, d0..d0+DC) of the quartet
            auto row = [&](int b) {
                double dbd[DC], dbc[NC];
#pragma unroll
                for (int d = 0; d < DC; d++) dbd[d] = Dl((long long)(fb + b) * n + fd + d0 + d);
#pragma unroll
                for (int c = 0; c < NC; c++) dbc[c] = Dl((long long)(fb + b) * n + fc + c);
                const double *r = q + (a * NB + b) * NCD + d0;
                const double dab = D[(long long)(fa + a) * n + fb + b];
                double jab = 0.0;
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int d = 0; d < DC; d++) {
                        const double v = act ? r[c * ND + d] : 0.0;   // r is readable either way
                        jab = fma(v, dcd[c * DC + d], jab);
                        jcd[c * DC + d] = fma(v, dab, jcd[c * DC + d]);
                        kac[c] = fma(v, dbd[d], kac[c]);
                        kad[d] = fma(v, dbc[c], kad[d]);
                        kbc[b][c] = fma(v, dad[d], kbc[b][c]);
                        kbd[b][d] = fma(v, dac[c], kbd[b][d]);
                    }
                if (jk.J) {
                    jab = wave_sum(f * jab);
                    if (lane == 0) unsafeAtomicAdd(jk.J + (long long)(fa + a) * n + fb + b, 4.0 * jab);
                }
            };
#pragma unroll
            for (int b = 0; b < NB; b++) row(b);
            if (jk.K && act) {
#pragma unroll
                for (int c = 0; c < NC; c++) addK(a, fc + c, g * kac[c]);
#pragma unroll
                for (int d = 0; d < DC; d++) addK(a, fd + d0 + d, g * kad[d]);
            }
        }
        if (act && jk.J) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int d = 0; d < DC; d++)
                    unsafeAtomicAdd(jk.J + (long long)(fc + c) * n + fd + d0 + d, 4.0 * f * jcd[c * DC + d]);
        }
        if (act && jk.K) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
#pragma unroll
                for (int c = 0; c < NC; c++) addK(na + b, fc + c, g * kbc[b][c]);
#pragma unroll
                for (int d = 0; d < DC; d++) addK(na + b, fd + d0 + d, g * kbd[b][d]);
            }
        }
    }
}

// one wavefront per work item
template <int NB, int NC, int ND, int DC>
__global__ void __launch_bounds__(256) jk_digest_t(const WorkItem *items, long long nitems, const long long *col,
                                                   const double *ints, int na, JkDev jk)
{
    const long long w = (long long)blockIdx.x * 4 + threadIdx.x / 64;
    if (w >= nitems) return;   // uniform over the wave
    digest_item<NB, NC, ND, DC>(items[w], threadIdx.x & 63, col, ints, na, jk);
}

// Doubles a lane of the per-bra kernel holds beyond the ket block's density
// and Coulomb sums when it keeps the second bra shell's exchange sums and
// density rows over all a and the integrals of two a at a time (held(): all
// loads of an a in flight together, each ket's cache lines read while they
// are in the L1 cache, and a row of the exchange added to the local data
// share once instead of na times).  With this, the loads a step ahead and
// J_ab summed per lane the digestion of 64 atoms takes 480 ms, 637 before; it
// is bound by the loads, 64 cache lines an instruction, and the adds into the
// local data share.
constexpr int kHeldDoubles = 108;
constexpr bool held(int nb, int nc, int dc)
{
    return 2 * nc * dc + 4 * (nc + dc) + 2 * nb * (nc + dc) + 2 * nb * nc * dc <= kHeldDoubles;
}

// Where it cannot, the next row's integrals are loaded ahead if two rows fit.
constexpr bool ahead(int nc, int dc) { return 4 * nc * dc + 4 * (nc + dc) <= 72; }

// Most threads of the per-bra kernel's block: two wavefronts a SIMD have 256
// registers each, which the f classes exceed.
constexpr int rows_threads(int nb, int nc, int nd) { return nb > 6 || nc > 6 || nd > 6 ? 256 : 512; }

// The per-bra kernel's work on one item: a in [a0, a1) of its quartets.  The
// exchange rows of the bra's functions, rows[r * nbf] (r < na: first shell),
// and the lanes' sums of J_ab, jsum[(a * NB + b) * 64 + lane], are in the
// local data share: both adds are fire and forget, where a sum over the
// wavefront for every (a, b) waited for twelve dependent exchanges.  Every
// wait is for loads issued a step ahead: the next a's integrals (held) or
// the next row's.
template <int NB, int NC, int ND, int DC>
__device__ __forceinline__ void digest_rows_item(const WorkItem &it, int lane, const long long *col,
                                                 const double *ints, int na, int a0, int a1, const JkDev &jk,
                                                 double *rows, double *jsum)
{
    static_assert(ND % DC == 0, "chunks of the second ket shell divide it");
    constexpr int NCD = NC * ND, NV = NC * DC;
    constexpr bool HOLD = held(NB, NC, DC), AHEAD = HOLD || ahead(NC, DC);
    constexpr int KB = HOLD ? NB : 1;
    constexpr int STEP = HOLD ? NB : 1;     // rows loaded at a time
    const int n = jk.nbf;
    const int fa = jk.bra_fun[2 * it.bra], fb = jk.bra_fun[2 * it.bra + 1];
    if (fa < 0 || fb < 0 || fa + na > n || fb + NB > n) return;
    bool act = lane >= it.lane_lo && lane < it.lane_hi;
    const long long k = act ? col[(long long)it.tile * 64 + lane] : -1;
    act = act && k >= 0;
    int fc = 0, fd = 0;
    if (act) {
        fc = jk.ket_fun[2 * k];
        fd = jk.ket_fun[2 * k + 1];
        act = fc >= 0 && fd >= 0 && fc + NC <= n && fd + ND <= n;
    }
    // idle lanes read a quartet of the item (its first lane's, which the
    // class kernel wrote) and density element 0, and add nothing
    const long long kq = act ? k : col[(long long)it.tile * 64 + it.lane_lo];
    const double *q = ints + it.obase + kq * (long long)(na * NB * NCD);
    const double *__restrict__ D = jk.D;
    auto Dl = [&](long long idx) { return D[act ? idx : 0]; };
    auto ldsadd = [](double *p, double v) {
        // the local data share, named as such so the add is a ds_add_f64
        atomicAdd((double *)(__attribute__((address_space(3))) double *)p, v);
    };
    auto addK = [&](int r, int c, double v) { ldsadd(rows + (long long)r * n + c, v); };
    double f = act ? 1.0 : 0.0;
    if (fa == fb) f *= 0.5;
    if (fc == fd) f *= 0.5;
    if (jk.same && k == it.bra) f *= 0.5;
    const double g = 2.0 * f;
    for (int d0 = 0; d0 < ND; d0 += DC) {
        double dcd[NV], jcd[NV], kbc[KB][NC], kbd[KB][DC], dbc[KB][NC], dbd[KB][DC];
        double cur[STEP * NV], nxt[AHEAD ? STEP * NV : 1];
        // rows r .. r + STEP of the quartet, columns of this chunk
        auto load = [&](double *v, int r) {
            const double *p = q + (long long)r * NCD + d0;
#pragma unroll
            for (int s = 0; s < STEP; s++)
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int d = 0; d < DC; d++) v[s * NV + c * DC + d] = p[s * NCD + c * ND + d];
        };
        auto load_db = [&](int kb, int b) {
#pragma unroll
            for (int c = 0; c < NC; c++) dbc[kb][c] = Dl((long long)(fb + b) * n + fc + c);
#pragma unroll
            for (int d = 0; d < DC; d++) dbd[kb][d] = Dl((long long)(fb + b) * n + fd + d0 + d);
        };
        auto clear_kb = [&](int kb) {
#pragma unroll
            for (int c = 0; c < NC; c++) kbc[kb][c] = 0.0;
#pragma unroll
            for (int d = 0; d < DC; d++) kbd[kb][d] = 0.0;
        };
        auto add_kb = [&](int kb, int b) {
            if (!jk.K || !act) return;
#pragma unroll
            for (int c = 0; c < NC; c++) addK(na + b, fc + c, g * kbc[kb][c]);
#pragma unroll
            for (int d = 0; d < DC; d++) addK(na + b, fd + d0 + d, g * kbd[kb][d]);
        };
        if constexpr (AHEAD) load(cur, a0 * NB);
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int d = 0; d < DC; d++) {
                dcd[c * DC + d] = Dl((long long)(fc + c) * n + fd + d0 + d);
                jcd[c * DC + d] = 0.0;
            }
        if constexpr (HOLD) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                load_db(b, b);
                clear_kb(b);
            }
        }
        for (int a = a0; a < a1; a++) {
            double dad[DC], dac[NC], kac[NC], kad[DC];
            if constexpr (HOLD) {
                if (a + 1 < a1) load(nxt, (a + 1) * NB);
            }
#pragma unroll
            for (int d = 0; d < DC; d++) {
                dad[d] = Dl((long long)(fa + a) * n + fd + d0 + d);
                kad[d] = 0.0;
            }
#pragma unroll
            for (int c = 0; c < NC; c++) {
                dac[c] = Dl((long long)(fa + a) * n + fc + c);
                kac[c] = 0.0;
            }
            // row (a, b) of the quartet, its values at v
            auto row = [&](int b, int kb, const double *v) {
                const double dab = D[(long long)(fa + a) * n + fb + b];
                double jab = 0.0;
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int d = 0; d < DC; d++) {
                        const double x = act ? v[c * DC + d] : 0.0;
                        jab = fma(x, dcd[c * DC + d], jab);
                        jcd[c * DC + d] = fma(x, dab, jcd[c * DC + d]);
                        kac[c] = fma(x, dbd[kb][d], kac[c]);
                        kad[d] = fma(x, dbc[kb][c], kad[d]);
                        kbc[kb][c] = fma(x, dad[d], kbc[kb][c]);
                        kbd[kb][d] = fma(x, dac[c], kbd[kb][d]);
                    }
                if (jk.J) {
                    if (jsum) {
                        ldsadd(jsum + (a * NB + b) * 64 + lane, f * jab);
                    } else {
                        jab = wave_sum(f * jab);
                        if (lane == 0) unsafeAtomicAdd(jk.J + (long long)(fa + a) * n + fb + b, 4.0 * jab);
                    }
                }
            };
            if constexpr (HOLD) {
#pragma unroll
                for (int b = 0; b < NB; b++) row(b, b, cur + b * NV);
#pragma unroll
                for (int i = 0; i < STEP * NV; i++) cur[i] = nxt[i];
            } else {
                // nothing is indexed by b: a loop, at most one row's loads ahead
#pragma unroll 1
                for (int b = 0; b < NB; b++) {
                    load_db(0, b);
                    clear_kb(0);
                    const int r = a * NB + b;
                    if constexpr (AHEAD) {
                        if (r + 1 < a1 * NB) load(nxt, r + 1);
                    } else {
                        load(cur, r);
                    }
                    row(b, 0, cur);
                    add_kb(0, b);
                    if constexpr (AHEAD) {
#pragma unroll
                        for (int i = 0; i < NV; i++) cur[i] = nxt[i];
                    }
                }
            }
            if (jk.K && act) {
#pragma unroll
                for (int c = 0; c < NC; c++) addK(a, fc + c, g * kac[c]);
#pragma unroll
                for (int d = 0; d < DC; d++) addK(a, fd + d0 + d, g * kad[d]);
            }
        }
        if (act && jk.J) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int d = 0; d < DC; d++)
                    unsafeAtomicAdd(jk.J + (long long)(fc + c) * n + fd + d0 + d, 4.0 * f * jcd[c * DC + d]);
        }
        if constexpr (HOLD) {
#pragma unroll
            for (int b = 0; b < NB; b++) add_kb(b, b);
        }
    }
}

// One block per bra pair of the launch: its wavefronts take the bra's work
// items (or, where the launch has few, parts of their a) in turn,
// and the exchange rows of the bra's functions and J_ab are summed over all
// its kets in the local data share ((na + NB) x nbf and na x NB x 64
// doubles, dynamic) and added to K and J once per touched element at the
// end -- never more global atomics than one per quartet and element, usually
// far fewer (every ket of the bra adds to the same rows).  Launched only
// with an exchange matrix to fill.
template <int NB, int NC, int ND, int DC>
__global__ void __launch_bounds__(rows_threads(NB, NC, ND)) jk_digest_rows(const WorkItem *items, long long nitems,
                                                      const long long *tstart, int nbra, const long long *col,
                                                      const double *ints, int na, int parts, int lanesum, JkDev jk)
{
    extern __shared__ double rows[];
    const int bi = blockIdx.x;
    const long long i0 = tstart[bi], i1 = bi + 1 < nbra ? tstart[bi + 1] : nitems;
    if (i0 >= i1) return;   // uniform over the block
    const int n = jk.nbf;
    const int R = na + NB;
    double *jsum = lanesum ? rows + R * n : nullptr;
    const int nlds = R * n + (lanesum ? na * NB * 64 : 0);   // at most 160 KB
    for (int e = threadIdx.x; e < nlds; e += blockDim.x) rows[e] = 0.0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64, nwave = blockDim.x / 64;
    for (int u = wave; u < (int)(i1 - i0) * parts; u += nwave) {
        const int w = u / parts, p = u - w * parts;
        digest_rows_item<NB, NC, ND, DC>(items[i0 + w], lane, col, ints, na, p * na / parts, (p + 1) * na / parts,
                                         jk, rows, jsum);
    }
    __syncthreads();
    const int bra = items[i0].bra;
    const int fa = jk.bra_fun[2 * bra], fb = jk.bra_fun[2 * bra + 1];
    if (fa < 0 || fb < 0 || fa + na > n || fb + NB > n) return;
    for (int e = threadIdx.x; e < R * n; e += blockDim.x) {
        const double v = rows[e];
        if (v == 0.0) continue;
        const int r = e / n, c = e - r * n;
        unsafeAtomicAdd(jk.K + (long long)(r < na ? fa + r : fb + r - na) * n + c, v);
    }
    if (!jk.J || !jsum) return;
    for (int r = wave; r < na * NB; r += nwave) {
        const double s = wave_sum(jsum[r * 64 + lane]);
        if (lane == 0) unsafeAtomicAdd(jk.J + (long long)(fa + r / NB) * n + fb + r % NB, 4.0 * s);
    }
}

constexpr int nc_of(int l) { return (l + 1) * (l + 2) / 2; }

// doubles per lane the specialised kernel holds for a chunk of dc
// components of the second ket shell: density and Coulomb sums of the ket
// block, the per-a and per-row vectors, and without the row accumulator the
// K_b. sums over a plus (a quarter of) the unrolled rows' loads in flight.
// Kept within kRegDoubles (gfx950 has 256 VGPRs per lane; the rest hold
// addresses and loads): every instance then runs without scratch.
constexpr int kRegDoubles = 96;
constexpr int reg_doubles(int nb, int nc, int dc, bool rows)
{
    return 2 * nc * dc + 4 * (nc + dc) + (rows ? 0 : nb * (nc + dc) + nb * nc * dc / 4);
}

// components of the second ket shell per chunk: the largest divisor of nd
// that fits; 0: none does (the generic kernel)
constexpr int pick_dc(int nb, int nc, int nd, bool rows)
{
    for (int dc = nd; dc >= 1; --dc)
        if (nd % dc == 0 && reg_doubles(nb, nc, dc, rows) <= kRegDoubles) return dc;
    return 0;
}

// exchange row accumulators of the per-bra kernel: at most this many bytes
// of the local data share per block (and no more than the device allows,
// 160 KB on gfx950).  A block above 80 KB holds its CU's share alone
// whatever its size, so the whole of it is offered.
constexpr long long kRowBytes = 160 * 1024;
// work items of a launch up to which the per-bra kernel's blocks have eight
// wavefronts and divide an item's components of the first bra shell between
// them: fewer items than one for every SIMD (10 atoms: 4.96 -> 4.80 ms of
// digestion, which is chains of dependent loads; single components a wavefront
// took 6.0)
constexpr long long kSplitItems = 1024;

std::atomic<int> g_rows_enabled{1};   // simint_hip_set_jk_rows

long long row_bytes_limit()
{
    static std::atomic<long long> lim{-1};
    long long v = lim.load(std::memory_order_relaxed);
    if (v < 0) {
        int dev = 0, a = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&a, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
            a = 65536;
        v = a < kRowBytes ? a : kRowBytes;
        lim.store(v, std::memory_order_relaxed);
    }
    return g_rows_enabled.load(std::memory_order_relaxed) ? v : 0;
}

struct Launch {
    const WorkItem *items;
    long long nitems;
    const long long *tstart;
    int nbra;
    const long long *col;
    const double *ints;
    int na;
};

template <int LB, int LC, int LD>
hipError_t launch_t(const Launch &L, const JkDev &d, hipStream_t s)
{
    constexpr int NB = nc_of(LB), NC = nc_of(LC), ND = nc_of(LD);
    const long long rbytes = 8LL * (L.na + NB) * d.nbf;
    constexpr int DCR = pick_dc(NB, NC, ND, true), DCG = pick_dc(NB, NC, ND, false);
    const WorkItem *items = L.items;
    const long long nitems = L.nitems;
    const long long *col = L.col;
    const double *ints = L.ints;
    const int na = L.na;
    const unsigned nwave_blocks = (unsigned)((nitems + 3) / 4);
    bool done = false;
    if constexpr (DCR > 0) {
        if (d.K && rbytes <= row_bytes_limit()) {
            // a block above half the local data share holds its CU alone: eight
            // wavefronts, two for every SIMD
            const long long lbytes = rbytes + 8LL * L.na * NB * 64;
            const int lanesum = lbytes <= row_bytes_limit();   // room for the lanes' sums of J_ab too
            const bool few = nitems <= kSplitItems;
            const int threads = few || lbytes > kRowBytes / 2 ? rows_threads(NB, NC, ND) : 256;
            const long long share = threads / 64 * (long long)L.nbra / nitems;   // wavefronts an item
            const int parts = few ? (int)std::max(1LL, std::min<long long>(na, share)) : 1;
            hipLaunchKernelGGL((jk_digest_rows<NB, NC, ND, DCR>), dim3((unsigned)L.nbra), dim3(threads),
                               (size_t)(lanesum ? lbytes : rbytes), s, items, nitems, L.tstart, L.nbra, col, ints,
                               na, parts, lanesum, d);
            done = true;
        }
    }
    if constexpr (DCG > 0) {
        if (!done) {
            hipLaunchKernelGGL((jk_digest_t<NB, NC, ND, DCG>), dim3(nwave_blocks), dim3(256), 0, s, items, nitems,
                               col, ints, na, d);
            done = true;
        }
    }
    if (!done)
        hipLaunchKernelGGL(jk_digest, dim3(nwave_blocks), dim3(256), 0, s, items, nitems, col, ints, na, NB, NC, ND,
                           d);
    return hipGetLastError();
}

template <int LB, int LC>
hipError_t launch_d(int ld, const Launch &L, const JkDev &d, hipStream_t s)
{
    switch (ld) {
    case 0: return launch_t<LB, LC, 0>(L, d, s);
    case 1: return launch_t<LB, LC, 1>(L, d, s);
    case 2: return launch_t<LB, LC, 2>(L, d, s);
    default: return launch_t<LB, LC, 3>(L, d, s);
    }
}

template <int LB>
hipError_t launch_c(int lc, int ld, const Launch &L, const JkDev &d, hipStream_t s)
{
    switch (lc) {
    case 0: return launch_d<LB, 0>(ld, L, d, s);
    case 1: return launch_d<LB, 1>(ld, L, d, s);
    case 2: return launch_d<LB, 2>(ld, L, d, s);
    default: return launch_d<LB, 3>(ld, L, d, s);
    }
}

// M <- (M + M^T)/2: thread (i, j) with i < j averages the pair
__global__ void __launch_bounds__(256) symmetrize(int n, double *M)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)n * n) return;
    const int i = (int)(t / n), j = (int)(t % n);
    if (i >= j) return;
    const double v = 0.5 * (M[(long long)i * n + j] + M[(long long)j * n + i]);
    M[(long long)i * n + j] = v;
    M[(long long)j * n + i] = v;
}

inline int ncart(int l) { return (l + 1) * (l + 2) / 2; }

}  // namespace

namespace simint_rt {

hipError_t launch_jk_digest(const int am[4], const WorkItem *items, long long nitems, const long long *tstart,
                            int nbra, const long long *col, const double *ints, const simint_hip_jk *jk,
                            hipStream_t s)
{
    JkDev d{jk->nbf, jk->same, jk->bra_fun, jk->ket_fun, jk->density, jk->J, jk->K};
    if (am[1] > 3 || am[2] > 3 || am[3] > 3) {
        hipLaunchKernelGGL(jk_digest, dim3((unsigned)((nitems + 3) / 4)), dim3(256), 0, s, items, nitems, col, ints,
                           ncart(am[0]), ncart(am[1]), ncart(am[2]), ncart(am[3]), d);
        return hipGetLastError();
    }
    const Launch L{items, nitems, tstart, nbra, col, ints, ncart(am[0])};
    switch (am[1]) {
    case 0: return launch_c<0>(am[2], am[3], L, d, s);
    case 1: return launch_c<1>(am[2], am[3], L, d, s);
    case 2: return launch_c<2>(am[2], am[3], L, d, s);
    default: return launch_c<3>(am[2], am[3], L, d, s);
    }
}

}  // namespace simint_rt

extern "C" {

int simint_hip_set_jk_rows(int enable)
{
    return g_rows_enabled.exchange(enable ? 1 : 0);
}

int simint_hip_jk_symmetrize(int nbf, double *d_J, double *d_K)
{
    if (nbf <= 0) return SIMINT_ERROR_ARGUMENT;
    if (!simint_rt::ensure_device()) return SIMINT_ERROR_NO_DEVICE;
    const hipStream_t s = simint_rt::stream();
    const long long nn = (long long)nbf * nbf;
    const unsigned nblk = (unsigned)((nn + 255) / 256);
    for (double *M : {d_J, d_K}) {
        if (!M) continue;
        hipLaunchKernelGGL(symmetrize, dim3(nblk), dim3(256), 0, s, nbf, M);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) { simint_rt::set_hip_error("symmetrize launch", e); return SIMINT_ERROR_HIP; }
    }
    return 0;
}

}  // extern "C"
