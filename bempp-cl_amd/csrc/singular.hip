// Singular (Sauter-Schwab) pairs, FP64, for gfx950: (test element, trial element) pairs that share a
// vertex, an edge or the whole triangle (bempp_cl/core/numba_kernels.py:1471-1526 scalar, 1973-2061
// EFIE), with 512 (vertex), 1280 (edge) or 1536 (coincident) Duffy points per pair at order 4.
//
// A workgroup of W waves takes 64 / G consecutive pairs; in every wave G lanes share a pair and the
// pair's points are split over the W G lanes. The pair table lists the pairs of one rule (kind and
// local vertices) together, so a wave's pairs share the points: the wave stages its part of them in LDS
// with coalesced loads and reads them as broadcasts (the pairs of a wave that spans several rules read
// their points from memory). Each lane accumulates the moment block S[a][b] = sum_k G_k w_k u_a(xi_k) u_b(eta_k),
// u = (1, xi_0, xi_1), of its points; the partial blocks are summed by shuffles and through LDS, scaled
// by J_test J_trial and turned into the local matrix block exactly as for regular pairs. The entries are
// added to the dense output with hardware atomics, real and imaginary part on neighbouring lanes (one
// memory-side request), which replaces the reference's host-side np.add.at scatter
// (bempp_cl/core/dense_assembler.py:78-98).
// Bound by FP64 arithmetic: 71 instructions a point for a complex single layer on P1, 26 for the
// Laplace one on DP0.
#include "bem_device.h"
#include "bem_internal.h"

namespace bem {

struct SingularArgs {
    SpaceArgs test, trial;
    int n_pairs;
    const int32_t *pairs;
    const double *tpts, *spts, *wts;
    double kr, ki;
    void *out;
    void *out2;  // DUAL: double layer (out: single layer)
    int64_t ld;
};

// LDS of one workgroup: the staged points, then the partial moments and the local blocks
template <int NV, int W, int G, int L>
union SingularShared {
    // points a wave stages at a time, with their loads in flight together
    static constexpr int kLoads = L, kChunk = 64 * kLoads;
    struct {
        double2 points[W][kChunk][2];  // (xi_0, xi_1), (eta_0, eta_1)
        double weights[W][kChunk];
    } st;
    double moments[W][NV][64 / G];
};

// DUAL: OP is a single layer; the double layer of the same family (sharing r and e^{ikr} at
// every point) goes to a.out2.
template <int OP, int NTS, int NSS, typename OutT, bool DUAL, int W, int G, int L>
__global__ __launch_bounds__(64 * W, (DUAL && NTS * NSS == 9) || L > 2 ? 2 : 3) void singular_kernel(const SingularArgs a) {
    constexpr bool CPLX = OpTraits<OP>::is_complex;
    constexpr int NC = CPLX ? 2 : 1, NB = NTS * NSS, NV = NB * NC, NOPS = DUAL ? 2 : 1;
    constexpr int PP = 64 / G;  // pairs per workgroup
    using Shared = SingularShared<NV, W, G, L>;
    __shared__ Shared sh;
    __shared__ int32_t rows[NTS][PP], cols[NSS][PP];
    __shared__ double mult[NTS + NSS][PP];
    const int lane = threadIdx.x & 63, p = lane % PP, sub = lane / PP;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = blockIdx.x * PP;
    const bool active = first + p < a.n_pairs;
    const int32_t *pd = a.pairs + 6 * (int64_t)(active ? first + p : first);
    const int e = pd[0], f = pd[1], toff = pd[2], soff = pd[3], woff = pd[4], np = pd[5];
    const double tnm = a.test.nmult ? (double)a.test.nmult[e] : 1.0;
    const double snm = a.trial.nmult ? (double)a.trial.nmult[f] : 1.0;
    // dofs and multipliers of the scatter, loaded together with the geometry
    if (wave == 0 && sub == 0) {
#pragma unroll
        for (int i = 0; i < NTS; ++i) {
            rows[i][p] = a.test.l2g[(int64_t)e * NTS + i];
            mult[i][p] = a.test.mult[(int64_t)e * NTS + i];
        }
#pragma unroll
        for (int j = 0; j < NSS; ++j) {
            cols[j][p] = a.trial.l2g[(int64_t)f * NSS + j];
            mult[NTS + j][p] = a.trial.mult[(int64_t)f * NSS + j];
        }
    }
    // the geometry rows in registers
    double gt[14], gf[14], nx[3], ny[3];
#pragma unroll
    for (int k = 0; k < 14; ++k) {
        gt[k] = a.test.geom[(int64_t)e * BEM_GEOM_STRIDE + k];
        gf[k] = a.trial.geom[(int64_t)f * BEM_GEOM_STRIDE + k];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        nx[d] = gt[9 + d] * tnm;
        ny[d] = gf[9 + d] * snm;
    }

    double S[NOPS][NC][NTS][NSS];
#pragma unroll
    for (int o = 0; o < NOPS; ++o)
#pragma unroll
        for (int z = 0; z < NC; ++z)
#pragma unroll
            for (int i = 0; i < NTS; ++i)
#pragma unroll
                for (int j = 0; j < NSS; ++j) S[o][z][i][j] = 0.0;

    auto points = [&](auto phase_tag) {
        constexpr int PH = decltype(phase_tag)::value;
        // one point: xi, eta and its weight
        auto point = [&](double xi0, double xi1, double et0, double et1, double w) {
            // the two points, then their difference: the swapped points of a coincident pair get exactly
            // opposite differences, so that its double layer cancels
            double d[3];
#pragma unroll
            for (int m = 0; m < 3; ++m)
                d[m] = fma(gf[6 + m], et1, fma(gf[3 + m], et0, gf[m])) -
                       fma(gt[6 + m], xi1, fma(gt[3 + m], xi0, gt[m]));
            const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            double g[2][2];
            green2<green_op<OP>(), DUAL, double, PH>(d[0], d[1], d[2], r2, nx, ny, a.kr, a.ki, g[0][0], g[0][1],
                                                     g[1][0], g[1][1]);
#pragma unroll
            for (int o = 0; o < NOPS; ++o)
#pragma unroll
                for (int z = 0; z < NC; ++z) {
                    const double t0 = g[o][z] * w;
                    const double t[3] = {t0, t0 * et0, t0 * et1};
#pragma unroll
                    for (int j = 0; j < NSS; ++j) {
                        S[o][z][0][j] += t[j];
                        if constexpr (NTS == 3) {
                            S[o][z][1][j] = fma(t[j], xi0, S[o][z][1][j]);
                            S[o][z][2][j] = fma(t[j], xi1, S[o][z][2][j]);
                        }
                    }
                }
        };
        // the rule of the first pair, and whether the wave's pairs share it
        const int to = __builtin_amdgcn_readfirstlane(toff), so = __builtin_amdgcn_readfirstlane(soff);
        const int wo = __builtin_amdgcn_readfirstlane(woff), n = __builtin_amdgcn_readfirstlane(np);
        if (!__all(!active || (toff == to && soff == so && woff == wo && np == n))) {
            // each pair reads its own rule
            if (active) {
                const int per = (np + W - 1) / W, k1 = min((wave + 1) * per, np);
                for (int k = wave * per + sub; k < k1; k += G) {
                    const double2 px = load_pair(a.tpts + 2 * ((int64_t)toff + k));
                    const double2 py = load_pair(a.spts + 2 * ((int64_t)soff + k));
                    point(px.x, px.y, py.x, py.y, a.wts[(int64_t)woff + k]);
                }
            }
            return;
        }
        const int per = (n + W - 1) / W, k0 = min(wave * per, n), k1 = min(k0 + per, n);
        for (int kb = k0; kb < k1; kb += Shared::kChunk) {
            const int count = min(Shared::kChunk, k1 - kb);
            // the wave's own part of LDS: its accesses complete in order, no barrier
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            double2 xt[Shared::kLoads], xs[Shared::kLoads];
            double xw[Shared::kLoads];
#pragma unroll
            for (int u = 0; u < Shared::kLoads; ++u) {
                const int64_t kk = kb + min(64 * u + lane, count - 1);
                xt[u] = load_pair(a.tpts + 2 * (to + kk));
                xs[u] = load_pair(a.spts + 2 * (so + kk));
                xw[u] = a.wts[wo + kk];
            }
#pragma unroll
            for (int u = 0; u < Shared::kLoads; ++u) {
                sh.st.points[wave][64 * u + lane][0] = xt[u];
                sh.st.points[wave][64 * u + lane][1] = xs[u];
                sh.st.weights[wave][64 * u + lane] = xw[u];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (!active) continue;
#pragma unroll 2
            for (int k = sub; k < count; k += G) {
                const double2 px = sh.st.points[wave][k][0], py = sh.st.points[wave][k][1];
                point(px.x, px.y, py.x, py.y, sh.st.weights[wave][k]);
            }
        }
    };
    // every distance within a pair is at most diam_t + diam_f (triangles sharing a vertex), so a
    // wave-uniform bound selects the phase mode: the series sin/cos without range reduction when
    // k r <= 1, else the branch-free reduction
    if constexpr (OpTraits<green_op<OP>()>::is_complex) {
        const double kd = fabs(a.kr) * (gt[13] + gf[13]);
        const bool small = __all(kd <= 1.0), reduced = __all(kd < 0x1p25), real = a.ki == 0.0;
        if (small && real) points(std::integral_constant<int, kPhSmall | kPhReal>{});
        else if (small) points(std::integral_constant<int, kPhSmall>{});
        else if (reduced && real) points(std::integral_constant<int, kPhReduced | kPhReal>{});
        else if (reduced) points(std::integral_constant<int, kPhReduced>{});
        else points(std::integral_constant<int, 0>{});
    } else {
        points(std::integral_constant<int, 0>{});
    }

    // sums over the lanes of a pair
#pragma unroll
    for (int o = 0; o < NOPS; ++o)
#pragma unroll
        for (int z = 0; z < NC; ++z)
#pragma unroll
            for (int i = 0; i < NTS; ++i)
#pragma unroll
                for (int j = 0; j < NSS; ++j)
#pragma unroll
                    for (int off = 32; off >= PP; off >>= 1) S[o][z][i][j] += __shfl_xor(S[o][z][i][j], off, 64);
    const double jj = gt[12] * gf[12];
#pragma unroll
    for (int o = 0; o < NOPS; ++o) {
        __syncthreads();  // the points (the previous operator's blocks) have been read
        if (sub == 0) {
#pragma unroll
            for (int z = 0; z < NC; ++z)
#pragma unroll
                for (int i = 0; i < NTS; ++i)
#pragma unroll
                    for (int j = 0; j < NSS; ++j) sh.moments[wave][(i * NSS + j) * NC + z][p] = S[o][z][i][j] * jj;
        }
        __syncthreads();
        // the sums over the waves: each thread its own values
        for (int idx = threadIdx.x; idx < NV * PP; idx += 64 * W) {
            double *m = &sh.moments[0][0][0] + idx;
            double sum = m[0];
#pragma unroll
            for (int k = 1; k < W; ++k) sum += m[k * NV * PP];
            m[0] = sum;
        }
        __syncthreads();
        // the local blocks [pair][entry][re, im], in the memory of the second wave's partial sums
        OutT *block = reinterpret_cast<OutT *>(&sh.moments[1][0][0]);
        C2d M[NTS][NSS];
#pragma unroll
        for (int i = 0; i < NTS; ++i)
#pragma unroll
            for (int j = 0; j < NSS; ++j) {
                M[i][j].re = sh.moments[0][(i * NSS + j) * NC][p];
                M[i][j].im = CPLX ? sh.moments[0][(i * NSS + j) * NC + NC - 1][p] : 0.0;
            }
        // the W G lanes of a pair share its entries
        for (int l = wave * G + sub; l < NB; l += W * G) {
            const int i = l / NSS, j = l % NSS;
            const double m = mult[i][p] * mult[NTS + j][p];
            C2d v = {0.0, 0.0};
            if (m != 0.0) {
                if constexpr (DUAL)
                    v = o ? local_value<OP + 1, NTS, NSS>(M, i, j, gt, gf, a.kr, a.ki)
                          : local_value<OP, NTS, NSS>(M, i, j, gt, gf, a.kr, a.ki);
                else
                    v = local_value<OP, NTS, NSS>(M, i, j, gt, gf, a.kr, a.ki, tnm * snm);
            }
            OutT *dst = block + (p * NB + l) * NC;
            dst[0] = (OutT)(v.re * m);
            if constexpr (CPLX) dst[1] = (OutT)(v.im * m);
        }
        __syncthreads();
        OutT *out = reinterpret_cast<OutT *>(o ? a.out2 : a.out);
        const int count = min(PP, a.n_pairs - first) * NV;
        for (int idx = threadIdx.x; idx < count; idx += 64 * W) {
            const int q = idx / NV, l = (idx - q * NV) / NC;
            const OutT v = block[idx];
            const int64_t at = (int64_t)rows[l / NSS][q] * a.ld + cols[l % NSS][q];
            if (v != (OutT)0) atomic_add(out + NC * at + idx % NC, v);
        }
    }
}

// Lanes of a wave per pair (G), waves (W = 4) and loads in flight per lane (L). The points of a pair are split
// W G ways. The coincident pairs' lanes form the longest chain (1536 / (W G) points), a split costs the set-up
// of more workgroups. Few pairs also leave waves whose pairs follow several rules; one rule after the other,
// with the other lanes idle, doubled and more the longest chain (6,400 pairs, electric field, G = 4: 54 against
// 32 us). Kernel times, G = 16 / 8 / 4 / 1, against lanes striding over a pair's points with loads of their
// own before (32 lanes a pair below 32,768 pairs, else 8), us:
//    pairs     Laplace P1 FP64       Laplace DP0 FP64     Helmholtz P1 SL + DL  electric field         Helmholtz DL P1 FP64
//     2,280   11/ 14/ 19  (14)       9/ 13/ 18  (12)      22/ 25/ 38  (28)     19/ 20/ 30  (21)      20/ 21/ 32  (23)
//     6,440   20/ 16/ 21  (19)      17/ 14/ 19  (17)      45/ 36/ 40  (46)     31/ 27/ 32  (31)      33/ 28/ 33  (43)
//    12,680   30/ 25/ 27/ 59 (29)   25/ 20/ 21/ 53 (25)   77/ 54/ 52/110 (65)  52/ 42/ 43/ 96 (52)   50/ 40/ 40/ 94 (59)
//    21,000   44/ 37/ 41/ 62 (45)   37/ 25/ 24/ 53 (38)  121/ 83/ 72/112 (102) 76/ 58/ 59/ 97 (103)  75/ 59/ 59/ 96 (89)
//    43,880   83/ 60/ 55/ 68 (75)   70/ 44/ 40/ 57 (68)  244/162/139/147 (177) 142/105/ 98/106 (140) 147/114/107/117 (155)
//    66,500       92/ 86/ 92 (109)      67/ 62/ 75 (91)      254/219/201 (257)     165/150/140 (206)     181/165/171 (226)
//   103,940      143/126/123 (157)     101/ 90/ 93 (136)     395/336/305 (404)     254/230/211 (306)     277/252/236 (346)
//   203,780      275/242/225 (284)     196/171/162 (243)     767/650/587 (735)     488/442/399 (584)     540/484/449 (644)
// G = 8 up to kSingMediumPairs (real operators kSingMediumPairsReal: 12,680 pairs, Laplace double layer 29.1 / 31.0,
// single and double layer 34.2 / 37.0 us with G = 8 / 4). The electric field operator takes G = 1 earlier.
// L: a vertex pair's part (128 points) in one step of two loads; G = 1 one load (10 registers less). Up to
// kSingWholePairs the chip holds at most two workgroups per CU, nothing hides the latency of a step, and a wave
// loads its whole part (384 points, 61 KB of LDS) at once. L = 2 / 6: 4,100 pairs, Helmholtz hypersingular
// 25.1 / 19.6 (22.0), electric field 22.4 / 19.3 (21.2), Laplace single and double layer 18.2 / 16.3 us (17.0);
// 4,500 pairs 26.5 / 20.8, 23.5 / 19.9, 20.1 / 18.3; 5,400 pairs 26.6 / 26.3, 23.5 / 25.8, 19.7 / 22.7 us.
constexpr int kSingLargePairs = 131072, kSingLargePairsEfie = 49152, kSingMediumPairs = 10240,
              kSingMediumPairsReal = 16384, kSingWholePairs = 4608, kSingSmallPairs = 3072;

template <int OP, typename OutT, bool DUAL, int W, int G, int L>
static int launch_sing_split(const SingularArgs &a, hipStream_t s) {
    constexpr int PP = 64 / G;
    const dim3 grid((unsigned)(((int64_t)a.n_pairs + PP - 1) / PP)), threads(64 * W);
    if constexpr (OP == kMaxwellEFIE) {
        hipLaunchKernelGGL((singular_kernel<OP, 3, 3, OutT, false, W, G, L>), grid, threads, 0, s, a);
    } else if constexpr (is_hypersingular<OP>()) {
        if (nshape_of(a.test.shape) != 3 || nshape_of(a.trial.shape) != 3) {
            set_error("hypersingular operators need P1 shape functions on both sides");
            return BEM_ERR_INVALID_ARGUMENT;
        }
        hipLaunchKernelGGL((singular_kernel<OP, 3, 3, OutT, false, W, G, L>), grid, threads, 0, s, a);
    } else {
        int nt = nshape_of(a.test.shape), ns = nshape_of(a.trial.shape);
        if (nt == 1 && ns == 1)
            hipLaunchKernelGGL((singular_kernel<OP, 1, 1, OutT, DUAL, W, G, L>), grid, threads, 0, s, a);
        else if (nt == 1 && ns == 3)
            hipLaunchKernelGGL((singular_kernel<OP, 1, 3, OutT, DUAL, W, G, L>), grid, threads, 0, s, a);
        else if (nt == 3 && ns == 1)
            hipLaunchKernelGGL((singular_kernel<OP, 3, 1, OutT, DUAL, W, G, L>), grid, threads, 0, s, a);
        else
            hipLaunchKernelGGL((singular_kernel<OP, 3, 3, OutT, DUAL, W, G, L>), grid, threads, 0, s, a);
    }
    return check_launch("singular_kernel");
}

template <int OP, typename OutT, bool DUAL>
static int launch_sing(const SingularArgs &a, hipStream_t s) {
    if (a.n_pairs == 0) return BEM_OK;
    if (a.n_pairs >= (OP == kMaxwellEFIE ? kSingLargePairsEfie : kSingLargePairs))
        return launch_sing_split<OP, OutT, DUAL, 4, 1, 1>(a, s);
    if (a.n_pairs >= (OpTraits<OP>::is_complex ? kSingMediumPairs : kSingMediumPairsReal))
        return launch_sing_split<OP, OutT, DUAL, 4, 4, 2>(a, s);
    if (a.n_pairs >= kSingWholePairs) return launch_sing_split<OP, OutT, DUAL, 4, 8, 2>(a, s);
    if (a.n_pairs >= kSingSmallPairs) return launch_sing_split<OP, OutT, DUAL, 4, 8, 6>(a, s);
    return launch_sing_split<OP, OutT, DUAL, 4, 16, 2>(a, s);
}

template <int OP, bool DUAL = false>
static int launch_sing_op(const SingularArgs &a, int out_dtype, hipStream_t s) {
    constexpr bool CPLX = OpTraits<OP>::is_complex;
    if (CPLX && out_dtype == BEM_C128) return launch_sing<OP, double, DUAL>(a, s);
    if (CPLX && out_dtype == BEM_C64) return launch_sing<OP, float, DUAL>(a, s);
    if (!CPLX && out_dtype == BEM_F64) return launch_sing<OP, double, DUAL>(a, s);
    if (!CPLX && out_dtype == BEM_F32) return launch_sing<OP, float, DUAL>(a, s);
    set_error("output dtype %d does not match operator %d", out_dtype, OP);
    return BEM_ERR_INVALID_ARGUMENT;
}

}  // namespace bem

using namespace bem;

static int singular_entry(int op, const bem_space_t *test, const bem_space_t *trial, int n_pairs,
                          const int32_t *pair_data, const double *test_points, const double *trial_points,
                          const double *weights, double k_re, double k_im, void *out, void *out2, int64_t ld,
                          int out_dtype, void *stream) {
    clear_error();
    if (!test || !trial || !out || (n_pairs > 0 && (!pair_data || !test_points || !trial_points || !weights))) {
        set_error("null argument");
        return BEM_ERR_INVALID_ARGUMENT;
    }
    if (n_pairs < 0) {
        set_error("negative pair count");
        return BEM_ERR_INVALID_ARGUMENT;
    }
    int rc;
    if ((rc = check_space(test, "test")) || (rc = check_space(trial, "trial"))) return rc;
    SingularArgs a;
    a.test = to_args(test);
    a.trial = to_args(trial);
    a.n_pairs = n_pairs;
    a.pairs = pair_data;
    a.tpts = test_points;
    a.spts = trial_points;
    a.wts = weights;
    a.kr = k_re;
    a.ki = k_im;
    a.out = out;
    a.out2 = out2;
    a.ld = ld;
    hipStream_t s = (hipStream_t)stream;
    if (out2) {
        if (op == BEM_LAPLACE_SINGLE_LAYER) return launch_sing_op<kLaplaceSL, true>(a, out_dtype, s);
        if (op == BEM_HELMHOLTZ_SINGLE_LAYER) return launch_sing_op<kHelmholtzSL, true>(a, out_dtype, s);
        set_error("the single/double layer pair needs a single-layer operator, got %d", op);
        return BEM_ERR_UNSUPPORTED;
    }
    switch (op) {
    case BEM_LAPLACE_SINGLE_LAYER: return launch_sing_op<kLaplaceSL>(a, out_dtype, s);
    case BEM_LAPLACE_DOUBLE_LAYER: return launch_sing_op<kLaplaceDL>(a, out_dtype, s);
    case BEM_LAPLACE_ADJOINT_DOUBLE_LAYER: return launch_sing_op<kLaplaceADL>(a, out_dtype, s);
    case BEM_HELMHOLTZ_SINGLE_LAYER: return launch_sing_op<kHelmholtzSL>(a, out_dtype, s);
    case BEM_HELMHOLTZ_DOUBLE_LAYER: return launch_sing_op<kHelmholtzDL>(a, out_dtype, s);
    case BEM_HELMHOLTZ_ADJOINT_DOUBLE_LAYER: return launch_sing_op<kHelmholtzADL>(a, out_dtype, s);
    case BEM_MAXWELL_ELECTRIC_FIELD: return launch_sing_op<kMaxwellEFIE>(a, out_dtype, s);
    case BEM_LAPLACE_HYPERSINGULAR: return launch_sing_op<kLaplaceHS>(a, out_dtype, s);
    case BEM_HELMHOLTZ_HYPERSINGULAR: return launch_sing_op<kHelmholtzHS>(a, out_dtype, s);
    case BEM_MAXWELL_MAGNETIC_FIELD:
        return mfie_singular_launch(a.test, a.trial, n_pairs, pair_data, test_points, trial_points, weights, k_re,
                                    k_im, out, ld, out_dtype, s);
    default: set_error("unsupported operator %d", op); return BEM_ERR_UNSUPPORTED;
    }
}

extern "C" int bem_singular_assemble(int op, const bem_space_t *test, const bem_space_t *trial, int n_pairs,
                                     const int32_t *pair_data, const double *test_points, const double *trial_points,
                                     const double *weights, double k_re, double k_im, void *out, int64_t ld,
                                     int out_dtype, void *stream) {
    return singular_entry(op, test, trial, n_pairs, pair_data, test_points, trial_points, weights, k_re, k_im, out,
                          nullptr, ld, out_dtype, stream);
}

extern "C" int bem_singular_assemble_sl_dl(int op, const bem_space_t *test, const bem_space_t *trial, int n_pairs,
                                           const int32_t *pair_data, const double *test_points,
                                           const double *trial_points, const double *weights, double k_re, double k_im,
                                           void *out_single, void *out_double, int64_t ld, int out_dtype,
                                           void *stream) {
    if (!out_double) {
        clear_error();
        set_error("null argument");
        return BEM_ERR_INVALID_ARGUMENT;
    }
    return singular_entry(op, test, trial, n_pairs, pair_data, test_points, trial_points, weights, k_re, k_im,
                          out_single, out_double, ld, out_dtype, stream);
}
