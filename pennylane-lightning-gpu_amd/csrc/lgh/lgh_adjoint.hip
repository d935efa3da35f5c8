// Adjoint Jacobian (arXiv:2009.02823) with the generator product and the
// overlap fused into the reverse step.
//
// Reference: AdjointJacobianGPU::adjointJacobian
// (pennylane_lightning_gpu/src/algorithms/AdjointDiffGPU.hpp:499-596), which
// per trainable op copies lambda into mu, applies U^dagger to lambda, applies
// the generator to mu, takes one cuBLAS dot per observable followed by a
// blocking device-to-host copy, and applies U^dagger to every observable
// state.  Here one kernel pass per trainable op reads lambda and every
// H|lambda_j>, accumulates Im<H lambda_j | G lambda> without materialising
// mu, and writes U^dagger lambda and U^dagger H|lambda_j>; the Jacobian stays
// on the device until one copy at the end.
//
//   jac[j][t] = -2 * s * (inverse ? -1 : 1) * Im<H lambda_j | G lambda>
//   (AdjointDiffGPU.hpp:132-162, :578-582; s from :96-114)
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "lgh_fused.hpp"
#include "lgh_internal.hpp"

using namespace lgh;

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kBras = 8; // observable states per launch
// bytes of lambda and partial sums of the fused sweeps that run side by side
constexpr size_t kSideBySide = size_t(9) << 28;
// groups of more than this ask how much memory is free
constexpr size_t kSideBySideAsk = size_t(64) << 20;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

template <int NV> __device__ __forceinline__ void block_sum(double (&v)[NV]) {
    __shared__ double sh[NV][kWaves];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double s = wave_sum(v[k]);
        if (lane == 0) sh[k][wid] = s;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double s = lane < kWaves ? sh[k][lane] : 0.0;
            v[k] = wave_sum(s);
        }
    }
}

template <class R> __device__ __forceinline__ cx<double> up(cx<R> a) { return cx<double>{double(a.re), double(a.im)}; }

// Im(conj(b) * q)
template <class R> __device__ __forceinline__ double im_dot(cx<R> b, cx<double> q) {
    return double(b.re) * q.im - double(b.im) * q.re;
}

// Dense generator step for one 1-target gate with optional controls: one
// amplitude pair per thread.  U^dagger in the state precision, G in double.
template <class R, int NB>
__global__ __launch_bounds__(kBlock) void k_adj_pair1(cx<R> *__restrict__ psi, cx<R> *const *__restrict__ bras, int nb,
                                                      int upd_psi, uint64_t ngroups, Fixed fx, uint64_t cmask,
                                                      uint64_t tbit, cx<R> u00, cx<R> u01, cx<R> u10, cx<R> u11,
                                                      int with_gen, cx<double> g00, cx<double> g01, cx<double> g10,
                                                      cx<double> g11, double *__restrict__ partials) {
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = 0.0;
    const uint64_t g = xcd_block() * kBlock + threadIdx.x;
    if (g < ngroups) {
        const uint64_t i0 = expand(g, fx) | cmask, i1 = i0 | tbit;
        const cx<R> a0 = ldnt(psi + i0), a1 = ldnt(psi + i1);
        const cx<double> q0 = cfma(g01, up(a1), cmul(g00, up(a0)));
        const cx<double> q1 = cfma(g11, up(a1), cmul(g10, up(a0)));
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j < nb) {
                cx<R> *bj = bras[j];
                const cx<R> b0 = ldnt(bj + i0), b1 = ldnt(bj + i1);
                acc[j] += im_dot(b0, q0) + im_dot(b1, q1);
                stnt(bj + i0, cfma(u01, b1, cmul(u00, b0)));
                stnt(bj + i1, cfma(u11, b1, cmul(u10, b0)));
            }
        }
        if (upd_psi) {
            stnt(psi + i0, cfma(u01, a1, cmul(u00, a0)));
            stnt(psi + i1, cfma(u11, a1, cmul(u10, a0)));
        }
    }
    if (!with_gen) return;
    block_sum<NB>(acc);
    if (threadIdx.x == 0)
        for (int j = 0; j < nb; ++j) partials[size_t(j) * gridDim.x + blockIdx.x] = acc[j];
}

// Same step for an uncontrolled target bit t < 6: each thread streams one
// amplitude of every state and takes its partner from lane ^ 2^t.
template <class R, int NB>
__global__ __launch_bounds__(kBlock) void k_adj_lane1(cx<R> *__restrict__ psi, cx<R> *const *__restrict__ bras, int nb,
                                                      int upd_psi, uint64_t len, int tmask, cx<R> u00, cx<R> u01,
                                                      cx<R> u10, cx<R> u11, int with_gen, cx<double> g00,
                                                      cx<double> g01, cx<double> g10, cx<double> g11,
                                                      double *__restrict__ partials) {
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = 0.0;
    const uint64_t i = xcd_block() * kBlock + threadIdx.x;
    const bool ok = i < len;
    const bool hi = (threadIdx.x & tmask) != 0;
    const cx<R> us = hi ? u11 : u00, up_ = hi ? u10 : u01;
    const cx<double> gs = hi ? g11 : g00, gp = hi ? g10 : g01;
    const cx<R> a = ok ? ldnt(psi + i) : cx<R>{R(0), R(0)};
    const cx<R> ap = shfl_xor_cx(a, tmask);
    const cx<double> q = cfma(gp, up(ap), cmul(gs, up(a)));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        if (j < nb) {
            cx<R> *bj = bras[j];
            const cx<R> b = ok ? ldnt(bj + i) : cx<R>{R(0), R(0)};
            const cx<R> bp = shfl_xor_cx(b, tmask);
            acc[j] += im_dot(b, q);
            if (ok) stnt(bj + i, cfma(up_, bp, cmul(us, b)));
        }
    }
    if (upd_psi && ok) stnt(psi + i, cfma(up_, ap, cmul(us, a)));
    if (!with_gen) return;
    block_sum<NB>(acc);
    if (threadIdx.x == 0)
        for (int j = 0; j < nb; ++j) partials[size_t(j) * gridDim.x + blockIdx.x] = acc[j];
}

// K-target dense step (K = 2, 4): matrices staged in LDS, one group per thread.
template <class R, int K, int NB>
__global__ __launch_bounds__(kBlock) void k_adj_dense(cx<R> *__restrict__ psi, cx<R> *const *__restrict__ bras, int nb,
                                                      int upd_psi, uint64_t ngroups, Fixed fx, uint64_t cmask,
                                                      const uint64_t *__restrict__ offs_g,
                                                      const cx<R> *__restrict__ udag_g,
                                                      const cx<double> *__restrict__ gen_g,
                                                      double *__restrict__ partials) {
    constexpr int D = 1 << K;
    __shared__ cx<R> U[D * D];
    __shared__ cx<double> G[D * D];
    __shared__ uint64_t O[D];
    for (int t = threadIdx.x; t < D * D; t += kBlock) {
        U[t] = udag_g[t];
        if (gen_g) G[t] = gen_g[t];
    }
    for (int t = threadIdx.x; t < D; t += kBlock) O[t] = offs_g[t];
    __syncthreads();
    const bool with_gen = gen_g != nullptr;
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = 0.0;
    const uint64_t g = xcd_block() * kBlock + threadIdx.x;
    if (g < ngroups) {
        const uint64_t base = expand(g, fx) | cmask;
        cx<R> a[D];
#pragma unroll
        for (int m = 0; m < D; ++m) a[m] = ldnt(psi + (base | O[m]));
        cx<double> q[D];
        if (with_gen) {
#pragma unroll
            for (int r = 0; r < D; ++r) {
                cx<double> s{0.0, 0.0};
#pragma unroll
                for (int c = 0; c < D; ++c) s = cfma(G[r * D + c], up(a[c]), s);
                q[r] = s;
            }
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j < nb) {
                cx<R> *bj = bras[j];
                cx<R> b[D];
#pragma unroll
                for (int m = 0; m < D; ++m) b[m] = ldnt(bj + (base | O[m]));
                if (with_gen) {
#pragma unroll
                    for (int m = 0; m < D; ++m) acc[j] += im_dot(b[m], q[m]);
                }
#pragma unroll
                for (int r = 0; r < D; ++r) {
                    cx<R> s{R(0), R(0)};
#pragma unroll
                    for (int c = 0; c < D; ++c) s = cfma(U[r * D + c], b[c], s);
                    stnt(bj + (base | O[r]), s);
                }
            }
        }
        if (upd_psi) {
#pragma unroll
            for (int r = 0; r < D; ++r) {
                cx<R> s{R(0), R(0)};
#pragma unroll
                for (int c = 0; c < D; ++c) s = cfma(U[r * D + c], a[c], s);
                stnt(psi + (base | O[r]), s);
            }
        }
    }
    if (!with_gen) return;
    block_sum<NB>(acc);
    if (threadIdx.x == 0)
        for (int j = 0; j < nb; ++j) partials[size_t(j) * gridDim.x + blockIdx.x] = acc[j];
}

template <class R, int NB>
__global__ __launch_bounds__(kBlock) void k_adj_diag(cx<R> *__restrict__ psi, cx<R> *const *__restrict__ bras, int nb,
                                                     int upd_psi, uint64_t count, Fixed fx, uint64_t cmask,
                                                     uint64_t pmask, cx<R> ue, cx<R> uo, int with_gen, double ge,
                                                     double go, double *__restrict__ partials) {
    double acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = 0.0;
    const uint64_t g = xcd_block() * kBlock + threadIdx.x;
    if (g < count) {
        const uint64_t i = expand(g, fx) | cmask;
        const bool odd = __popcll(i & pmask) & 1;
        const cx<R> a = ldnt(psi + i);
        const cx<R> u = odd ? uo : ue;
        const double gv = odd ? go : ge;
        const cx<double> q{gv * double(a.re), gv * double(a.im)};
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j < nb) {
                const cx<R> b = ldnt(bras[j] + i);
                acc[j] += im_dot(b, q);
                stnt(bras[j] + i, cmul(u, b));
            }
        }
        if (upd_psi) stnt(psi + i, cmul(u, a));
    }
    if (!with_gen) return;
    block_sum<NB>(acc);
    if (threadIdx.x == 0)
        for (int j = 0; j < nb; ++j) partials[size_t(j) * gridDim.x + blockIdx.x] = acc[j];
}

// The step for a gate that mixes pairs of basis states (KOp::npair): reads and
// writes the pairs' amplitudes only, in the order of operations of k_adj_dense;
// blockIdx.y: the sweep, each with a lambda and an observable state of its own.
// A double excitation on 18 qubits: k_adj_dense 21 us and two more launches
// for its sum (8 us), 4.4 us here, the sums of a run of gates stored together.
template <class R> struct PairGen {
    cx<double> g[2][4];
};
template <class R, int NP>
__global__ __launch_bounds__(kBlock) void k_adj_pairs(void *lam_one, void *bra_one,
                                                      const AdjArrays *__restrict__ table, PairArgs<R> p,
                                                      PairGen<R> gen, int with_gen, double *__restrict__ partials,
                                                      uint64_t stride) {
    cx<R> *psi = static_cast<cx<R> *>(table ? table[blockIdx.y].lam : lam_one);
    cx<R> *bra = static_cast<cx<R> *>(table ? table[blockIdx.y].bra : bra_one);
    double acc[1] = {0.0};
    const uint64_t g = xcd_block() * kBlock + threadIdx.x;
    if (g < p.ngroups) {
        const uint64_t base = expand(g, p.fx) | p.cmask;
        cx<R> a0[NP], a1[NP], b0[NP], b1[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint64_t i = base | p.lo[q], j = base | p.hi[q];
            a0[q] = ldnt(psi + i);
            a1[q] = ldnt(psi + j);
            b0[q] = ldnt(bra + i);
            b1[q] = ldnt(bra + j);
        }
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint64_t i = base | p.lo[q], j = base | p.hi[q];
            const cx<R> *m = p.m[q];
            if (with_gen) {
                const cx<double> *gm = gen.g[q];
                acc[0] += im_dot(b0[q], cfma(gm[1], up(a1[q]), cmul(gm[0], up(a0[q]))));
                acc[0] += im_dot(b1[q], cfma(gm[3], up(a1[q]), cmul(gm[2], up(a0[q]))));
            }
            stnt(bra + i, cfma(m[1], b1[q], cmul(m[0], b0[q])));
            stnt(bra + j, cfma(m[3], b1[q], cmul(m[2], b0[q])));
            stnt(psi + i, cfma(m[1], a1[q], cmul(m[0], a0[q])));
            stnt(psi + j, cfma(m[3], a1[q], cmul(m[2], a0[q])));
        }
    }
    if (!with_gen) return;
    block_sum<1>(acc);
    if (threadIdx.x == 0) partials[blockIdx.y * stride + blockIdx.x] = acc[0];
}

template <class R>
void adj_pairs_t(StreamCtx *ctx, int n, const KOp &udag, const KGen *gen, const AdjArrays &one, const AdjArrays *table,
                 int count, double *partials, uint64_t stride) {
    const PairArgs<R> p = pair_args<R>(udag, n);
    PairGen<R> pg{};
    const size_t D = size_t(1) << udag.k;
    for (int q = 0; gen && q < udag.npair; ++q) {
        const size_t r = size_t(udag.pair_row[q]), s = r ^ size_t(udag.pair_flip);
        pg.g[q][0] = to_cx<double>(gen->mat[r * D + r]);
        pg.g[q][1] = to_cx<double>(gen->mat[r * D + s]);
        pg.g[q][2] = to_cx<double>(gen->mat[s * D + r]);
        pg.g[q][3] = to_cx<double>(gen->mat[s * D + s]);
    }
    auto kern = udag.npair == 1 ? k_adj_pairs<R, 1> : k_adj_pairs<R, 2>;
    hipLaunchKernelGGL(kern, dim3(unsigned((p.ngroups + kBlock - 1) / kBlock), unsigned(count)), dim3(kBlock), 0,
                       ctx->stream, one.lam, one.bra, table, p, pg, int(gen != nullptr), partials, stride);
    LGH_LAUNCH_CHECK();
}

// Row sums of the per-workgroup partials in two deterministic stages:
// k_row_chunks sums fixed contiguous slices of each row (grid: slices x rows),
// k_jac_store sums the slice results of row j and scales them into the
// Jacobian column.
constexpr int kSlices = 256;

__global__ __launch_bounds__(kBlock) void k_row_chunks(const double *__restrict__ partials, int nparts,
                                                       double *__restrict__ slices) {
    const int row = blockIdx.y;
    const int per = (nparts + kSlices - 1) / kSlices;
    const int lo = blockIdx.x * per, hi = min(lo + per, nparts);
    const double *p = partials + size_t(row) * nparts;
    double v[1] = {0.0};
    for (int b = lo + threadIdx.x; b < hi; b += kBlock) v[0] += p[b];
    block_sum<1>(v);
    if (threadIdx.x == 0) slices[size_t(row) * kSlices + blockIdx.x] = v[0];
}

__global__ __launch_bounds__(kBlock) void k_jac_store(const double *__restrict__ slices, double *__restrict__ jac,
                                                      int64_t ntp, int64_t col, double factor) {
    double v[1] = {threadIdx.x < kSlices ? slices[size_t(blockIdx.x) * kSlices + threadIdx.x] : 0.0};
    block_sum<1>(v);
    if (threadIdx.x == 0) jac[blockIdx.x * ntp + col] = factor * v[0];
}

bool is_prep(const lgh_op &op) { return op.gate < 0; }

// Launch geometry of one fused step: workgroups of kBlock threads, one
// amplitude (lane kernel), pair or group per thread.
struct StepShape {
    enum Kind { LANE1, PAIR1, DENSE, DIAG } kind;
    Fixed fx;
    uint64_t count;
    unsigned blocks;
};

StepShape step_shape(int n, const KOp &udag) {
    StepShape s{};
    if (udag.kind == KOp::DIAG) {
        s.kind = StepShape::DIAG;
        s.fx = make_fixed(udag.cbits);
    } else {
        std::vector<int> fixed_bits = udag.cbits;
        for (int i = 0; i < udag.k; ++i) fixed_bits.push_back(udag.tbits[i]);
        s.fx = make_fixed(fixed_bits);
        if (udag.k == 1)
            s.kind = (udag.cmask == 0 && udag.tbits[0] < 6 && n >= 6) ? StepShape::LANE1 : StepShape::PAIR1;
        else
            s.kind = StepShape::DENSE;
    }
    s.count = s.kind == StepShape::LANE1 ? (1ull << n) : (1ull << (n - s.fx.cnt));
    s.blocks = unsigned((s.count + kBlock - 1) / kBlock);
    return s;
}

// Calls f(std::integral_constant<int, NB>) with the smallest NB in {1, 2, 4, 8} >= nb.
template <class F> void with_nb(int nb, F &&f) {
    if (nb <= 1)
        f(std::integral_constant<int, 1>{});
    else if (nb <= 2)
        f(std::integral_constant<int, 2>{});
    else if (nb <= 4)
        f(std::integral_constant<int, 4>{});
    else
        f(std::integral_constant<int, 8>{});
}

template <class R>
void fused_step(lgh_sv *lam, cx<R> **bras_dev, int nobs, const KOp &udag, const KGen *gen, double *partials) {
    StreamCtx *ctx = lam->ctx;
    hipStream_t st = ctx->stream;
    cx<R> *psi = static_cast<cx<R> *>(lam->data);
    const int nbatches = std::max(1, (nobs + kBras - 1) / kBras);
    const StepShape sh = step_shape(lam->n, udag);
    const int wg = gen ? 1 : 0;
    auto batch = [&](int b, auto launch) {
        const int nb = std::max(0, std::min(kBras, nobs - b * kBras));
        launch(bras_dev + b * kBras, nb, int(b == nbatches - 1), partials + size_t(b) * kBras * sh.blocks);
        LGH_LAUNCH_CHECK();
    };
    if (sh.kind == StepShape::DIAG) {
        const double ge = gen ? gen->g_even : 0.0, go = gen ? gen->g_odd : 0.0;
        for (int b = 0; b < nbatches; ++b)
            batch(b, [&](cx<R> **bp, int nb, int upd, double *pb) {
                with_nb(nb, [&](auto NBc) {
                    hipLaunchKernelGGL((k_adj_diag<R, decltype(NBc)::value>), dim3(sh.blocks), dim3(kBlock), 0, st,
                                       psi, bp, nb, upd, sh.count, sh.fx, udag.cmask, udag.pmask,
                                       to_cx<R>(udag.d_even), to_cx<R>(udag.d_odd), wg, ge, go, pb);
                });
            });
        return;
    }
    if (sh.kind != StepShape::DENSE) {
        const cx<R> u00 = to_cx<R>(udag.mat[0]), u01 = to_cx<R>(udag.mat[1]), u10 = to_cx<R>(udag.mat[2]),
                    u11 = to_cx<R>(udag.mat[3]);
        cx<double> gm[4] = {};
        if (gen)
            for (int i = 0; i < 4; ++i) gm[i] = to_cx<double>(gen->mat[size_t(i)]);
        for (int b = 0; b < nbatches; ++b)
            batch(b, [&](cx<R> **bp, int nb, int upd, double *pb) {
                with_nb(nb, [&](auto NBc) {
                    constexpr int NB = decltype(NBc)::value;
                    if (sh.kind == StepShape::LANE1)
                        hipLaunchKernelGGL((k_adj_lane1<R, NB>), dim3(sh.blocks), dim3(kBlock), 0, st, psi, bp, nb,
                                           upd, sh.count, 1 << udag.tbits[0], u00, u01, u10, u11, wg, gm[0], gm[1],
                                           gm[2], gm[3], pb);
                    else
                        hipLaunchKernelGGL((k_adj_pair1<R, NB>), dim3(sh.blocks), dim3(kBlock), 0, st, psi, bp, nb,
                                           upd, sh.count, sh.fx, udag.cmask, 1ull << udag.tbits[0], u00, u01, u10,
                                           u11, wg, gm[0], gm[1], gm[2], gm[3], pb);
                });
            });
        return;
    }
    // DENSE with K in {2, 4}: one upload of offsets | U^dagger | G
    const int D = 1 << udag.k;
    const size_t b_off = sizeof(uint64_t) * D, b_u = sizeof(cx<R>) * D * D, b_g = sizeof(cx<double>) * D * D;
    const size_t o_u = (b_off + 15) & ~size_t(15), o_g = (o_u + b_u + 15) & ~size_t(15);
    std::vector<unsigned char> blob(o_g + b_g);
    uint64_t *offs = reinterpret_cast<uint64_t *>(blob.data());
    for (int m = 0; m < D; ++m) {
        uint64_t o = 0;
        for (int j = 0; j < udag.k; ++j)
            if ((m >> (udag.k - 1 - j)) & 1) o |= 1ull << udag.tbits[j];
        offs[m] = o;
    }
    cx<R> *u = reinterpret_cast<cx<R> *>(blob.data() + o_u);
    cx<double> *gmat = reinterpret_cast<cx<double> *>(blob.data() + o_g);
    for (int i = 0; i < D * D; ++i) {
        u[i] = to_cx<R>(udag.mat[size_t(i)]);
        gmat[i] = gen ? to_cx<double>(gen->mat[size_t(i)]) : cx<double>{0.0, 0.0};
    }
    unsigned char *dblob = static_cast<unsigned char *>(ctx->upload(blob.data(), blob.size()));
    const uint64_t *d_off = reinterpret_cast<const uint64_t *>(dblob);
    const cx<R> *d_u = reinterpret_cast<const cx<R> *>(dblob + o_u);
    const cx<double> *d_g = gen ? reinterpret_cast<const cx<double> *>(dblob + o_g) : nullptr;
    for (int b = 0; b < nbatches; ++b)
        batch(b, [&](cx<R> **bp, int nb, int upd, double *pb) {
            if (udag.k != 2 && udag.k != 4)
                throw Error(LGH_ERR_UNSUPPORTED, "no fused adjoint kernel for a " + std::to_string(udag.k) +
                                                     "-target generator");
            with_nb(nb, [&](auto NBc) {
                constexpr int NB = decltype(NBc)::value;
                if (udag.k == 2)
                    hipLaunchKernelGGL((k_adj_dense<R, 2, NB>), dim3(sh.blocks), dim3(kBlock), 0, st, psi, bp, nb,
                                       upd, sh.count, sh.fx, udag.cmask, d_off, d_u, d_g, pb);
                else
                    hipLaunchKernelGGL((k_adj_dense<R, 4, NB>), dim3(sh.blocks), dim3(kBlock), 0, st, psi, bp, nb,
                                       upd, sh.count, sh.fx, udag.cmask, d_off, d_u, d_g, pb);
            });
        });
}

// dst = Z-word(zmask) src: the sign (-1)^popcount(i & zmask) per amplitude
template <class R>
__global__ __launch_bounds__(kBlock) void k_zsign(cx<R> *__restrict__ dst, const cx<R> *__restrict__ src, uint64_t len,
                                                  uint64_t zmask) {
    const uint64_t i = xcd_block() * kBlock + threadIdx.x;
    if (i >= len) return;
    const cx<R> a = ldnt(src + i);
    stnt(dst + i, (__popcll(i & zmask) & 1) ? cx<R>{-a.re, -a.im} : a);
}

template <class R> void zsign(lgh_sv *dst, const void *src, uint64_t zmask, hipStream_t stream) {
    const uint64_t len = dst->length();
    hipLaunchKernelGGL(k_zsign<R>, dim3(unsigned((len + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                       static_cast<cx<R> *>(dst->data), static_cast<const cx<R> *>(src), len, zmask);
    LGH_LAUNCH_CHECK();
}

// zmasks (nullable): observable j is the Z word zmasks[j] and bras[j] is
// scratch that the sweep fills with Z_j psi (inside its first reverse pass
// where that pass is fused).
template <class R>
void adjoint_t(const lgh_sv *psi_in, lgh_sv *const *bras_in, int nobs, const lgh_op *ops, int64_t nops,
               const int64_t *tp, int64_t ntp, bool apply_ops, double *jac_host, const uint64_t *zmasks) {
    const int n = psi_in->n;
    StreamCtx *ctx = psi_in->ctx;
    // The observable states may belong to other streams: what those still do is
    // waited for, and the sweep works on them in psi's stream throughout (the
    // gates that run on their own too), which it waits for before it returns.
    std::vector<lgh_sv> views;
    std::vector<lgh_sv *> bras;
    views.reserve(size_t(nobs));
    for (int j = 0; j < nobs; ++j) {
        if (bras_in[j]->ctx != ctx) bras_in[j]->ctx->sync();
        views.push_back(*bras_in[j]);
        views.back().ctx = ctx;
        bras.push_back(&views.back());
    }
    const bool fused_path = fusion_enabled() && fused_partials_bytes(n, psi_in->device) > 0 && nobs > 0;
    // Working copies of psi, freed once the stream has been waited for.
    struct Buffers {
        const lgh_sv *like;
        std::vector<void *> ptrs;
        void *take() {
            ptrs.reserve(ptrs.size() + 1);
            ptrs.push_back(pool_alloc(like->device, like->bytes));
            return ptrs.back();
        }
        // gives back all but the first `keep`, none of which has been used yet
        void trim(size_t keep) {
            for (; ptrs.size() > keep; ptrs.pop_back()) pool_free(like->device, ptrs.back(), like->bytes);
        }
        ~Buffers() {
            (void)hipStreamSynchronize(like->ctx->stream);
            trim(0);
        }
    } buffers{psi_in, {}};
    // The fused sweep reads lambda's starting values from psi itself when no
    // forward application is asked for; the other forms work on a copy.
    lgh_sv lam = *psi_in;
    const void *start = psi_in->data;
    if (!fused_path || apply_ops) {
        start = lam.data = buffers.take();
        LGH_HIP(hipMemcpyAsync(lam.data, psi_in->data, psi_in->bytes, hipMemcpyDeviceToDevice, ctx->stream));
    }
    if (apply_ops)
        for (int64_t i = 0; i < nops; ++i)
            if (!is_prep(ops[i])) launch_kop(&lam, compile_op(ops[i], n, false));
    // Z-word observable states: formed here unless the fused sweep forms them
    if (zmasks && !fused_path)
        for (int j = 0; j < nobs; ++j) zsign<R>(bras[j], lam.data, zmasks[j], ctx->stream);

    // Sweeps that run side by side in the fused path share the launches of a
    // pass: a small state leaves the device idle on its own, a large one at
    // the end of every pass.  Two layers of StronglyEntanglingLayers with
    // <Z_w> on every wire, complex128, one sweep after another and side by
    // side: 12 qubits 3180 and 570 us (the sweeps of a 4-layer ring circuit),
    // 18 qubits 3329 and 1269, 20 qubits 4677 and 2785, 22 qubits 12.3 and
    // 10.0 ms, 24 qubits 43 and 40.5 ms.  The limit bounds what the call itself
    // takes for them, a lambda and the partial sums of each; a group that
    // needs much takes at most half of the memory that is free, so that the
    // rest is left to the runtime and to other streams.
    const size_t b_one = fused_path ? fused_partials_bytes(n, psi_in->device) : 0;
    const size_t per_sweep = psi_in->bytes + b_one + AdjPasses::kTableBytes;
    int group = fused_path ? int(std::max<size_t>(1, std::min<size_t>({size_t(nobs), size_t(65535),
                                                                             kSideBySide / per_sweep})))
                                 : 1;
    if (size_t(group) * per_sweep > kSideBySideAsk) {
        size_t free_bytes = 0, total_bytes = 0;
        if (hipMemGetInfo(&free_bytes, &total_bytes) == hipSuccess)
            group = int(std::max<size_t>(1, std::min<size_t>(size_t(group), free_bytes / 2 / per_sweep)));
        else
            (void)hipGetLastError();
    }
    // workspace: [jac (nobs*ntp) | bra pointers | partials of the steps | slices | fused partials | sweep table]
    // the widest step shape has one thread per amplitude
    const unsigned max_blocks = unsigned(((1ull << n) + kBlock - 1) / kBlock);
    const int nbatches = std::max(1, (nobs + kBras - 1) / kBras);
    auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t b_jac = al(sizeof(double) * size_t(std::max<int64_t>(1, nobs * ntp)));
    const size_t b_ptr = al(sizeof(void *) * size_t(nbatches * kBras));
    // the fused path's standalone steps take one observable at a time
    const size_t b_part = al(sizeof(double) * (fused_path ? 1 : size_t(nbatches) * kBras) * max_blocks);
    const size_t b_slices = al(sizeof(double) * kBras * kSlices);
    // lambda per sweep of a group; a single sweep may use up the forward state formed above
    const bool own = fused_path && apply_ops && nobs == 1;
    const size_t held = buffers.ptrs.size();
    size_t b_fused = 0;
    char *ws = nullptr;
    for (;;) {
        b_fused = al(b_one * size_t(group));
        const size_t b_tab = fused_path ? al(AdjPasses::kTableBytes * size_t(group)) : 0;
        try {
            while (fused_path && !own && buffers.ptrs.size() < held + size_t(group)) (void)buffers.take();
            ws = static_cast<char *>(ctx->workspace(b_jac + b_ptr + b_part + b_slices + b_fused + b_tab));
            break;
        } catch (const Error &e) {
            if (group == 1 || e.code != LGH_ERR_OUT_OF_MEMORY) throw;
            group /= 2; // what memory is left takes fewer at a time
            buffers.trim(held + size_t(group));
        }
    }
    double *jac_dev = reinterpret_cast<double *>(ws);
    cx<R> **bras_dev = reinterpret_cast<cx<R> **>(ws + b_jac);
    double *partials = reinterpret_cast<double *>(ws + b_jac + b_ptr);
    double *slices = reinterpret_cast<double *>(ws + b_jac + b_ptr + b_part);
    double *fpartials = reinterpret_cast<double *>(ws + b_jac + b_ptr + b_part + b_slices);
    void *table = ws + b_jac + b_ptr + b_part + b_slices + b_fused;
    std::vector<void *> hp(size_t(nbatches * kBras), nullptr);
    for (int j = 0; j < nobs; ++j) hp[size_t(j)] = bras[j]->data;
    // The pointer table is copied before the first step that reads it.  Most
    // fused sweeps have none, and a copy as the stream's first command after a
    // wait cost a lone 12-qubit sweep 17 us.
    bool bras_there = false;
    auto need_bras = [&] {
        if (!bras_there) ctx->copy_in(bras_dev, hp.data(), sizeof(void *) * hp.size());
        bras_there = true;
    };
    LGH_HIP(hipMemsetAsync(jac_dev, 0, sizeof(double) * size_t(std::max<int64_t>(1, nobs * ntp)), ctx->stream));

    if (fused_path) {
        // Fused reverse sweeps.  Ops before the earliest trainable one are never visited.
        std::vector<KOp> udag;
        std::vector<KGen> gens;
        std::vector<int> slot;
        std::vector<double> fac;
        int64_t pidx = -1, k = 0;
        bool started = false;
        for (int64_t i = 0; i < nops; ++i) {
            const lgh_op &o = ops[i];
            if (is_prep(o)) continue;
            int col = -1;
            if (o.num_params > 0) {
                ++pidx;
                if (k < ntp && pidx == tp[k]) col = int(k++);
            }
            if (col < 0 && !started) continue;
            started = true;
            udag.push_back(compile_op(o, n, true));
            if (col >= 0) {
                gens.push_back(compile_generator(o, n, udag.back()));
                fac.push_back(-2.0 * gens.back().scale * (o.inverse ? -1.0 : 1.0));
            } else {
                gens.emplace_back();
                fac.push_back(0.0);
            }
            slot.push_back(col);
        }
        AdjPasses passes(psi_in, udag, gens, slot, fac, nobs > group);
        std::vector<lgh_sv> lams(size_t(group), *psi_in);
        for (int j = 0; j < group; ++j) lams[size_t(j)].data = own ? lam.data : buffers.ptrs[held + size_t(j)];
        auto standalone = [&](const AdjSweep &sw, const KOp &u, const KGen *g, int64_t col, double f) {
            const bool fusedk = u.kind == KOp::DIAG || (u.kind == KOp::DENSE && (u.k == 1 || u.k == 2 || u.k == 4));
            if (!fusedk) {
                launch_kop(sw.lam, u);
                launch_kop(sw.bra, u);
                return;
            }
            const ptrdiff_t j = (sw.jac_row - jac_dev) / ntp;
            need_bras();
            fused_step<R>(sw.lam, bras_dev + j, 1, u, g, partials);
            if (g) {
                const unsigned blocks = step_shape(n, u).blocks;
                hipLaunchKernelGGL(k_row_chunks, dim3(kSlices, 1), dim3(kBlock), 0, ctx->stream, partials, int(blocks),
                                   slices);
                hipLaunchKernelGGL(k_jac_store, dim3(1), dim3(kBlock), 0, ctx->stream, slices, sw.jac_row, ntp, col, f);
                LGH_LAUNCH_CHECK();
            }
        };
        for (int j0 = 0; j0 < nobs; j0 += group) {
            std::vector<AdjSweep> sweeps;
            for (int j = j0; j < std::min(nobs, j0 + group); ++j) {
                AdjSweep sw;
                sw.lam = &lams[size_t(j - j0)];
                sw.lam_src = own ? nullptr : start;
                sw.bra = bras[j];
                sw.jac_row = jac_dev + size_t(j) * size_t(ntp);
                if (zmasks) {
                    sw.bra_from_z = true;
                    sw.zmask = zmasks[j];
                    sw.materialize = [&, j] { zsign<R>(bras[j], start, zmasks[j], ctx->stream); };
                }
                sweeps.push_back(std::move(sw));
            }
            passes.run(sweeps.data(), int(sweeps.size()), fpartials, table, standalone);
        }
        if (nobs * ntp > 0)
            LGH_HIP(hipMemcpyAsync(jac_host, jac_dev, sizeof(double) * size_t(nobs * ntp), hipMemcpyDeviceToHost,
                                   ctx->stream));
        ctx->sync();
        return;
    }

    need_bras();
    ctx->sync(); // the first kernels start sooner behind a copy that has been waited for (see above)
    int64_t num_param_ops = 0;
    for (int64_t i = 0; i < nops; ++i)
        if (!is_prep(ops[i]) && ops[i].num_params > 0) ++num_param_ops;
    int64_t tp_pos = ntp - 1;
    int64_t param_idx = num_param_ops - 1;
    for (int64_t op = nops - 1; op >= 0; --op) {
        const lgh_op &o = ops[op];
        if (is_prep(o)) continue;
        if (tp_pos < 0) break;
        const KOp udag = compile_op(o, n, true);
        const bool trainable = o.num_params > 0 && param_idx == tp[tp_pos];
        if (trainable && nobs > 0) {
            const KGen gen = compile_generator(o, n, udag);
            if (udag.kind == KOp::DENSE && udag.k != 1 && udag.k != 2 && udag.k != 4)
                throw Error(LGH_ERR_UNSUPPORTED, "no fused adjoint kernel for this operation");
            fused_step<R>(&lam, bras_dev, nobs, udag, &gen, partials);
            const unsigned blocks = step_shape(n, udag).blocks;
            const double factor = -2.0 * gen.scale * (o.inverse ? -1.0 : 1.0);
            for (int b = 0; b < nbatches; ++b) {
                const int nb = std::min(kBras, nobs - b * kBras);
                if (nb <= 0) break;
                hipLaunchKernelGGL(k_row_chunks, dim3(kSlices, nb), dim3(kBlock), 0, ctx->stream,
                                   partials + size_t(b) * kBras * blocks, int(blocks), slices);
                hipLaunchKernelGGL(k_jac_store, dim3(nb), dim3(kBlock), 0, ctx->stream, slices,
                                   jac_dev + size_t(b) * kBras * ntp, ntp, tp_pos, factor);
                LGH_LAUNCH_CHECK();
            }
        } else if (udag.kind == KOp::DIAG ||
                   (udag.kind == KOp::DENSE && (udag.k == 1 || udag.k == 2 || udag.k == 4))) {
            fused_step<R>(&lam, bras_dev, nobs, udag, nullptr, partials); // U^dagger on every state, one pass
        } else if (udag.kind != KOp::NOP) {
            launch_kop(&lam, udag);
            for (int j = 0; j < nobs; ++j) launch_kop(bras[j], udag);
        }
        if (trainable) --tp_pos;
        if (o.num_params > 0) --param_idx;
    }
    if (nobs * ntp > 0) {
        LGH_HIP(hipMemcpyAsync(jac_host, jac_dev, sizeof(double) * size_t(nobs * ntp), hipMemcpyDeviceToHost,
                               ctx->stream));
    }
    ctx->sync();
}

} // namespace

namespace lgh {

unsigned adj_pairs_blocks(int n, const KOp &udag) {
    const uint64_t groups = 1ull << (n - udag.k - int(udag.cbits.size()));
    return unsigned((groups + kBlock - 1) / kBlock);
}

void launch_adj_pairs(StreamCtx *ctx, lgh_dtype dtype, int n, const KOp &udag, const KGen *gen, const AdjArrays &one,
                      const AdjArrays *table, int count, double *partials, uint64_t stride) {
    if (dtype == LGH_C128)
        adj_pairs_t<double>(ctx, n, udag, gen, one, table, count, partials, stride);
    else
        adj_pairs_t<float>(ctx, n, udag, gen, one, table, count, partials, stride);
}

} // namespace lgh

extern "C" {

static void adjoint_entry(const lgh_sv *psi, lgh_sv *const *bras, int32_t num_obs, const lgh_op *ops,
                      int64_t num_ops, const int64_t *trainable, int64_t num_trainable, int32_t apply_operations,
                      double *jac, const uint64_t *zmasks) {
    LGH_REQUIRE(psi, "null state");
    LGH_REQUIRE(num_trainable > 0, "No trainable parameters provided.");
    LGH_REQUIRE(trainable && (num_obs == 0 || (bras && jac)) && (num_ops == 0 || ops), "null pointer");
    LGH_REQUIRE(num_obs >= 0, "negative observable count");
    for (int32_t j = 0; j < num_obs; ++j) {
        LGH_REQUIRE(bras[j], "null observable state");
        LGH_REQUIRE(bras[j]->n == psi->n && bras[j]->dtype == psi->dtype && bras[j]->device == psi->device,
                    "observable state does not match psi");
    }
    for (int64_t i = 1; i < num_trainable; ++i)
        LGH_REQUIRE(trainable[i] > trainable[i - 1], "trainable parameters must be sorted and unique");
    for (int64_t i = 0; i < num_ops; ++i) {
        if (ops[i].gate < 0) continue; // state preparation: skipped by the reverse sweep
        LGH_REQUIRE(ops[i].num_params <= 1,
                    "The operation is not supported using the adjoint differentiation method");
        validate_op(ops[i], psi->n);
    }
    if (zmasks)
        for (int32_t j = 0; j < num_obs; ++j)
            LGH_REQUIRE((zmasks[j] >> psi->n) == 0, "Z-word mask beyond the state's qubits");
    DeviceGuard g(psi->device);
    if (psi->dtype == LGH_C128)
        adjoint_t<double>(psi, bras, num_obs, ops, num_ops, trainable, num_trainable, apply_operations != 0, jac,
                          zmasks);
    else
        adjoint_t<float>(psi, bras, num_obs, ops, num_ops, trainable, num_trainable, apply_operations != 0, jac,
                         zmasks);
}

lgh_status lgh_adjoint_jacobian(const lgh_sv *psi, lgh_sv *const *bras, int32_t num_obs, const lgh_op *ops,
                                int64_t num_ops, const int64_t *trainable, int64_t num_trainable,
                                int32_t apply_operations, double *jac) {
    return guard([&] {
        Range rg("lgh_adjoint_jacobian");
        adjoint_entry(psi, bras, num_obs, ops, num_ops, trainable, num_trainable, apply_operations, jac, nullptr);
    });
}

lgh_status lgh_adjoint_jacobian_zwords(const lgh_sv *psi, lgh_sv *const *bras, const uint64_t *zmasks,
                                       int32_t num_obs, const lgh_op *ops, int64_t num_ops, const int64_t *trainable,
                                       int64_t num_trainable, int32_t apply_operations, double *jac) {
    return guard([&] {
        Range rg("lgh_adjoint_jacobian_zwords");
        LGH_REQUIRE(num_obs == 0 || zmasks, "null pointer");
        adjoint_entry(psi, bras, num_obs, ops, num_ops, trainable, num_trainable, apply_operations, jac, zmasks);
    });
}

} // extern "C"
