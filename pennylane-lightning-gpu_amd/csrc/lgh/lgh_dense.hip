// Dense matrices on four to thirteen target bits: application to a state
// (QubitUnitary and the like, StateVectorCudaManaged.hpp:1400-1472) and
// expectation values (getExpectationValueDeviceMatrix, :1649-1713).
//
// With the 2^k amplitudes of a group (all values of the target bits for one
// value of the others) as a column, both are a product M X of the 2^k x 2^k
// matrix with the 2^k x 2^(n-k) matrix of all groups: a contraction, done on
// the matrix cores in double precision (also for complex64 states, whose
// amplitudes are widened when they are staged).
#include <algorithm>

#include "lgh_internal.hpp"

using namespace lgh;

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

// A workgroup forms a tile of 16 H WR rows x 16 WC columns of M X, each of its
// four wavefronts 16 H x 16 of it as H blocks of 16 x 16: with the real and
// the imaginary parts 2 H independent chains of v_mfma_f64_16x16x4, of two
// each per four columns of M.  M and X pass through LDS in chunks of 16
// columns (rows of X), double-buffered: the next chunk is loaded into
// registers while the matrix cores work on this one.  64 x 32 (H = 2; 51 KiB
// of LDS, three workgroups per CU) from six target bits on, 32 x 64 with
// five, 16 x 64 (H = 1, one chunk) with four.  Bound by the double-precision
// matrix rate above 2^6 rows, below that by the state's reads and writes.
// 20 qubits, complex128, one workgroup per group of amplitudes with M read
// from global memory by every group before, the product now: 9 wires <H>
// 342 -> 124 us, a 6-wire unitary 52 -> 24 us.
constexpr int kChunk = 16;

typedef double d4 __attribute__((ext_vector_type(4)));

// Index bit of each matrix-index bit, least significant first (0 beyond the
// matrix's).  The loops over them have a fixed length, so that the kernel
// arguments they read are loaded once, together: a loop of as many steps as
// there are targets waited for a scalar load in every one of them.
struct Tbits {
    int k;
    int b[kMaxLdsK];
};
__device__ __forceinline__ uint64_t deposit(uint32_t m, const Tbits &tb) {
    uint64_t o = 0;
#pragma unroll
    for (int j = 0; j < kMaxLdsK; ++j) o |= uint64_t((m >> j) & 1u) << tb.b[j];
    return o;
}
__device__ __forceinline__ uint64_t column_base(uint64_t g, const Fixed &f) {
#pragma unroll
    for (int k = 0; k < kMaxFixed; ++k)
        if (k < f.cnt) g = ((g >> f.pos[k]) << (f.pos[k] + 1)) | (g & ((1ull << f.pos[k]) - 1ull));
    return g;
}

struct DenseArgs {
    uint64_t ngroups;     // columns of X
    uint64_t col0, ncols; // the launch's columns
    Fixed fx;
    uint64_t cmask;
    Tbits tb;
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Mode 0: M X into the state where X was read (all rows in one workgroup);
// 1: into tmp[row][column - col0]; 2: partial sums of conj(X) . (M X).
template <class R, int H, int WR, int WC, int Mode>
__global__ __launch_bounds__(kBlock) void k_dense_mm(const cx<R> *sv, cx<R> *dst, const cx<double> *__restrict__ mat,
                                                     double *__restrict__ partials, DenseArgs g) {
    static_assert(WR * WC == kWaves, "four wavefronts");
    constexpr int MT = 16 * H * WR, NT = 16 * WC;
    constexpr int kBufs = MT == 16 ? 1 : 2; // 16 rows: the matrix has one chunk
    constexpr int kA = MT * kChunk / kBlock, kB = (NT * kChunk + kBlock - 1) / kBlock; // loads per thread and chunk
    __shared__ cx<double> As[kBufs][MT][kChunk + 1];
    __shared__ cx<double> Bs[kBufs][kChunk][NT + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t D = 1u << g.tb.k;
    const uint32_t nrt = D / MT;
    const uint32_t row0 = (blockIdx.x % nrt) * MT;
    const uint64_t c0 = g.col0 + uint64_t(blockIdx.x / nrt) * NT;
    const uint64_t cend = g.col0 + g.ncols;

    // this thread's elements of a chunk: M[row0 + ar + ..][ac], X[bk + ..][bc]
    const int ac = tid % kChunk, ar = tid / kChunk;
    const int bc = tid % NT, bk = tid / NT;
    constexpr int kBStep = kBlock / NT;
    const bool bin = c0 + bc < cend;
    const uint64_t colbase = bin ? (column_base(c0 + bc, g.fx) | g.cmask) : 0;
    uint64_t boff[kB];
#pragma unroll
    for (int e = 0; e < kB; ++e) boff[e] = colbase | deposit(uint32_t(bk + e * kBStep), g.tb);
    cx<double> av[kA];
    cx<R> bv[kB];
    auto load = [&](uint32_t kc) {
        const uint64_t hi = deposit(kc, g.tb); // the chunk's high row bits: uniform
#pragma unroll
        for (int e = 0; e < kA; ++e)
            av[e] = mat[uint64_t(row0 + ar + e * (kBlock / kChunk)) * D + kc + ac];
#pragma unroll
        for (int e = 0; e < kB; ++e) bv[e] = bin ? sv[boff[e] | hi] : cx<R>{R(0), R(0)};
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int e = 0; e < kA; ++e) As[buf][ar + e * (kBlock / kChunk)][ac] = av[e];
#pragma unroll
        for (int e = 0; e < kB; ++e)
            Bs[buf][bk + e * kBStep][bc] = cx<double>{double(bv[e].re), double(bv[e].im)};
    };
    static_assert(NT * kChunk % kBlock == 0 && kBlock % NT == 0 && kBlock % kChunk == 0, "whole loads");

    const int wr = (w % WR) * 16 * H, wc = (w / WR) * 16;
    const int li = lane & 15, lk = lane >> 4;
    d4 yr[H] = {}, yi[H] = {};
    load(0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (uint32_t kc = 0; kc < D; kc += kChunk, buf ^= 1) {
        const bool more = kBufs > 1 && kc + kChunk < D;
        if (more) load(kc + kChunk);
#pragma unroll
        for (int kk = 0; kk < kChunk; kk += 4) {
            const cx<double> b = Bs[buf][kk + lk][wc + li];
            const double nbi = -b.im;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const cx<double> a = As[buf][wr + 16 * h + li][kk + lk];
                yr[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, yr[h], 0, 0, 0);
                yi[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, yi[h], 0, 0, 0);
                yr[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, nbi, yr[h], 0, 0, 0);
                yi[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, yi[h], 0, 0, 0);
            }
        }
        if (more) stage(buf ^ 1);
        __syncthreads(); // also: every read of X is done before the state is written
    }

    // block h, element r of a lane: row 16 h + (lane / 16) + 4 r, column lane % 16
    const uint64_t col = c0 + wc + li;
    const bool in = col < cend;
    if constexpr (Mode == 1) {
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = row0 + wr + 16 * h + lk + 4 * r;
                if (in) dst[uint64_t(row) * g.ncols + (col - g.col0)] = cx<R>{R(yr[h][r]), R(yi[h][r])};
            }
    } else {
        const uint64_t base = (in ? (column_base(col, g.fx) | g.cmask) : 0) | deposit(row0 + wr, g.tb) |
                              uint64_t(lk & 1) << g.tb.b[0] | uint64_t(lk >> 1) << g.tb.b[1];
        double er = 0.0, ei = 0.0;
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint64_t i = base | uint64_t(r & 1) << g.tb.b[2] | uint64_t(r >> 1) << g.tb.b[3] |
                                   uint64_t(h) << g.tb.b[4];
                if constexpr (Mode == 0) {
                    if (in) dst[i] = cx<R>{R(yr[h][r]), R(yi[h][r])};
                } else if (in) {
                    const cx<R> x = sv[i];
                    er += double(x.re) * yr[h][r] + double(x.im) * yi[h][r];
                    ei += double(x.re) * yi[h][r] - double(x.im) * yr[h][r];
                }
            }
        if constexpr (Mode == 2) {
            __shared__ double sh[2][kWaves];
            er = wave_sum(er);
            ei = wave_sum(ei);
            if (lane == 0) {
                sh[0][w] = er;
                sh[1][w] = ei;
            }
            __syncthreads();
            if (tid < 2) {
                double s = 0.0;
                for (int q = 0; q < kWaves; ++q) s += sh[tid][q];
                partials[uint64_t(tid) * gridDim.x + blockIdx.x] = s;
            }
        }
    }
}

// tmp[row][column - col0] back to the state
template <class R>
__global__ __launch_bounds__(kBlock) void k_dense_store(const cx<R> *__restrict__ tmp, cx<R> *__restrict__ sv,
                                                        DenseArgs g) {
    const uint64_t e = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    const uint64_t row = e / g.ncols, col = e - row * g.ncols;
    if (row >= (1ull << g.tb.k)) return;
    sv[column_base(g.col0 + col, g.fx) | g.cmask | deposit(uint32_t(row), g.tb)] = tmp[e];
}

DenseArgs dense_args(int n, const int *tbits, int k, const std::vector<int> &cbits, uint64_t cmask) {
    DenseArgs g{};
    std::vector<int> fixed = cbits;
    g.tb.k = k;
    for (int j = 0; j < k; ++j) {
        g.tb.b[k - 1 - j] = tbits[j];
        fixed.push_back(tbits[j]);
    }
    g.fx = make_fixed(fixed);
    g.cmask = cmask;
    g.ngroups = g.ncols = 1ull << (n - g.fx.cnt);
    return g;
}

// workgroups of a launch over g.ncols columns
// Five and six target bits with few columns: the time is one tile's chain of
// matrix instructions, and tiles of half the size with half the chain (H = 1)
// run on CUs that would be idle. A 6-wire unitary on 12 qubits, complex128: 40.3
// us a call with the large tiles, 38.4 here (44.8 with a thread per row of M);
// 2^18 amplitudes 43.4 and 39.6, 2^19 42.9 and 45.4.
constexpr uint64_t kDenseNarrow = 1 << 18; // amplitudes
bool dense_narrow(const DenseArgs &g) { return g.tb.k <= 6 && (g.ncols << g.tb.k) <= kDenseNarrow; }
unsigned dense_blocks(const DenseArgs &g) {
    const uint64_t mt = std::min(64, 1 << g.tb.k);
    const uint64_t nt = dense_narrow(g) && g.tb.k > 4 ? (g.tb.k == 5 ? 32 : 16) : g.tb.k <= 5 ? 64 : 32;
    return unsigned(((1ull << g.tb.k) / mt) * ((g.ncols + nt - 1) / nt));
}
template <class R, int Mode>
void dense_launch(hipStream_t st, const cx<R> *sv, cx<R> *dst, const cx<double> *mat, double *partials,
                  const DenseArgs &g) {
    auto kern = g.tb.k == 4   ? k_dense_mm<R, 1, 1, 4, Mode>
                : g.tb.k == 5 ? (dense_narrow(g) ? k_dense_mm<R, 1, 2, 2, Mode> : k_dense_mm<R, 2, 1, 4, Mode>)
                              : (dense_narrow(g) ? k_dense_mm<R, 1, 4, 1, Mode> : k_dense_mm<R, 2, 2, 2, Mode>);
    hipLaunchKernelGGL(kern, dim3(dense_blocks(g)), dim3(kBlock), 0, st, sv, dst, mat, partials, g);
    LGH_LAUNCH_CHECK();
}

constexpr size_t kSmallMatrix = size_t(1) << 20; // bytes that go through the pinned upload ring
// Columns whose rows do not all fit one workgroup (seven target bits and
// more) are formed in a buffer of at most this many amplitudes, small enough
// to stay in the last-level cache, and stored from there.
constexpr uint64_t kDenseTmp = 1ull << 22;

size_t al256(size_t b) { return (b + 255) & ~size_t(255); }

template <class R> void dense_apply_t(lgh_sv *sv, const KOp &op) {
    StreamCtx *ctx = sv->ctx;
    cx<R> *data = static_cast<cx<R> *>(sv->data);
    DenseArgs g = dense_args(sv->n, op.tbits, op.k, op.cbits, op.cmask);
    const uint64_t D = 1ull << op.k;
    const size_t mbytes = sizeof(cx<double>) * D * D;
    const bool small = mbytes <= kSmallMatrix, whole = op.k <= 6;
    const uint64_t chunk = std::min<uint64_t>(g.ngroups, std::max<uint64_t>(32, kDenseTmp / D));
    // Neither buffer is the workspace, which the adjoint sweep holds while it
    // applies a gate.  The rows' is bounded (64 MiB) and kept; a large
    // matrix's is given back once the stream has passed it.
    struct Matrix {
        StreamCtx *ctx;
        size_t bytes;
        void *p = nullptr;
        ~Matrix() {
            if (!p) return;
            (void)hipStreamSynchronize(ctx->stream);
            pool_free(ctx->device, p, bytes);
        }
    } large{ctx, mbytes};
    const cx<double> *mat;
    if (small) {
        mat = static_cast<const cx<double> *>(ctx->upload(op.mat.data(), mbytes));
    } else {
        large.p = pool_alloc(ctx->device, mbytes);
        LGH_HIP(hipMemcpyAsync(large.p, op.mat.data(), mbytes, hipMemcpyHostToDevice, ctx->stream));
        mat = static_cast<const cx<double> *>(large.p);
    }
    if (whole) {
        dense_launch<R, 0>(ctx->stream, data, data, mat, nullptr, g);
    } else {
        cx<R> *tmp = static_cast<cx<R> *>(ctx->gate_scratch(sizeof(cx<R>) * chunk * D));
        for (uint64_t c = 0; c < g.ngroups; c += chunk) {
            g.col0 = c;
            g.ncols = std::min(chunk, g.ngroups - c);
            dense_launch<R, 1>(ctx->stream, data, tmp, mat, nullptr, g);
            hipLaunchKernelGGL(k_dense_store<R>, dim3(unsigned((g.ncols * D + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                               ctx->stream, tmp, data, g);
            LGH_LAUNCH_CHECK();
        }
    }
    if (!small) ctx->sync(); // op.mat may go out of scope
}

template <class R>
void dense_expval_t(const lgh_sv *sv, const int *tbits, int k, const double *matrix, double *re_im) {
    StreamCtx *ctx = sv->ctx;
    const DenseArgs g = dense_args(sv->n, tbits, k, {}, 0);
    const size_t mbytes = sizeof(cx<double>) << (2 * k);
    const unsigned blocks = dense_blocks(g);
    char *ws = static_cast<char *>(ctx->workspace(al256(mbytes) + 2 * sizeof(double) * blocks));
    double *partials = reinterpret_cast<double *>(ws + al256(mbytes));
    double *host = static_cast<double *>(ctx->host_buffer(2 * sizeof(double)));
    const cx<double> *mat;
    if (mbytes <= kSmallMatrix) {
        mat = static_cast<const cx<double> *>(ctx->upload(matrix, mbytes));
    } else {
        LGH_HIP(hipMemcpyAsync(ws, matrix, mbytes, hipMemcpyHostToDevice, ctx->stream));
        mat = reinterpret_cast<const cx<double> *>(ws);
    }
    dense_launch<R, 2>(ctx->stream, static_cast<const cx<R> *>(sv->data), nullptr, mat, partials, g);
    launch_reduce(ctx, partials, int(blocks), 2, host);
    ctx->sync();
    re_im[0] = host[0];
    re_im[1] = host[1];
}

} // namespace

namespace lgh {

void dense_apply(lgh_sv *sv, const KOp &op) {
    if (sv->dtype == LGH_C128)
        dense_apply_t<double>(sv, op);
    else
        dense_apply_t<float>(sv, op);
}

void dense_expval(const lgh_sv *sv, const int *tbits, int k, const double *matrix, double *re_im) {
    if (sv->dtype == LGH_C128)
        dense_expval_t<double>(sv, tbits, k, matrix, re_im);
    else
        dense_expval_t<float>(sv, tbits, k, matrix, re_im);
}

} // namespace lgh
