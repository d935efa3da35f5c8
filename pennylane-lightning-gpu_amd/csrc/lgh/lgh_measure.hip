// Measurements and BLAS-like helpers: inner products, axpy/scale, dense and
// Pauli-word expectation values, resident CSR SpMV (+ fused dot),
// probabilities and the seeded sampler.
//
// Reference counterparts (pennylane_lightning_gpu/src/...):
//   innerProdC_CUDA / scaleAndAddC_CUDA / scaleC_CUDA   util/cuda_helpers.hpp:456-560
//   getExpectationValueDeviceMatrix                    simulator/StateVectorCudaManaged.hpp:1649-1713
//   getExpectationValuePauliWords                      simulator/StateVectorCudaManaged.hpp:1071-1148
//   getExpectationValueOnSparseSpMV                    simulator/StateVectorCudaManaged.hpp:795-922
//   SparseHamiltonianGPU::applyInPlace                 algorithms/ObservablesGPU.hpp:469-587
//   probability                                        simulator/StateVectorCudaManaged.hpp:931-970
//   generate_samples                                   simulator/StateVectorCudaManaged.hpp:982-1061
//
// Every reduction is deterministic for a given problem size: each workgroup
// reduces a fixed contiguous chunk (wavefront shuffles, then an LDS tree) to
// one partial, and a second kernel sums the partials in a fixed order.
#include <algorithm>
#include <cstring>
#include <map>
#include <type_traits>
#include <utility>

#include "lgh_internal.hpp"

namespace lgh {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Block-wide sums of NV values; the results are valid in thread 0.
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
            s = wave_sum(s);
            v[k] = s;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_final_reduce(const double *__restrict__ partials, int nparts,
                                                         double *__restrict__ out) {
    // one workgroup per value
    const double *p = partials + size_t(blockIdx.x) * nparts;
    double v[1] = {0.0};
    for (int b = threadIdx.x; b < nparts; b += kBlock) v[0] += p[b];
    block_sum<1>(v);
    if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

// chunked partitioning of [0, count) over a bounded number of workgroups
struct Chunks {
    uint64_t chunk;
    unsigned blocks;
};
Chunks chunks_for(uint64_t count, int device, uint64_t per_thread = 4) {
    const uint64_t max_blocks = uint64_t(std::max(1, sm_count(device))) * 8;
    uint64_t blocks = (count + kBlock * per_thread - 1) / (kBlock * per_thread);
    blocks = std::max<uint64_t>(1, std::min(blocks, max_blocks));
    uint64_t chunk = (count + blocks - 1) / blocks;
    blocks = (count + chunk - 1) / chunk;
    return {chunk, unsigned(std::max<uint64_t>(1, blocks))};
}

} // namespace

void launch_reduce(StreamCtx *ctx, const double *partials, int nparts, int nvals, double *out_dev) {
    hipLaunchKernelGGL(k_final_reduce, dim3(nvals), dim3(kBlock), 0, ctx->stream, partials, nparts, out_dev);
    LGH_LAUNCH_CHECK();
}

// Reduction workspace: partials (nvals * nparts).
struct RedBuf {
    double *partials;
};
static RedBuf red_buf(StreamCtx *ctx, int nvals, int nparts) {
    return {static_cast<double *>(ctx->workspace(sizeof(double) * size_t(nvals) * nparts))};
}

// Sums each of the nvals rows of partials and returns the values: the
// reduction writes them into pinned host memory itself, so no copy follows
// it (a copy of 16 bytes is one more 4 us launch in a chain of three).
static void reduce_to_host(StreamCtx *ctx, const double *partials, int nparts, int nvals, double *out) {
    double *h = static_cast<double *>(ctx->host_buffer(sizeof(double) * nvals));
    launch_reduce(ctx, partials, nparts, nvals, h);
    ctx->sync();
    std::memcpy(out, h, sizeof(double) * nvals);
}

} // namespace lgh

using namespace lgh;

namespace {

// ---------------------------------------------------------------- BLAS-like

template <class R>
__global__ __launch_bounds__(kBlock) void k_inner(const cx<R> *__restrict__ a, const cx<R> *__restrict__ b,
                                                  uint64_t len, uint64_t chunk, double *__restrict__ partials) {
    const uint64_t lo = uint64_t(blockIdx.x) * chunk, hi = min(lo + chunk, len);
    double v[2] = {0.0, 0.0};
    for (uint64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const cx<R> x = a[i], y = b[i];
        v[0] += double(x.re) * y.re + double(x.im) * y.im;
        v[1] += double(x.re) * y.im - double(x.im) * y.re;
    }
    block_sum<2>(v);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = v[0];
        partials[gridDim.x + blockIdx.x] = v[1];
    }
}

template <class R>
__global__ __launch_bounds__(kBlock) void k_axpy(cx<R> *__restrict__ y, const cx<R> *__restrict__ x, uint64_t len,
                                                 cx<R> a) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < len) y[i] = cfma(a, x[i], y[i]);
}

// dst = P src for the Pauli word P with X/Y bits xmask, Y/Z bits zmask and
// ny Y factors: (P src)[i] = i^ny (-1)^popcount(j & zmask) src[j], j = i ^ xmask.
// One read and one write per amplitude; the reads of a wavefront stay in the
// same cache lines as its writes when xmask has only low bits, and are whole
// lines otherwise.
template <class R>
__global__ __launch_bounds__(kBlock) void k_pauli_from(cx<R> *__restrict__ dst, const cx<R> *__restrict__ src,
                                                       uint64_t len, uint64_t xmask, uint64_t zmask, int ny) {
    const uint64_t i = xcd_block() * kBlock + threadIdx.x;
    if (i >= len) return;
    const uint64_t j = i ^ xmask;
    cx<R> v = ldnt(src + j);
    if (ny & 2) v = cx<R>{-v.re, -v.im};       // i^2 = -1
    if (ny & 1) v = cx<R>{-v.im, v.re};        // times i
    if (__popcll(j & zmask) & 1) v = cx<R>{-v.re, -v.im};
    stnt(dst + i, v);
}

template <class R>
__global__ __launch_bounds__(kBlock) void k_scale(cx<R> *__restrict__ x, uint64_t len, cx<R> a) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < len) x[i] = cmul(a, x[i]);
}

// ---------------------------------------------------------------- dense expval

template <int K> struct Offs {
    uint64_t o[1 << K];
};

template <class R, int K>
__global__ __launch_bounds__(kBlock) void k_expval_reg(const cx<R> *__restrict__ sv, uint64_t ngroups, uint64_t chunk,
                                                       Fixed fx, Offs<K> offs, const cx<double> *__restrict__ mat,
                                                       double *__restrict__ partials) {
    constexpr int D = 1 << K;
    __shared__ cx<double> sm[D * D];
    for (int t = threadIdx.x; t < D * D; t += kBlock) sm[t] = mat[t];
    __syncthreads();
    const uint64_t lo = uint64_t(blockIdx.x) * chunk, hi = min(lo + chunk, ngroups);
    double acc[2] = {0.0, 0.0};
    for (uint64_t g = lo + threadIdx.x; g < hi; g += kBlock) {
        const uint64_t base = expand(g, fx);
        cx<double> v[D];
#pragma unroll
        for (int m = 0; m < D; ++m) {
            cx<R> t = sv[base | offs.o[m]];
            v[m] = cx<double>{double(t.re), double(t.im)};
        }
#pragma unroll
        for (int r = 0; r < D; ++r) {
            cx<double> y{0.0, 0.0};
#pragma unroll
            for (int c = 0; c < D; ++c) y = cfma(sm[r * D + c], v[c], y);
            acc[0] += v[r].re * y.re + v[r].im * y.im;
            acc[1] += v[r].re * y.im - v[r].im * y.re;
        }
    }
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = acc[0];
        partials[gridDim.x + blockIdx.x] = acc[1];
    }
}

// ---------------------------------------------------------------- Pauli words
//
// <P> for a word with X/Y bits f (flip mask), Z/Y bits zy and nY factors Y:
// P|i> = i^nY (-1)^popcount(i & zy) |i ^ f>, so
//   <P> = Re( i^nY sum_i (-1)^popcount(i & zy) conj(psi_{i^f}) psi_i ),
// real for a Hermitian word.  Kernels accumulate the term's real and
// imaginary parts and keep the one i^nY turns into the real part (`phase` =
// nY mod 4: +re, -im, -re, +im).
//
// Words are grouped into passes by tiles: a pass holds a set of index bits
// (the three lowest, so that loads cover 128-byte runs, and up to nine more
// chosen per pass); a workgroup stages each tile of 2^12 amplitudes (all
// combinations of the pass's bits for one value of the others) in LDS, and
// every word of the pass whose flip bits are tile bits finds each partner
// i ^ f in the tile.  One read of the state then serves every word of the
// pass, whatever their flip masks.  Words with more flip bits than a tile
// holds take the pair kernel below, one pass per flip mask.
//
// Each wavefront of a workgroup has words of its own and walks the whole tile
// for them, 64 pairs (i, i ^ f) at a time in 32 steps:
//  - the terms of i and i ^ f are equal, so one bit of f (the pivot) is kept
//    clear in i, and the sum over pairs counts twice;
//  - words of one flip mask (and the same parity of nY) that a wavefront holds
//    share the pair products conj(psi_{i^f}) psi_i, kept in registers; words
//    without flips take |psi_i|^2 of two amplitudes a step;
//  - a word's sign is (-1)^parity of the index bits outside the tile (one
//    scalar per tile), of the five bits that the steps run over (one FMA with
//    +1 or -1 per level of a binary tree over the 32 products) and of the
//    lane's bits (a constant of the whole sum, applied once at the end).
// So a word costs 31 FMAs a lane and tile, a flip mask 64 LDS reads and 64
// FMAs more.  64 KiB of LDS: two workgroups of eight wavefronts per CU.
// Bound by the state reads, one per launch.  24 qubits, 256 words,
// complex128: 3712 us in 16 launches with tiles of 2^11 and an LDS read per
// word and amplitude, 1091 us in 13 launches here.
constexpr int kPTileBits = 12;       // amplitudes per tile: 2^12
constexpr int kPFixedBits = 3;       // lowest index bits in every tile
constexpr int kPBlock = 512;
constexpr int kPWaves = kPBlock / 64;
constexpr int kPSlots = 8;           // words per wavefront and launch
constexpr int kPassWords = kPWaves * kPSlots;
constexpr int kPSteps = 1 << (kPTileBits - 7);
constexpr int kPLevels = kPTileBits - 7; // bits the steps run over
constexpr int kMaxWordsPerPass = 8;  // words per pair-kernel launch

enum : uint32_t { kPEven = 0, kPOdd = 1, kPSquare = 2, kPSquareDiff = 3 }; // products of a flip mask

// One word of a launch, in device memory; read with scalar loads.
struct alignas(16) PWord {
    double sign[kPLevels]; // +1 / -1 by the Z/Y mask over the bits that the steps run over
    double scale;          // real part of i^nY or -i^nY, times two for pairs
    uint64_t zy;           // Z/Y mask over the index bits outside the tile
    uint32_t flip;         // flip mask in tile-local bits (the pivot bit where the word has no flips)
    uint32_t pivot;        // the bit kept clear
    uint32_t zlane;        // Z/Y mask over the lane's bits
    uint32_t kind;         // kPEven..kPSquareDiff; bit 4: first word of its products in the wavefront
    uint32_t row;          // row of the partials
    uint32_t pad;
};
// the launch's words, [wavefront][slot]
struct PLaunch {
    uint32_t slots[kPWaves];
    PWord word[kPWaves][kPSlots];
};
typedef __attribute__((address_space(4))) const PWord CPWord;
typedef __attribute__((address_space(4))) const PLaunch CPLaunch;

// tile-local bit r is global index bit bit[r] (ascending)
struct PTile {
    int g;
    int bit[kPTileBits];
};

// Half of a launch's words as kernel arguments, and the kernel that writes them
// to device memory: for callers that may neither allocate nor wait.
struct PHalf {
    uint32_t w[sizeof(PLaunch) / 8];
};
static_assert(sizeof(PLaunch) % 8 == 0 && sizeof(PHalf) <= 3072, "two halves, each within the kernel arguments");
__global__ __launch_bounds__(256) void k_pauli_put(uint32_t *__restrict__ dst, PHalf h) {
    for (unsigned i = threadIdx.x; i < sizeof(PHalf) / 4; i += 256) dst[i] = h.w[i];
}

// The products of a flip mask, 32 pairs per lane.
template <class R, uint32_t Kind>
__device__ __forceinline__ void pair_products(const char *tile, uint32_t pivot, uint32_t flip, int lane,
                                              double (&x)[kPSteps]) {
    constexpr uint32_t A = sizeof(cx<R>);
    // the lane's part of i: its six bits around the pivot; then the steps
    // count in the bits above, around the pivot too
    const uint32_t low = uint32_t(lane) & ((1u << pivot) - 1u), high = uint32_t(lane) >> pivot;
    const uint32_t at = pivot < 6 ? (high << (pivot + 1)) | low : uint32_t(lane);
    const uint32_t pm = pivot < 6 ? 0u : A << pivot, step = pivot < 6 ? 128 * A : 64 * A, fl = flip * A;
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kPSteps; ++k) {
        const uint32_t i = at * A + c;
        const cx<R> a = *reinterpret_cast<const cx<R> *>(tile + i);
        const cx<R> b = *reinterpret_cast<const cx<R> *>(tile + (i ^ fl));
        if constexpr (Kind == kPEven)
            x[k] = double(b.re) * a.re + double(b.im) * a.im;
        else if constexpr (Kind == kPOdd)
            x[k] = double(b.re) * a.im - double(b.im) * a.re;
        else if constexpr (Kind == kPSquare)
            x[k] = (double(a.re) * a.re + double(a.im) * a.im) + (double(b.re) * b.re + double(b.im) * b.im);
        else
            x[k] = (double(a.re) * a.re + double(a.im) * a.im) - (double(b.re) * b.re + double(b.im) * b.im);
        c = ((c | pm) + step) & ~pm;
    }
}

template <class R>
__global__ __launch_bounds__(kPBlock, 4) void k_pauli_tile(const cx<R> *__restrict__ sv, uint64_t ntiles,
                                                           uint64_t tiles_per_block, Fixed tfx, PTile tm,
                                                           const PLaunch *__restrict__ launch,
                                                           double *__restrict__ partials) {
    __shared__ cx<R> tile[1 << kPTileBits];
    constexpr int kPer = (1 << kPTileBits) / kPBlock;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const CPLaunch *cl = (const CPLaunch *)launch;
    const CPWord *cw = &cl->word[w][0];
    const int slots = int(cl->slots[w]);
    const uint32_t tsz = 1u << tm.g;
    uint64_t off = 0, koff[3];
#pragma unroll
    for (int r = 0; r < 9; ++r)
        if (r < tm.g && ((tid >> r) & 1)) off |= 1ull << tm.bit[r];
#pragma unroll
    for (int r = 0; r < 3; ++r) koff[r] = 9 + r < tm.g ? 1ull << tm.bit[9 + r] : 0;
    static_assert(kPBlock == 512 && kPer == 8, "nine bits on the threads, three on the loads");
    double acc[kPSlots];
#pragma unroll
    for (int q = 0; q < kPSlots; ++q) acc[q] = 0.0;
    const uint64_t t0 = uint64_t(blockIdx.x) * tiles_per_block, t1 = min(t0 + tiles_per_block, ntiles);
    for (uint64_t t = t0; t < t1; ++t) {
        const uint64_t base = expand(t, tfx);
        {
            cx<R> v[kPer];
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const uint64_t ko = (k & 1 ? koff[0] : 0) | (k & 2 ? koff[1] : 0) | (k & 4 ? koff[2] : 0);
                v[k] = uint32_t(tid + k * kPBlock) < tsz ? ldnt(sv + (base | off | ko)) : cx<R>{R(0), R(0)};
            }
#pragma unroll
            for (int k = 0; k < kPer; ++k) tile[tid + k * kPBlock] = v[k];
        }
        __syncthreads();
        double x[kPSteps];
#pragma unroll 1
        for (int q = 0; q < slots; ++q) {
            const uint32_t kind = cw[q].kind;
            if (kind & 16u) {
                const char *tp = reinterpret_cast<const char *>(tile);
                const uint32_t pivot = cw[q].pivot, flip = cw[q].flip;
                switch (kind & 3u) {
                case kPEven: pair_products<R, kPEven>(tp, pivot, flip, lane, x); break;
                case kPOdd: pair_products<R, kPOdd>(tp, pivot, flip, lane, x); break;
                case kPSquare: pair_products<R, kPSquare>(tp, pivot, flip, lane, x); break;
                default: pair_products<R, kPSquareDiff>(tp, pivot, flip, lane, x); break;
                }
            }
            // sum over the steps with the sign of each of their bits
            double y[kPSteps / 2];
#pragma unroll
            for (int k = 0; k < kPSteps / 2; ++k) y[k] = fma(x[2 * k + 1], cw[q].sign[0], x[2 * k]);
#pragma unroll
            for (int l = 1; l < kPLevels; ++l)
#pragma unroll
                for (int k = 0; k < (kPSteps >> (l + 1)); ++k) y[k] = fma(y[2 * k + 1], cw[q].sign[l], y[2 * k]);
            const double s = (__popcll(base & cw[q].zy) & 1) ? -y[0] : y[0];
#pragma unroll
            for (int u = 0; u < kPSlots; ++u)
                if (u == q) acc[u] += s;
        }
        __syncthreads(); // the next tile overwrites the LDS copy
    }
#pragma unroll
    for (int q = 0; q < kPSlots; ++q) {
        if (q >= slots) break;
        const bool neg = __popc(uint32_t(lane) & cw[q].zlane) & 1;
        const double s = wave_sum(neg ? -acc[q] : acc[q]);
        if (lane == 0) partials[size_t(cw[q].row) * gridDim.x + blockIdx.x] = cw[q].scale * s;
    }
}

struct WordSet {
    int count;
    uint64_t zy[kMaxWordsPerPass];
    uint32_t phase[kMaxWordsPerPass];
};

// <P_w> for words that share one flip mask f.  With f != 0 each pair
// (i, i^f) is read once: its two terms s_i conj(psi_j) psi_i and
// s_j conj(psi_i) psi_j are added together.
template <class R>
__global__ __launch_bounds__(kBlock) void k_pauli(const cx<R> *__restrict__ sv, uint64_t count, uint64_t chunk,
                                                  int pivot, uint64_t flip, WordSet ws,
                                                  double *__restrict__ partials) {
    const uint64_t lo = uint64_t(blockIdx.x) * chunk, hi = min(lo + chunk, count);
    double acc[2 * kMaxWordsPerPass];
#pragma unroll
    for (int k = 0; k < 2 * kMaxWordsPerPass; ++k) acc[k] = 0.0;
    for (uint64_t g = lo + threadIdx.x; g < hi; g += kBlock) {
        if (pivot < 0) {
            const cx<R> a = sv[g];
            const double p = double(a.re) * a.re + double(a.im) * a.im;
#pragma unroll
            for (int w = 0; w < kMaxWordsPerPass; ++w)
                if (w < ws.count) acc[2 * w] += (__popcll(g & ws.zy[w]) & 1) ? -p : p;
        } else {
            const uint64_t lo_bits = g & ((1ull << pivot) - 1ull);
            const uint64_t i = ((g >> pivot) << (pivot + 1)) | lo_bits;
            const uint64_t j = i ^ flip;
            const cx<R> a = sv[i], b = sv[j];
            // conj(b) a and conj(a) b = conj(conj(b) a)
            const double re = double(b.re) * a.re + double(b.im) * a.im;
            const double im = double(b.re) * a.im - double(b.im) * a.re;
#pragma unroll
            for (int w = 0; w < kMaxWordsPerPass; ++w) {
                if (w < ws.count) {
                    const double si = (__popcll(i & ws.zy[w]) & 1) ? -1.0 : 1.0;
                    const double sj = (__popcll(j & ws.zy[w]) & 1) ? -1.0 : 1.0;
                    acc[2 * w] += (si + sj) * re;
                    acc[2 * w + 1] += (si - sj) * im;
                }
            }
        }
    }
    double val[kMaxWordsPerPass];
#pragma unroll
    for (int w = 0; w < kMaxWordsPerPass; ++w) {
        const uint32_t ph = w < ws.count ? ws.phase[w] : 0u;
        const double re = acc[2 * w], im = acc[2 * w + 1];
        val[w] = ph == 0 ? re : ph == 1 ? -im : ph == 2 ? -re : im;
    }
    block_sum<kMaxWordsPerPass>(val);
    if (threadIdx.x == 0)
        for (int w = 0; w < ws.count; ++w) partials[size_t(w) * gridDim.x + blockIdx.x] = val[w];
}

// ---------------------------------------------------------------- sums of Pauli words
//
// dst = sum_w c_w P_w src: (P src)_i = i^nY (-1)^popcount(j & zy) src_j with
// j = i ^ f.  The words are grouped into tile passes as above; a thread keeps
// eight amplitudes of the result.  Words of one flip mask first add up their
// coefficient per amplitude (real for even nY, imaginary for odd), then the
// partner is read from LDS once for all of them.  Every pass but the first
// adds to dst.  18 qubits, 64 random words, complex128: 3 passes of 22 us; two
// launches per word before, some 500 us.
constexpr int kSPer = (1 << kPTileBits) / kPBlock;

// One word of a pass, in device memory.
struct alignas(16) SWord {
    double c;      // coefficient, with the sign of i^nY
    uint64_t zy;   // Z/Y mask over the index bits outside the tile
    uint32_t flip; // flip mask in tile-local bits
    uint32_t zl;   // Z/Y mask over the tile's bits; bit 16: nY odd; 17: last word of its flip mask
    double pad;
};
typedef __attribute__((address_space(4))) const SWord CSWord;

template <class R>
__global__ __launch_bounds__(kPBlock) void k_pauli_sum(cx<R> *__restrict__ dst, const cx<R> *__restrict__ src,
                                                       uint64_t ntiles, Fixed tfx, PTile tm,
                                                       const SWord *__restrict__ words, int count, int add) {
    __shared__ cx<R> tile[1 << kPTileBits];
    const uint32_t tid = threadIdx.x, tsz = 1u << tm.g;
    const CSWord *cw = (const CSWord *)words;
    uint64_t off = 0, koff[3];
#pragma unroll
    for (int r = 0; r < 9; ++r)
        if (r < tm.g && ((tid >> r) & 1)) off |= 1ull << tm.bit[r];
#pragma unroll
    for (int r = 0; r < 3; ++r) koff[r] = 9 + r < tm.g ? 1ull << tm.bit[9 + r] : 0;
    auto kindex = [&](int k) { return (k & 1 ? koff[0] : 0) | (k & 2 ? koff[1] : 0) | (k & 4 ? koff[2] : 0); };
    const uint64_t base = expand(blockIdx.x, tfx);
#pragma unroll
    for (int k = 0; k < kSPer; ++k)
        if (tid + k * kPBlock < tsz) tile[tid + k * kPBlock] = src[base | off | kindex(k)];
    __syncthreads();
    cx<double> y[kSPer];
    double re[kSPer], im[kSPer];
#pragma unroll
    for (int k = 0; k < kSPer; ++k) {
        y[k] = cx<double>{0.0, 0.0};
        re[k] = im[k] = 0.0;
    }
#pragma unroll 1
    for (int q = 0; q < count; ++q) {
        const uint32_t f = cw[q].flip, zl = cw[q].zl;
        // the sign of j = i ^ f: outside the tile that of i
        const uint32_t outer = uint32_t(__popcll(base & cw[q].zy)) + uint32_t(__popc((tid ^ f) & zl & (kPBlock - 1)));
        const double c = (outer & 1) ? -cw[q].c : cw[q].c;
        const uint32_t zk = (zl & 0xffffu) >> 9, fk = f >> 9;
        if ((zl >> 16) & 1u) {
#pragma unroll
            for (int k = 0; k < kSPer; ++k) im[k] += (__popc((uint32_t(k) ^ fk) & zk) & 1) ? -c : c;
        } else {
#pragma unroll
            for (int k = 0; k < kSPer; ++k) re[k] += (__popc((uint32_t(k) ^ fk) & zk) & 1) ? -c : c;
        }
        if ((zl >> 17) & 1u) {
#pragma unroll
            for (int k = 0; k < kSPer; ++k) {
                if (tid + k * kPBlock < tsz) {
                    const cx<R> p = tile[(tid + k * kPBlock) ^ f];
                    y[k] = cfma(cx<double>{re[k], im[k]}, cx<double>{double(p.re), double(p.im)}, y[k]);
                }
                re[k] = im[k] = 0.0;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kSPer; ++k)
        if (tid + k * kPBlock < tsz) {
            const uint64_t i = base | off | kindex(k);
            if (add) {
                const cx<R> o = dst[i];
                y[k].re += double(o.re);
                y[k].im += double(o.im);
            }
            dst[i] = cx<R>{R(y[k].re), R(y[k].im)};
        }
}

// A word that flips more bits than a tile has: dst (+)= c P src.
template <class R>
__global__ __launch_bounds__(kBlock) void k_pauli_add(cx<R> *__restrict__ dst, const cx<R> *__restrict__ src,
                                                      uint64_t len, uint64_t flip, uint64_t zy, int odd, double c,
                                                      int add) {
    const uint64_t i = xcd_block() * kBlock + threadIdx.x;
    if (i >= len) return;
    const uint64_t j = i ^ flip;
    const cx<R> p = src[j];
    const double s = (__popcll(j & zy) & 1) ? -c : c;
    cx<double> y = odd ? cx<double>{-s * double(p.im), s * double(p.re)} : cx<double>{s * double(p.re), s * double(p.im)};
    if (add) {
        y.re += double(dst[i].re);
        y.im += double(dst[i].im);
    }
    dst[i] = cx<R>{R(y.re), R(y.im)};
}

// The sum without words.  Written, not scaled: dst may hold infinities and NaN.
template <class R> __global__ __launch_bounds__(kBlock) void k_zero(cx<R> *__restrict__ dst, uint64_t len) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < len) stnt(dst + i, cx<R>{R(0), R(0)});
}

// ---------------------------------------------------------------- CSR

// Short rows (see csr_streams): a workgroup takes kBlock / T consecutive rows,
// whose entries lie together, and stages them in LDS as one stream, every load
// full and all loads of a step in flight at once.  From there neighbouring
// lanes walk neighbouring rows, each of the T parts of the workgroup every
// T-th entry of its row: the columns of neighbouring rows at one place of the
// row are near each other in an operator on qubits, so a load of x touches
// few cache lines.  Rows of any length are right; a long one only leaves the
// other rows' lanes idle while it streams.  T follows the average, so that a
// workgroup's rows fill about one step.
// Bound by reading the matrix (70 us of the 89 it takes at the first of these
// sizes).  <H> of the 21-entry rows of a transverse-field Ising chain on 20
// qubits, call to call: 150 -> 100 us in complex128 (32-bit indices; with 64
// the matrix has 528 MB for 440), 119 -> 82 in complex64, against 16 lanes
// per row, whose loads of x took a cache line per lane and whose second round
// had 5 of 16 lanes at work.
constexpr int kCsrItems = 6;
__global__ __launch_bounds__(kBlock) void k_narrow(int32_t *__restrict__ dst, const int64_t *__restrict__ src,
                                                   int64_t count) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < count) dst[i] = int32_t(src[i]);
}

// Rows of random columns, 2^18 of 30 and 44 entries: 90 and 121 us, with 32
// lanes per row 92 and 136, in complex128; in complex64 73 and 95, with 32
// lanes 71 and 89.  Of 18 entries and less the stream is faster in both.
//
// A long row among short ones is walked by T lanes of its workgroup, or by the
// 32 of a row: 90 and 140 ns an entry and lane.  The rest of the matrix takes
// the time of reading it as a stream, and with 32 lanes per row 2 us for every
// 16384 rows, the grid's, in each of which the same workgroup may get a long
// one.  One dense row above a diagonal, complex128: 1050 us as a stream, 115 with
// 32 lanes on 2^14 rows, 20 and 3.7 ms on 2^18; every 256th row of 2000 entries, the
// others of one: 111 and 40 us on 2^14 rows, 280 and 590 on 2^18.
inline int csr_parts(double avg) { return avg <= 6 ? 1 : avg <= 12 ? 2 : avg <= 24 ? 4 : 8; }
template <class R> bool csr_streams(const lgh_csr *csr) {
    const double avg = csr->avg_row, longest = double(csr->longest_row);
    if (avg > (sizeof(R) == 8 ? 48 : 24)) return false;
    if (longest <= 4 * avg + 16) return true;
    const double stream = 2.2e-4 * double(csr->b_val + csr->b_idx) + 90.0 * longest / csr_parts(avg);
    const double lanes = (2000.0 + 140.0 * longest / 32) * std::max(1.0, double(csr->rows) / 16384);
    return stream <= lanes;
}
constexpr int kCsrPerCu = 5; // workgroups per CU that the LDS allows
template <class I, class R, int T>
__global__ __launch_bounds__(kBlock) void k_csr_stream(const I *__restrict__ indptr, const I *__restrict__ indices,
                                                       const cx<R> *__restrict__ vals, const cx<R> *__restrict__ x,
                                                       cx<R> *__restrict__ y, int64_t rows,
                                                       double *__restrict__ partials) {
    constexpr int kRows = kBlock / T, kStep = kCsrItems * kBlock, kAhead = 3;
    __shared__ __align__(16) cx<R> s_val[kStep];
    __shared__ I s_col[kStep];
    cx<double> *const s_sum = reinterpret_cast<cx<double> *>(s_val); // after the last step
    const int tid = threadIdx.x, part = tid / kRows;
    double acc[2] = {0.0, 0.0};
    for (int64_t r0 = int64_t(blockIdx.x) * kRows; r0 < rows; r0 += int64_t(gridDim.x) * kRows) {
        const int64_t row = r0 + tid % kRows;
        const bool live = row < rows;
        const int64_t b = live ? int64_t(indptr[row]) : 0, e = live ? int64_t(indptr[row + 1]) : 0;
        const int64_t kb = indptr[r0], ke = indptr[r0 + kRows < rows ? r0 + kRows : rows];
        const cx<R> xr = live ? x[row] : cx<R>{R(0), R(0)};
        double yr = 0.0, yi = 0.0;
        for (int64_t k0 = kb; k0 < ke; k0 += kStep) {
            const int n = int(ke - k0 < kStep ? ke - k0 : kStep);
            cx<R> v[kCsrItems];
            I col[kCsrItems];
#pragma unroll
            for (int q = 0; q < kCsrItems; ++q)
                if (q * kBlock + tid < n) {
                    col[q] = __builtin_nontemporal_load(indices + k0 + q * kBlock + tid);
                    v[q] = ldnt(vals + k0 + q * kBlock + tid);
                }
            __syncthreads(); // the step before has been read
#pragma unroll
            for (int q = 0; q < kCsrItems; ++q)
                if (q * kBlock + tid < n) {
                    s_col[q * kBlock + tid] = col[q];
                    s_val[q * kBlock + tid] = v[q];
                }
            __syncthreads();
            const int lo = int((b > k0 ? b : k0) - k0), hi = int((e < k0 + n ? e : k0 + n) - k0);
            for (int k = lo + part; k < hi; k += kAhead * T) {
                cx<R> xv[kAhead], m[kAhead];
#pragma unroll
                for (int q = 0; q < kAhead; ++q) {
                    const int at = k + q * T < hi ? k + q * T : k;
                    xv[q] = x[s_col[at]];
                    m[q] = s_val[at];
                }
#pragma unroll
                for (int q = 0; q < kAhead; ++q)
                    if (k + q * T < hi) {
                        yr += double(m[q].re) * xv[q].re - double(m[q].im) * xv[q].im;
                        yi += double(m[q].re) * xv[q].im + double(m[q].im) * xv[q].re;
                    }
            }
        }
        if (!y) { // every part on its own: the sum over rows takes them all
            if (part == 0 || b + part < e) {
                acc[0] += double(xr.re) * yr + double(xr.im) * yi;
                acc[1] += double(xr.re) * yi - double(xr.im) * yr;
            }
            continue;
        }
        if constexpr (T > 1) {
            __syncthreads();
            s_sum[tid] = cx<double>{yr, yi};
            __syncthreads();
            if (part == 0)
                for (int q = 1; q < T; ++q) {
                    yr += s_sum[q * kRows + tid].re;
                    yi += s_sum[q * kRows + tid].im;
                }
        }
        if (live && part == 0) y[row] = cx<R>{R(yr), R(yi)};
        __syncthreads();
    }
    if (y) return;
    block_sum<2>(acc);
    if (tid == 0) {
        partials[blockIdx.x] = acc[0];
        partials[gridDim.x + blockIdx.x] = acc[1];
    }
}

// Longer rows: L lanes per row.
template <class I, class R, int L>
__global__ __launch_bounds__(kBlock) void k_csr(const I *__restrict__ indptr, const I *__restrict__ indices,
                                                const cx<R> *__restrict__ vals, const cx<R> *__restrict__ x,
                                                cx<R> *__restrict__ y, int64_t rows, double *__restrict__ partials) {
    // L lanes per row; rows assigned round-robin over all sub-groups
    const int lane = threadIdx.x & (L - 1);
    const int64_t sub = (int64_t(blockIdx.x) * kBlock + threadIdx.x) / L;
    const int64_t nsub = int64_t(gridDim.x) * kBlock / L;
    double acc[2] = {0.0, 0.0};
    for (int64_t r = sub; r < rows; r += nsub) {
        const int64_t b = indptr[r], e = indptr[r + 1];
        double yr = 0.0, yi = 0.0;
        for (int64_t k = b + lane; k < e; k += L) {
            const cx<R> v = vals[k];
            const cx<R> xv = x[indices[k]];
            yr += double(v.re) * xv.re - double(v.im) * xv.im;
            yi += double(v.re) * xv.im + double(v.im) * xv.re;
        }
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) {
            yr += __shfl_xor(yr, off, L);
            yi += __shfl_xor(yi, off, L);
        }
        if (lane == 0) {
            if (y) {
                y[r] = cx<R>{R(yr), R(yi)};
            } else {
                const cx<R> p = x[r];
                acc[0] += double(p.re) * yr + double(p.im) * yi;
                acc[1] += double(p.re) * yi - double(p.im) * yr;
            }
        }
    }
    if (y) return;
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = acc[0];
        partials[gridDim.x + blockIdx.x] = acc[1];
    }
}

// ---------------------------------------------------------------- probabilities

// Marginal probabilities.  A wavefront's 64 lanes read the amplitudes of six
// index bits with the other wires of the output fixed, and add up |a|^2 in
// registers over the index bits that are summed out; the
// summed bits among the lanes are added with shuffles at the end, so each
// output value of the wavefront costs one store and nothing is accumulated
// in memory.  The summed bits above the lanes are split over `splits`
// wavefronts where the output alone has too few values to fill the device;
// up to 16 of them meet in LDS, k_probs_sum adds the rest in a fixed order.
// Bound by reading the state.  24 qubits, 10 wires, complex128: 118 us as an
// LDS histogram with one atomic per amplitude (135 us a call), 57 us a call here;
// 11 wires took 5.3 ms with one thread per output value, 57 us here.
constexpr int kProbsLoads = 8;         // loads in flight per lane
constexpr int kProbsBlock = 1024;      // 16 wavefronts, which add their splits before one of them stores
constexpr int kProbsLogWaves = 4;
constexpr int kProbsSumBins = 16;      // bins per workgroup of k_probs_sum: 128 consecutive bytes a row
constexpr int kProbsMaxWaves = 8192;   // 8 wavefronts per SIMD of 256 CUs
constexpr int kProbsHostBins = 4096;   // results written by the kernel into pinned host memory

// Outputs of at least 128 KiB that are no less than a 128th of the state's
// length: the lanes hold the lowest index bits (runs of 128 bytes) and those
// of output bits 0..2 (stores of 64 bytes) instead of index bits 0..5.  The
// output's low bits are the state's high bits for wires in increasing order,
// so with lanes on bits 0..5 every 8-byte store has a cache line of its own
// (26 qubits, the first 20 wires: 1341 against 806 us).  Smaller outputs are
// bound by the reads, which are faster in runs of 1 KiB (26 qubits complex64,
// 14 wires: 113 against 193 us).
constexpr int kProbsWide = 14;
constexpr int kProbsWideRest = 7;

struct ProbsMap {
    int lane_bit[6];    // index bit of each lane position
    int nkeep;          // output wires above the lane bits
    int keep_bit[32];   // their index bits, ascending
    int keep_out[32];   // their output bits
    uint32_t lane_sum;  // lane positions that are summed out
    int lane_out[6];    // output bit of a kept lane position, -1: none
    int nsum;           // summed bits above the lanes
    int log_splits;
    int sum_bit[64];    // their index bits, ascending
};

template <class R>
__global__ __launch_bounds__(kProbsBlock) void k_probs(const cx<R> *__restrict__ sv, uint64_t len, uint64_t nwaves,
                                                       ProbsMap pm, double *__restrict__ out, uint64_t bins) {
    __shared__ double sh[1 << kProbsLogWaves][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t wave = (uint64_t(blockIdx.x) << kProbsLogWaves) + w;
    const bool live = wave < nwaves;
    const uint64_t split = wave & ((1ull << pm.log_splits) - 1), kept = live ? wave >> pm.log_splits : 0;
    uint64_t g = 0, o = 0;
    for (int j = 0; j < pm.nkeep; ++j) {
        const uint64_t bit = (kept >> j) & 1ull;
        g |= bit << pm.keep_bit[j];
        o |= bit << pm.keep_out[j];
    }
    // the split's share: the highest summed bits are fixed to its number
    const int nloop = pm.nsum - pm.log_splits;
    uint64_t loop_mask = 0;
    for (int j = 0; j < nloop; ++j) loop_mask |= 1ull << pm.sum_bit[j];
    for (int j = 0; j < pm.log_splits; ++j) g |= ((split >> j) & 1ull) << pm.sum_bit[nloop + j];
    const uint64_t iters = 1ull << nloop;
    const bool in = uint64_t(lane) < len; // states of fewer than 6 qubits
    double s = 0.0;
    uint64_t c = 0; // the loop's bits at their places in the index
#pragma unroll
    for (int b = 0; b < 6; ++b) g |= uint64_t((lane >> b) & 1) << pm.lane_bit[b];
    const cx<R> *p = sv + g;
    if (live && iters >= kProbsLoads) {
        for (uint64_t it = 0; it < iters; it += kProbsLoads) {
            cx<R> v[kProbsLoads];
#pragma unroll
            for (int k = 0; k < kProbsLoads; ++k) {
                v[k] = ldnt(p + c);
                c = ((c | ~loop_mask) + 1) & loop_mask;
            }
#pragma unroll
            for (int k = 0; k < kProbsLoads; ++k) s += double(v[k].re) * v[k].re + double(v[k].im) * v[k].im;
        }
    } else if (live) {
        for (uint64_t it = 0; it < iters; ++it) {
            const cx<R> v = in ? ldnt(p + c) : cx<R>{R(0), R(0)};
            s += double(v.re) * v.re + double(v.im) * v.im;
            c = ((c | ~loop_mask) + 1) & loop_mask;
        }
    }
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        if ((pm.lane_sum >> b) & 1u) s += __shfl_xor(s, 1 << b, 64);
        else if (pm.lane_out[b] >= 0) o |= uint64_t((lane >> b) & 1) << pm.lane_out[b];
    }
    // neighbouring wavefronts hold the splits of one set of output values
    const int meet = 1 << min(pm.log_splits, kProbsLogWaves);
    if (meet > 1) {
        sh[w][lane] = s;
        __syncthreads();
        if ((w & (meet - 1)) == 0)
            for (int q = 1; q < meet; ++q) s += sh[w + q][lane];
    }
    if (live && (w & (meet - 1)) == 0 && in && (uint32_t(lane) & pm.lane_sum) == 0)
        out[(split / unsigned(meet)) * bins + o] = s;
}

// out[b] = sum over the splits of partials[split][b]
__global__ __launch_bounds__(kBlock) void k_probs_sum(const double *__restrict__ partials, uint64_t bins, int splits,
                                                      double *__restrict__ out) {
    constexpr int kGroups = kBlock / kProbsSumBins; // threads per bin
    __shared__ double sh[kGroups][kProbsSumBins];
    const int q = threadIdx.x / kProbsSumBins, j = threadIdx.x % kProbsSumBins;
    const uint64_t b = uint64_t(blockIdx.x) * kProbsSumBins + j;
    double s = 0.0;
    if (b < bins) {
#pragma unroll 8
        for (int k = q; k < splits; k += kGroups) s += partials[uint64_t(k) * bins + b];
    }
    sh[q][j] = s;
    __syncthreads();
    if (q == 0 && b < bins) {
        for (int k = 1; k < kGroups; ++k) s += sh[k][j];
        out[b] = s;
    }
}

// ---------------------------------------------------------------- sampler

// Philox4x32-10 (Salmon et al., SC'11); counter = (shot lo, shot hi, 0, 0),
// key = (seed lo, seed hi).
__device__ __forceinline__ void philox(uint64_t seed, uint64_t ctr, uint32_t out[4]) {
    uint32_t c0 = uint32_t(ctr), c1 = uint32_t(ctr >> 32), c2 = 0, c3 = 0;
    uint32_t k0 = uint32_t(seed), k1 = uint32_t(seed >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = uint64_t(0xD2511F53u) * c0;
        const uint64_t p1 = uint64_t(0xCD9E8D57u) * c2;
        const uint32_t n0 = uint32_t(p1 >> 32) ^ c1 ^ k0, n1 = uint32_t(p1);
        const uint32_t n2 = uint32_t(p0 >> 32) ^ c3 ^ k1, n3 = uint32_t(p0);
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

constexpr double kFixedScale = 1152921504606846976.0; // 2^60

// |a|^2 in 2^-60 fixed point with explicit roundings (no contraction), so
// that the value is the same bit pattern the oracle computes.
template <class R> __device__ __forceinline__ uint64_t fixed_prob(cx<R> a) {
    const double re = double(a.re), im = double(a.im);
    const double p = __dadd_rn(__dmul_rn(re, re), __dmul_rn(im, im));
    return uint64_t(__dmul_rn(p, kFixedScale));
}

// Sampling by inverse CDF.  Shot s draws a threshold t_s below the total mass
// (fixed point, so that the order of summation does not matter) and takes the
// first index whose inclusive prefix sum exceeds t_s; the indices are returned
// in ascending order.  The CDF is formed per tile of 2^11 amplitudes and never
// written out: the tiles' sums are scanned, every shot finds its tile in them
// and goes to its bin (up to 8192 bins of consecutive tiles), and one
// workgroup per bin forms the prefix sums of each tile that got shots in LDS,
// counts the shots per amplitude and writes them in order.  The counts come
// out sorted, so nothing is sorted.  The shots are binned with counters in
// LDS and a scan: one global counter per tile, added to by every shot, took
// 0.7 ms at 2^13 tiles and 3 ms at 8.
// Bound by two reads of the state (the second only of tiles that got shots).
// 24 qubits, 10^6 shots, complex128: 710 us of kernels with a stored CDF,
// a search of all of it per shot and a radix sort; 185 us here (the copy of the indices to the host, 450 us, not
// counted).
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;
constexpr int kSampleBins = 8192;
// Shots of one bin handled by one workgroup.  A bin with more (a state with
// few large amplitudes) is shared by several, which add their counts in
// global memory and write their parts of its output in a second launch.
constexpr int kLogBinShots = 12;
// shots per workgroup of the binning kernels
constexpr int kAssignBlock = 1024;
constexpr int kAssignShots = 8 * kAssignBlock;

__device__ __forceinline__ uint64_t wave_incl_scan(uint64_t v, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t u = __shfl_up(v, off, 64);
        if (lane >= off) v += u;
    }
    return v;
}
// Exclusive prefix of v over the workgroup's threads (W wavefronts); total:
// the sum over all of them.
template <int W> __device__ __forceinline__ uint64_t block_excl_scan(uint64_t v, uint64_t &total) {
    __shared__ uint64_t sh[W];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t incl = wave_incl_scan(v, lane);
    __syncthreads(); // sh is free again
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < W; ++q) {
        if (q < w) before += sh[q];
        all += sh[q];
    }
    total = all;
    return before + incl - v;
}

// A call's device arrays, in the workspace.
struct SampleBufs {
    uint64_t *tile_off;    // [ntiles] tile sums, then their exclusive prefix
    uint64_t *total;       // total mass
    uint32_t *hist;        // [nassign][nbins] shots per bin of a binning workgroup, then their prefix over workgroups
    uint32_t *bin_off;     // [nbins + 1] first output position of a bin
    uint2 *heavy;          // [nheavy_max] (bin, part) of shared bins
    uint32_t *heavy_id;    // [nbins] row of heavy_count
    uint32_t *heavy_count; // [nrows][tiles of a bin][kScanTile] shots per amplitude of a shared bin
    uint32_t *nitems;      // parts of shared bins, shared bins
    uint32_t *where;       // [shots] bin << 16 | rank among the workgroup's shots of that bin
    uint64_t *thresh;      // [shots] thresholds, by bin
    uint64_t ntiles, nbins, nassign, shots, seed;
    uint64_t bin_shots;    // shots per workgroup of a bin: 2^log_bin_shots
    int log_bin_shots;
    uint32_t nrows;
    int log_bin_tiles;     // tiles per bin
};

template <class R>
__global__ __launch_bounds__(kBlock) void k_sample_sums(const cx<R> *__restrict__ sv, uint64_t len, SampleBufs sb) {
    const uint64_t base = uint64_t(blockIdx.x) * kScanTile;
    cx<R> a[kScanItems];
#pragma unroll
    for (int e = 0; e < kScanItems; ++e) {
        const uint64_t i = base + uint64_t(e) * kBlock + threadIdx.x;
        a[e] = i < len ? sv[i] : cx<R>{R(0), R(0)};
    }
    uint64_t s = 0, total;
#pragma unroll
    for (int e = 0; e < kScanItems; ++e) s += fixed_prob(a[e]);
    block_excl_scan<kWaves>(s, total);
    if (threadIdx.x == 0) sb.tile_off[blockIdx.x] = total;
    if (blockIdx.x == 0 && threadIdx.x < 2) sb.nitems[threadIdx.x] = 0;
    const uint64_t nzero = (uint64_t(sb.nrows) << sb.log_bin_tiles) * kScanTile;
    for (uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x; i < nzero; i += uint64_t(gridDim.x) * kBlock)
        sb.heavy_count[i] = 0;
}

// Exclusive prefix of the tile sums, in place, by one workgroup.
constexpr int kScanBlock = 1024;
__global__ __launch_bounds__(kScanBlock) void k_sample_offsets(SampleBufs sb, uint64_t *total_host) {
    const uint64_t ntiles = sb.ntiles;
    constexpr int kPer = 8; // consecutive sums per thread
    uint64_t run = 0;
    for (uint64_t b = 0; b < ntiles; b += kScanBlock * kPer) {
        const uint64_t i = b + uint64_t(threadIdx.x) * kPer;
        uint64_t v[kPer], s = 0, sum;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            v[e] = i + e < ntiles ? sb.tile_off[i + e] : 0;
            s += v[e];
        }
        uint64_t x = run + block_excl_scan<kScanBlock / 64>(s, sum);
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            if (i + e < ntiles) sb.tile_off[i + e] = x;
            x += v[e];
        }
        run += sum;
    }
    if (threadIdx.x == 0) *sb.total = *total_host = run;
}

// t = floor(u53 * total / 2^53) with a 128-bit product
__device__ __forceinline__ uint64_t threshold(uint64_t seed, uint64_t shot, uint64_t total) {
    uint32_t r[4];
    philox(seed, shot, r);
    const uint64_t u53 = ((uint64_t(r[1]) << 32) | r[0]) >> 11;
    const uint64_t hi = __umul64hi(u53, total), lo = u53 * total;
    return (hi << 11) | (lo >> 53);
}

// The bin of every shot and its rank among the workgroup's shots of the bin.
// Lanes of one bin add to its counter together (two bins a wavefront, then
// one by one): a state with few large amplitudes sends a wavefront's shots to
// few bins.  The ranks depend on timing, the output does not: it only counts
// the shots of an amplitude.
__global__ __launch_bounds__(kAssignBlock) void k_sample_assign(SampleBufs sb) {
    __shared__ uint32_t cnt[kSampleBins];
    __shared__ uint64_t off[kSampleBins]; // offsets of the bins' first tiles
    for (unsigned q = threadIdx.x; q < sb.nbins; q += kAssignBlock) {
        cnt[q] = 0;
        off[q] = sb.tile_off[uint64_t(q) << sb.log_bin_tiles];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const uint64_t total = *sb.total, s0 = uint64_t(blockIdx.x) * kAssignShots;
    for (int e = 0; e < kAssignShots / kAssignBlock; ++e) {
        const uint64_t s = s0 + uint64_t(e) * kAssignBlock + threadIdx.x;
        const bool live = s < sb.shots;
        uint32_t bin = 0;
        if (live) {
            const uint64_t t = threshold(sb.seed, s, total);
            for (uint32_t step = uint32_t(sb.nbins >> 1); step > 0; step >>= 1) // nbins is a power of two
                if (off[bin + step] <= t) bin += step; // the last bin whose offset is at most t
        }
        uint32_t rank = 0;
        bool todo = live;
        for (int round = 0; round < 2; ++round) {
            const uint64_t open = __ballot(todo);
            if (!open) break;
            const int leader = __ffsll((unsigned long long)open) - 1;
            const uint32_t lb = __shfl(bin, leader, 64);
            const bool mine = todo && bin == lb;
            const uint64_t group = __ballot(mine);
            uint32_t first = 0;
            if (lane == leader) first = atomicAdd(&cnt[lb], uint32_t(__popcll(group)));
            first = __shfl(first, leader, 64);
            if (mine) {
                rank = first + uint32_t(__popcll(group & ((1ull << lane) - 1ull)));
                todo = false;
            }
        }
        if (todo) rank = atomicAdd(&cnt[bin], 1u);
        if (live) sb.where[s] = bin << 16 | rank; // at most kAssignShots shots: 16 bits
    }
    __syncthreads();
    for (unsigned q = threadIdx.x; q < sb.nbins; q += kAssignBlock) sb.hist[blockIdx.x * sb.nbins + q] = cnt[q];
}
static_assert(kAssignShots <= 1 << 16 && kSampleBins <= 1 << 16, "bin and rank share a word");

// Per bin: the prefix of its counts over the binning workgroups, in place,
// and its total (to bin_off, scanned by the next kernel).
__global__ __launch_bounds__(kBlock) void k_sample_columns(SampleBufs sb) {
    // a wavefront takes 8 bins (32 consecutive bytes), 8 rows at a time
    const int lane = threadIdx.x & 63, r = lane >> 3;
    const uint64_t wave = (uint64_t(blockIdx.x) * kBlock + threadIdx.x) >> 6;
    const uint64_t bin = wave * 8 + (lane & 7);
    uint32_t run = 0;
    for (uint64_t b = 0; b < sb.nassign; b += 8) {
        const bool in = bin < sb.nbins && b + r < sb.nassign;
        const uint32_t c = in ? sb.hist[(b + r) * sb.nbins + bin] : 0;
        uint32_t x = c;
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) {
            const uint32_t u = __shfl_up(x, off, 64);
            if (lane >= off) x += u;
        }
        if (in) sb.hist[(b + r) * sb.nbins + bin] = run + x - c;
        run += __shfl(x, 56 + (lane & 7), 64);
    }
    if (r == 0 && bin < sb.nbins) sb.bin_off[bin] = run;
}

// Output positions of the bins, by one workgroup, and the parts of shared
// bins (their order does not matter).
__global__ __launch_bounds__(kScanBlock) void k_sample_items(SampleBufs sb) {
    constexpr int kPer = 8; // consecutive bins per thread
    uint32_t run = 0;
    for (uint64_t b = 0; b < sb.nbins; b += kScanBlock * kPer) {
        const uint64_t i = b + uint64_t(threadIdx.x) * kPer;
        uint32_t c[kPer];
        uint64_t s = 0, sum;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            c[e] = i + e < sb.nbins ? sb.bin_off[i + e] : 0;
            s += c[e];
        }
        uint32_t x = run + uint32_t(block_excl_scan<kScanBlock / 64>(s, sum));
        bool shared = false;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            if (i + e < sb.nbins) sb.bin_off[i + e] = x;
            x += c[e];
            shared |= c[e] > sb.bin_shots;
        }
        run += uint32_t(sum);
        if (shared) {
#pragma unroll 1
            for (int e = 0; e < kPer && i + e < sb.nbins; ++e) {
                const uint64_t n = (i + e + 1 < sb.nbins && e + 1 < kPer ? sb.bin_off[i + e + 1] : x) - sb.bin_off[i + e];
                if (n <= sb.bin_shots) continue;
                const uint32_t parts = uint32_t((n + sb.bin_shots - 1) >> sb.log_bin_shots);
                const uint32_t at = atomicAdd(&sb.nitems[0], parts);
                sb.heavy_id[i + e] = atomicAdd(&sb.nitems[1], 1u);
                for (uint32_t p = 0; p < parts; ++p) sb.heavy[at + p] = make_uint2(uint32_t(i + e), p);
            }
        }
    }
    if (threadIdx.x == 0) sb.bin_off[sb.nbins] = run;
}

// Every shot's threshold to its bin.
__global__ __launch_bounds__(kBlock) void k_sample_scatter(SampleBufs sb) {
    const uint64_t s = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (s >= sb.shots) return;
    const uint32_t w = sb.where[s], bin = w >> 16;
    const uint64_t at = uint64_t(sb.bin_off[bin]) + sb.hist[(s / kAssignShots) * sb.nbins + bin] + (w & 0xffffu);
    sb.thresh[at] = threshold(sb.seed, s, *sb.total);
}

// one u64 of padding per 8: a thread's 8 consecutive entries start on banks
// of their own
__device__ __forceinline__ int pad8(int i) { return i + (i >> 3); }

// Writes the part of a tile's output that lies in positions [lo, hi): the
// tile's shots have positions from `at` on, amplitude a's start at at + first[a].
__device__ __forceinline__ void emit(const uint32_t *first, uint64_t base, uint64_t at, uint64_t count, uint64_t lo,
                                     uint64_t hi, uint64_t *__restrict__ out) {
    const uint64_t p0 = max(at, lo), p1 = min(at + count, hi);
    for (uint64_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
        const uint32_t r = uint32_t(p - at);
        int a = 0; // the last amplitude whose first position is at most p
#pragma unroll
        for (int step = kScanTile / 2; step > 0; step >>= 1)
            if (first[a + step] <= r) a += step;
        out[p] = base + uint64_t(a);
    }
}

// Counts per amplitude become the first position of each amplitude's shots;
// returns the tile's shots.
__device__ __forceinline__ uint32_t scan_counts(uint32_t *cnt) {
    uint32_t c[kScanItems];
    uint64_t s = 0, total;
#pragma unroll
    for (int e = 0; e < kScanItems; ++e) {
        c[e] = cnt[threadIdx.x * kScanItems + e];
        s += c[e];
    }
    uint32_t run = uint32_t(block_excl_scan<kWaves>(s, total));
#pragma unroll
    for (int e = 0; e < kScanItems; ++e) {
        cnt[threadIdx.x * kScanItems + e] = run;
        run += c[e];
    }
    __syncthreads();
    return uint32_t(total);
}

// One workgroup per bin, and after those one per part of a shared bin.
template <class R>
__global__ __launch_bounds__(kBlock) void k_sample_bins(const cx<R> *__restrict__ sv, uint64_t len, SampleBufs sb,
                                                        uint64_t *__restrict__ out) {
    __shared__ uint64_t cdf[kScanTile + kScanTile / 8];
    __shared__ uint32_t cnt[kScanTile];
    const bool light = blockIdx.x < sb.nbins;
    if (!light && blockIdx.x - sb.nbins >= sb.nitems[0]) return;
    const uint2 it = light ? make_uint2(blockIdx.x, 0u) : sb.heavy[blockIdx.x - sb.nbins];
    const int tid = threadIdx.x;
    // the item's shots: positions [lo, hi)
    const uint64_t bin_lo = sb.bin_off[it.x], bin_hi = sb.bin_off[it.x + 1];
    if (light && (bin_hi == bin_lo || bin_hi - bin_lo > sb.bin_shots)) return; // no shots, or a shared bin
    const uint64_t lo = bin_lo + uint64_t(it.y) * sb.bin_shots, hi = min(lo + sb.bin_shots, bin_hi);
    const uint64_t t0 = uint64_t(it.x) << sb.log_bin_tiles, t1 = min(t0 + (1ull << sb.log_bin_tiles), sb.ntiles);
    uint64_t at = bin_lo; // output position of the tile
    for (uint64_t tile = t0; tile < t1; ++tile) {
        // thresholds of the tile: [off, end); the bin's first and last tiles take what lies beyond as well
        const uint64_t off = sb.tile_off[tile];
        const uint64_t end = tile + 1 < sb.ntiles ? sb.tile_off[tile + 1] : *sb.total;
        const bool first = tile == t0, last = tile + 1 == t1;
        bool any = first && last;
        for (uint64_t p = lo + tid; p < hi && !any; p += kBlock) {
            const uint64_t t = sb.thresh[p];
            any = (first || t >= off) && (last || t < end);
        }
        if (!__syncthreads_or(any)) continue;
        const uint64_t base = tile * kScanTile;
#pragma unroll
        for (int e = 0; e < kScanItems; ++e) {
            const int j = e * kBlock + tid;
            const uint64_t i = base + uint64_t(j);
            cdf[pad8(j)] = i < len ? fixed_prob(sv[i]) : 0;
            cnt[j] = 0;
        }
        __syncthreads();
        uint64_t q[kScanItems], s = 0, total;
#pragma unroll
        for (int e = 0; e < kScanItems; ++e) {
            q[e] = cdf[pad8(tid * kScanItems + e)];
            s += q[e];
        }
        uint64_t run = block_excl_scan<kWaves>(s, total);
#pragma unroll
        for (int e = 0; e < kScanItems; ++e) {
            run += q[e];
            cdf[pad8(tid * kScanItems + e)] = run;
        }
        __syncthreads();
        const int top = int(min(uint64_t(kScanTile), len - base)) - 1;
        for (uint64_t p = lo + tid; p < hi; p += kBlock) {
            const uint64_t t = sb.thresh[p];
            if (!((first || t >= off) && (last || t < end))) continue;
            int a = 0; // the first amplitude whose inclusive prefix exceeds t - off
#pragma unroll
            for (int step = kScanTile / 2; step > 0; step >>= 1)
                if (cdf[pad8(a + step - 1)] <= t - off) a += step;
            atomicAdd(&cnt[min(a, top)], 1u);
        }
        __syncthreads();
        if (light) {
            const uint32_t c = scan_counts(cnt);
            emit(cnt, base, at, c, bin_lo, bin_hi, out);
            at += c;
            __syncthreads(); // the next tile clears the counts
        } else {
            uint32_t *row = sb.heavy_count +
                            ((uint64_t(sb.heavy_id[it.x]) << sb.log_bin_tiles) + (tile - t0)) * kScanTile;
            for (int j = tid; j < kScanTile; j += kBlock)
                if (cnt[j]) atomicAdd(&row[j], cnt[j]);
            __syncthreads();
        }
    }
}

// The output of shared bins, once their counts are complete.
__global__ __launch_bounds__(kBlock) void k_sample_shared(SampleBufs sb, uint64_t *__restrict__ out) {
    __shared__ uint32_t cnt[kScanTile];
    if (blockIdx.x >= sb.nitems[0]) return;
    const uint2 it = sb.heavy[blockIdx.x];
    const uint64_t bin_lo = sb.bin_off[it.x], bin_hi = sb.bin_off[it.x + 1];
    const uint64_t lo = bin_lo + uint64_t(it.y) * sb.bin_shots, hi = min(lo + sb.bin_shots, bin_hi);
    const uint64_t t0 = uint64_t(it.x) << sb.log_bin_tiles, t1 = min(t0 + (1ull << sb.log_bin_tiles), sb.ntiles);
    uint64_t at = bin_lo;
    for (uint64_t tile = t0; tile < t1 && at < hi; ++tile) {
        const uint32_t *row =
            sb.heavy_count + ((uint64_t(sb.heavy_id[it.x]) << sb.log_bin_tiles) + (tile - t0)) * kScanTile;
        for (int j = threadIdx.x; j < kScanTile; j += kBlock) cnt[j] = row[j];
        __syncthreads();
        const uint32_t c = scan_counts(cnt);
        emit(cnt, tile * kScanTile, at, c, lo, hi, out);
        at += c;
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void k_expand_bits(const uint64_t *__restrict__ idx, uint64_t shots, int n,
                                                        uint64_t *__restrict__ bits) {
    const uint64_t t = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= shots * uint64_t(n)) return;
    const uint64_t s = t / n;
    const int col = int(t - s * n);
    bits[t] = (idx[s] >> (n - 1 - col)) & 1ull;
}

// ---------------------------------------------------------------- host helpers

template <class R> const cx<R> *cdata(const lgh_sv *sv) { return static_cast<const cx<R> *>(sv->data); }
template <class R> cx<R> *mdata(lgh_sv *sv) { return static_cast<cx<R> *>(sv->data); }

template <class R> void inner_t(const lgh_sv *a, const lgh_sv *b, double *re, double *im) {
    StreamCtx *ctx = a->ctx;
    Chunks ch = chunks_for(a->length(), a->device);
    RedBuf rb = red_buf(ctx, 2, ch.blocks);
    hipLaunchKernelGGL(k_inner<R>, dim3(ch.blocks), dim3(kBlock), 0, ctx->stream, cdata<R>(a), cdata<R>(b),
                       a->length(), ch.chunk, rb.partials);
    LGH_LAUNCH_CHECK();
    double out[2];
    reduce_to_host(ctx, rb.partials, ch.blocks, 2, out);
    *re = out[0];
    *im = out[1];
}

template <class R> void expval_t(const lgh_sv *sv, const int32_t *wires, int k, const double *matrix, double *re,
                                 double *im) {
    StreamCtx *ctx = sv->ctx;
    const int n = sv->n;
    const int D = 1 << k;
    std::vector<int> tb(k);
    for (int j = 0; j < k; ++j) tb[j] = n - 1 - wires[j];
    if (k <= kMaxRegK) {
        const Fixed fx = make_fixed(tb);
        const uint64_t ngroups = 1ull << (n - k);
        std::vector<cx<double>> m(size_t(D) * D);
        for (size_t i = 0; i < m.size(); ++i) m[i] = cx<double>{matrix[2 * i], matrix[2 * i + 1]};
        const cx<double> *dm = static_cast<const cx<double> *>(ctx->upload(m.data(), m.size() * sizeof(m[0])));
        Chunks ch = chunks_for(ngroups, sv->device, 2);
        RedBuf rb = red_buf(ctx, 2, ch.blocks);
        auto run = [&](auto offs, auto kern) {
            for (int mi = 0; mi < D; ++mi) {
                uint64_t o = 0;
                for (int j = 0; j < k; ++j)
                    if ((mi >> (k - 1 - j)) & 1) o |= 1ull << tb[j];
                offs.o[mi] = o;
            }
            hipLaunchKernelGGL(kern, dim3(ch.blocks), dim3(kBlock), 0, ctx->stream, cdata<R>(sv), ngroups, ch.chunk,
                               fx, offs, dm, rb.partials);
        };
        if (k == 1) run(Offs<1>{}, k_expval_reg<R, 1>);
        else if (k == 2) run(Offs<2>{}, k_expval_reg<R, 2>);
        else run(Offs<3>{}, k_expval_reg<R, 3>);
        LGH_LAUNCH_CHECK();
        double out[2];
        reduce_to_host(ctx, rb.partials, ch.blocks, 2, out);
        *re = out[0];
        *im = out[1];
        return;
    }
    double out[2];
    dense_expval(sv, tb.data(), k, matrix, out);
    *re = out[0];
    *im = out[1];
}

// sum_w Re(c_w <P_w>) with <P_w> real, in word order; per_word (nullable) gets <P_w>
double weighted_total(int64_t nwords, const double *coeffs, const double *vals, double *per_word) {
    double tot = 0.0;
    for (int64_t w = 0; w < nwords; ++w) {
        tot += coeffs[2 * w] * vals[w];
        if (per_word) per_word[w] = vals[w];
    }
    return tot;
}

// Parses word w into its flip mask, Z/Y mask and number of Y factors.
void parse_word(int n, const char *paulis, const int32_t *wires, int64_t b, int64_t e, uint64_t &flip,
                uint64_t &zy, int32_t &ny) {
    flip = zy = 0;
    ny = 0;
    for (int64_t j = b; j < e; ++j) {
        const int wire = wires[j];
        LGH_REQUIRE(wire >= 0 && wire < n, "Pauli word wire out of range");
        const uint64_t bit = 1ull << (n - 1 - wire);
        switch (paulis[j]) {
        case 'I': break;
        case 'X': flip |= bit; break;
        case 'Y': flip |= bit; zy |= bit; ny++; break;
        case 'Z': zy |= bit; break;
        default: LGH_REQUIRE(false, "unknown Pauli factor (words use I, X, Y, Z)");
        }
    }
}

// Tile geometry of the Pauli passes on an n-qubit state.
struct PGeo {
    int g;          // tile bits
    int fixed;      // lowest index bits in every tile
    int chosen_max; // bits chosen per pass
};
PGeo pauli_geo(int n) {
    PGeo p;
    p.g = std::min(kPTileBits, n);
    p.fixed = std::min(kPFixedBits, n);
    p.chosen_max = p.g - p.fixed;
    return p;
}

// Groups words into tile passes without allocating: pass_of[w] gets the pass
// of word w (-1: its flip bits do not fit a tile), pass_mask[p] the chosen
// bits of pass p; returns the number of passes.  Each pass is filled first
// with the uncovered words of most flip bits that still fit the pass's
// budget of chosen bits (first fit, decreasing), then takes every
// uncovered word whose flip bits lie in the tile.
int64_t plan_pauli_tiles(int n, int64_t nwords, const uint64_t *flip, int32_t *pass_of, uint64_t *pass_mask) {
    const PGeo geo = pauli_geo(n);
    const uint64_t fixed_mask = (1ull << geo.fixed) - 1ull;
    int64_t left = 0;
    for (int64_t w = 0; w < nwords; ++w) {
        const int c = __builtin_popcountll(flip[w] & ~fixed_mask);
        pass_of[w] = c <= geo.chosen_max ? -2 : -1; // -2: still to place
        left += pass_of[w] == -2;
    }
    int64_t np = 0;
    while (left > 0) {
        uint64_t chosen = 0;
        for (int c = geo.chosen_max; c >= 0; --c)
            for (int64_t w = 0; w < nwords; ++w) {
                if (pass_of[w] != -2) continue;
                const uint64_t rest = flip[w] & ~fixed_mask;
                if (__builtin_popcountll(rest) == c && __builtin_popcountll(chosen | rest) <= geo.chosen_max)
                    chosen |= rest;
            }
        for (int b = geo.fixed; b < n && __builtin_popcountll(chosen) < geo.chosen_max; ++b) chosen |= 1ull << b;
        for (int64_t w = 0; w < nwords; ++w)
            if (pass_of[w] == -2 && ((flip[w] & ~fixed_mask) & ~chosen) == 0) {
                pass_of[w] = int32_t(np);
                --left;
            }
        pass_mask[np++] = chosen;
    }
    return np;
}

// Workgroups of a tile launch: the two that a CU holds.
constexpr unsigned kPauliBlocksPerCU = 2;

// Tile-local bits of a pass, ascending.
PTile pauli_layout(const PGeo &geo, int n, uint64_t chosen) {
    PTile tm{};
    tm.g = geo.g;
    int r = 0;
    for (int b = 0; b < n; ++b)
        if (b < geo.fixed || ((chosen >> b) & 1)) tm.bit[r++] = b;
    LGH_REQUIRE(r == geo.g, "Pauli tile: bad bit count");
    return tm;
}

uint32_t to_tile(const PTile &tm, uint64_t mask) {
    uint32_t m = 0;
    for (int q = 0; q < tm.g; ++q) m |= uint32_t((mask >> tm.bit[q]) & 1u) << q;
    return m;
}

// One word's record for the pivot bit `pivot`.
PWord pauli_word(const PTile &tm, uint64_t tile_mask, uint64_t flip, uint64_t zy, int32_t ny, uint32_t pivot) {
    PWord pw{};
    const uint32_t fl = to_tile(tm, flip), zl = to_tile(tm, zy), ph = uint32_t(ny & 3);
    pw.pivot = pivot;
    pw.flip = fl ? fl : 1u << pivot;
    pw.kind = fl ? (ph & 1u ? kPOdd : kPEven) : (zl >> pivot) & 1u ? kPSquareDiff : kPSquare;
    // lane bits, then step bits, are the tile's bits without the pivot
    int at = 0;
    for (uint32_t b = 0; b < uint32_t(kPTileBits); ++b) {
        if (b == pivot) continue;
        const bool z = (zl >> b) & 1u;
        if (at < 6)
            pw.zlane |= uint32_t(z) << at;
        else
            pw.sign[at - 6] = z ? -1.0 : 1.0;
        ++at;
    }
    // i^nY: +re, -im, -re, +im
    pw.scale = (ph == 1 || ph == 2 ? -1.0 : 1.0) * (fl ? 2.0 : 1.0);
    pw.zy = zy & ~tile_mask;
    return pw;
}

// Records of up to kPassWords words (sorted by flip mask and parity of nY)
// spread over the wavefronts: words that share products stay together, in
// groups of at most the wavefronts' mean, each group on the wavefront with
// the least to do (products weigh as three words) that has room.
void pauli_fill(PLaunch &l, const PTile &tm, uint64_t tile_mask, const int32_t *words, int count, const uint64_t *flip,
                const uint64_t *zy, const int32_t *ny) {
    l = PLaunch{};
    int load[kPWaves] = {};
    const int most = std::min(kPSlots, (count + kPWaves - 1) / kPWaves);
    for (int s = 0; s < count;) {
        // the pivot: the highest flipped bit; without flips the highest bit
        // outside the word's own mask, kept while the next words allow it
        const int32_t w0 = words[s];
        const uint32_t fl = to_tile(tm, flip[w0]), z0 = to_tile(tm, zy[w0]), all = (1u << kPTileBits) - 1u;
        const uint32_t from = fl ? fl : (~z0 & all) ? (~z0 & all) : all;
        const uint32_t pivot = 31u - uint32_t(__builtin_clz(from));
        const uint32_t kind = pauli_word(tm, tile_mask, flip[w0], zy[w0], ny[w0], pivot).kind;
        int best = -1;
        for (int w = 0; w < kPWaves; ++w)
            if (l.slots[w] < uint32_t(kPSlots) && (best < 0 || load[w] < load[best])) best = w;
        LGH_REQUIRE(best >= 0, "Pauli words: no room");
        load[best] += 3;
        for (int taken = 0; s < count && taken < most && l.slots[best] < uint32_t(kPSlots); ++taken, ++s) {
            const int32_t w = words[s];
            if (flip[w] != flip[w0]) break;
            PWord pw = pauli_word(tm, tile_mask, flip[w], zy[w], ny[w], pivot);
            if (pw.kind != kind) break;
            pw.kind |= taken == 0 ? 16u : 0u;
            pw.row = uint32_t(s);
            l.word[best][l.slots[best]++] = pw;
            ++load[best];
        }
    }
}

struct PauliBufs {
    double *partials; // device, partials_cap doubles
    size_t partials_cap;
    double *results;  // one double per word: device memory or pinned host memory
    // copies a launch's records to the device (stream ordered) and returns their address there
    const PLaunch *(*upload)(StreamCtx *ctx, const PLaunch &launch, void *arg);
    void *arg;
};

// Device doubles of reduction partials the Pauli passes of an n-qubit state need.
size_t pauli_partials_doubles(int n, int device) {
    const uint64_t len = 1ull << n;
    const unsigned pair_blocks = chunks_for(len, device).blocks;
    const unsigned tile_blocks = unsigned(std::max(1, sm_count(device))) * kPauliBlocksPerCU;
    return std::max(size_t(kMaxWordsPerPass) * pair_blocks, size_t(kPassWords) * tile_blocks);
}

// Launches every pass of the words (tile passes first, in pass order, then
// pair passes in ascending flip mask) and their reductions into
// bufs.results; slot_word[s] is the word whose value lands in result slot s.
// Needs no allocation: the caller provides every array (nwords entries each).
template <class R>
void pauli_run(const lgh_sv *sv, int64_t nwords, const uint64_t *flip, const uint64_t *zy, const int32_t *ny,
               int32_t *pass_of, uint64_t *pass_mask, bool *done, int32_t *slot_word, const PauliBufs &bufs) {
    StreamCtx *ctx = sv->ctx;
    const int n = sv->n;
    const uint64_t len = sv->length();
    const PGeo geo = pauli_geo(n);
    const int64_t npasses = plan_pauli_tiles(n, nwords, flip, pass_of, pass_mask);
    int64_t nslots = 0;
    // tile passes
    const uint64_t ntiles = len >> geo.g;
    const unsigned max_blocks = unsigned(std::max(1, sm_count(sv->device))) * kPauliBlocksPerCU;
    const uint64_t per_block = (ntiles + max_blocks - 1) / max_blocks;
    const unsigned tblocks = unsigned((ntiles + per_block - 1) / per_block);
    LGH_REQUIRE(size_t(kPassWords) * tblocks <= bufs.partials_cap, "Pauli partials buffer too small");
    // the words of each pass, by flip mask (slot_word: result slot -> word)
    for (int64_t p = 0; p < npasses; ++p) {
        const int64_t first = nslots;
        for (int64_t w = 0; w < nwords; ++w)
            if (pass_of[w] == p) slot_word[nslots++] = int32_t(w);
        std::sort(slot_word + first, slot_word + nslots, [&](int32_t x, int32_t y) {
            if (flip[x] != flip[y]) return flip[x] < flip[y];
            if ((ny[x] & 1) != (ny[y] & 1)) return (ny[x] & 1) < (ny[y] & 1);
            return x < y;
        });
    }
    for (int64_t first = 0, end; first < nslots; first = end) {
        const int32_t p = pass_of[slot_word[first]];
        for (end = first; end < nslots && pass_of[slot_word[end]] == p;) ++end;
        const PTile tm = pauli_layout(geo, n, pass_mask[p]);
        uint64_t tile_mask = 0;
        Fixed tfx{};
        tfx.cnt = geo.g;
        for (int q = 0; q < geo.g; ++q) {
            tfx.pos[q] = tm.bit[q];
            tile_mask |= 1ull << tm.bit[q];
        }
        for (int64_t s = first; s < end; s += kPassWords) {
            const int nw = int(std::min<int64_t>(kPassWords, end - s));
            PLaunch launch;
            pauli_fill(launch, tm, tile_mask, slot_word + s, nw, flip, zy, ny);
            const PLaunch *dl = bufs.upload(ctx, launch, bufs.arg);
            hipLaunchKernelGGL(k_pauli_tile<R>, dim3(tblocks), dim3(kPBlock), 0, ctx->stream, cdata<R>(sv), ntiles,
                               per_block, tfx, tm, dl, bufs.partials);
            LGH_LAUNCH_CHECK();
            launch_reduce(ctx, bufs.partials, int(tblocks), nw, bufs.results + s);
        }
    }
    // words wider than a tile: one pair pass per flip mask, ascending
    for (int64_t w = 0; w < nwords; ++w) done[w] = pass_of[w] >= 0;
    for (;;) {
        bool any = false;
        uint64_t f = 0;
        for (int64_t w = 0; w < nwords; ++w)
            if (!done[w] && (!any || flip[w] < f)) {
                f = flip[w];
                any = true;
            }
        if (!any) break;
        const int pivot = f ? __builtin_ctzll(f) : -1;
        const uint64_t count = f ? len / 2 : len;
        const Chunks ch = chunks_for(count, sv->device);
        LGH_REQUIRE(size_t(kMaxWordsPerPass) * ch.blocks <= bufs.partials_cap, "Pauli partials buffer too small");
        WordSet ws{};
        auto launch = [&] {
            hipLaunchKernelGGL(k_pauli<R>, dim3(ch.blocks), dim3(kBlock), 0, ctx->stream, cdata<R>(sv), count,
                               ch.chunk, pivot, f, ws, bufs.partials);
            LGH_LAUNCH_CHECK();
            launch_reduce(ctx, bufs.partials, ch.blocks, ws.count, bufs.results + (nslots - ws.count));
            ws.count = 0;
        };
        for (int64_t w = 0; w < nwords; ++w) {
            if (done[w] || flip[w] != f) continue;
            done[w] = true;
            ws.zy[ws.count] = zy[w];
            ws.phase[ws.count] = uint32_t(ny[w] & 3);
            ++ws.count;
            slot_word[nslots++] = int32_t(w);
            if (ws.count == kMaxWordsPerPass) launch();
        }
        if (ws.count > 0) launch();
    }
    LGH_REQUIRE(nslots == nwords, "Pauli words: every word gets one result slot");
}

template <class R>
void pauli_t(const lgh_sv *sv, int64_t nwords, const char *paulis, const int32_t *wires, const int64_t *offsets,
             const double *coeffs, double *per_word, double *result) {
    StreamCtx *ctx = sv->ctx;
    const size_t nw = size_t(nwords);
    std::vector<uint64_t> flip(nw), zy(nw), pass_mask(std::max<size_t>(1, nw));
    std::vector<int32_t> ny(nw), pass_of(nw), slot_word(nw);
    std::unique_ptr<bool[]> done(new bool[std::max<size_t>(1, nw)]);
    for (int64_t w = 0; w < nwords; ++w)
        parse_word(sv->n, paulis, wires, offsets[w], offsets[w + 1], flip[size_t(w)], zy[size_t(w)], ny[size_t(w)]);
    const size_t pcap = pauli_partials_doubles(sv->n, sv->device);
    double *partials = static_cast<double *>(ctx->workspace(sizeof(double) * pcap));
    // the reductions write the words' values into pinned host memory
    double *host = static_cast<double *>(ctx->host_buffer(sizeof(double) * std::max<size_t>(1, nw)));
    PauliBufs bufs{partials, pcap, host,
                   [](StreamCtx *c, const PLaunch &l, void *) {
                       return static_cast<const PLaunch *>(c->upload(&l, sizeof(l)));
                   },
                   nullptr};
    if (nwords > 0)
        pauli_run<R>(sv, nwords, flip.data(), zy.data(), ny.data(), pass_of.data(), pass_mask.data(), done.get(),
                     slot_word.data(), bufs);
    std::vector<double> vals(std::max<size_t>(1, nw));
    ctx->sync();
    for (size_t q = 0; q < nw; ++q) vals[size_t(slot_word[q])] = host[q];
    *result = weighted_total(nwords, coeffs, vals.data(), per_word);
}

template <class R>
void pauli_sum_t(lgh_sv *dst, const lgh_sv *src, int64_t nwords, const char *paulis, const int32_t *wires,
                 const int64_t *offsets, const double *coeffs) {
    StreamCtx *ctx = dst->ctx;
    const int n = dst->n;
    const uint64_t len = dst->length();
    const size_t nw = size_t(nwords);
    std::vector<uint64_t> flip(nw), zy(nw), pass_mask(std::max<size_t>(1, nw));
    std::vector<int32_t> ny(nw), pass_of(nw);
    for (size_t w = 0; w < nw; ++w) parse_word(n, paulis, wires, offsets[w], offsets[w + 1], flip[w], zy[w], ny[w]);
    const PGeo geo = pauli_geo(n);
    const int64_t npasses = nwords ? plan_pauli_tiles(n, nwords, flip.data(), pass_of.data(), pass_mask.data()) : 0;
    // real part or, for odd nY, imaginary part of c i^nY: +1, +i, -1, -i
    auto coeff = [&](size_t w) { return (ny[w] & 2) ? -coeffs[w] : coeffs[w]; };
    int add = 0;
    for (int64_t p = 0; p < npasses; ++p) {
        std::vector<size_t> words;
        for (size_t w = 0; w < nw; ++w)
            if (pass_of[w] == p) words.push_back(w);
        std::sort(words.begin(), words.end(),
                  [&](size_t a, size_t b) { return flip[a] != flip[b] ? flip[a] < flip[b] : a < b; });
        const PTile tm = pauli_layout(geo, n, pass_mask[size_t(p)]);
        Fixed tfx{};
        tfx.cnt = geo.g;
        uint64_t tile_mask = 0;
        for (int q = 0; q < geo.g; ++q) {
            tfx.pos[q] = tm.bit[q];
            tile_mask |= 1ull << tm.bit[q];
        }
        std::vector<SWord> rec(words.size());
        for (size_t k = 0; k < words.size(); ++k) {
            const size_t w = words[k];
            const bool last = k + 1 == words.size() || flip[words[k + 1]] != flip[w];
            rec[k] = {coeff(w), zy[w] & ~tile_mask, to_tile(tm, flip[w]),
                      to_tile(tm, zy[w]) | uint32_t(ny[w] & 1) << 16 | uint32_t(last) << 17, 0.0};
        }
        const SWord *drec = static_cast<const SWord *>(ctx->upload(rec.data(), rec.size() * sizeof(SWord)));
        hipLaunchKernelGGL(k_pauli_sum<R>, dim3(unsigned(len >> geo.g)), dim3(kPBlock), 0, ctx->stream, mdata<R>(dst),
                           cdata<R>(src), len >> geo.g, tfx, tm, drec, int(rec.size()), add);
        LGH_LAUNCH_CHECK();
        add = 1;
    }
    for (size_t w = 0; w < nw; ++w) {
        if (pass_of[w] >= 0) continue;
        hipLaunchKernelGGL(k_pauli_add<R>, dim3(unsigned((len + kBlock - 1) / kBlock)), dim3(kBlock), 0, ctx->stream,
                           mdata<R>(dst), cdata<R>(src), len, flip[w], zy[w], int(ny[w] & 1), coeff(w), add);
        LGH_LAUNCH_CHECK();
        add = 1;
    }
    if (!add) { // no words
        hipLaunchKernelGGL(k_zero<R>, dim3(unsigned((len + kBlock - 1) / kBlock)), dim3(kBlock), 0, ctx->stream,
                           mdata<R>(dst), len);
        LGH_LAUNCH_CHECK();
    }
}

// ---------------------------------------------------------------- Pauli words without allocation
//
// lgh_expval_pauli_words_noalloc runs the passes of pauli_t (same kernels,
// same grouping, same chunking, so the same results bit for bit) with its
// reduction partials and word results in `scratch`, a device array of fixed
// size that every call on one device shares.  The host side keeps its
// bookkeeping in fixed-size arrays on the stack.  Nothing is allocated after
// the first call on a device, which looks up the array's device address (and
// the device's CU count used to size the passes).
//
// Layout of `scratch` for one call: reduction partials of one launch |
// one result per word | the launch's word records.  Every entry a call reads was written earlier in the
// same call (each launch writes all its partials, each reduction its
// words' results), so nothing needs clearing; two calls that overlap on one
// device race on the array.

constexpr size_t kNoAllocScratchBytes = size_t(512) << 10;
constexpr int64_t kNoAllocMaxWords = 1024;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

std::mutex g_scratch_mu;
void *g_scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on `device` (the current device), looked up once
// per device.  The array's host-side name is not a device address.
void *scratch_on(int device) {
    LGH_REQUIRE(device >= 0 && device < kMaxDevices, "device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[device]) {
        void *p = nullptr;
        LGH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        LGH_REQUIRE(p != nullptr, "scratch array has no device address");
        (void)sm_count(device); // cached from here on: later calls only read it
        g_scratch_dev[device] = p;
    }
    return g_scratch_dev[device];
}

template <class R>
void pauli_noalloc_t(const lgh_sv *sv, int64_t nwords, const char *paulis, const int32_t *wires,
                     const int64_t *offsets, const double *coeffs, double *per_word, double *result) {
    LGH_REQUIRE(nwords <= kNoAllocMaxWords, "lgh_expval_pauli_words_noalloc takes at most " +
                                                std::to_string(kNoAllocMaxWords) + " words (got " +
                                                std::to_string(nwords) + ")");
    StreamCtx *ctx = sv->ctx;
    char *base = static_cast<char *>(scratch_on(sv->device));
    uint64_t flip[kNoAllocMaxWords], zy[kNoAllocMaxWords], pass_mask[kNoAllocMaxWords];
    int32_t ny[kNoAllocMaxWords], pass_of[kNoAllocMaxWords], slot_word[kNoAllocMaxWords];
    bool done[kNoAllocMaxWords];
    for (int64_t w = 0; w < nwords; ++w) parse_word(sv->n, paulis, wires, offsets[w], offsets[w + 1], flip[w], zy[w], ny[w]);
    const size_t pcap = pauli_partials_doubles(sv->n, sv->device);
    // partials | results | a launch's records
    const size_t o_words = (sizeof(double) * (pcap + size_t(nwords)) + 255) & ~size_t(255);
    const size_t need = o_words + sizeof(PLaunch);
    LGH_REQUIRE(need <= kNoAllocScratchBytes, "lgh_expval_pauli_words_noalloc: " + std::to_string(need) +
                                                  " bytes of scratch needed, " +
                                                  std::to_string(kNoAllocScratchBytes) + " available");
    PauliBufs bufs{reinterpret_cast<double *>(base), pcap, reinterpret_cast<double *>(base) + pcap,
                   [](StreamCtx *c, const PLaunch &l, void *dst) {
                       for (int q = 0; q < 2; ++q) {
                           PHalf h;
                           std::memcpy(&h, reinterpret_cast<const char *>(&l) + q * sizeof(h), sizeof(h));
                           hipLaunchKernelGGL(k_pauli_put, dim3(1), dim3(256), 0, c->stream,
                                              static_cast<uint32_t *>(dst) + q * (sizeof(h) / 4), h);
                           LGH_LAUNCH_CHECK();
                       }
                       return static_cast<const PLaunch *>(dst);
                   },
                   base + o_words};
    if (nwords > 0) pauli_run<R>(sv, nwords, flip, zy, ny, pass_of, pass_mask, done, slot_word, bufs);
    double out[kNoAllocMaxWords];
    double vals[kNoAllocMaxWords];
    if (nwords > 0) {
        LGH_HIP(hipMemcpyAsync(out, bufs.results, sizeof(double) * size_t(nwords), hipMemcpyDeviceToHost,
                               ctx->stream));
        ctx->sync();
    }
    for (int64_t q = 0; q < nwords; ++q) vals[slot_word[q]] = out[q];
    *result = weighted_total(nwords, coeffs, vals, per_word);
}

// Host offsets or indices that fit 32 bits, narrowed on the device piece by
// piece (on the host it took 13 ms of a 45 ms upload of 22 million entries);
// a single piece on the host, where the staging costs more (2^12 rows of 13
// entries: 105 us to create the matrix, 86 without).
void upload_narrow(int device, int32_t *dst, const int64_t *src, int64_t count) {
    if (count <= 0) return;
    constexpr int64_t kPiece = int64_t(1) << 22;
    if (count <= kPiece) {
        const std::vector<int32_t> v(src, src + count);
        LGH_HIP(hipMemcpy(dst, v.data(), sizeof(int32_t) * size_t(count), hipMemcpyHostToDevice));
        return;
    }
    const size_t bytes = sizeof(int64_t) * size_t(std::min(count, kPiece));
    struct Piece {
        int device;
        size_t bytes;
        void *p;
        ~Piece() {
            (void)hipStreamSynchronize(nullptr);
            pool_free(device, p, bytes);
        }
    } piece{device, bytes, pool_alloc(device, bytes)};
    for (int64_t at = 0; at < count; at += kPiece) {
        const int64_t n = std::min(kPiece, count - at);
        LGH_HIP(hipMemcpy(piece.p, src + at, sizeof(int64_t) * size_t(n), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_narrow, dim3(unsigned((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, nullptr, dst + at,
                           static_cast<const int64_t *>(piece.p), n);
        LGH_LAUNCH_CHECK();
    }
}

template <class I, class R>
void csr_launch(const lgh_csr *csr, const cx<R> *x, cx<R> *y, StreamCtx *ctx, double *partials, unsigned blocks) {
    const I *ip = static_cast<const I *>(csr->indptr);
    const I *ix = static_cast<const I *>(csr->indices);
    const cx<R> *vv = static_cast<const cx<R> *>(csr->values);
    auto stream = [&](auto t) {
        hipLaunchKernelGGL((k_csr_stream<I, R, decltype(t)::value>), dim3(blocks), dim3(kBlock), 0, ctx->stream, ip, ix,
                           vv, x, y, csr->rows, partials);
    };
    switch (csr_streams<R>(csr) ? csr_parts(csr->avg_row) : 0) {
    case 1: stream(std::integral_constant<int, 1>{}); break;
    case 2: stream(std::integral_constant<int, 2>{}); break;
    case 4: stream(std::integral_constant<int, 4>{}); break;
    case 8: stream(std::integral_constant<int, 8>{}); break;
    default:
        hipLaunchKernelGGL((k_csr<I, R, 32>), dim3(blocks), dim3(kBlock), 0, ctx->stream, ip, ix, vv, x, y, csr->rows,
                           partials);
    }
    LGH_LAUNCH_CHECK();
}

template <class R> void csr_run(const lgh_csr *csr, const lgh_sv *x, lgh_sv *y, double *re, double *im) {
    StreamCtx *ctx = x->ctx;
    const int per_cu = csr_streams<R>(csr) ? kCsrPerCu : 8;
    const unsigned blocks = unsigned(std::max<int64_t>(
        1, std::min<int64_t>((csr->rows * 16 + kBlock - 1) / kBlock, int64_t(sm_count(x->device)) * per_cu)));
    if (y) {
        if (csr->idx64)
            csr_launch<int64_t, R>(csr, cdata<R>(x), mdata<R>(y), ctx, nullptr, blocks);
        else
            csr_launch<int32_t, R>(csr, cdata<R>(x), mdata<R>(y), ctx, nullptr, blocks);
        return;
    }
    RedBuf rb = red_buf(ctx, 2, int(blocks));
    if (csr->idx64)
        csr_launch<int64_t, R>(csr, cdata<R>(x), nullptr, ctx, rb.partials, blocks);
    else
        csr_launch<int32_t, R>(csr, cdata<R>(x), nullptr, ctx, rb.partials, blocks);
    double out[2];
    reduce_to_host(ctx, rb.partials, int(blocks), 2, out);
    *re = out[0];
    *im = out[1];
}

template <class R> void probs_t(const lgh_sv *sv, const int32_t *wires, int k, double *out) {
    StreamCtx *ctx = sv->ctx;
    const int n = sv->n;
    std::vector<int> out_of(size_t(n), -1); // output bit of an index bit
    for (int j = 0; j < k; ++j) out_of[size_t(n - 1 - wires[j])] = j;
    ProbsMap pm{};
    // the lanes' index bits
    uint64_t lanes = 0;
    int nl = 0;
    auto lane = [&](int bit) {
        if (nl < 6 && bit < n && !((lanes >> bit) & 1)) {
            lanes |= 1ull << bit;
            pm.lane_bit[nl++] = bit;
        }
    };
    if (k >= kProbsWide && n - k <= kProbsWideRest) {
        for (int b = 0; b < (sizeof(R) == 8 ? 3 : 4); ++b) lane(b);
        for (int j = 0; j < 3; ++j) lane(n - 1 - wires[j]);
    }
    for (int b = 0; b < n; ++b) lane(b);
    for (int b = nl; b < 6; ++b) pm.lane_bit[b] = b; // a state of fewer than 6 qubits: those lanes read nothing
    for (int b = 0; b < 6; ++b) pm.lane_out[b] = -1;
    for (int b = 0; b < nl; ++b) {
        if (out_of[size_t(pm.lane_bit[b])] >= 0)
            pm.lane_out[b] = out_of[size_t(pm.lane_bit[b])];
        else
            pm.lane_sum |= 1u << b;
    }
    for (int b = 0; b < n; ++b) {
        if ((lanes >> b) & 1) continue;
        if (out_of[size_t(b)] >= 0) {
            pm.keep_bit[pm.nkeep] = b;
            pm.keep_out[pm.nkeep++] = out_of[size_t(b)];
        } else {
            pm.sum_bit[pm.nsum++] = b;
        }
    }
    // Splits of the summed bits: enough wavefronts to fill the device, each
    // with at least kProbsLoads loads (one group in flight).
    while (pm.log_splits < pm.nsum - 3 && (1ull << (pm.nkeep + pm.log_splits + 1)) <= uint64_t(kProbsMaxWaves))
        ++pm.log_splits;
    static_assert(kProbsLoads == 8, "three loop bits per group of loads");
    const uint64_t nwaves = 1ull << (pm.nkeep + pm.log_splits), bins = 1ull << k;
    // rows of partial sums that the workgroups leave
    const int splits = 1 << (pm.log_splits - std::min(pm.log_splits, kProbsLogWaves));
    const unsigned blocks = unsigned((nwaves + (1u << kProbsLogWaves) - 1) >> kProbsLogWaves);
    const bool to_host = bins <= uint64_t(kProbsHostBins);
    double *host = to_host ? static_cast<double *>(ctx->host_buffer(sizeof(double) * bins)) : nullptr;
    double *ws = static_cast<double *>(ctx->workspace(sizeof(double) * bins * size_t(splits > 1 ? splits + 1 : 1)));
    double *partials = ws, *result = to_host ? host : splits > 1 ? ws + bins * uint64_t(splits) : ws;
    hipLaunchKernelGGL(k_probs<R>, dim3(blocks), dim3(kProbsBlock), 0, ctx->stream, cdata<R>(sv), sv->length(), nwaves,
                       pm, splits > 1 ? partials : result, bins);
    LGH_LAUNCH_CHECK();
    if (splits > 1) {
        const unsigned sblocks = unsigned((bins + kProbsSumBins - 1) / kProbsSumBins);
        hipLaunchKernelGGL(k_probs_sum, dim3(sblocks), dim3(kBlock), 0, ctx->stream, partials, bins, splits, result);
        LGH_LAUNCH_CHECK();
    }
    if (!to_host)
        LGH_HIP(hipMemcpyAsync(out, result, sizeof(double) * bins, hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    if (to_host) std::memcpy(out, host, sizeof(double) * bins);
}

// Returns the device pointer of the sorted indices (in the workspace).
template <class R> uint64_t *sample_t(const lgh_sv *sv, uint64_t shots, uint64_t seed) {
    StreamCtx *ctx = sv->ctx;
    const uint64_t len = sv->length();
    SampleBufs sb{};
    sb.shots = shots;
    sb.seed = seed;
    sb.ntiles = (len + kScanTile - 1) / kScanTile;
    sb.nbins = std::min<uint64_t>(sb.ntiles, kSampleBins); // powers of two
    while ((sb.nbins << sb.log_bin_tiles) < sb.ntiles) ++sb.log_bin_tiles;
    sb.nassign = (shots + kAssignShots - 1) / kAssignShots;
    // at most 256 shared bins however many the shots
    sb.log_bin_shots = kLogBinShots;
    while ((shots >> sb.log_bin_shots) > 256) ++sb.log_bin_shots;
    sb.bin_shots = 1ull << sb.log_bin_shots;
    const uint64_t rows = std::min<uint64_t>(sb.nbins, shots / sb.bin_shots); // bins with more shots than that
    // parts of shared bins: each bin's last one may be short
    const uint32_t nheavy = rows ? uint32_t(shots / sb.bin_shots + rows) : 0;
    sb.nrows = uint32_t(rows);
    auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t size[] = {al(sb.ntiles * 8),
                           256,
                           al(sb.nassign * sb.nbins * 4),
                           al((sb.nbins + 1) * 4),
                           al(nheavy * 8ull),
                           al(sb.nbins * 4),
                           al((rows << sb.log_bin_tiles) * kScanTile * 4),
                           256,
                           al(shots * 4),
                           al(shots * 8),
                           al(shots * 8)};
    size_t bytes = 0;
    for (size_t b : size) bytes += b;
    char *p = static_cast<char *>(ctx->workspace(bytes));
    int k = 0;
    auto take = [&](auto *&dst) {
        dst = reinterpret_cast<std::remove_reference_t<decltype(dst)>>(p);
        p += size[k++];
    };
    uint64_t *out = nullptr;
    take(sb.tile_off);
    take(sb.total);
    take(sb.hist);
    take(sb.bin_off);
    take(sb.heavy);
    take(sb.heavy_id);
    take(sb.heavy_count);
    take(sb.nitems);
    take(sb.where);
    take(sb.thresh);
    take(out);
    uint64_t *total = static_cast<uint64_t *>(ctx->host_buffer(sizeof(uint64_t)));
    const dim3 block(kBlock);
    hipStream_t st = ctx->stream;
    hipLaunchKernelGGL(k_sample_sums<R>, dim3(unsigned(sb.ntiles)), block, 0, st, cdata<R>(sv), len, sb);
    hipLaunchKernelGGL(k_sample_offsets, dim3(1), dim3(kScanBlock), 0, st, sb, total);
    hipLaunchKernelGGL(k_sample_assign, dim3(unsigned(sb.nassign)), dim3(kAssignBlock), 0, st, sb);
    hipLaunchKernelGGL(k_sample_columns, dim3(unsigned((sb.nbins + 31) / 32)), block, 0, st, sb);
    hipLaunchKernelGGL(k_sample_items, dim3(1), dim3(kScanBlock), 0, st, sb);
    hipLaunchKernelGGL(k_sample_scatter, dim3(unsigned((shots + kBlock - 1) / kBlock)), block, 0, st, sb);
    hipLaunchKernelGGL(k_sample_bins<R>, dim3(unsigned(sb.nbins) + nheavy), block, 0, st, cdata<R>(sv), len, sb, out);
    if (nheavy) hipLaunchKernelGGL(k_sample_shared, dim3(nheavy), block, 0, st, sb, out);
    LGH_LAUNCH_CHECK();
    return out;
}

// Waits for the sampler; a state with no probability mass cannot be sampled
// (the indices formed for it are not returned).
void wait_sampled(const lgh_sv *sv) {
    sv->ctx->sync();
    LGH_REQUIRE(*static_cast<const uint64_t *>(sv->ctx->host) > 0, "cannot sample from a zero state");
}

template <class F> void by_dtype(const lgh_sv *sv, F &&f) {
    if (sv->dtype == LGH_C128)
        f(double{});
    else
        f(float{});
}

} // namespace

extern "C" {

lgh_status lgh_inner(const lgh_sv *a, const lgh_sv *b, double *re, double *im) {
    return guard([&] {
        LGH_REQUIRE(a && b && re && im, "null pointer");
        LGH_REQUIRE(a->n == b->n && a->dtype == b->dtype, "states differ in size or precision");
        DeviceGuard g(a->device);
        if (b->ctx != a->ctx) b->ctx->sync();
        by_dtype(a, [&](auto r) { inner_t<decltype(r)>(a, b, re, im); });
    });
}

lgh_status lgh_axpy(lgh_sv *y, double are, double aim, const lgh_sv *x) {
    return guard([&] {
        LGH_REQUIRE(x && y, "null state");
        LGH_REQUIRE(x->n == y->n && x->dtype == y->dtype, "states differ in size or precision");
        DeviceGuard g(y->device);
        if (x->ctx != y->ctx) x->ctx->sync();
        const unsigned blocks = unsigned((y->length() + kBlock - 1) / kBlock);
        by_dtype(y, [&](auto r) {
            using R = decltype(r);
            hipLaunchKernelGGL(k_axpy<R>, dim3(blocks), dim3(kBlock), 0, y->ctx->stream, mdata<R>(y), cdata<R>(x),
                               y->length(), cx<R>{R(are), R(aim)});
        });
        LGH_LAUNCH_CHECK();
    });
}

lgh_status lgh_sv_pauli_word_from(lgh_sv *dst, const lgh_sv *src, const char *paulis, const int32_t *wires,
                                  int32_t num_wires) {
    return guard([&] {
        LGH_REQUIRE(dst && src, "null state");
        LGH_REQUIRE(dst != src && dst->data != src->data, "source and destination must differ");
        LGH_REQUIRE(dst->n == src->n && dst->dtype == src->dtype, "states differ in size or precision");
        LGH_REQUIRE(num_wires >= 0 && (num_wires == 0 || (paulis && wires)), "null Pauli word");
        const int n = dst->n;
        uint64_t xmask = 0, zmask = 0, seen = 0;
        int ny = 0;
        for (int32_t k = 0; k < num_wires; ++k) {
            LGH_REQUIRE(wires[k] >= 0 && wires[k] < n, "wire out of range");
            const uint64_t bit = 1ull << (n - 1 - wires[k]);
            LGH_REQUIRE(!(seen & bit), "repeated wire in a Pauli word");
            seen |= bit;
            switch (paulis[k]) {
            case 'I': break;
            case 'X': xmask |= bit; break;
            case 'Y': xmask |= bit; zmask |= bit; ++ny; break;
            case 'Z': zmask |= bit; break;
            default: throw Error(LGH_ERR_INVALID_ARGUMENT, "Pauli word letters are I, X, Y, Z");
            }
        }
        DeviceGuard g(dst->device);
        if (src->ctx != dst->ctx) src->ctx->sync();
        const uint64_t len = dst->length();
        unsigned blocks = unsigned((len + kBlock - 1) / kBlock);
        if (blocks >= 8) blocks = (blocks + 7) / 8 * 8; // whole XCD rounds for the block order
        by_dtype(dst, [&](auto r) {
            using R = decltype(r);
            hipLaunchKernelGGL(k_pauli_from<R>, dim3(blocks), dim3(kBlock), 0, dst->ctx->stream, mdata<R>(dst),
                               cdata<R>(src), len, xmask, zmask, ny & 3);
        });
        LGH_LAUNCH_CHECK();
    });
}

lgh_status lgh_sv_pauli_sum_from(lgh_sv *dst, const lgh_sv *src, int64_t num_words, const char *paulis,
                                 const int32_t *wires, const int64_t *offsets, const double *coeffs) {
    return guard([&] {
        LGH_REQUIRE(dst && src, "null state");
        LGH_REQUIRE(dst != src && dst->data != src->data, "source and destination must differ");
        LGH_REQUIRE(dst->n == src->n && dst->dtype == src->dtype && dst->device == src->device,
                    "states differ in size or precision");
        LGH_REQUIRE(num_words >= 0, "negative word count");
        LGH_REQUIRE(num_words == 0 || (paulis && offsets && coeffs), "null pointer");
        for (int64_t w = 0; w < num_words; ++w) {
            LGH_REQUIRE(offsets[w + 1] >= offsets[w] && (offsets[w + 1] == offsets[w] || wires),
                        "bad Pauli word offsets");
            for (int64_t a = offsets[w]; a < offsets[w + 1]; ++a)
                for (int64_t b = offsets[w]; b < a; ++b)
                    LGH_REQUIRE(wires[a] != wires[b], "repeated wire in a Pauli word");
        }
        DeviceGuard g(dst->device);
        if (src->ctx != dst->ctx) src->ctx->sync();
        by_dtype(dst, [&](auto r) {
            pauli_sum_t<decltype(r)>(dst, src, num_words, paulis, wires, offsets, coeffs);
        });
    });
}

lgh_status lgh_scale(lgh_sv *x, double are, double aim) {
    return guard([&] {
        LGH_REQUIRE(x, "null state");
        DeviceGuard g(x->device);
        const unsigned blocks = unsigned((x->length() + kBlock - 1) / kBlock);
        by_dtype(x, [&](auto r) {
            using R = decltype(r);
            hipLaunchKernelGGL(k_scale<R>, dim3(blocks), dim3(kBlock), 0, x->ctx->stream, mdata<R>(x), x->length(),
                               cx<R>{R(are), R(aim)});
        });
        LGH_LAUNCH_CHECK();
    });
}

lgh_status lgh_expval_matrix(const lgh_sv *sv, const int32_t *wires, int32_t num_wires, const double *matrix,
                             double *re, double *im) {
    return guard([&] {
        Range rg("lgh_expval_matrix");
        LGH_REQUIRE(sv && wires && matrix && re && im, "null pointer");
        LGH_REQUIRE(num_wires >= 1 && num_wires <= kMaxLdsK && num_wires <= sv->n,
                    "observable must act on 1..13 wires of the state");
        for (int i = 0; i < num_wires; ++i) {
            LGH_REQUIRE(wires[i] >= 0 && wires[i] < sv->n, "wire index out of range");
            for (int j = 0; j < i; ++j) LGH_REQUIRE(wires[i] != wires[j], "repeated wire");
        }
        DeviceGuard g(sv->device);
        by_dtype(sv, [&](auto r) { expval_t<decltype(r)>(sv, wires, num_wires, matrix, re, im); });
    });
}

lgh_status lgh_expval_pauli_words(const lgh_sv *sv, int64_t num_words, const char *paulis, const int32_t *wires,
                                  const int64_t *offsets, const double *coeffs, double *per_word, double *result) {
    return guard([&] {
        Range rg("lgh_expval_pauli_words");
        LGH_REQUIRE(sv && result, "null pointer");
        LGH_REQUIRE(num_words >= 0, "negative word count");
        LGH_REQUIRE(num_words == 0 || (paulis && offsets && coeffs), "null pointer");
        for (int64_t w = 0; w < num_words; ++w)
            LGH_REQUIRE(offsets[w + 1] >= offsets[w] && (offsets[w + 1] == offsets[w] || wires),
                        "bad Pauli word offsets");
        DeviceGuard g(sv->device);
        by_dtype(sv, [&](auto r) {
            pauli_t<decltype(r)>(sv, num_words, paulis, wires, offsets, coeffs, per_word, result);
        });
    });
}

lgh_status lgh_pauli_plan(int32_t num_qubits, int64_t num_words, const char *paulis, const int32_t *wires,
                          const int64_t *offsets, int32_t *tile_passes, int32_t *tile_launches,
                          int32_t *pair_launches) {
    return guard([&] {
        LGH_REQUIRE(num_qubits >= 1 && num_qubits <= 36, "num_qubits must be in [1, 36]");
        LGH_REQUIRE(num_words >= 0 && (num_words == 0 || (paulis && offsets)), "bad word list");
        const size_t nw = size_t(num_words);
        std::vector<uint64_t> flip(nw), zy(nw), mask(std::max<size_t>(1, nw));
        std::vector<int32_t> ny(nw), pass_of(nw);
        for (int64_t w = 0; w < num_words; ++w) {
            LGH_REQUIRE(offsets[w + 1] >= offsets[w] && (offsets[w + 1] == offsets[w] || wires), "bad Pauli word offsets");
            parse_word(num_qubits, paulis, wires, offsets[w], offsets[w + 1], flip[size_t(w)], zy[size_t(w)],
                       ny[size_t(w)]);
        }
        const int64_t np = num_words ? plan_pauli_tiles(num_qubits, num_words, flip.data(), pass_of.data(), mask.data()) : 0;
        std::vector<int64_t> per(size_t(std::max<int64_t>(1, np)), 0);
        std::map<uint64_t, int64_t> pair;
        for (size_t w = 0; w < nw; ++w) {
            if (pass_of[w] >= 0)
                ++per[size_t(pass_of[w])];
            else
                ++pair[flip[w]];
        }
        int64_t tl = 0, pl = 0;
        for (int64_t p = 0; p < np; ++p) tl += (per[size_t(p)] + kPassWords - 1) / kPassWords;
        for (auto &kv : pair) pl += (kv.second + kMaxWordsPerPass - 1) / kMaxWordsPerPass;
        if (tile_passes) *tile_passes = int32_t(np);
        if (tile_launches) *tile_launches = int32_t(tl);
        if (pair_launches) *pair_launches = int32_t(pl);
    });
}

lgh_status lgh_expval_pauli_words_noalloc(const lgh_sv *sv, int64_t num_words, const char *paulis,
                                          const int32_t *wires, const int64_t *offsets, const double *coeffs,
                                          double *per_word, double *result) {
    return guard([&] {
        LGH_REQUIRE(sv && result, "null pointer");
        LGH_REQUIRE(num_words >= 0, "negative word count");
        LGH_REQUIRE(num_words == 0 || (paulis && offsets && coeffs), "null pointer");
        for (int64_t w = 0; w < num_words; ++w)
            LGH_REQUIRE(offsets[w + 1] >= offsets[w] && (offsets[w + 1] == offsets[w] || wires),
                        "bad Pauli word offsets");
        DeviceGuard g(sv->device);
        by_dtype(sv, [&](auto r) {
            pauli_noalloc_t<decltype(r)>(sv, num_words, paulis, wires, offsets, coeffs, per_word, result);
        });
    });
}

lgh_status lgh_csr_create(lgh_csr **out, int device, lgh_dtype dtype, int64_t num_rows, const int64_t *indptr,
                          const int64_t *indices, const double *values, int64_t nnz) {
    return guard([&] {
        LGH_REQUIRE(out && indptr && (nnz == 0 || (indices && values)), "null pointer");
        LGH_REQUIRE(num_rows >= 1, "CSR matrix needs at least one row");
        LGH_REQUIRE(indptr[0] == 0 && indptr[num_rows] == nnz, "CSR offsets do not match nnz");
        // the longest row; a negative length is the longest of all, unsigned
        uint64_t len[4] = {};
        int64_t r = 0;
        for (; r + 4 <= num_rows; r += 4)
            for (int q = 0; q < 4; ++q) len[q] = std::max(len[q], uint64_t(indptr[r + q + 1]) - uint64_t(indptr[r + q]));
        for (; r < num_rows; ++r) len[0] = std::max(len[0], uint64_t(indptr[r + 1]) - uint64_t(indptr[r]));
        const uint64_t longest = std::max({len[0], len[1], len[2], len[3]});
        LGH_REQUIRE(longest <= uint64_t(INT64_MAX), "CSR offsets must not decrease");
        for (int64_t k = 0; k < nnz; ++k)
            LGH_REQUIRE(indices[k] >= 0 && indices[k] < num_rows, "CSR column index out of range");
        auto c = std::make_unique<lgh_csr>();
        c->device = device;
        c->dtype = dtype;
        c->rows = num_rows;
        c->nnz = nnz;
        c->avg_row = double(nnz) / double(num_rows);
        c->longest_row = int64_t(longest);
        // 32-bit indices where they fit: a sixth of a complex128 matrix's bytes
        c->idx64 = num_rows >= (int64_t(1) << 31) || nnz >= (int64_t(1) << 31);
        DeviceGuard g(device);
        const size_t isz = c->idx64 ? 8 : 4;
        c->b_ptr = isz * size_t(num_rows + 1);
        c->b_idx = isz * size_t(std::max<int64_t>(nnz, 1));
        c->b_val = (dtype == LGH_C128 ? 16 : 8) * size_t(std::max<int64_t>(nnz, 1));
        LGH_HIP(hipMalloc(&c->indptr, c->b_ptr));
        LGH_HIP(hipMalloc(&c->indices, c->b_idx));
        LGH_HIP(hipMalloc(&c->values, c->b_val));
        if (c->idx64) {
            LGH_HIP(hipMemcpy(c->indptr, indptr, c->b_ptr, hipMemcpyHostToDevice));
            if (nnz) LGH_HIP(hipMemcpy(c->indices, indices, 8 * size_t(nnz), hipMemcpyHostToDevice));
        } else {
            upload_narrow(device, static_cast<int32_t *>(c->indptr), indptr, num_rows + 1);
            upload_narrow(device, static_cast<int32_t *>(c->indices), indices, nnz);
        }
        if (dtype == LGH_C128) {
            if (nnz) LGH_HIP(hipMemcpy(c->values, values, 16 * size_t(nnz), hipMemcpyHostToDevice));
        } else {
            std::vector<float> v(2 * size_t(nnz));
            for (size_t i = 0; i < v.size(); ++i) v[i] = float(values[i]);
            if (nnz) LGH_HIP(hipMemcpy(c->values, v.data(), 8 * size_t(nnz), hipMemcpyHostToDevice));
        }
        *out = c.release();
    });
}

lgh_status lgh_csr_destroy(lgh_csr *csr) {
    return guard([&] {
        if (!csr) return;
        DeviceGuard g(csr->device);
        (void)hipDeviceSynchronize();
        (void)hipFree(csr->indptr);
        (void)hipFree(csr->indices);
        (void)hipFree(csr->values);
        delete csr;
    });
}

lgh_status lgh_expval_csr(const lgh_sv *sv, const lgh_csr *csr, double *re, double *im) {
    return guard([&] {
        Range rg("lgh_expval_csr");
        LGH_REQUIRE(sv && csr && re && im, "null pointer");
        LGH_REQUIRE(csr->rows == int64_t(sv->length()), "CSR dimension does not match the state");
        LGH_REQUIRE(csr->dtype == sv->dtype && csr->device == sv->device, "CSR precision/device mismatch");
        DeviceGuard g(sv->device);
        by_dtype(sv, [&](auto r) { csr_run<decltype(r)>(csr, sv, nullptr, re, im); });
    });
}

lgh_status lgh_apply_csr(lgh_sv *out, const lgh_csr *csr, const lgh_sv *in) {
    return guard([&] {
        LGH_REQUIRE(out && csr && in, "null pointer");
        LGH_REQUIRE(out != in, "in-place CSR product is not supported");
        LGH_REQUIRE(csr->rows == int64_t(in->length()) && out->n == in->n && out->dtype == in->dtype,
                    "CSR dimension does not match the state");
        LGH_REQUIRE(csr->dtype == in->dtype && csr->device == in->device, "CSR precision/device mismatch");
        DeviceGuard g(in->device);
        if (in->ctx != out->ctx) in->ctx->sync();
        by_dtype(in, [&](auto r) { csr_run<decltype(r)>(csr, in, out, nullptr, nullptr); });
    });
}

lgh_status lgh_probs(const lgh_sv *sv, const int32_t *wires, int32_t num_wires, double *out) {
    return guard([&] {
        Range rg("lgh_probs");
        LGH_REQUIRE(sv && out && (num_wires == 0 || wires), "null pointer");
        LGH_REQUIRE(num_wires >= 0 && num_wires <= sv->n && num_wires <= 30, "bad wire count");
        for (int i = 0; i < num_wires; ++i) {
            LGH_REQUIRE(wires[i] >= 0 && wires[i] < sv->n, "wire index out of range");
            for (int j = 0; j < i; ++j) LGH_REQUIRE(wires[i] != wires[j], "repeated wire");
        }
        DeviceGuard g(sv->device);
        by_dtype(sv, [&](auto r) { probs_t<decltype(r)>(sv, wires, num_wires, out); });
    });
}

lgh_status lgh_sample(const lgh_sv *sv, uint64_t shots, uint64_t seed, uint64_t *indices) {
    return guard([&] {
        Range rg("lgh_sample");
        LGH_REQUIRE(sv && (shots == 0 || indices), "null pointer");
        LGH_REQUIRE(shots < (1ull << 32), "too many shots in one call");
        if (shots == 0) return;
        DeviceGuard g(sv->device);
        uint64_t *d = nullptr;
        by_dtype(sv, [&](auto r) { d = sample_t<decltype(r)>(sv, shots, seed); });
        wait_sampled(sv);
        LGH_HIP(hipMemcpyAsync(indices, d, 8 * shots, hipMemcpyDeviceToHost, sv->ctx->stream));
        sv->ctx->sync();
    });
}

lgh_status lgh_sample_bits(const lgh_sv *sv, uint64_t shots, uint64_t seed, uint64_t *bits) {
    return guard([&] {
        LGH_REQUIRE(sv && (shots == 0 || bits), "null pointer");
        LGH_REQUIRE(shots < (1ull << 32), "too many shots in one call");
        if (shots == 0) return;
        DeviceGuard g(sv->device);
        uint64_t *d = nullptr;
        by_dtype(sv, [&](auto r) { d = sample_t<decltype(r)>(sv, shots, seed); });
        wait_sampled(sv);
        const uint64_t total = shots * uint64_t(sv->n);
        // the expanded bits go to a separate buffer (the workspace holds the indices)
        uint64_t *dbits = static_cast<uint64_t *>(pool_alloc(sv->device, 8 * total));
        hipLaunchKernelGGL(k_expand_bits, dim3(unsigned((total + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                           sv->ctx->stream, d, shots, sv->n, dbits);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(bits, dbits, 8 * total, hipMemcpyDeviceToHost, sv->ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(sv->ctx->stream);
        pool_free(sv->device, dbits, 8 * total);
        LGH_HIP(e);
    });
}

} // extern "C"
