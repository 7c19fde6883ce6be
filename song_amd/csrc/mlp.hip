// Learned form: the entry-vertex / stop-step MLP on the matrix cores (include/song_learned.h).
//
// Matrix products use v_mfma_f32_16x16x16_bf16 (BF16 inputs, FP32 accumulation).  Fragment
// layout of one 16x16x16 product for wave lane l (verified by the GEMM test against numpy):
//   A[i][k]: i = l % 16, k = 4*(l/16) + j     (j = 0..3, the 4 bf16 of the lane's operand)
//   B[k][n]: n = l % 16, k = 4*(l/16) + j
//   D[i][n]: n = l % 16, i = 4*(l/16) + j
// Training runs as separate kernels (GEMM with bias/ReLU/mask epilogues, softmax
// cross-entropy, column sums, Adam); inference is one fused kernel, 16 queries per workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/song_learned.h"

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

static thread_local std::string g_mlp_err;

static int mfail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_mlp_err = buf;
    return code;
}

#define MHIP(expr)                                                                          \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) return mfail(-2, "%s: %s", #expr, hipGetErrorString(e_));    \
    } while (0)

extern "C" const char *song_mlp_last_error(void) { return g_mlp_err.c_str(); }

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// ---------------------------------------------------------------- GEMM

struct GemmArgs {
    int M, N, K;
    const uint16_t *A;
    long long sam, sak;
    const uint16_t *B;
    long long sbk, sbn;
    float *C;
    int ldc;
    float alpha;
};

constexpr int GBM = 64, GBN = 64, GBK = 16;

// C[m][n] = alpha * sum_k A(m,k) B(k,n), A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn], any
// strides (song_gemm_bf16; the network's own products are tile_kernel's).  256 threads: 2x2 waves of
// 32x32, each 2x2 MFMA tiles.
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g) {
    __shared__ uint16_t As[GBM][GBK + 4];
    __shared__ uint16_t Bs[GBN][GBK + 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    v4f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < g.K; k0 += GBK) {
        for (int e = tid; e < GBM * GBK; e += 256) {
            const int r = e / GBK, c = e % GBK, m = m0 + r, k = k0 + c;
            As[r][c] = (m < g.M && k < g.K) ? g.A[(long long)m * g.sam + (long long)k * g.sak] : (uint16_t)0;
        }
        for (int e = tid; e < GBN * GBK; e += 256) {
            const int r = e / GBK, c = e % GBK, n = n0 + r, k = k0 + c;
            Bs[r][c] = (n < g.N && k < g.K) ? g.B[(long long)k * g.sbk + (long long)n * g.sbn] : (uint16_t)0;
        }
        __syncthreads();
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                v4s a, b;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a[j] = (short)As[wm + mi * 16 + (lane & 15)][4 * (lane >> 4) + j];
                    b[j] = (short)Bs[wn + ni * 16 + (lane & 15)][4 * (lane >> 4) + j];
                }
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[mi][ni], 0, 0, 0);
            }
        __syncthreads();
    }
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + wm + mi * 16 + 4 * (lane >> 4) + j;
                const int n = n0 + wn + ni * 16 + (lane & 15);
                if (m < g.M && n < g.N) g.C[(long long)m * g.ldc + n] = g.alpha * acc[mi][ni][j];
            }
}

// ---------------------------------------------------------------- the network's products

// The training products: operands whose rows are 16-byte aligned along one of their two directions.
// A block computes BM x BN with 2 x 2 waves, BK of the contraction at a time, through two LDS buffers
// of k-contiguous rows; the next PF tiles' global loads are in flight while one is multiplied.  An
// operand that is contiguous along the contraction is stored as it is loaded; one that is contiguous
// across it (the transposed factors of the weight gradients and of the backward products) is turned
// in registers (Stage).  Each output is one accumulator chain over ascending k in steps of 16 (no split of
// the contraction), so results equal gemm_kernel's bit for bit.  Bound: the latency of the k loop --
// the shapes give each CU one or two blocks -- not the matrix cores.  Against gemm_kernel, which reads
// two bytes per lane and load, 12 training steps (batch 1,024, 136-256-256-4,097) and one read of the
// parameters went from 19.8 to 1.37 ms, with the loss and update kernels below.
enum Along { ALONG_K, ALONG_ROW };  // what is contiguous in memory: the contraction, or the operand's rows

struct TileArgs {
    int M, N, K;
    const uint16_t *A;
    int lda;  // elements between rows (ALONG_K) or between k (ALONG_ROW)
    const uint16_t *B;
    int ldb;
    float *C;  // float32 output or null
    int ldc;
    uint16_t *Cb;  // bf16 output or null
    int ldcb;
    const float *bias;     // per column, or null
    const uint16_t *mask;  // zero the output where mask[m][n] <= 0 (ReLU backward), or null
    int ldm;
    int relu;
    float *rowsum;  // sum over k of A per row m, ascending k (the bias gradient), or null
};

// BR rows x BK of one operand, by 128 threads (t = 0..127): global memory -> registers -> LDS.  A unit
// is 8 k of one row (ALONG_K, one 16-byte load) or 4 k of 4 rows (ALONG_ROW, four 8-byte loads turned
// into four 8-byte k runs).  Each unit keeps its pointer and advances by a tile, so a load costs no
// address arithmetic; k past K (the last tile only) reads as zero; rows past R read a valid row,
// whose outputs are not stored.
// The two operands' movers share one state (Mover): half the block's waves run one, half the other.
template <int NP> struct Mover {
    const uint16_t *ptr[NP];
    size_t ld, step;
    int t;
};
template <int BR, int BK, Along AL> struct Stage {
    // LDS row stride: 2 words more than a multiple of 32, so that the 16 rows of a fragment read, and
    // the 4 x 4 units that 16 lanes of a turned store write, fall on different banks (a stride of BK + 8
    // elements had 14 of 22 LDS cycles per access in conflicts, and LDS was what bound the backward)
    static constexpr int LD = BK + 4;
    static constexpr int UNITS = AL == ALONG_K ? BR * BK / 8 : BR * BK / 16;
    static constexpr int PER = UNITS / 128;              // units per thread
    static constexpr int REGS = AL == ALONG_K ? PER : 2 * PER;  // 16-byte registers per tile
    static_assert(UNITS % 128 == 0, "whole units per thread");
    // 16 lanes of turned units take 4 row groups x 4 k groups
    __device__ __forceinline__ static int row_of(int u) {
        return AL == ALONG_K ? u / (BK / 8) : (((u >> 4) % (BR / 16)) * 4 + (u & 3)) * 4;
    }
    __device__ __forceinline__ static int k_of(int u) {
        return AL == ALONG_K ? (u % (BK / 8)) * 8 : (((u >> 4) / (BR / 16)) * 4 + ((u >> 2) & 3)) * 4;
    }
    template <int NP>
    __device__ __forceinline__ static void init(Mover<NP> &c, const uint16_t *X, int ldx, int r0, int R) {
        const size_t ld = (size_t)ldx;
        c.ld = ld;
        c.step = AL == ALONG_K ? (size_t)BK : (size_t)BK * ld;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int u = c.t + 128 * i;
            const int r = AL == ALONG_K ? min(r0 + row_of(u), R - 1) : min(r0 + row_of(u), (R - 1) & ~3);
            c.ptr[i] = AL == ALONG_K ? X + (size_t)r * ld + k_of(u) : X + (size_t)k_of(u) * ld + r;
        }
    }
    // the tile the pointers stand at (its first k is k0)
    template <int NP, int NV> __device__ __forceinline__ static void load(Mover<NP> &c, uint4 (&v)[NV], int k0, int K) {
        const size_t ld = c.ld;
        if (k0 + BK <= K) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if constexpr (AL == ALONG_K) {
                    v[i] = *reinterpret_cast<const uint4 *>(c.ptr[i]);
                } else {
                    const uint2 a = *reinterpret_cast<const uint2 *>(c.ptr[i]);
                    const uint2 b = *reinterpret_cast<const uint2 *>(c.ptr[i] + ld);
                    const uint2 e = *reinterpret_cast<const uint2 *>(c.ptr[i] + 2 * ld);
                    const uint2 d = *reinterpret_cast<const uint2 *>(c.ptr[i] + 3 * ld);
                    v[2 * i] = make_uint4(a.x, a.y, b.x, b.y);
                    v[2 * i + 1] = make_uint4(e.x, e.y, d.x, d.y);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int k = k0 + k_of(c.t + 128 * i);
                if constexpr (AL == ALONG_K) {
                    v[i] = k < K ? *reinterpret_cast<const uint4 *>(c.ptr[i]) : make_uint4(0u, 0u, 0u, 0u);
                    const auto cut = [&](uint32_t w, int e) {  // elements e, e + 1 of the unit
                        return (k + e < K ? w & 0x0000ffffu : 0u) | (k + e + 1 < K ? w & 0xffff0000u : 0u);
                    };
                    v[i] = make_uint4(cut(v[i].x, 0), cut(v[i].y, 2), cut(v[i].z, 4), cut(v[i].w, 6));
                } else {
                    const auto one = [&](int j) {
                        return k + j < K ? *reinterpret_cast<const uint2 *>(c.ptr[i] + j * ld) : make_uint2(0u, 0u);
                    };
                    const uint2 a = one(0), b = one(1), e = one(2), d = one(3);
                    v[2 * i] = make_uint4(a.x, a.y, b.x, b.y);
                    v[2 * i + 1] = make_uint4(e.x, e.y, d.x, d.y);
                }
            }
        }
    }
    template <int NP, int NV>
    __device__ __forceinline__ static void store(const Mover<NP> &c, const uint4 (&v)[NV], uint16_t *lds) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int u = c.t + 128 * i;
            uint16_t *o = lds + row_of(u) * LD + k_of(u);
            if constexpr (AL == ALONG_K) {
                *reinterpret_cast<uint2 *>(o) = make_uint2(v[i].x, v[i].y);
                *reinterpret_cast<uint2 *>(o + 4) = make_uint2(v[i].z, v[i].w);
            } else {
                const uint32_t k0[2] = {v[2 * i].x, v[2 * i].y}, k1[2] = {v[2 * i].z, v[2 * i].w};
                const uint32_t k2[2] = {v[2 * i + 1].x, v[2 * i + 1].y}, k3[2] = {v[2 * i + 1].z, v[2 * i + 1].w};
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t sel = (r & 1) ? 0x07060302u : 0x05040100u;
                    uint2 x;
                    x.x = __builtin_amdgcn_perm(k1[r >> 1], k0[r >> 1], sel);
                    x.y = __builtin_amdgcn_perm(k3[r >> 1], k2[r >> 1], sel);
                    *reinterpret_cast<uint2 *>(o + r * LD) = x;
                }
            }
        }
    }
};

template <int BM, int BN, int BK, Along AA, Along AB, int PF>
__device__ __forceinline__ void tile_gemm(const TileArgs &g, int bm, int bn, uint16_t *lds) {
    using SA = Stage<BM, BK, AA>;
    using SB = Stage<BN, BK, AB>;
    constexpr int LD = SA::LD, TM = BM / 32, TN = BN / 32, BUF = (BM + BN) * LD;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = bm * BM, n0 = bn * BN;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    v4f acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    // one block more per row of blocks adds A's rows and multiplies nothing: the sums are a serial
    // chain as long as the contraction, which in a multiplying block came on top of its products
    const bool sums = n0 >= g.N;
    float rs = 0.0f;
    // waves 0 and 1 move A, waves 2 and 3 move B
    const bool first = wave < 2;
    constexpr bool SAME = AA == AB && BM == BN;
    constexpr int NP = SA::PER > SB::PER ? SA::PER : SB::PER;
    Mover<NP> mv;
#pragma unroll
    for (int i = 0; i < NP; ++i) mv.ptr[i] = g.A;
    uint4 v[PF][SA::REGS > SB::REGS ? SA::REGS : SB::REGS];
    mv.t = tid & 127;
    if (SAME) SA::init(mv, first ? g.A : g.B, first ? g.lda : g.ldb, first ? m0 : n0, first ? g.M : g.N);
    else if (first) SA::init(mv, g.A, g.lda, m0, g.M);
    else SB::init(mv, g.B, g.ldb, n0, g.N);
    const int nk = (g.K + BK - 1) / BK;
    const auto fetch = [&](int slot, int it) __attribute__((always_inline)) {
        if (it < nk) {
            if (SAME || first) SA::load(mv, v[slot], it * BK, g.K);
            else SB::load(mv, v[slot], it * BK, g.K);
#pragma unroll
            for (int i = 0; i < NP; ++i) mv.ptr[i] += mv.step;
        }
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) fetch(p, p);
    for (int it0 = 0; it0 < nk; it0 += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int it = it0 + p;
            if (it >= nk) break;
            // two buffers and one barrier per tile: a wave that writes tile it + 1 has passed the barrier
            // of tile it, so every wave is done with the buffer of tile it - 1
            uint16_t *As = lds + (it & 1) * BUF, *Bs = As + BM * LD;
            if (SAME) SA::store(mv, v[p], first ? As : Bs);
            else if (first) SA::store(mv, v[p], As);
            else SB::store(mv, v[p], Bs);
            __syncthreads();
            fetch(p, it + PF);
#pragma unroll
            for (int kk = 0; kk < BK; kk += 16) {
                if (sums) break;
                v4s a[TM], b[TN];
#pragma unroll
                for (int mi = 0; mi < TM; ++mi)
                    a[mi] = *reinterpret_cast<const v4s *>(As + (wm + mi * 16 + (lane & 15)) * LD + kk + 4 * (lane >> 4));
#pragma unroll
                for (int ni = 0; ni < TN; ++ni)
                    b[ni] = *reinterpret_cast<const v4s *>(Bs + (wn + ni * 16 + (lane & 15)) * LD + kk + 4 * (lane >> 4));
#pragma unroll
                for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[mi], b[ni], acc[mi][ni], 0, 0, 0);
            }
            if (sums && tid < BM) {
#pragma unroll
                for (int k = 0; k < BK; k += 4) {
                    const uint2 x = *reinterpret_cast<const uint2 *>(As + tid * LD + k);
                    const uint32_t w[2] = {x.x, x.y};
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        rs += __uint_as_float(w[t] << 16);
                        rs += __uint_as_float(w[t] & 0xffff0000u);
                    }
                }
            }
        }
    }
    if (sums) {
        if (tid < BM && m0 + tid < g.M) g.rowsum[m0 + tid] = rs;
        return;
    }
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + wm + mi * 16 + 4 * (lane >> 4) + j;
                const int n = n0 + wn + ni * 16 + (lane & 15);
                if (m < g.M && n < g.N) {
                    float v = acc[mi][ni][j];
                    if (g.bias) v += g.bias[n];
                    if (g.relu) v = fmaxf(v, 0.0f);
                    if (g.mask && bf2f(g.mask[(size_t)m * g.ldm + n]) <= 0.0f) v = 0.0f;
                    if (g.C) g.C[(size_t)m * g.ldc + n] = v;
                    if (g.Cb) g.Cb[(size_t)m * g.ldcb + n] = f2bf(v);
                }
            }
}

template <int BM, int BN, int BK, Along AA, Along AB, int PF>
__global__ __launch_bounds__(256) void tile_kernel(TileArgs g) {
    __shared__ __align__(16) uint16_t lds[2 * (BM + BN) * (BK + 4)];
    tile_gemm<BM, BN, BK, AA, AB, PF>(g, blockIdx.y, blockIdx.x, lds);
}

// Two independent products of one backward stage in one launch, blocks of the first before those of
// the second: the input gradient (rows along k, weights across it) and the weight gradient (both
// across it).  Neither fills the device alone.
template <int BM1, int BN1, int BK1, int PF1, int BM2, int BN2, int BK2, int PF2>
__global__ __launch_bounds__(256) void tile_pair_kernel(TileArgs g1, int nb1, int nn1, TileArgs g2, int nn2) {
    constexpr int L1 = 2 * (BM1 + BN1) * (BK1 + 4), L2 = 2 * (BM2 + BN2) * (BK2 + 4);
    __shared__ __align__(16) uint16_t lds[L1 > L2 ? L1 : L2];
    const int b = blockIdx.x;
    if (b < nb1)
        tile_gemm<BM1, BN1, BK1, ALONG_K, ALONG_ROW, PF1>(g1, b / nn1, b % nn1, lds);
    else
        tile_gemm<BM2, BN2, BK2, ALONG_ROW, ALONG_ROW, PF2>(g2, (b - nb1) / nn2, (b - nb1) % nn2, lds);
}

static int tiles(int n, int b) { return (n + b - 1) / b; }
// blocks along n: the products' and, with row sums, one for those
static int tiles_n(const TileArgs &g, int b) { return tiles(g.N, b) + (g.rowsum ? 1 : 0); }

template <int BM, int BN, int BK, Along AA, Along AB, int PF>
static int tile_launch(const TileArgs &g, hipStream_t st) {
    hipLaunchKernelGGL((tile_kernel<BM, BN, BK, AA, AB, PF>), dim3(tiles_n(g, BN), tiles(g.M, BM)), dim3(256), 0, st, g);
    MHIP(hipGetLastError());
    return 0;
}

extern "C" int song_gemm_bf16(int M, int N, int K, const uint16_t *d_a, int sam, int sak, const uint16_t *d_b, int sbk,
                              int sbn, float *d_c, int ldc, float alpha, void *stream) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const GemmArgs g{M, N, K, d_a, sam, sak, d_b, sbk, sbn, d_c, ldc, alpha};
    hipLaunchKernelGGL(gemm_kernel, dim3(tiles(N, GBN), tiles(M, GBM)), dim3(256), 0, (hipStream_t)stream, g);
    MHIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------- loss, sums, Adam

// One block of four waves per row: softmax cross-entropy over the first C logits against the label,
// squared error of logit C against the stop target; writes dZ (bf16) and the row's share of the batch
// means of both losses.  Every exponential is computed once, by all waves, and kept in LDS (C + 1
// floats); the first wave adds them, lane l the columns l, l + 64, ... in ascending order and then
// the lanes in halving steps, the order a single wave per row has, so the sum does not depend on the
// waves.  Rows too wide for LDS (IN_LDS false) compute the exponentials again where they are used.
// One wave per row that computed each exponential twice took 64 us for 1,024 rows of 4,097; four waves
// that added the losses to one pair of floats took 39 us, most of it those 2,048 atomics; now 10 us.
constexpr int LOSS_LDS_CLASSES = 12288;  // 48 KB: three blocks fit a CU's LDS
template <bool IN_LDS>
__global__ __launch_bounds__(256) void loss_kernel(const float *Z, int ldz, int C, const int *labels, const float *stop_t,
                                                   int B, float stop_w, uint16_t *dZ, int lddz, float2 *row_loss) {
    extern __shared__ __align__(16) float ex[];
    __shared__ float red[8];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *z = Z + (long long)row * ldz;
    uint16_t *dz = dZ + (long long)row * lddz;
    const int C4 = C & ~3;  // columns taken four at a time (rows are 16-byte aligned), then the rest
    float mx = -INFINITY;
    for (int c = 4 * tid; c < C4; c += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(z + c);
        if (IN_LDS) *reinterpret_cast<float4 *>(ex + c) = v;
        mx = fmaxf(fmaxf(fmaxf(mx, v.x), fmaxf(v.y, v.z)), v.w);
    }
    if (C4 + tid < C) {
        const float v = z[C4 + tid];
        if (IN_LDS) ex[C4 + tid] = v;
        mx = fmaxf(mx, v);
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    if (IN_LDS) {
        for (int c = tid; c < C; c += 256) ex[c] = expf(ex[c] - mx);
        __syncthreads();
    }
    if (wave == 0) {
        float se = 0.0f;
        int c = lane;
        if (IN_LDS)
            for (; c + 7 * 64 < C; c += 512) {  // eight reads in flight, added in order
                float e[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) e[t] = ex[c + 64 * t];
#pragma unroll
                for (int t = 0; t < 8; ++t) se += e[t];
            }
        for (; c < C; c += 64) se += IN_LDS ? ex[c] : expf(z[c] - mx);
        for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o);
        if (lane == 0) red[4] = se;
    }
    __syncthreads();
    const float se = red[4];
    const int lab = labels[row];
    const float inv = 1.0f / (float)B;
    const auto grad = [&](float e, int c) { return f2bf((e / se - (c == lab ? 1.0f : 0.0f)) * inv); };
    for (int c = 4 * tid; c < C4; c += 1024) {
        float4 e = *reinterpret_cast<const float4 *>(IN_LDS ? ex + c : z + c);
        if (!IN_LDS) e = make_float4(expf(e.x - mx), expf(e.y - mx), expf(e.z - mx), expf(e.w - mx));
        *reinterpret_cast<ushort4 *>(dz + c) = make_ushort4(grad(e.x, c), grad(e.y, c + 1), grad(e.z, c + 2), grad(e.w, c + 3));
    }
    if (C4 + tid < C) {
        const int c = C4 + tid;
        dz[c] = grad(IN_LDS ? ex[c] : expf(z[c] - mx), c);
    }
    if (tid == 0) {
        const float diff = z[C] - stop_t[row];
        dz[C] = f2bf(2.0f * stop_w * diff * inv);
        row_loss[row] = make_float2((logf(se) + mx - z[lab]) * inv, diff * diff * inv);
    }
}

// the batch's losses from its rows', when they are asked for
__global__ __launch_bounds__(256) void loss_sum_kernel(const float2 *row_loss, int B, float *loss) {
    __shared__ float2 part[4];
    const int tid = threadIdx.x;
    float2 s = make_float2(0.0f, 0.0f);
    for (int i = tid; i < B; i += 256) {
        s.x += row_loss[i].x;
        s.y += row_loss[i].y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        s.x += __shfl_xor(s.x, o);
        s.y += __shfl_xor(s.y, o);
    }
    if ((tid & 63) == 0) part[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        loss[0] = (part[0].x + part[1].x) + (part[2].x + part[3].x);
        loss[1] = (part[0].y + part[1].y) + (part[2].y + part[3].y);
    }
}

// The parameter vector's segments (W1 b1 W2 b2 W3 b3) and the bf16 copies of its weights
struct ParamCopies {
    long long off[6], cnt[6];
    uint16_t *Wb[3];
    uint16_t *W3i;  // the output weights in the layout infer_kernel reads (see refresh_kernel)
    int rows3, hidden, npad;
};
struct AdamArgs {
    float *p;
    const float *g;
    float *m, *v;
    float lr, b1, b2, c1, c2, eps;
};

__device__ __forceinline__ void adam_one(const AdamArgs &a, float gi, float &p, float &m, float &v) {
    // contracted as written (the compiler would choose per use, and the two loops would differ)
    m = fmaf(1.0f - a.b1, gi, a.b1 * m);
    v = fmaf(gi, (1.0f - a.b2) * gi, a.b2 * v);
    p -= a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
}

// Every parameter once: with ADAM the update, then the bf16 copies of the weights, the output
// weights twice -- row by row for the products, and for inference in pairs of k quads: W3[n][32s + 4q
// .. +4) and W3[n][32s + 16 + 4q .. +4) at W3i[((4s + q) * npad + n) * 8], zero for n >= rows3 and past
// the last hidden unit, so that a lane reads its fragments of two k-steps in one 16-byte load and the
// 16 columns of a lane group are one aligned 256-byte run.  The first blocks
// take W3 in tiles of 16 rows x 64 columns, four columns per lane (64-byte runs of the float arrays,
// half-filled 256-byte runs of W3i); the rest take the other segments in order.  Bound by memory: 30 bytes per
// parameter.  As five kernels (update, three conversions, interleave) a step took 26 us at 1.16
// million parameters and read the new weights three times.
template <bool ADAM>
__global__ __launch_bounds__(256) void refresh_kernel(AdamArgs a, ParamCopies c, int w3_blocks) {
    const int tid = threadIdx.x;
    if ((int)blockIdx.x < w3_blocks) {
        const int kt = (c.hidden + 63) / 64;
        const int n = ((int)blockIdx.x / kt) * 16 + (tid & 15), k = ((int)blockIdx.x % kt) * 64 + (tid >> 4) * 4;
        if (k >= c.hidden) return;
        uint16_t h[4] = {0, 0, 0, 0};
        if (n < c.rows3) {
            const long long i = c.off[4] + (long long)n * c.hidden + k;  // (a multiple of four: so are all segments)
            float4 p = *reinterpret_cast<const float4 *>(a.p + i);
            if constexpr (ADAM) {
                const float4 gr = *reinterpret_cast<const float4 *>(a.g + i);
                float4 mo = *reinterpret_cast<const float4 *>(a.m + i), vo = *reinterpret_cast<const float4 *>(a.v + i);
                adam_one(a, gr.x, p.x, mo.x, vo.x);
                adam_one(a, gr.y, p.y, mo.y, vo.y);
                adam_one(a, gr.z, p.z, mo.z, vo.z);
                adam_one(a, gr.w, p.w, mo.w, vo.w);
                *reinterpret_cast<float4 *>(a.p + i) = p;
                *reinterpret_cast<float4 *>(a.m + i) = mo;
                *reinterpret_cast<float4 *>(a.v + i) = vo;
            }
            h[0] = f2bf(p.x), h[1] = f2bf(p.y), h[2] = f2bf(p.z), h[3] = f2bf(p.w);
            *reinterpret_cast<ushort4 *>(c.Wb[2] + (long long)n * c.hidden + k) = make_ushort4(h[0], h[1], h[2], h[3]);
        }
        const long long sq = (long long)(k >> 5) * 4 + ((k >> 2) & 3);
        *reinterpret_cast<ushort4 *>(c.W3i + (sq * c.npad + n) * 8 + ((k >> 4) & 1) * 4) = make_ushort4(h[0], h[1], h[2], h[3]);
        return;
    }
    // W1 b1 W2 b2 are one run, b3 is the last
    const long long run = c.off[4];
    long long i = ((long long)blockIdx.x - w3_blocks) * 256 + tid;
    if (i >= run) i += c.cnt[4];
    if (i >= c.off[5] + c.cnt[5]) return;
    float p = a.p[i];
    if constexpr (ADAM) {
        float mo = a.m[i], vo = a.v[i];
        adam_one(a, a.g[i], p, mo, vo);
        a.p[i] = p;
        a.m[i] = mo;
        a.v[i] = vo;
    }
    if (i < c.cnt[0]) c.Wb[0][i] = f2bf(p);
    else if (i >= c.off[2] && i < c.off[2] + c.cnt[2]) c.Wb[1][i - c.off[2]] = f2bf(p);
}

// ---------------------------------------------------------------- features

__global__ __launch_bounds__(64) void features_kernel(const float *Q, int dim, const float *mean, const float *inv_std,
                                                      const float *v0, float f0, float f1, float f2, float f3,
                                                      float f4, float f5, float f6, float f7, uint16_t *X,
                                                      int width) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const float *q = Q + (long long)row * dim;
    uint16_t *x = X + (long long)row * width;
    float s = 0.f, s2 = 0.f, dv = 0.f, mn = INFINITY, mx = -INFINITY, nz = 0.f;
    for (int i = lane; i < dim; i += 64) {
        const float v = q[i];
        x[i] = f2bf((v - mean[i]) * inv_std[i]);
        s += v;
        s2 += v * v;
        const float d = v - v0[i];
        dv += d * d;
        mn = fminf(mn, v);
        mx = fmaxf(mx, v);
        nz += (v == 0.0f) ? 1.0f : 0.0f;
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o);
        s2 += __shfl_xor(s2, o);
        dv += __shfl_xor(dv, o);
        mn = fminf(mn, __shfl_xor(mn, o));
        mx = fmaxf(mx, __shfl_xor(mx, o));
        nz += __shfl_xor(nz, o);
    }
    if (lane < 8) {
        const float meanq = s / dim;
        const float var = fmaxf(s2 / dim - meanq * meanq, 0.0f);
        float f;
        switch (lane) {
        case 0: f = sqrtf(s2) * f0; break;
        case 1: f = sqrtf(dv) * f1; break;
        case 2: f = meanq * f2; break;
        case 3: f = sqrtf(var) * f3; break;
        case 4: f = mn * f4; break;
        case 5: f = mx * f5; break;
        case 6: f = nz / dim * f6; break;
        default: f = f7; break;
        }
        x[dim + lane] = f2bf(f);
    }
    for (int i = dim + 8 + lane; i < width; i += 64) x[i] = 0;
}

// ---------------------------------------------------------------- fused inference

struct InferArgs {
    const uint16_t *X;
    int batch, width, hidden, C;
    const uint16_t *W1, *W2, *W3;
    const uint16_t *W3i;  // W3 in the layout of refresh_kernel, npad columns
    int npad;
    const float *b1, *b2, *b3;
    int *top2;  // batch x 2 pivot indices (best first)
    float *conf, *stop, *logits;
    const int *nbr;  // C x n_nbr pivot neighbourhoods (row a starts with a) or null
    int n_nbr;
    int x16;  // 1: X can be read in 16-byte units
};

// exp(x) for finite x <= REF_SPAN to within an ulp or two: 2^(x log2 e) by the hardware's exponential, the
// product's rounding error carried along and put back as a first-order factor
__device__ __forceinline__ float exp_mid(float x) {
    const float L = 1.44269502f, Ll = 1.92596303e-8f, ln2 = 0.693147182f;  // L + Ll = log2 e
    const float hi = x * L;
    const float lo = fmaf(x, Ll, fmaf(x, L, -hi));
    const float e = __builtin_amdgcn_exp2f(hi);
    return fmaf(e, lo * ln2, e);
}

// One hidden layer on the LDS tile: out[r][n] = relu(in[r] . W[n] + bias[n]) for this block's rows,
// the waves taking 16 columns at a time.  The weight fragments of eight k-steps are loaded together,
// so a tile waits for memory once or twice, not once per step.
template <int MI, int WAVES>
__device__ __forceinline__ void hidden_layer(const uint16_t *in, int ldin, int K, const uint16_t *W, const float *bias,
                                             int N, uint16_t *out, int ldo) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kq = 4 * (lane >> 4);
    const uint16_t *arow = in + (lane & 15) * ldin + kq;
    for (int n0 = wave * 16; n0 < N; n0 += WAVES * 16) {  // (N is a multiple of 16)
        const int n = n0 + (lane & 15);
        const uint16_t *w = W + (size_t)n * K + kq;
        v4f acc[MI];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[mi] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < K; k0 += 128) {
            v4s b[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) b[t] = *reinterpret_cast<const v4s *>(w + min(k0 + 16 * t, K - 16));
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if (k0 + 16 * t >= K) break;
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
                    acc[mi] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                        *reinterpret_cast<const v4s *>(arow + mi * 16 * ldin + k0 + 16 * t), b[t], acc[mi], 0, 0, 0);
            }
        }
        const float bn = bias[n];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                out[(mi * 16 + 4 * (lane >> 4) + t) * ldo + n] = f2bf(fmaxf(acc[mi][t] + bn, 0.0f));
    }
}

// softmax state of a row: top two (value, index) and the sum of exp(v - v1)
struct Soft {
    float v1, v2, s;
    int a1, a2;
};
__device__ __forceinline__ bool better(float v, int a, float w, int b) { return v > w || (v == w && a < b); }
__device__ __forceinline__ Soft soft_empty() { return Soft{-INFINITY, -INFINITY, 0.0f, 0x7fffffff, 0x7fffffff}; }
__device__ __forceinline__ Soft soft_merge(const Soft &x, const Soft &y) {
    if (y.v1 == -INFINITY) return x;
    if (x.v1 == -INFINITY) return y;
    Soft t;
    const bool xf = better(x.v1, x.a1, y.v1, y.a1);
    // field by field (a conditional over the two structs would select their addresses, which
    // puts them in scratch memory)
    Soft hi, lo;
    hi.v1 = xf ? x.v1 : y.v1;
    hi.v2 = xf ? x.v2 : y.v2;
    hi.s = xf ? x.s : y.s;
    hi.a1 = xf ? x.a1 : y.a1;
    hi.a2 = xf ? x.a2 : y.a2;
    lo.v1 = xf ? y.v1 : x.v1;
    lo.v2 = xf ? y.v2 : x.v2;
    lo.s = xf ? y.s : x.s;
    lo.a1 = xf ? y.a1 : x.a1;
    lo.a2 = xf ? y.a2 : x.a2;
    t.v1 = hi.v1;
    t.a1 = hi.a1;
    t.s = hi.s + lo.s * expf(lo.v1 - hi.v1);
    if (better(hi.v2, hi.a2, lo.v1, lo.a1)) {
        t.v2 = hi.v2;
        t.a2 = hi.a2;
    } else {
        t.v2 = lo.v1;
        t.a2 = lo.a1;
    }
    return t;
}

// A row's running state over the columns one lane owns, in ascending order: the top two, and the sum
// of exp(v - ref) for a reference that only moves when a value exceeds it by REF_SPAN (the sum of at
// most 2^31 terms below e^REF_SPAN stays finite), so that a value costs one exponential.
constexpr float REF_SPAN = 40.0f;
struct Lane {
    float v1, v2, s, ref;
    int a1, a2;
};
// `v` of column `a`, larger than every column before it (a tie keeps the earlier one), into the top two
__device__ __forceinline__ void lane_top(Lane &t, float v, int a) {
    const bool b1 = v > t.v1, b2 = v > t.v2;
    t.a2 = b1 ? t.a1 : (b2 ? a : t.a2);
    t.a1 = b1 ? a : t.a1;
    t.v2 = b1 ? t.v1 : (b2 ? v : t.v2);
    t.v1 = b1 ? v : t.v1;
}
// one value into the sum, whatever it is (NaN stays NaN, -inf adds nothing)
__device__ __forceinline__ void lane_sum(Lane &t, float v) {
    if (v - t.ref > REF_SPAN) {
        t.s *= expf(t.ref - v);
        t.ref = v;
    }
    t.s += expf(v - t.ref);
}

// Fused inference of 16 MI queries per block by WAVES waves: two hidden layers, the output layer with a
// running softmax, the confidence.  In the output layer a wave takes 64 columns at a time (4 column
// tiles x MI row tiles of accumulators); its weights come from W3i 16 bytes per lane, two k-steps per
// load, one step ahead across the column groups, so the softmax of a group covers the first loads of
// the next.  Bound: the vector instructions of the softmax (about 17 per logit) and the L2 reads of the
// weights (each block reads all of them), 136-256-256-4,097: 10,000 queries 213 -> 101 us, 33 queries
// 197 -> 47 us against four waves per 16 rows with two bytes of X, eight of W per load and five
// library exponentials per four logits.
template <int MI, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void infer_kernel(InferArgs a) {
    constexpr int IQ = 16 * MI, IT = 64 * WAVES;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r0 = blockIdx.x * IQ;
    const int kp = (a.hidden + 31) & ~31;  // contraction of the output layer, padded with zeros
    const int ldx = a.width + 8, ldh = kp + 8;
    uint16_t *H2 = reinterpret_cast<uint16_t *>(smem);
    float *stp = reinterpret_cast<float *>(H2 + IQ * ldh);  // [IQ]
    uint16_t *X = reinterpret_cast<uint16_t *>(stp + IQ);
    uint16_t *H1 = X + IQ * ldx;
    // once the hidden layers are done, in their place:
    Soft *part = reinterpret_cast<Soft *>(X);  // [WAVES][IQ]
    Soft *run = part + WAVES * IQ;             // [IQ]

    if (a.x16) {
        const int u = a.width / 8;
        for (int e = tid; e < IQ * u; e += IT) {
            const int r = e / u, c = (e % u) * 8;
            *reinterpret_cast<uint4 *>(X + r * ldx + c) =
                r0 + r < a.batch ? *reinterpret_cast<const uint4 *>(a.X + (size_t)(r0 + r) * a.width + c)
                                 : make_uint4(0u, 0u, 0u, 0u);
        }
    } else {
        for (int e = tid; e < IQ * a.width; e += IT) {
            const int r = e / a.width, c = e % a.width;
            X[r * ldx + c] = (r0 + r < a.batch) ? a.X[(size_t)(r0 + r) * a.width + c] : (uint16_t)0;
        }
    }
    if (kp > a.hidden)
        for (int e = tid; e < IQ * 16; e += IT) H2[(e >> 4) * ldh + a.hidden + (e & 15)] = 0;
    __syncthreads();
    hidden_layer<MI, WAVES>(X, ldx, a.width, a.W1, a.b1, a.hidden, H1, ldh);
    __syncthreads();
    hidden_layer<MI, WAVES>(H1, ldh, a.hidden, a.W2, a.b2, a.hidden, H2, ldh);
    __syncthreads();

    const int NO = a.C + 1, S = kp / 32, q = lane >> 4;
    const int groups = (NO + 63) / 64;
    Lane ts[MI][4];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int j = 0; j < 4; ++j) ts[mi][j] = Lane{-INFINITY, -INFINITY, 0.0f, -FLT_MAX, 0x7fffffff, 0x7fffffff};
    const uint16_t *arow = H2 + (lane & 15) * ldh + 4 * q;
    const size_t sstep = (size_t)32 * a.npad;  // elements of W3i per two k-steps
    const uint16_t *wp = a.W3i + ((size_t)q * a.npad + wave * 64 + (lane & 15)) * 8;
    uint4 b[4];
    if (wave < groups) {
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) b[ni] = *reinterpret_cast<const uint4 *>(wp + ni * 128);
    }
    for (int g = wave; g < groups; g += WAVES) {
        v4f acc[MI][4];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = v4f{0.f, 0.f, 0.f, 0.f};
        float bias[4];
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) bias[ni] = a.b3[min(g * 64 + ni * 16 + (lane & 15), NO - 1)];
        const int tiles_n = min(4, (NO - g * 64 + 15) / 16);  // the last group may hold fewer columns
        for (int st = 0; st < S; ++st) {
            // the next two k-steps' weights, or the next group's first (the last group reads its own again)
            const uint16_t *np = st + 1 < S ? wp + (size_t)(st + 1) * sstep : g + WAVES < groups ? wp + (size_t)WAVES * 512 : wp;
            uint4 nb[4];
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) nb[ni] = *reinterpret_cast<const uint4 *>(np + ni * 128);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v4s af[MI];
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
                    af[mi] = *reinterpret_cast<const v4s *>(arow + mi * 16 * ldh + st * 32 + h * 16);
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) {
                    if (ni > 0 && ni >= tiles_n) break;
                    const uint2 w = h == 0 ? make_uint2(b[ni].x, b[ni].y) : make_uint2(b[ni].z, b[ni].w);
#pragma unroll
                    for (int mi = 0; mi < MI; ++mi)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(af[mi], __builtin_bit_cast(v4s, w),
                                                                                acc[mi][ni], 0, 0, 0);
                }
            }
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) b[ni] = nb[ni];
        }
        wp += (size_t)WAVES * 512;
        const bool whole = g * 64 + 64 <= a.C;  // every column of the group is a pivot's
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = mi * 16 + 4 * q + j;
                Lane &t = ts[mi][j];
                float v[4];
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) {
                    v[ni] = acc[mi][ni][j] + bias[ni];
                    const int n = g * 64 + ni * 16 + (lane & 15);
                    if (a.logits && n < NO && r0 + r < a.batch) a.logits[(size_t)(r0 + r) * NO + n] = v[ni];
                }
                if (whole) {
                    // the sum's usual case -- finite values near the reference -- without a branch per value
                    const float hi = fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
                    const float lo = fminf(fminf(v[0], v[1]), fminf(v[2], v[3]));
                    if (hi - t.ref <= REF_SPAN && lo >= -FLT_MAX) {
#pragma unroll
                        for (int ni = 0; ni < 4; ++ni) t.s += exp_mid(v[ni] - t.ref);
                    } else {
#pragma unroll
                        for (int ni = 0; ni < 4; ++ni) lane_sum(t, v[ni]);
                    }
#pragma unroll
                    for (int ni = 0; ni < 4; ++ni) lane_top(t, v[ni], g * 64 + ni * 16 + (lane & 15));
                } else {
#pragma unroll
                    for (int ni = 0; ni < 4; ++ni) {
                        const int n = g * 64 + ni * 16 + (lane & 15);
                        if (n < a.C) {
                            lane_sum(t, v[ni]);
                            lane_top(t, v[ni], n);
                        } else if (n == a.C) {
                            stp[r] = v[ni];
                        }
                    }
                }
            }
    }
    // the 16 lanes of a row, then the waves
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = mi * 16 + 4 * q + j;
            const Lane &l = ts[mi][j];
            Soft t{l.v1, l.v2, l.v1 == -INFINITY ? 0.0f : l.s * expf(l.ref - l.v1), l.a1, l.a2};
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                Soft u;
                u.v1 = __shfl_xor(t.v1, o);
                u.v2 = __shfl_xor(t.v2, o);
                u.s = __shfl_xor(t.s, o);
                u.a1 = __shfl_xor(t.a1, o);
                u.a2 = __shfl_xor(t.a2, o);
                t = soft_merge(t, u);
            }
            if ((lane & 15) == 0) part[wave * IQ + r] = t;
        }
    __syncthreads();
    if (tid < IQ) {
        Soft t = soft_empty();
        for (int w = 0; w < WAVES; ++w) t = soft_merge(t, part[w * IQ + tid]);
        run[tid] = t;
    }
    __syncthreads();
    // confidence: softmax mass of the best pivot's neighbourhood, its logits recomputed from the last
    // hidden layer by the TPR threads of a row, eight hidden units at a time; without neighbourhoods,
    // the mass of the top two
    {
        constexpr int TPR = IT >= 64 * IQ ? 64 : IT >= 32 * IQ ? 32 : IT >= 16 * IQ ? 16 : IT >= 8 * IQ ? 8 : 4;
        const int row = tid / TPR, part_of = tid % TPR;
        if (row < IQ) {
            const Soft t = run[row];
            float mass = 0.0f;
            if (a.nbr && t.a1 >= 0 && t.a1 < a.C) {  // (no valid best pivot: non-finite logits)
                for (int e = 0; e < a.n_nbr; ++e) {
                    const int p = a.nbr[(size_t)t.a1 * a.n_nbr + e];
                    const uint16_t *w = a.W3 + (size_t)p * a.hidden;
                    float z = 0.0f;
                    for (int h = part_of * 8; h < a.hidden; h += TPR * 8) {
                        const uint4 wv = *reinterpret_cast<const uint4 *>(w + h);
                        const uint4 hv = *reinterpret_cast<const uint4 *>(H2 + row * ldh + h);
                        const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w}, hh[4] = {hv.x, hv.y, hv.z, hv.w};
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            z += __uint_as_float(hh[u] << 16) * __uint_as_float(ww[u] << 16);
                            z += __uint_as_float(hh[u] & 0xffff0000u) * __uint_as_float(ww[u] & 0xffff0000u);
                        }
                    }
#pragma unroll
                    for (int o = 1; o < TPR; o <<= 1) z += __shfl_xor(z, o);
                    mass += expf(fminf(z + a.b3[p] - t.v1, 0.0f));
                }
            } else if (!a.nbr) {
                mass = 1.0f + (t.v2 == -INFINITY ? 0.0f : expf(t.v2 - t.v1));
            }
            if (part_of == 0 && r0 + row < a.batch) {
                a.top2[2 * (r0 + row)] = t.a1;
                a.top2[2 * (r0 + row) + 1] = t.a2;
                a.conf[r0 + row] = fminf(mass / t.s, 1.0f);
                a.stop[r0 + row] = stp[row];
            }
        }
    }
}

template <int MI, int WAVES> static size_t infer_lds(const InferArgs &a) {
    constexpr int IQ = 16 * MI;
    const size_t ldh = (size_t)((a.hidden + 31) & ~31) + 8;
    const size_t layers = (size_t)IQ * (a.width + 8 + ldh) * 2, soft = (size_t)(WAVES + 1) * IQ * sizeof(Soft);
    return (size_t)IQ * ldh * 2 + IQ * 4 + std::max(layers, soft);
}
template <int MI, int WAVES> static int infer_launch(const InferArgs &a, hipStream_t st) {
    constexpr int IQ = 16 * MI;
    const size_t lds = infer_lds<MI, WAVES>(a);
    if (lds > 65536)
        MHIP(hipFuncSetAttribute((const void *)infer_kernel<MI, WAVES>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((infer_kernel<MI, WAVES>), dim3((a.batch + IQ - 1) / IQ), dim3(64 * WAVES), lds, st, a);
    MHIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------- host object

struct song_mlp {
    int in_dim = 0, width = 0, hidden = 0, C = 0, max_batch = 0;
    long long off[6] = {0}, cnt[6] = {0}, total = 0;  // W1 b1 W2 b2 W3 b3
    float *P = nullptr, *G = nullptr, *Mo = nullptr, *Vo = nullptr;
    uint16_t *Wb[3] = {nullptr, nullptr, nullptr};
    uint16_t *W3i = nullptr;  // inference copy of the output weights (refresh_kernel)
    int npad = 0;             // its column count: C + 1 rounded up to 64
    int n_cu = 1;             // compute units of the device
    size_t max_lds = 65536;
    int ldz = 0;              // row stride of Z and dZ: C + 1 rounded up to 8 (16-byte rows)
    uint16_t *H1 = nullptr, *H2 = nullptr, *dZ = nullptr, *dH2 = nullptr, *dH1 = nullptr;
    float *Z = nullptr, *loss = nullptr;
    float2 *row_loss = nullptr;  // each row's share of the two losses
    uint16_t *Xa = nullptr;  // aligned copy of inputs that are not
    int t = 0;
};

static uint64_t splitmix(uint64_t &s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

template <bool ADAM> static int refresh(song_mlp *m, AdamArgs a, hipStream_t st) {
    ParamCopies c{};
    for (int i = 0; i < 6; ++i) {
        c.off[i] = m->off[i];
        c.cnt[i] = m->cnt[i];
    }
    for (int l = 0; l < 3; ++l) c.Wb[l] = m->Wb[l];
    c.W3i = m->W3i;
    c.rows3 = m->C + 1;
    c.hidden = m->hidden;
    c.npad = m->npad;
    const int w3 = (m->npad / 16) * ((m->hidden + 63) / 64);
    const long long rest = m->total - m->cnt[4];
    hipLaunchKernelGGL(refresh_kernel<ADAM>, dim3((unsigned)(w3 + (rest + 255) / 256)), dim3(256), 0, st, a, c, w3);
    MHIP(hipGetLastError());
    return 0;
}
static int refresh_bf16(song_mlp *m, hipStream_t st) {
    AdamArgs a{};
    a.p = m->P;
    return refresh<false>(m, a, st);
}

extern "C" int song_mlp_create(int in_dim, int hidden, int n_classes, int max_batch, uint64_t seed, song_mlp **out) {
    if (!out || in_dim < 1 || hidden < 16 || hidden % 16 != 0 || n_classes < 2 || max_batch < 1)
        return mfail(-1, "bad MLP shape in=%d hidden=%d classes=%d batch=%d", in_dim, hidden, n_classes, max_batch);
    song_mlp *m = new song_mlp();
    m->in_dim = in_dim;
    m->width = (in_dim + 15) & ~15;
    m->hidden = hidden;
    m->C = n_classes;
    m->max_batch = max_batch;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) {
        m->n_cu = std::max(1, prop.multiProcessorCount);
        m->max_lds = std::max<size_t>(65536, prop.sharedMemPerBlock);
    }
    const long long sizes[6] = {(long long)hidden * m->width, hidden, (long long)hidden * hidden, hidden,
                                (long long)(n_classes + 1) * hidden, n_classes + 1};
    long long o = 0;
    for (int i = 0; i < 6; ++i) {
        m->off[i] = o;
        m->cnt[i] = sizes[i];
        o += sizes[i];
    }
    m->total = o;
    std::vector<float> init(o, 0.0f);
    uint64_t s = seed;
    const int fan[3] = {in_dim, hidden, hidden};
    for (int l = 0; l < 3; ++l) {
        const float lim = std::sqrt(6.0f / (float)fan[l]);
        const int rows = (int)(sizes[2 * l] / (l == 0 ? m->width : hidden));
        const int cols = l == 0 ? m->width : hidden;
        for (int r = 0; r < rows; ++r)
            for (int c = 0; c < cols; ++c) {
                const double u = (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
                init[m->off[2 * l] + (long long)r * cols + c] = (l == 0 && c >= in_dim) ? 0.0f : (float)((2.0 * u - 1.0) * lim);
            }
    }
    auto bad = [&](const char *what) {
        song_mlp_destroy(m);
        return mfail(-2, "hipMalloc %s", what);
    };
    if (hipMalloc(&m->P, o * 4) || hipMalloc(&m->G, o * 4) || hipMalloc(&m->Mo, o * 4) || hipMalloc(&m->Vo, o * 4))
        return bad("params");
    for (int l = 0; l < 3; ++l)
        if (hipMalloc(&m->Wb[l], m->cnt[2 * l] * 2)) return bad("bf16 weights");
    m->npad = (n_classes + 1 + 63) & ~63;
    const size_t w3i = (size_t)m->npad * ((hidden + 31) & ~31) * 2;
    if (hipMalloc(&m->W3i, w3i) || hipMemset(m->W3i, 0, w3i)) return bad("interleaved output weights");
    m->ldz = (n_classes + 1 + 7) & ~7;
    const long long B = max_batch, LZ = m->ldz;
    if (hipMalloc(&m->H1, B * hidden * 2) || hipMalloc(&m->H2, B * hidden * 2) || hipMalloc(&m->dZ, B * LZ * 2) ||
        hipMalloc(&m->dH2, B * hidden * 2) || hipMalloc(&m->dH1, B * hidden * 2) || hipMalloc(&m->Z, B * LZ * 4) ||
        hipMalloc(&m->loss, 8) || hipMalloc(&m->Xa, B * m->width * 2) ||
        hipMalloc(&m->row_loss, B * sizeof(float2)))
        return bad("activations");
    if (hipMemcpy(m->P, init.data(), o * 4, hipMemcpyHostToDevice) || hipMemset(m->Mo, 0, o * 4) ||
        hipMemset(m->Vo, 0, o * 4) || hipMemset(m->G, 0, o * 4)) {
        song_mlp_destroy(m);
        return mfail(-2, "init upload");
    }
    if (refresh_bf16(m, 0) || hipDeviceSynchronize()) {
        song_mlp_destroy(m);
        return mfail(-2, "init bf16");
    }
    *out = m;
    return 0;
}

extern "C" int song_mlp_destroy(song_mlp *m) {
    if (!m) return 0;
    void *ptrs[] = {m->P, m->G, m->Mo, m->Vo, m->Wb[0], m->Wb[1], m->Wb[2], m->W3i, m->H1, m->H2, m->dZ, m->dH2,
                    m->dH1, m->Z, m->loss, m->row_loss, m->Xa};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    delete m;
    return 0;
}

extern "C" int song_mlp_input_width(const song_mlp *m) { return m ? m->width : 0; }

extern "C" int song_mlp_param_count(const song_mlp *m, uint64_t *count) {
    if (!m || !count) return mfail(-1, "null");
    *count = (uint64_t)m->total;
    return 0;
}

extern "C" int song_mlp_get_params(const song_mlp *m, float *host) {
    if (!m || !host) return mfail(-1, "null");
    MHIP(hipMemcpy(host, m->P, m->total * 4, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int song_mlp_set_params(song_mlp *m, const float *host) {
    if (!m || !host) return mfail(-1, "null");
    MHIP(hipMemcpy(m->P, host, m->total * 4, hipMemcpyHostToDevice));
    if (refresh_bf16(m, 0)) return -2;
    MHIP(hipDeviceSynchronize());
    return 0;
}

extern "C" int song_mlp_loss_grad(song_mlp *m, const uint16_t *d_x, const int *d_labels, const float *d_stop, int batch,
                                  float stop_weight, float *loss_out, float *grads_host, void *stream) {
    if (!m || !d_x || !d_labels || !d_stop) return mfail(-1, "null argument");
    if (batch < 1 || batch > m->max_batch) return mfail(-1, "batch %d outside [1, %d]", batch, m->max_batch);
    hipStream_t st = (hipStream_t)stream;
    const int W = m->width, Hd = m->hidden, NO = m->C + 1, LZ = m->ldz;
    float *b1 = m->P + m->off[1], *b2 = m->P + m->off[3], *b3 = m->P + m->off[5], *G = m->G;
    // the tile kernels read the inputs in 16-byte units; the network's own buffers are aligned
    const uint16_t *x = d_x;
    if (((uintptr_t)d_x & 15) != 0) {
        MHIP(hipMemcpyAsync(m->Xa, d_x, (size_t)batch * W * 2, hipMemcpyDeviceToDevice, st));
        x = m->Xa;
    }
    const auto args = [](int M, int N, int K, const uint16_t *A, int lda, const uint16_t *B, int ldb) {
        TileArgs g{};
        g.M = M;
        g.N = N;
        g.K = K;
        g.A = A;
        g.lda = lda;
        g.B = B;
        g.ldb = ldb;
        return g;
    };
    // forward: H1 = relu(X W1^T + b1), H2 = relu(H1 W2^T + b2), Z = H2 W3^T + b3
    TileArgs g = args(batch, Hd, W, x, W, m->Wb[0], W);
    g.Cb = m->H1;
    g.ldcb = Hd;
    g.bias = b1;
    g.relu = 1;
    if (tile_launch<32, 32, 64, ALONG_K, ALONG_K, 2>(g, st)) return -2;
    g = args(batch, Hd, Hd, m->H1, Hd, m->Wb[1], Hd);
    g.Cb = m->H2;
    g.ldcb = Hd;
    g.bias = b2;
    g.relu = 1;
    if (tile_launch<32, 32, 64, ALONG_K, ALONG_K, 2>(g, st)) return -2;
    g = args(batch, NO, Hd, m->H2, Hd, m->Wb[2], Hd);
    g.C = m->Z;
    g.ldc = LZ;
    g.bias = b3;
    if (tile_launch<64, 64, 32, ALONG_K, ALONG_K, 2>(g, st)) return -2;
    const bool in_lds = m->C <= LOSS_LDS_CLASSES;
    hipLaunchKernelGGL(in_lds ? loss_kernel<true> : loss_kernel<false>, dim3(batch), dim3(256),
                       in_lds ? (size_t)m->C * sizeof(float) : 0, st, m->Z, LZ, m->C, d_labels, d_stop, batch,
                       stop_weight, m->dZ, LZ, m->row_loss);
    MHIP(hipGetLastError());
    // backward: dH2 = dZ W3 * (H2 > 0) beside dW3 = dZ^T H2 and db3, then dH1 beside dW2 and db2, then dW1
    TileArgs gi = args(batch, Hd, NO, m->dZ, LZ, m->Wb[2], Hd);
    gi.Cb = m->dH2;
    gi.ldcb = Hd;
    gi.mask = m->H2;
    gi.ldm = Hd;
    TileArgs gw = args(NO, Hd, batch, m->dZ, LZ, m->H2, Hd);
    gw.C = G + m->off[4];
    gw.ldc = Hd;
    gw.rowsum = G + m->off[5];
    {
        const int nb1 = tiles(batch, 32) * tiles(Hd, 32), nb2 = tiles(NO, 64) * tiles_n(gw, 64);
        hipLaunchKernelGGL((tile_pair_kernel<32, 32, 128, 2, 64, 64, 32, 2>), dim3(nb1 + nb2), dim3(256), 0, st, gi, nb1,
                           tiles(Hd, 32), gw, tiles_n(gw, 64));
        MHIP(hipGetLastError());
    }
    gi = args(batch, Hd, Hd, m->dH2, Hd, m->Wb[1], Hd);
    gi.Cb = m->dH1;
    gi.ldcb = Hd;
    gi.mask = m->H1;
    gi.ldm = Hd;
    gw = args(Hd, Hd, batch, m->dH2, Hd, m->H1, Hd);
    gw.C = G + m->off[2];
    gw.ldc = Hd;
    gw.rowsum = G + m->off[3];
    {
        const int nb1 = tiles(batch, 32) * tiles(Hd, 32), nb2 = tiles(Hd, 32) * tiles_n(gw, 32);
        hipLaunchKernelGGL((tile_pair_kernel<32, 32, 128, 2, 32, 32, 128, 2>), dim3(nb1 + nb2), dim3(256), 0, st, gi, nb1,
                           tiles(Hd, 32), gw, tiles_n(gw, 32));
        MHIP(hipGetLastError());
    }
    g = args(Hd, W, batch, m->dH1, Hd, x, W);
    g.C = G + m->off[0];
    g.ldc = W;
    g.rowsum = G + m->off[1];
    if (tile_launch<32, 32, 128, ALONG_ROW, ALONG_ROW, 2>(g, st)) return -2;
    if (loss_out) {
        hipLaunchKernelGGL(loss_sum_kernel, dim3(1), dim3(256), 0, st, m->row_loss, batch, m->loss);
        MHIP(hipGetLastError());
        MHIP(hipMemcpyAsync(loss_out, m->loss, 8, hipMemcpyDeviceToHost, st));
        MHIP(hipStreamSynchronize(st));
    }
    if (grads_host) {
        MHIP(hipMemcpyAsync(grads_host, G, m->total * 4, hipMemcpyDeviceToHost, st));
        MHIP(hipStreamSynchronize(st));
    }
    return 0;
}

extern "C" int song_mlp_adam_step(song_mlp *m, float lr, void *stream) {
    if (!m) return mfail(-1, "null");
    hipStream_t st = (hipStream_t)stream;
    m->t += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)m->t), c2 = 1.0f - std::pow(b2, (float)m->t);
    return refresh<true>(m, AdamArgs{m->P, m->G, m->Mo, m->Vo, lr, b1, b2, c1, c2, 1e-8f}, st);
}

extern "C" int song_mlp_infer(song_mlp *m, const uint16_t *d_x, int batch, int *d_top2, float *d_conf, float *d_stop,
                              float *d_logits, void *stream) {
    return song_mlp_infer_nbr(m, d_x, batch, nullptr, 0, d_top2, d_conf, d_stop, d_logits, stream);
}

extern "C" int song_mlp_infer_nbr(song_mlp *m, const uint16_t *d_x, int batch, const int *d_nbr, int n_nbr, int *d_top2,
                                  float *d_conf, float *d_stop, float *d_logits, void *stream) {
    if (d_nbr && (n_nbr < 1 || n_nbr > 64)) return mfail(-1, "n_nbr=%d not in [1,64]", n_nbr);
    if (!m || !d_x || !d_top2 || !d_conf || !d_stop) return mfail(-1, "null argument");
    if (batch < 1) return 0;
    InferArgs a{};
    a.X = d_x;
    a.batch = batch;
    a.width = m->width;
    a.hidden = m->hidden;
    a.C = m->C;
    a.W1 = m->Wb[0];
    a.W2 = m->Wb[1];
    a.W3 = m->Wb[2];
    a.W3i = m->W3i;
    a.npad = m->npad;
    a.b1 = m->P + m->off[1];
    a.b2 = m->P + m->off[3];
    a.b3 = m->P + m->off[5];
    a.top2 = d_top2;
    a.conf = d_conf;
    a.stop = d_stop;
    a.logits = d_logits;
    a.nbr = d_nbr;
    a.n_nbr = n_nbr;
    a.x16 = ((uintptr_t)d_x & 15) == 0;
    // Block shape by how many 16-row tiles the batch has per compute unit.  Up to one each, a tile on 16
    // waves is the shortest (33 rows: 47 us; on 8 waves 49, on 4 waves 113).  Beyond, two blocks of 8
    // waves share a unit and take a tile each in about 67 us, or one block of 8 waves takes three tiles,
    // each weight fragment serving three products, in 100 us: the cheaper of the two by whole rounds
    // over the device (8,200-12,288 rows: 101 against 118 us; 6,000: 80 against 99; 60,000: 493 with
    // one tile a block).
    const long long t = (batch + 15) / 16, n = m->n_cu;
    if (t <= n) return infer_launch<1, 16>(a, (hipStream_t)stream);
    const long long rest = t % (2 * n);
    const long long one = 67 * (t / (2 * n)) + (rest == 0 ? 0 : rest <= n ? 52 : 70), three = 100 * ((t + 3 * n - 1) / (3 * n));
    if (three < one && infer_lds<3, 8>(a) <= m->max_lds) return infer_launch<3, 8>(a, (hipStream_t)stream);
    return infer_launch<1, 8>(a, (hipStream_t)stream);
}

__global__ __launch_bounds__(256) void plan_kernel(const int *top2, const float *conf, const float *stop, int batch,
                                                   const int *nbr, int n_nbr, const int *pivot_vertex, int npiv, float thr,
                                                   float scale, float add, int fcap, int pq_l, int pq_f, int *pq,
                                                   int *entry, int *caps, unsigned char *ok) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= batch) return;
    const int best = top2[2 * i];
    // no valid best pivot (non-finite logits): the fallback
    const bool good = conf[i] >= thr && best >= 0 && best < npiv;
    int *row = entry + (long long)i * n_nbr;
    for (int e = 0; e < n_nbr; ++e) row[e] = good ? pivot_vertex[nbr[(long long)best * n_nbr + e]] : -1;
    const float c = fminf(fmaxf(scale * (exp2f(stop[i]) - 1.0f) + add, 1.0f), 1.0e6f);
    caps[i] = good ? (int)c : (fcap > 0 ? fcap : 1000000);
    pq[i] = good ? pq_l : pq_f;
    ok[i] = good ? 1 : 0;
}

extern "C" int song_mlp_plan(const int *d_top2, const float *d_conf, const float *d_stop, int batch, const int *d_nbr,
                             int n_nbr, const int *d_pivot_vertex, int n_pivots, float conf_threshold,
                             float step_scale, float step_add, int fallback_cap, int pq_learned, int pq_fallback, int *d_pq,
                             int *d_entry, int *d_caps, unsigned char *d_ok, void *stream) {
    if (!d_top2 || !d_conf || !d_stop || !d_nbr || !d_pivot_vertex || !d_pq || !d_entry || !d_caps || !d_ok)
        return mfail(-1, "null argument");
    if (n_nbr < 1 || pq_learned < 1 || pq_fallback < 1 || fallback_cap < 0)
        return mfail(-1, "bad plan arguments n_nbr=%d pq=%d/%d cap=%d", n_nbr, pq_learned, pq_fallback, fallback_cap);
    if (batch < 1) return 0;
    hipLaunchKernelGGL(plan_kernel, dim3((unsigned)((batch + 255) / 256)), dim3(256), 0, (hipStream_t)stream, d_top2,
                       d_conf, d_stop, batch, d_nbr, n_nbr, d_pivot_vertex, n_pivots, conf_threshold, step_scale,
                       step_add,
                       fallback_cap, pq_learned, pq_fallback, d_pq, d_entry, d_caps, d_ok);
    MHIP(hipGetLastError());
    return 0;
}

extern "C" int song_mlp_features(const float *d_queries, int nq, int dim, const float *d_mean, const float *d_inv_std,
                                 const float *d_v0, const float *fs, uint16_t *d_x, int width, void *stream) {
    if (!d_queries || !d_mean || !d_inv_std || !d_v0 || !fs || !d_x) return mfail(-1, "null argument");
    if (width < dim + 8) return mfail(-1, "width %d < dim + 8", width);
    if (nq < 1) return 0;
    hipLaunchKernelGGL(features_kernel, dim3(nq), dim3(64), 0, (hipStream_t)stream, d_queries, dim, d_mean, d_inv_std,
                       d_v0, fs[0], fs[1], fs[2], fs[3], fs[4], fs[5], fs[6], fs[7], d_x, width);
    MHIP(hipGetLastError());
    return 0;
}
