// C ABI of the graph search (include/song_amd.h): index upload, launch planning,
// overflow re-runs.  Everything that touches the search runs on the GPU; there is no
// CPU search path in this library.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "index_internal.hpp"

using namespace song;

namespace song {

static thread_local std::string g_err;

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

}  // namespace song

// visited spill tables: 2^13 u32 (32 KB) per launch slot, launches of at most kChunk queries
static constexpr int kGhlog = 13;
static constexpr unsigned kChunk = 32768;

static int ensure_gvis(song_index *ix, void *stream, size_t slots, uint32_t **out) {
    std::lock_guard<std::mutex> g(ix->spill_mu);
    song_index::Spill &sp = ix->spill[stream];
    if (sp.slots < slots) {
        if (sp.d) {
            // the previous buffer may still be read by work queued on this stream
            HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
            HIP_TRY(hipFree(sp.d));
        }
        sp.d = nullptr;
        sp.slots = 0;
        HIP_TRY(hipMalloc(&sp.d, slots * ((size_t)4 << kGhlog)));
        sp.slots = slots;
    }
    *out = sp.d;
    return SONG_OK;
}

// queue bags: `stride` bytes (qcap keys) per launch slot, grown on demand like the tables
static int ensure_gbag(song_index *ix, void *stream, size_t slots, size_t stride, unsigned char **out) {
    std::lock_guard<std::mutex> g(ix->spill_mu);
    song_index::Spill &sp = ix->spill[stream];
    const size_t need = slots * stride;
    if (sp.bag_bytes < need) {
        if (sp.bag) {
            HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
            HIP_TRY(hipFree(sp.bag));
        }
        sp.bag = nullptr;
        sp.bag_bytes = 0;
        HIP_TRY(hipMalloc(&sp.bag, need));
        sp.bag_bytes = need;
    }
    *out = sp.bag;
    return SONG_OK;
}

extern "C" const char *song_last_error(void) { return song::g_err.c_str(); }

extern "C" void song_search_opts_default(song_search_opts *o) {
    o->mode = SONG_MODE_AUTO;
    o->slack = 128;
    o->hash_log2 = 0;
    o->max_steps = 0;
    o->retry = 1;
    o->storage = SONG_STORE_F32;
    o->rerank = 1;
    o->visited_bits = 0;
    o->bloom_k = 0;
    o->best_in_global = -1;
}

// Low-precision copy of one row per thread: BF16 with a power-of-two scale (round to
// nearest even), or FP8-E4M3 with scale max|x|/448 (hardware conversion of the clamped
// value).  The scale of an all-zero row is 1.
__global__ void quantize_kernel(const float *data, uint64_t n, int dim, int ld, int store, uint8_t *out,
                                size_t stride, float *scale) {
    uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const float *r = data + v * (uint64_t)ld;
    float amax = 0.0f;
    for (int i = 0; i < dim; ++i) amax = fmaxf(amax, fabsf(r[i]));
    float s = 1.0f;
    if (amax > 0.0f) {
        if (store == SONG_STORE_BF16) {
            int e;
            frexpf(amax, &e);
            s = ldexpf(1.0f, e);
        } else {
            s = amax / 448.0f;
        }
    }
    scale[v] = s;
    uint32_t *o = reinterpret_cast<uint32_t *>(out + v * stride);
    const int words = (int)(stride / 4);
    for (int w = 0; w < words; ++w) {
        uint32_t word = 0u;
        if (store == SONG_STORE_BF16) {
            for (int t = 0; t < 2; ++t) {
                const int i = 2 * w + t;
                const float x = i < dim ? r[i] / s : 0.0f;
                const uint32_t u = __float_as_uint(x);
                const uint32_t code = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
                word |= (code & 0xffffu) << (16 * t);
            }
        } else {
            float y[4];
            for (int t = 0; t < 4; ++t) {
                const int i = 4 * w + t;
                y[t] = i < dim ? fminf(fmaxf(r[i] / s, -448.0f), 448.0f) : 0.0f;
            }
            int lo = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
            word = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], lo, true);
        }
        o[w] = word;
    }
}

// squared norm per base row with one sequential fmaf chain (data.h:54 as the reference
// build contracts it), the `lena` of the cosine distance
__global__ void norms_kernel(const float *data, uint64_t n, int dim, int ld, float *out) {
    uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const float *r = data + v * (uint64_t)ld;
    float s = 0.0f;
    for (int i = 0; i < dim; ++i) s = fmaf(r[i], r[i], s);
    out[v] = s;
}

// integer-valued test and range of a float array, one result per block: out[3b] = 1 if any is not an
// integer, out[3b + 1] / out[3b + 2] = min / max as orderable bits.  The host folds the blocks'
// results, so nothing is cleared beforehand and no atomics meet.
constexpr int kRangeBlocks = 512;
__global__ __launch_bounds__(256) void range_kernel(const float *x, uint64_t count, unsigned *out) {
    __shared__ unsigned part[4][3];
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned nonint = 0, mn = 0xffffffffu, mx = 0u;
    for (; i < count; i += stride) {
        const float v = x[i];
        if (v != rintf(v)) nonint = 1;
        const unsigned o = ord32(v);
        mn = min(mn, o);
        mx = max(mx, o);
    }
    for (int o = 32; o > 0; o >>= 1) {
        nonint |= (unsigned)__shfl_xor((int)nonint, o);
        mn = min(mn, (unsigned)__shfl_xor((int)mn, o));
        mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        part[w][0] = nonint;
        part[w][1] = mn;
        part[w][2] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[3 * blockIdx.x] = part[0][0] | part[1][0] | part[2][0] | part[3][0];
        out[3 * blockIdx.x + 1] = min(min(part[0][1], part[1][1]), min(part[2][1], part[3][1]));
        out[3 * blockIdx.x + 2] = max(max(part[0][2], part[1][2]), max(part[2][2], part[3][2]));
    }
}

static float unord_host(unsigned o) {
    unsigned u = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

static unsigned ord_host(float f) {
    unsigned u;
    memcpy(&u, &f, 4);
    if (f == 0.0f) u = 0u;
    if (f != f) u = 0x7f800000u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// A call's workspace, kept by the index between calls: device memory, and pinned host memory for the
// copies of calls of up to kPinned bytes (larger copies go from and to the caller's memory or a plain
// vector: pinning takes longer than it saves).  A call takes one from the pool (or makes one) and
// gives it back when its stream is done with it, so calls from several threads and streams have
// different ones; the pool holds at most kPool of them, none above kPoolBytes, and the index frees
// them.  Against four allocations and frees, a cleared range buffer and seven copies per call, one
// query on 1M x 128 went from 341 to 267 us and 3,001 device queries, whose range test allocated too,
// from 1.50 to 1.35 ms.
static constexpr size_t kPool = 4, kPoolBytes = (size_t)8 << 20, kPinned = (size_t)1 << 20;

namespace {
struct Workspace {
    const song_index *ix;
    song_index::Work w;
    explicit Workspace(const song_index *index) : ix(index) {}
    int take(size_t bytes) {
        {
            std::lock_guard<std::mutex> g(ix->work_mu);
            for (size_t i = 0; i < ix->work.size(); ++i)
                if (ix->work[i].bytes >= bytes) {
                    w = ix->work[i];
                    ix->work.erase(ix->work.begin() + (long)i);
                    return SONG_OK;
                }
        }
        // sizes in powers of two, so that a slightly larger call finds one
        size_t b = 65536;
        while (b < bytes) b <<= 1;
        if (b > kPoolBytes) b = bytes;
        if (hipMalloc(&w.dev, b) != hipSuccess || (b <= kPinned && hipHostMalloc(&w.host, b) != hipSuccess))
            return fail(SONG_E_HIP, "search workspace of %zu bytes", b);
        w.bytes = b;
        return SONG_OK;
    }
    ~Workspace() {
        if (w.bytes > 0 && w.bytes <= kPoolBytes) {
            std::lock_guard<std::mutex> g(ix->work_mu);
            if (ix->work.size() < kPool) {
                ix->work.push_back(w);
                return;
            }
        }
        if (w.dev) (void)hipFree(w.dev);
        if (w.host) (void)hipHostFree(w.host);
    }
};
}  // namespace

int song::device_range(const song_index *ix, const float *d, uint64_t count, int *integer, float *vmin, float *vmax,
                       hipStream_t st) {
    Workspace ws(ix);
    const size_t bytes = kRangeBlocks * 3 * sizeof(unsigned);
    int rc = ws.take(bytes);
    if (rc != SONG_OK) return rc;
    std::vector<unsigned> plain(ws.w.host ? 0 : kRangeBlocks * 3);  // (a larger call's workspace has no pinned part)
    const int blocks = (int)std::min<uint64_t>(kRangeBlocks, (count + 1023) / 1024 + 1);
    unsigned *out = reinterpret_cast<unsigned *>(ws.w.dev), *res = ws.w.host ? reinterpret_cast<unsigned *>(ws.w.host) : plain.data();
    hipLaunchKernelGGL(range_kernel, dim3(blocks), dim3(256), 0, st, d, count, out);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(res, out, blocks * 3 * sizeof(unsigned), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    unsigned nonint = 0, mn = 0xffffffffu, mx = 0u;
    for (int b = 0; b < blocks; ++b) {
        nonint |= res[3 * b];
        mn = std::min(mn, res[3 * b + 1]);
        mx = std::max(mx, res[3 * b + 2]);
    }
    *integer = nonint == 0u;
    *vmin = unord_host(mn);
    *vmax = unord_host(mx);
    return SONG_OK;
}

extern "C" int song_index_create(const float *data, uint64_t n, int dim, const uint64_t *graph, int shift,
                                 int metric, song_index **out) {
    if (!out) return fail(SONG_E_ARG, "out is null");
    *out = nullptr;
    if (!data || !graph) return fail(SONG_E_ARG, "data/graph is null");
    if (n == 0 || n >= 0xFFFFFFFFull) return fail(SONG_E_ARG, "n=%llu out of range", (unsigned long long)n);
    if (dim < 1 || dim > 16384) return fail(SONG_E_ARG, "dim=%d out of range", dim);
    if (shift < 1 || shift > 6) return fail(SONG_E_ARG, "shift=%d not in [1,6]", shift);
    if (metric < SONG_L2 || metric > SONG_COS) return fail(SONG_E_ARG, "metric=%d", metric);
    const int slots = 1 << shift;
    const int gstride = slots <= 32 ? 32 : 64;
    std::vector<uint32_t> g32((size_t)n * gstride, 0u);
    for (uint64_t v = 0; v < n; ++v) {
        const uint64_t *r = graph + v * (uint64_t)slots;
        uint64_t deg = r[0];
        if (deg >= (uint64_t)slots)
            return fail(SONG_E_ARG, "vertex %llu: degree %llu >= %d", (unsigned long long)v,
                        (unsigned long long)deg, slots);
        uint32_t *o = &g32[(size_t)v * gstride];
        o[0] = (uint32_t)deg;
        for (uint64_t j = 1; j <= deg; ++j) {
            if (r[j] >= n)
                return fail(SONG_E_ARG, "vertex %llu: neighbour id %llu >= n", (unsigned long long)v,
                            (unsigned long long)r[j]);
            o[j] = (uint32_t)r[j];
        }
    }

    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(SONG_E_NODEV, "no GPU visible");

    song_index *ix = new song_index();
    ix->n = n;
    ix->dim = dim;
    ix->ld = (dim + 3) & ~3;
    ix->metric = metric;
    ix->shift = shift;
    ix->gstride = gstride;
    ix->idbits = n <= 1 ? 1 : 64 - __builtin_clzll((unsigned long long)(n - 1));
    auto cleanup = [&](int code) {
        song_index_destroy(ix);
        return code;
    };
    if (hipGetDevice(&ix->device) != hipSuccess) return cleanup(fail(SONG_E_HIP, "hipGetDevice failed"));
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, ix->device) == hipSuccess) {
        ix->max_lds = std::max<size_t>(65536, prop.sharedMemPerBlock);
        ix->n_cu = std::max(1, prop.multiProcessorCount);
    }

    size_t dbytes = (size_t)n * ix->ld * sizeof(float);
    if (hipMalloc(&ix->d_data, dbytes) != hipSuccess) return cleanup(fail(SONG_E_HIP, "hipMalloc data %zu", dbytes));
    // rows of a multiple of four floats go up as they lie; others are padded with zeros, cleared
    // before the copy starts
    if (ix->ld == dim) {
        if (hipMemcpy(ix->d_data, data, dbytes, hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(fail(SONG_E_HIP, "upload data"));
    } else {
        if (hipMemset(ix->d_data, 0, dbytes) != hipSuccess || hipDeviceSynchronize() != hipSuccess)
            return cleanup(fail(SONG_E_HIP, "hipMemset data"));
        if (hipMemcpy2D(ix->d_data, ix->ld * sizeof(float), data, dim * sizeof(float), dim * sizeof(float), n,
                        hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(fail(SONG_E_HIP, "upload data"));
    }
    size_t gbytes = g32.size() * sizeof(uint32_t);
    if (hipMalloc(&ix->d_graph, gbytes) != hipSuccess) return cleanup(fail(SONG_E_HIP, "hipMalloc graph"));
    if (hipMemcpy(ix->d_graph, g32.data(), gbytes, hipMemcpyHostToDevice) != hipSuccess)
        return cleanup(fail(SONG_E_HIP, "upload graph"));
    if (metric == SONG_COS) {
        if (hipMalloc(&ix->d_norms, n * sizeof(float)) != hipSuccess) return cleanup(fail(SONG_E_HIP, "hipMalloc norms"));
        hipLaunchKernelGGL(norms_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, ix->d_data, n, dim,
                           ix->ld, ix->d_norms);
        if (hipGetLastError() != hipSuccess) return cleanup(fail(SONG_E_HIP, "norms kernel"));
    }
    int rc = device_range(ix, ix->d_data, (uint64_t)n * ix->ld, &ix->integer_valued, &ix->vmin, &ix->vmax, 0);
    if (rc != SONG_OK) return cleanup(rc);
    if (hipDeviceSynchronize() != hipSuccess) return cleanup(fail(SONG_E_HIP, "index upload sync"));
    *out = ix;
    return SONG_OK;
}

extern "C" int song_index_add_storage(song_index *ix, int store) {
    if (!ix) return fail(SONG_E_ARG, "index is null");
    if (store != SONG_STORE_BF16 && store != SONG_STORE_FP8) return fail(SONG_E_ARG, "storage=%d", store);
    if (ix->d_lp[store]) return SONG_OK;
    const int epu = store == SONG_STORE_BF16 ? 8 : 16;
    const size_t esz = store == SONG_STORE_BF16 ? 2 : 1;
    const size_t stride = (size_t)((ix->dim + epu - 1) / epu) * epu * esz;
    HIP_TRY(hipMalloc(&ix->d_lp[store], stride * ix->n));
    HIP_TRY(hipMalloc(&ix->d_scale[store], sizeof(float) * ix->n));
    hipLaunchKernelGGL(quantize_kernel, dim3((unsigned)((ix->n + 255) / 256)), dim3(256), 0, 0, ix->d_data, ix->n,
                       ix->dim, ix->ld, store, ix->d_lp[store], stride, ix->d_scale[store]);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    ix->lp_stride[store] = stride;
    return SONG_OK;
}

extern "C" int song_index_get_storage(const song_index *ix, int store, void *codes, float *scales,
                                      uint64_t *row_bytes) {
    if (!ix || store < SONG_STORE_BF16 || store > SONG_STORE_FP8 || !ix->d_lp[store])
        return fail(SONG_E_ARG, "storage %d not built", store);
    if (row_bytes) *row_bytes = ix->lp_stride[store];
    if (codes) HIP_TRY(hipMemcpy(codes, ix->d_lp[store], ix->lp_stride[store] * ix->n, hipMemcpyDeviceToHost));
    if (scales) HIP_TRY(hipMemcpy(scales, ix->d_scale[store], sizeof(float) * ix->n, hipMemcpyDeviceToHost));
    return SONG_OK;
}

extern "C" int song_index_destroy(song_index *ix) {
    if (!ix) return SONG_OK;
    for (int i = 0; i < 3; ++i) {
        if (ix->d_lp[i]) (void)hipFree(ix->d_lp[i]);
        if (ix->d_scale[i]) (void)hipFree(ix->d_scale[i]);
    }
    if (ix->d_data) (void)hipFree(ix->d_data);
    if (ix->d_graph) (void)hipFree(ix->d_graph);
    if (ix->d_norms) (void)hipFree(ix->d_norms);
    for (auto &kv : ix->spill) {
        if (kv.second.d) (void)hipFree(kv.second.d);
        if (kv.second.bag) (void)hipFree(kv.second.bag);
    }
    for (auto &w : ix->work) {
        (void)hipFree(w.dev);
        if (w.host) (void)hipHostFree(w.host);
    }
    delete ix;
    return SONG_OK;
}

extern "C" int song_index_integer_valued(const song_index *ix) { return ix ? ix->integer_valued : 0; }

// ---------------------------------------------------------------- launch planning

// must match the per-wave layout of search_query: visited (2^hlog slots of 4 or, compact, 2
// bytes) | best (pq rounded to even; not with bglob) | 256
// candidate ids / radix bins | query (the head is in registers, the bag in global memory) | with
// seq_stage (make_plan adds it) the exact sums' stage
size_t song::lds_bytes(bool exact, int pq, int qcap, int hlog, int qld, int vis16, int bloom_k, int bag_lds,
                       int bglob) {
    size_t key = exact ? 16 : 8;
    const size_t vis = bloom_k > 0 ? ((size_t)4 << hlog) : ((size_t)(vis16 ? 2 : 4) << hlog);
    return vis + (bglob ? 0 : (size_t)((pq + 1) & ~1) * key) + 256 * 4 + (size_t)qld * 4 +
           (bag_lds ? (size_t)qcap * key : 0);
}

// auto_tune_bloom.cc:65-86 restated: n = 12.897 pq expected insertions; the smallest filter of
// m = 64 * 2^i bits (i = 1..15) whose false-positive rate p = (1 - e^(-k/r))^k, r = m / n,
// k = round(ln 2 * r) (auto_tune_bloom.cc:6-37) is below 0.03, else i = 15.  Returned as
// 2^(i + 1) 32-bit words and k (at most 9, the kernel's limit).
void song::bloom_size(int pq, int *hlog32, int *k) {
    const double n = (double)pq * 12.897;
    int bi = 15;
    double bk = 0;
    for (int i = 1; i <= 15; ++i) {
        const double m = 64.0 * (double)(1 << i);
        const double r = m / n;
        const double kk = std::round(std::log(2.0) * r);
        const double p = std::pow(1.0 - std::exp(-kk / r), kk);
        bi = i;
        bk = kk;
        if (p < 0.03) break;
    }
    *hlog32 = bi + 1;
    *k = (int)std::max(1.0, std::min(9.0, bk));
}

extern "C" int song_bloom_size(int pq, int *hash_log2, int *bloom_k) {
    if (pq < 1 || !hash_log2 || !bloom_k) return fail(SONG_E_ARG, "pq=%d", pq);
    bloom_size(pq, hash_log2, bloom_k);
    return SONG_OK;
}

size_t song::bag_stride(const Plan &p) {
    const size_t key = p.exact ? 16 : 8;
    const size_t bag = ((size_t)p.qcap * key + 255) & ~(size_t)255;  // as bag_bytes in the kernel
    return p.bglob ? bag + (((size_t)p.pq * key + 255) & ~(size_t)255) : bag;
}

size_t song::group_lds_bytes(bool exact, int pq, int slack, int hlog, int qld, int vis16, int lanes) {
    const size_t key = exact ? 16 : 8;
    const size_t qc = (size_t)pq + (size_t)slack + 2 * (size_t)lanes;
    return ((size_t)(vis16 ? 2 : 4) << hlog) + qc * key + (size_t)((pq + 1) & ~1) * key + 64 * key + 64 * 4 +
           (size_t)qld * 4;
}

int song::make_plan(const song_index *ix, bool exact, int store, int pq, int slack, int hlog, Plan *p, int shape,
                    int visited_bits, int bloom_k, int queries_per_wave, int bag_lds, int waves_per_query,
                    int best_in_global, uint64_t nq_hint) {
    if (pq > 4096) return fail(SONG_E_ARG, "pq=%d exceeds 4096", pq);
    if (queries_per_wave != 1 && queries_per_wave != 2 && queries_per_wave != 4)
        return fail(SONG_E_ARG, "queries_per_wave=%d not 1, 2 or 4", queries_per_wave);
    if (queries_per_wave > 1 && bloom_k != 0)
        return fail(SONG_E_ARG, "several queries per wave use the exact visited table (bloom_k must be 0)");
    if (queries_per_wave > 1 && ix->gstride != 32)
        return fail(SONG_E_ARG, "several queries per wave need graph rows of 32 slots (shift <= 5)");
    p->lanes = 64 / queries_per_wave;
    if (bag_lds && (queries_per_wave > 1 || store != SONG_STORE_F32))
        return fail(SONG_E_ARG, "an LDS bag needs one query per wave and float32 rows");
    p->bag_lds = bag_lds ? 1 : 0;
    if (waves_per_query != 1 && waves_per_query != 2)
        return fail(SONG_E_ARG, "waves_per_query=%d not 1 or 2", waves_per_query);
    if (waves_per_query == 2 && (exact || store != SONG_STORE_F32 || bloom_k != 0 || queries_per_wave > 1 || bag_lds))
        return fail(SONG_E_ARG, "two waves per query need FP32 mode on float32 rows, the exact visited table, one "
                                "query per wave and the bag in global memory");
    p->duo = waves_per_query == 2 ? 1 : 0;
    if (best_in_global < -1 || best_in_global > 1) return fail(SONG_E_ARG, "best_in_global=%d", best_in_global);
    const bool bglob_ok = queries_per_wave == 1 && !bag_lds && store == SONG_STORE_F32;
    if (best_in_global == 1 && !bglob_ok)
        return fail(SONG_E_ARG, "the best list in global memory needs one query per wave, float32 rows and the bag "
                                "in global memory");
    p->pq = pq;
    if (bloom_k < -1 || bloom_k > 9) return fail(SONG_E_ARG, "bloom_k=%d not in [-1,9]", bloom_k);
    if (bloom_k != 0) {
        int bh = 0, bk = 0;
        bloom_size(pq, &bh, &bk);
        if (hlog <= 0) hlog = bh;
        if (bloom_k < 0) bloom_k = bk;
        if (hlog < 1 || hlog > 15) return fail(SONG_E_ARG, "Bloom filter of 2^%d words", hlog);
    }
    p->bloom_k = bloom_k;
    if (store != SONG_STORE_F32 && !ix->d_lp[store]) return fail(SONG_E_ARG, "storage %d not built", store);
    p->exact = exact && store == SONG_STORE_F32;
    p->store = store;
    const int units = store == SONG_STORE_F32 ? ix->ld / 4 : (int)(ix->lp_stride[store] / 16);
    p->shape = shape >= 0 ? std::min(shape, 4) : shape_for_units(units);
    p->hlog = hlog;
    p->slack = slack;
    // queue buffer: pq + slack live entries, 64 of merge room, 64 of head room
    p->qcap = pq + slack + 128;
    p->qld = (ix->dim + 15) & ~15;
    // compact visited slots when an id's bits beyond the group index (groups of 8) number 0..13
    const int lob = ix->idbits - (hlog - 3);
    p->vis16 = (bloom_k == 0 && visited_bits != 32 && hlog >= 4 && lob >= 0 && lob <= 13) ? 1 : 0;
    p->bglob = best_in_global == 1 ? 1 : 0;
    p->seq_stage = 0;
    if (best_in_global < 0 && bglob_ok) {
        const size_t lds_front = lds_granted(lds_bytes(p->exact, pq, p->qcap, hlog, p->qld, p->vis16, bloom_k, 0, 0));
        const uint64_t per_cu = std::max<uint64_t>(1, ix->max_lds / lds_front);
        p->bglob = (nq_hint == 0 || nq_hint > per_cu * (uint64_t)ix->n_cu) ? 1 : 0;
    }
    if (p->lanes < 64) {
        p->shape = std::min(p->shape, 3);  // a row's lanes must lie in one sub-group
        p->lds = group_lds_bytes(p->exact, pq, slack, hlog, p->qld, p->vis16, p->lanes);
    } else {
        p->lds = lds_bytes(p->exact, pq, p->qcap, hlog, p->qld, p->vis16, bloom_k, p->bag_lds, p->bglob);
        // exact sums of wide rows (the shapes that share a row among 16 or more lanes) are done again
        // through LDS, where the slice has room for it
        const size_t more = SEQ_STAGE * sizeof(float);
        if (p->exact && p->shape >= 3 && p->lds + more <= ix->max_lds) {
            p->seq_stage = 1;
            p->lds += more;
        }
    }
    if (p->lds > ix->max_lds)
        return fail(SONG_E_OVERFLOW, "search needs %zu bytes of LDS per query (> %zu)", p->lds, ix->max_lds);
    return SONG_OK;
}

// LDS visited-table size by budget, the fastest on the 1M x 128 workload: 2^12 slots (8 KB with
// the compact 16-bit table) keep the ~1-3k vertices a search discovers up to pq ~ 1000 in LDS
// at 3/4 load; the few queries that discover more continue in the global table, and queries
// whose global table overflows are re-run.
int song::default_hlog(int pq) { return pq > 1024 ? 13 : 12; }

// waves of a plan that one CU holds, by its LDS and by the kernel's registers; 0 = unknown
static int waves_per_cu(const song_index *ix, const Plan &p, bool persistent) {
    const SearchFn fn = search_fn(ix->metric, p, persistent);
    const size_t lds = (p.lds + 15) & ~(size_t)15;
    int n = 0;
    if (!fn || lds > 65536 ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *)fn, 64, lds) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return (int)std::min<size_t>((size_t)n, ix->max_lds / lds_granted(lds));
}

// The default table of a plain or no-allocation call.  Results do not depend on the size.
//
// Where its nq queries leave LDS free: as large as leaves all of them in flight at once, up to 2^14
// slots.  A fuller table costs second probes (at half load one of 31 neighbours finds its group full in
// most expansions) and, at the end, the global one.
//
// Where they do not fit at once: half the table if a CU then holds at least a sixth more waves and these
// take them in fewer rounds.  The kernels of rows up to 32 floats, and of narrow 16- and 8-bit rows,
// leave registers for 20 to 24 waves where 2^12 slots leave LDS for 16.  Up to 100k rows and pq 128 few
// searches outgrow 2^11 slots: cosine 15k x 16, 5000 queries at pq 100, exact 668 -> 574 us; 100k x 32
// uniform rows, 9000 queries at pq 100, 935 -> 877 us, bf16 943 -> 892.  As many rounds as before lose
// (the same set, 7000 queries: 778 -> 811), and so do a few more waves over many rounds (100k x 96 in
// bf16, 14 -> 16 waves, 30,000 queries at pq 100: 3866 -> 4080), larger budgets (50k x 24, 20,000 queries
// at pq 256: 3499 -> 3689), larger sets (1M x 32, 4500 queries at pq 100: 929 -> 1138) and 2^10 slots.
int song::roomy_hlog(const song_index *ix, bool exact, int store, int pq, int slack, uint64_t nq, int visited_bits,
                     int best_in_global, bool persistent) {
    int h = default_hlog(pq);
    const uint64_t per_cu = std::max<uint64_t>(1, (nq + ix->n_cu - 1) / ix->n_cu);
    auto plan = [&](int hlog, Plan *p) {
        return make_plan(ix, exact, store, pq, slack, hlog, p, -1, visited_bits, 0, 1, 0, 1, best_in_global, nq) == SONG_OK;
    };
    Plan p;
    while (h < 14 && plan(h + 1, &p) && lds_granted(p.lds) * per_cu <= ix->max_lds) ++h;
    Plan half;
    if (h == default_hlog(pq) && pq <= 128 && ix->n <= 100000 && plan(h, &p) && plan(h - 1, &half)) {
        const uint64_t now = waves_per_cu(ix, p, persistent), more = waves_per_cu(ix, half, persistent);
        if (now > 0 && 6 * more >= 7 * now && (per_cu + more - 1) / more < (per_cu + now - 1) / now) --h;
    }
    return h;
}

SearchFn song::search_fn(int metric, const Plan &p, bool persistent) {
    if (p.duo && persistent) {
        switch (metric) {
        case SONG_L2: return duo_fn_l2(p.shape, p.bglob);
        case SONG_IP: return duo_fn_ip(p.shape, p.bglob);
        default: return duo_fn_cos(p.shape, p.bglob);
        }
    }
    if (p.lanes < 64) {
        switch (metric) {
        case SONG_L2: return group_fn_l2(p.exact, p.store, p.shape, p.lanes);
        case SONG_IP: return group_fn_ip(p.exact, p.store, p.shape, p.lanes);
        default: return group_fn_cos(p.exact, p.store, p.shape, p.lanes);
        }
    }
    const bool bagl = p.bag_lds && persistent;
    switch (metric) {
    case SONG_L2: return search_fn_l2(p.exact, p.store, p.shape, persistent, bagl, p.bglob);
    case SONG_IP: return search_fn_ip(p.exact, p.store, p.shape, persistent, bagl, p.bglob);
    default: return search_fn_cos(p.exact, p.store, p.shape, persistent, bagl, p.bglob);
    }
}

static int launch(song_index *ix, const Plan &p, SearchParams sp, unsigned count, hipStream_t st,
                  uint32_t *gvis) {
    SearchFn fn = search_fn(ix->metric, p);
    const size_t stride = bag_stride(p);
    int rc = ensure_gbag(ix, (void *)st, std::min(count, kChunk), stride, &sp.gbag);
    if (rc != SONG_OK) return rc;
    sp.gbag_stride = stride;
    sp.hlog = p.hlog;
    sp.slack = p.slack;
    sp.qcap = p.qcap;
    sp.gvis = gvis;
    sp.ghlog = kGhlog;
    sp.qld = p.qld;
    sp.wave_lds = (uint32_t)p.lds;
    sp.vis16 = p.vis16;
    sp.seq_stage = p.seq_stage;
    sp.bloom_k = p.bloom_k;
    sp.idbits = ix->idbits;
    sp.data_lp = ix->d_lp[p.store];
    sp.scale = ix->d_scale[p.store];
    sp.lp_stride = ix->lp_stride[p.store];
    if (p.lds > 65536)
        HIP_TRY(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds));
    for (unsigned q0 = 0; q0 < count; q0 += kChunk) {
        sp.qbase = (int)q0;
        hipLaunchKernelGGL(fn, dim3(std::min(kChunk, count - q0)), dim3(64), p.lds, st, sp);
        HIP_TRY(hipGetLastError());
    }
    return SONG_OK;
}

// FP32 accumulation is exact when every product and every partial sum is an integer
// below 2^24: integer-valued data and queries with dim * span^2 < 2^24 (L2) or
// dim * max|x| * max|q| < 2^24 (IP).
bool song::fp32_exact(const song_index *ix, int q_integer, float qmin, float qmax) {
    if (!ix->integer_valued || !q_integer || ix->metric == SONG_COS) return false;
    double lim = 16777216.0;
    if (ix->metric == SONG_L2) {
        double span = std::max((double)ix->vmax, (double)qmax) - std::min((double)ix->vmin, (double)qmin);
        return (double)ix->dim * span * span < lim;
    }
    double ax = std::max(std::fabs((double)ix->vmin), std::fabs((double)ix->vmax));
    double aq = std::max(std::fabs((double)qmin), std::fabs((double)qmax));
    return (double)ix->dim * ax * aq < lim;
}

extern "C" int song_search_device(song_index *ix, const float *d_queries, uint64_t nq, int pq, int k,
                                  const int *d_pq, const int *d_k, uint32_t *d_ids, float *d_dist, int k_ld,
                                  uint32_t *d_flags, uint32_t *d_stats, const song_search_opts *opts_in,
                                  void *stream) {
    song_query_params qp{};
    qp.pq = d_pq;
    qp.k = d_k;
    qp.n_entry = 1;
    return song_search_device_ex(ix, d_queries, nq, pq, k, &qp, d_ids, d_dist, k_ld, d_flags, d_stats, opts_in,
                                 stream);
}

extern "C" int song_search_device_ex(song_index *ix, const float *d_queries, uint64_t nq, int pq, int k,
                                     const song_query_params *qp_in, uint32_t *d_ids, float *d_dist, int k_ld,
                                     uint32_t *d_flags, uint32_t *d_stats, const song_search_opts *opts_in,
                                     void *stream) {
    song_query_params qp{};
    qp.n_entry = 1;
    if (qp_in) qp = *qp_in;
    const int *d_pq = qp.pq, *d_k = qp.k;
    const uint32_t *d_entry = qp.entry;
    const int n_entry = qp.entry ? qp.n_entry : 1, *d_steps = qp.steps;
    if (n_entry < 1 || n_entry > 64) return fail(SONG_E_ARG, "n_entry=%d not in [1,64]", n_entry);
    const uint64_t nrun = qp.subset ? qp.n_subset : nq;
    if (!ix) return fail(SONG_E_ARG, "index is null");
    if (nq == 0) return SONG_OK;
    if (!d_queries || !d_ids) return fail(SONG_E_ARG, "queries/ids are null");
    if (pq < 1 || k < 1 || k_ld < k) return fail(SONG_E_ARG, "pq=%d k=%d k_ld=%d", pq, k, k_ld);
    if (nq > 0x7fffffffull) return fail(SONG_E_ARG, "nq too large");
    song_search_opts opts;
    song_search_opts_default(&opts);
    if (opts_in) opts = *opts_in;
    if (opts.slack < 0) opts.slack = 0;
    if (opts.max_steps <= 0) opts.max_steps = 1000000;
    hipStream_t st = (hipStream_t)stream;

    if (opts.storage < SONG_STORE_F32 || opts.storage > SONG_STORE_FP8)
        return fail(SONG_E_ARG, "storage=%d", opts.storage);
    if (opts.visited_bits != 0 && opts.visited_bits != 16 && opts.visited_bits != 32)
        return fail(SONG_E_ARG, "visited_bits=%d not 0, 16 or 32", opts.visited_bits);
    bool exact = true;
    if (opts.storage != SONG_STORE_F32 || opts.mode == SONG_MODE_FP32) {
        exact = false;
    } else if (opts.mode == SONG_MODE_AUTO && ix->integer_valued && ix->metric != SONG_COS) {
        int qint = 0;
        float qmin = 0.f, qmax = 0.f;
        int rc = device_range(ix, d_queries, nq * (uint64_t)ix->dim, &qint, &qmin, &qmax, st);
        if (rc != SONG_OK) return rc;
        exact = !fp32_exact(ix, qint, qmin, qmax);
    }

    uint32_t *gvis = nullptr;
    int rcg = ensure_gvis(ix, stream, (size_t)std::min<uint64_t>(nrun ? nrun : 1, kChunk), &gvis);
    if (rcg != SONG_OK) return rcg;
    int hlog = opts.hash_log2 > 0 ? opts.hash_log2
                                  : roomy_hlog(ix, exact, opts.storage, pq, opts.slack, nrun, opts.visited_bits,
                                               opts.best_in_global, false);
    hlog = std::max(8, std::min(hlog, 16));
    if (opts.bloom_k != 0) hlog = opts.hash_log2 > 0 ? std::min(opts.hash_log2, 15) : 0;  // 0: sized for pq
    Plan plan;
    int rc = make_plan(ix, exact, opts.storage, pq, opts.slack, hlog, &plan, -1, opts.visited_bits, opts.bloom_k, 1, 0,
                       1, opts.best_in_global, nrun);
    if (rc != SONG_OK) return rc;

    uint32_t *flags = d_flags;
    uint32_t *tmp_flags = nullptr;
    if (!flags && opts.retry) {
        HIP_TRY(hipMalloc(&tmp_flags, nq * sizeof(uint32_t)));
        flags = tmp_flags;
    }
    SearchParams sp{};
    sp.data = ix->d_data;
    sp.graph = ix->d_graph;
    sp.norms = ix->d_norms;
    sp.queries = d_queries;
    sp.entry = d_entry;
    sp.n_entry = n_entry;
    sp.steps_arr = d_steps;
    sp.pq_arr = d_pq;
    sp.k_arr = d_k;
    sp.qidx = qp.subset;
    sp.out_ids = d_ids;
    sp.out_dist = d_dist;
    sp.out_flags = flags;
    sp.out_stats = d_stats;
    sp.n = ix->n;
    sp.dim = ix->dim;
    sp.ld = ix->ld;
    sp.gstride = ix->gstride;
    sp.int_rows = ix->integer_valued;
    sp.row_min = ix->vmin;
    sp.row_max = ix->vmax;
    sp.nq = (int)nq;
    sp.pq = pq;
    sp.k = k;
    sp.out_ld = k_ld;
    sp.max_steps = opts.max_steps;
    sp.rerank = opts.rerank;
    if (nrun == 0) {
        if (tmp_flags) (void)hipFree(tmp_flags);
        return SONG_OK;
    }
    rc = launch(ix, plan, sp, (unsigned)nrun, st, gvis);
    if (rc == SONG_OK && opts.retry) {
        // re-run queries whose LDS tables overflowed, with 4x larger tables, until none remain
        std::vector<uint32_t> hf(nq);
        std::vector<uint32_t> run_ids;
        if (qp.subset) {
            run_ids.resize(nrun);
            if (hipMemcpyAsync(run_ids.data(), qp.subset, nrun * 4, hipMemcpyDeviceToHost, st) != hipSuccess)
                rc = fail(SONG_E_HIP, "subset readback");
        }
        uint32_t *d_idx = nullptr;
        for (int round = 0; rc == SONG_OK; ++round) {
            if (hipMemcpyAsync(hf.data(), flags, nq * sizeof(uint32_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipStreamSynchronize(st) != hipSuccess) {
                rc = fail(SONG_E_HIP, "flag readback");
                break;
            }
            std::vector<uint32_t> redo;
            bool vis = false, que = false;
            for (uint64_t j = 0; j < nrun; ++j) {
                const uint64_t i = run_ids.empty() ? j : run_ids[j];
                if (hf[i] & (SONG_FLAG_VISITED_OVF | SONG_FLAG_QUEUE_OVF)) {
                    redo.push_back((uint32_t)i);
                    vis |= (hf[i] & SONG_FLAG_VISITED_OVF) != 0;
                    que |= (hf[i] & SONG_FLAG_QUEUE_OVF) != 0;
                }
            }
            if (redo.empty()) break;
            if (round == 4) {
                rc = fail(SONG_E_OVERFLOW, "%zu queries still overflow after 4 re-runs", redo.size());
                break;
            }
            Plan p2;
            int h2 = vis ? plan.hlog + 2 : plan.hlog;
            int s2 = que ? plan.slack * 4 + 64 : plan.slack;
            rc = make_plan(ix, exact, opts.storage, pq, s2, std::min(h2, plan.bloom_k ? 15 : 16), &p2, -1,
                           opts.visited_bits, plan.bloom_k, 1, 0, 1, opts.best_in_global, redo.size());
            if (rc != SONG_OK) break;
            plan = p2;
            if (!d_idx && hipMalloc(&d_idx, nq * sizeof(uint32_t)) != hipSuccess) {
                rc = fail(SONG_E_HIP, "hipMalloc retry index");
                break;
            }
            if (hipMemcpyAsync(d_idx, redo.data(), redo.size() * 4, hipMemcpyHostToDevice, st) != hipSuccess) {
                rc = fail(SONG_E_HIP, "retry index upload");
                break;
            }
            SearchParams sp2 = sp;
            sp2.qidx = d_idx;
            rc = launch(ix, plan, sp2, (unsigned)redo.size(), st, gvis);
            if (rc != SONG_OK) break;
        }
        if (d_idx) (void)hipFree(d_idx);
    }
    if (tmp_flags) (void)hipFree(tmp_flags);
    return rc;
}

extern "C" int song_search(song_index *ix, const float *queries, uint64_t nq, int pq, int k, uint64_t *out_ids,
                           float *out_dist, uint32_t *out_flags, const song_search_opts *opts) {
    if (!ix) return fail(SONG_E_ARG, "index is null");
    if (nq == 0) return SONG_OK;
    if (!queries || !out_ids) return fail(SONG_E_ARG, "queries/out_ids are null");
    if (pq < 1 || k < 1) return fail(SONG_E_ARG, "pq=%d k=%d", pq, k);
    // rows keep the caller's stride k; a search returns at most pq entries, so columns
    // [pq, k) are padding (UINT64_MAX, +inf) like a list shorter than k
    const int kk = std::min(k, pq);
    // one workspace: queries, then ids, distances and flags, which come back in one copy
    const size_t qb = (nq * (size_t)ix->dim * sizeof(float) + 255) & ~(size_t)255, n = nq * (size_t)k;
    const size_t rb = (2 * n + nq) * 4;
    Workspace ws(ix);
    int rc = ws.take(qb + rb);
    if (rc != SONG_OK) return rc;
    float *d_q = reinterpret_cast<float *>(ws.w.dev);
    uint32_t *d_i = reinterpret_cast<uint32_t *>(ws.w.dev + qb), *d_f = d_i + 2 * n;
    float *d_d = reinterpret_cast<float *>(d_i + n);
    const bool pinned = ws.w.host != nullptr;
    std::vector<uint32_t> plain(pinned ? 0 : rb / 4);
    uint32_t *h_i = pinned ? reinterpret_cast<uint32_t *>(ws.w.host + qb) : plain.data(), *h_f = h_i + 2 * n;
    const float *h_d = reinterpret_cast<const float *>(h_i + n);
    song_search_opts o;
    song_search_opts_default(&o);
    if (opts) o = *opts;
    // the queries' range here, where they are, for what fits in a few microseconds; the GPU's otherwise
    if (o.mode == SONG_MODE_AUTO && o.storage == SONG_STORE_F32 && ix->integer_valued && ix->metric != SONG_COS &&
        nq * (size_t)ix->dim <= 32768) {
        unsigned mn = 0xffffffffu, mx = 0u;
        int whole = 1;
        for (size_t i = 0; i < nq * (size_t)ix->dim; ++i) {
            whole &= queries[i] == std::rint(queries[i]);
            mn = std::min(mn, ord_host(queries[i]));
            mx = std::max(mx, ord_host(queries[i]));
        }
        o.mode = fp32_exact(ix, whole, unord_host(mn), unord_host(mx)) ? SONG_MODE_FP32 : SONG_MODE_EXACT;
    }
    const void *src = queries;
    if (pinned) src = memcpy(ws.w.host, queries, nq * (size_t)ix->dim * sizeof(float));
    HIP_TRY(hipMemcpyAsync(d_q, src, nq * (size_t)ix->dim * sizeof(float), hipMemcpyHostToDevice, nullptr));
    // searched once and read back with the flags; only when a query overflowed, again with re-runs
    const int retry = o.retry;
    for (int pass = 0; pass < 2; ++pass) {
        o.retry = pass;
        rc = song_search_device(ix, d_q, nq, pq, kk, nullptr, nullptr, d_i, d_d, k, d_f, nullptr, &o, nullptr);
        if (rc != SONG_OK) return rc;
        HIP_TRY(hipMemcpyAsync(h_i, d_i, rb, hipMemcpyDeviceToHost, nullptr));
        HIP_TRY(hipStreamSynchronize(nullptr));
        bool over = false;
        for (uint64_t i = 0; i < nq; ++i) over |= (h_f[i] & (SONG_FLAG_VISITED_OVF | SONG_FLAG_QUEUE_OVF)) != 0;
        if (!over || !retry) break;
    }
    for (uint64_t r = 0; r < nq; ++r)
        for (int c = 0; c < k; ++c) {
            const size_t i = r * (size_t)k + c;
            out_ids[i] = (c >= kk || h_i[i] == 0xFFFFFFFFu) ? UINT64_MAX : (uint64_t)h_i[i];
            if (out_dist) out_dist[i] = c >= kk ? INFINITY : h_d[i];
        }
    if (out_flags) memcpy(out_flags, h_f, nq * sizeof(uint32_t));
    return SONG_OK;
}

extern "C" int song_astar_multi_start_search_batch(const float *h_queries, uint64_t nq, int pq, uint64_t *results,
                                                   const float *h_data, const uint64_t *h_graph,
                                                   int vertex_offset_shift, uint64_t num, int dim, int metric) {
    song_index *ix = nullptr;
    int rc = song_index_create(h_data, num, dim, h_graph, vertex_offset_shift, metric, &ix);
    if (rc != SONG_OK) return rc;
    song_search_opts o;
    song_search_opts_default(&o);
    o.mode = SONG_MODE_EXACT;
    rc = song_search(ix, h_queries, nq, pq, pq, results, nullptr, nullptr, &o);
    song_index_destroy(ix);
    return rc;
}
