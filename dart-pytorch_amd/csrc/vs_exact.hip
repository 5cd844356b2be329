// vs_exact.hip -- exact top-k without the MFMA selection: every (query, row)
// score in the reference's fp64 arithmetic as a 64-bit key, then per-query
// selection of the k smallest keys.  Serves searches so small that a key
// matrix costs less than the selection's bookkeeping, every k the fused
// selection's lists cannot hold, and the queries it could not prove.
#include <algorithm>

#include "vs_device.h"

namespace vs {

// ---------------------------------------------------------------------------
// Queries as fp64 rows [nq][ldd], zero past d (the fp32 values promoted), so
// that the tile kernel reads them with scalar loads.  Row qi's flag word
// holds kFlagNonFinite if a value is NaN or infinite; such a row becomes zero.
// One workgroup per query: the values may sit in host memory, where every
// dependent round trip costs over a microsecond.
// ---------------------------------------------------------------------------
template <typename TS>
__global__ __launch_bounds__(256) void exact_queries_kernel(const TS *__restrict__ src,
                                                            int64_t stride, int64_t d, int64_t ldd,
                                                            double *__restrict__ qd,
                                                            uint32_t *__restrict__ rowflags) {
    const int64_t q = blockIdx.x;
    bool bad = false;
    for (int64_t j0 = threadIdx.x; j0 < ldd; j0 += 4 * 256) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t j = j0 + u * 256;
            v[u] = 0.0f;
            if (j < d) {
                if constexpr (sizeof(TS) == 2)
                    v[u] = bf16_to_f32(src[q * stride + j]);
                else
                    v[u] = src[q * stride + j];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            bad |= !__builtin_isfinite(v[u]);
            if (j0 + u * 256 < ldd) qd[q * ldd + j0 + u * 256] = (double)v[u];
        }
    }
    bad = __syncthreads_or(bad);
    if (bad)
        for (int64_t j = threadIdx.x; j < ldd; j += 256) qd[q * ldd + j] = 0.0;
    if (rowflags && threadIdx.x == 0) rowflags[q] = bad ? kFlagNonFinite : 0u;
}

int64_t exact_ldd(int64_t d) { return (d + 63) / 64 * 64; }

hipError_t launch_exact_queries(const void *src, int src_dtype, int64_t stride, int64_t nq,
                                int64_t d, double *qd, uint32_t *rowflags, hipStream_t st) {
    if (nq <= 0) return hipSuccess;
    if (nq > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)nq), block(256);
    if (src_dtype == 0)
        exact_queries_kernel<float><<<grid, block, 0, st>>>((const float *)src, stride, d,
                                                            exact_ldd(d), qd, rowflags);
    else
        exact_queries_kernel<uint16_t><<<grid, block, 0, st>>>((const uint16_t *)src, stride, d,
                                                               exact_ldd(d), qd, rowflags);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// keys[q][r] = enc_order(key) << 32 | r, key = fp32 score (L2) or -fp32 score
// (IP) of query q and row r, the score being the fp64 sum in dimension order
// (index_flat.dart:75-90).
//
// Bound by the fp64 rate: one product of two promoted fp32 values is exact
// in fp64, so IP takes one fused multiply-add per element (the same bits as
// a multiply and an add); L2 takes subtract, multiply, add.  A workgroup
// covers 64 rows by 4 QT queries: the rows are staged through LDS in
// 64-element chunks with coalesced loads (the next chunk in flight while one
// is summed), each lane sums one row against its wave's QT queries, whose
// values are wave-uniform and come through scalar loads as fp64, so the
// vector units convert each row value once for QT products.  QT = 4: 16
// scalars per 4 elements leave room for the next ones in flight.
// Measured: 100 queries x 200,000 x 128, L2: 300 us, 8.5e12 products/s, two
// thirds of the fp64 rate (one thread per row and query: 1,814 us); 100 x
// 10,000 x 384, IP: 37 us; one query x 10,000 x 384: 17 us.
// ---------------------------------------------------------------------------
// (the constant address space makes uniform loads scalar ones)
typedef const __attribute__((address_space(4))) double *const_f64_t;

constexpr int kWaitLgkm0 = 0xC07F;  // s_waitcnt lgkmcnt(0) alone

constexpr int kExactRows = 64, kExactK = 64, kExactPad = 4;

struct ExactTileArgs {
    const void *xb;
    int64_t ld, d, ldd;
    const double *qd;
    int64_t nq, n;
    uint64_t *keys;
    int64_t kstride;
};

template <int ST, int METRIC, int QT>
__global__ __launch_bounds__(256) void exact_tile_kernel(ExactTileArgs a) {
    __shared__ __align__(16) float xs[kExactRows][kExactK + kExactPad];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t r0 = (int64_t)blockIdx.x * kExactRows;
    const int64_t qb = ((int64_t)blockIdx.y * 4 + w) * QT;
    const bool active = qb < a.nq;
    const_f64_t qrow[QT];
#pragma unroll
    for (int u = 0; u < QT; ++u)
        qrow[u] = (const_f64_t)(uintptr_t)(a.qd + min(qb + u, a.nq - 1) * a.ldd);
    double acc[QT];
#pragma unroll
    for (int u = 0; u < QT; ++u) acc[u] = 0.0;

    // a thread's 16-byte pieces of a chunk (rows past n are slack rows)
    constexpr int PE = ST == 1 ? 8 : 4;                  // elements per piece
    constexpr int TPR = kExactK / PE;                    // threads per row
    constexpr int NP = kExactRows * kExactK / PE / 256;  // pieces per thread
    const int prow = tid / TPR, pcol = (tid % TPR) * PE;
    u32x4_t piece[NP];
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int64_t e = (r0 + prow + i * (256 / TPR)) * a.ld + k0 + pcol;
            piece[i] = *(const u32x4_t *)((const char *)a.xb + e * (ST == 1 ? 2 : 4));
        }
    };
    load(0);
    for (int64_t k0 = 0; k0 < a.d; k0 += kExactK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            float *dst = &xs[prow + i * (256 / TPR)][pcol];
            if constexpr (ST == 1) {
                const u32x4_t p = piece[i];  // element 2u is the low half of word u
                const u32x4_t lo = {p.x << 16, p.x & 0xFFFF0000u, p.y << 16, p.y & 0xFFFF0000u};
                const u32x4_t hi = {p.z << 16, p.z & 0xFFFF0000u, p.w << 16, p.w & 0xFFFF0000u};
                *(u32x4_t *)dst = lo;
                *(u32x4_t *)(dst + 4) = hi;
            } else {
                *(u32x4_t *)dst = piece[i];
            }
        }
        __syncthreads();
        if (k0 + kExactK < a.d) load(k0 + kExactK);
        if (active) {
            // (elements past d are zero on both sides: their terms add +0)
            // 8 elements at a time; the queries' values of the next 4 are
            // requested before the current 4 are summed, which hides the
            // scalar cache's latency where few waves share a SIMD
            const int jn = (int)min((int64_t)kExactK, (a.d - k0 + 7) & ~(int64_t)7);
            double qa[QT][4], qn[QT][4];
            auto fetch = [&](double (&dst)[QT][4], int j) {
#pragma unroll
                for (int u = 0; u < QT; ++u)
#pragma unroll
                    for (int c = 0; c < 4; ++c) dst[u][c] = qrow[u][k0 + j + c];
            };
            auto sum = [&](const double (&q)[QT][4], const float4 &x4) {
                const double x[4] = {(double)x4.x, (double)x4.y, (double)x4.z, (double)x4.w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
#pragma unroll
                    for (int u = 0; u < QT; ++u) {
                        if constexpr (METRIC == 0) {
                            const double diff = q[u][c] - x[c];
                            acc[u] = acc[u] + diff * diff;
                        } else {
                            acc[u] = __builtin_fma(q[u][c], x[c], acc[u]);
                        }
                    }
                }
            };
            fetch(qa, 0);
            float4 xa = *(const float4 *)&xs[lane][0];
            for (int j = 0; j < jn; j += 8) {
                // (scalar loads return out of order, so waiting for the current
                // values has to come before the next request)
                __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
                const float4 xb4 = *(const float4 *)&xs[lane][j + 4];
                fetch(qn, j + 4);
                __builtin_amdgcn_sched_barrier(0);
                sum(qa, xa);
                // (the last fetch re-reads the chunk's first elements)
                const int jj = j + 8 < jn ? j + 8 : 0;
                __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
                xa = *(const float4 *)&xs[lane][jj];
                fetch(qa, jj);
                __builtin_amdgcn_sched_barrier(0);
                sum(qn, xb4);
            }
        }
    }
    const int64_t r = r0 + lane;
    if (active && r < a.n) {
#pragma unroll
        for (int u = 0; u < QT; ++u) {
            if (qb + u < a.nq) {
                const float key = METRIC == 0 ? (float)acc[u] : -(float)acc[u];
                a.keys[(qb + u) * a.kstride + r] =
                    ((uint64_t)enc_order(key) << 32) | (uint32_t)r;
            }
        }
    }
}

hipError_t launch_exact_tile(const void *xb, int storage, int64_t ld, int64_t d, int metric,
                             const double *qd, int64_t nq, int64_t n, uint64_t *keys,
                             int64_t kstride, hipStream_t st) {
    if (nq <= 0 || n <= 0) return hipSuccess;
    if (n > (int64_t)UINT32_MAX) return hipErrorInvalidValue;
    const int qt = nq <= 4 ? 1 : 4;
    const int64_t nx = (n + kExactRows - 1) / kExactRows, ny = (nq + 4 * qt - 1) / (4 * qt);
    if (nx > INT32_MAX || ny > 65535) return hipErrorInvalidValue;
    ExactTileArgs a{xb, ld, d, exact_ldd(d), qd, nq, n, keys, kstride};
    void (*fn)(ExactTileArgs);
    if (storage == 1)
        fn = metric == 0 ? (qt == 1 ? exact_tile_kernel<1, 0, 1> : exact_tile_kernel<1, 0, 4>)
                         : (qt == 1 ? exact_tile_kernel<1, 1, 1> : exact_tile_kernel<1, 1, 4>);
    else
        fn = metric == 0 ? (qt == 1 ? exact_tile_kernel<0, 0, 1> : exact_tile_kernel<0, 0, 4>)
                         : (qt == 1 ? exact_tile_kernel<0, 1, 1> : exact_tile_kernel<0, 1, 4>);
    hipLaunchKernelGGL(fn, dim3((unsigned)nx, (unsigned)ny), dim3(256), 0, st, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The k smallest of a segment's keys, sorted.  One workgroup per (query,
// segment).  kNoKey entries (no row) are ignored.
//
// Bound by reading the keys, three times in the usual case: once for their
// smallest and largest, once for a histogram of 2048 equal steps between
// those (the distances of a query spread over few exponents, so bins on the
// keys' top bits would hold nearly all of them), once to collect the keys up
// to the k-th's bin into LDS, where they are sorted.  While that bin holds
// more than the buffer takes, it is divided again, at the end down to one key
// (a subset may name a row more than once).
// Measured: k = 1000 of 200,000 keys for 100 queries: 117 us (a device radix
// sort per query: 7 ms); k = 10 of 10,000 keys: 10 us.
// ---------------------------------------------------------------------------
constexpr uint64_t kNoKey = ~0ull;
constexpr int kSelBins = 2048, kSelThreads = 1024, kSelRegKeys = 10;
// Places in a segment of up to INT32_MAX keys.  The walk looks up to eight
// rounds past the last key, which 32 signed bits do not count to.
typedef uint32_t sel_pos_t;
constexpr int kSelUnroll = 8;
static_assert((uint64_t)INT32_MAX + 2ull * kSelUnroll * kSelThreads <= (sel_pos_t)~(sel_pos_t)0 &&
                  (sel_pos_t)~(sel_pos_t)0 > 0,
              "a place past the last key neither wraps nor turns negative");

struct SelectKeysArgs {
    const uint64_t *keys;
    int64_t n, kstride;
    int64_t seglen;
    int nseg;
    int64_t k;
    int cap;  // keys the LDS buffer holds (a power of two >= 2 k)
    int metric;
    float *D;        // [nq][k] results (outk null)
    int32_t *I;
    uint64_t *outk;  // [nq][nseg][k] keys, kNoKey past the segment's
    // flags of every query of the call (or null): with any set, D and I are
    // left alone; *hflags (host-visible) receives their union
    const uint32_t *rowflags;
    int64_t nflags;
    uint32_t *hflags;
    // groups instead of equal rows of keys (off non-null): query q's keys are
    // keys[off[q] .. + cnt[q]); kFlagShort goes to *short_flag (or null) for
    // one of fewer than k
    const int32_t *off, *cnt;
    uint32_t *short_flag;
};

__device__ __forceinline__ void sort_keys_block(uint64_t *b, int n) {
    for (int size = 2; size <= n; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < (n >> 1); t += kSelThreads) {
                const int i = 2 * t - (t & (stride - 1)), j = i + stride;
                const uint64_t vi = b[i], vj = b[j];
                if ((vi > vj) == ((i & size) == 0)) {
                    b[i] = vj;
                    b[j] = vi;
                }
            }
            __syncthreads();
        }
    }
}

// REG: the segment's keys (at most kSelRegKeys per thread) stay in registers
// after one read; otherwise every pass reads them again.
template <bool REG>
__global__ __launch_bounds__(kSelThreads) void select_keys_kernel(SelectKeysArgs a) {
    extern __shared__ __align__(16) char smem[];
    uint64_t *buf = (uint64_t *)smem;        // [cap]
    int *hist = (int *)(buf + a.cap);        // [kSelBins]
    __shared__ uint64_t s_lo[16], s_hi[16];
    __shared__ int s_n[16];
    __shared__ int s_bin, s_before, s_in, s_fill, s_eq;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t q = blockIdx.x / a.nseg;
    const int seg = (int)(blockIdx.x % a.nseg);
    const int64_t k0 = (int64_t)seg * a.seglen;
    const int m = a.off ? a.cnt[q] : (int)max((int64_t)0, min(a.seglen, a.n - k0));
    const uint64_t *kp = a.keys + (a.off ? (int64_t)a.off[q] : q * a.kstride + k0);
    if (a.short_flag && tid == 0 && m < a.k) atomicOr(a.short_flag, kFlagShort);

    uint32_t flag = 0;
    if (a.rowflags) {
        for (int64_t t = tid; t < a.nflags; t += kSelThreads) flag |= a.rowflags[t];
        flag = __syncthreads_or((int)flag);
        if (tid == 0 && blockIdx.x == 0) *a.hflags = flag;
    }

    uint64_t reg[kSelRegKeys];
    if constexpr (REG) {
#pragma unroll
        for (int u = 0; u < kSelRegKeys; ++u) {
            const int t = u * kSelThreads + tid;
            reg[u] = t < m ? kp[t] : kNoKey;
        }
    }
    auto each = [&](auto &&f) {  // f(key) for every key of the thread
        if constexpr (REG) {
#pragma unroll
            for (int u = 0; u < kSelRegKeys; ++u)
                if (reg[u] != kNoKey) f(reg[u]);
        } else {
            const sel_pos_t end = (sel_pos_t)m;
            for (sel_pos_t t0 = tid; t0 < end; t0 += kSelUnroll * kSelThreads) {
                uint64_t v[kSelUnroll];  // that many loads in flight
#pragma unroll
                for (int u = 0; u < kSelUnroll; ++u) {
                    const sel_pos_t t = t0 + u * kSelThreads;
                    v[u] = t < end ? kp[t] : kNoKey;
                }
#pragma unroll
                for (int u = 0; u < kSelUnroll; ++u)
                    if (v[u] != kNoKey) f(v[u]);
            }
        }
    };
    // smallest and largest key, and how many there are
    uint64_t lo = kNoKey, hi = 0;
    int cnt = 0;
    each([&](uint64_t v) {
        lo = min(lo, v);
        hi = max(hi, v);
        ++cnt;
    });
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint64_t)__shfl_xor((unsigned long long)lo, o));
        hi = max(hi, (uint64_t)__shfl_xor((unsigned long long)hi, o));
        cnt += __shfl_xor(cnt, o);
    }
    if (lane == 0) {
        s_lo[wave] = lo;
        s_hi[wave] = hi;
        s_n[wave] = cnt;
    }
    if (tid == 0) s_fill = s_eq = 0;
    __syncthreads();
    lo = s_lo[0];
    hi = s_hi[0];
    cnt = s_n[0];
    for (int i = 1; i < 16; ++i) {
        lo = min(lo, s_lo[i]);
        hi = max(hi, s_hi[i]);
        cnt += s_n[i];
    }

    uint64_t top = hi;  // every key up to top is collected
    int take = cnt;
    int eq_want = INT_MAX;  // of those equal to top, this many
    if (cnt > a.cap) {
        int rank = (int)a.k, below = 0;  // (k <= cap < cnt)
        for (;;) {
            const uint64_t range = hi - lo;
            const int shift = max(0, 64 - (int)__clzll((unsigned long long)(range | 1)) - 11);
            for (int t = tid; t < kSelBins; t += kSelThreads) hist[t] = 0;
            __syncthreads();
            each([&](uint64_t v) {
                if (v >= lo && v <= hi) atomicAdd(&hist[(int)((v - lo) >> shift)], 1);
            });
            __syncthreads();
            // prefix sums: a thread owns bins 2 tid and 2 tid + 1
            const int c0 = hist[2 * tid], c1 = hist[2 * tid + 1];
            int inc = c0 + c1;
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(inc, o);
                if (lane >= o) inc += y;
            }
            if (lane == 63) s_n[wave] = inc;
            __syncthreads();
            int base = 0;
            for (int i = 0; i < wave; ++i) base += s_n[i];
            const int end = base + inc, mid = end - c1, begin = mid - c0;
            if (begin < rank && rank <= end) {  // one thread
                const bool first = rank <= mid;
                s_bin = 2 * tid + (first ? 0 : 1);
                s_before = first ? begin : mid;
                s_in = first ? c0 : c1;
            }
            __syncthreads();
            const int bin = s_bin, before = s_before, in = s_in;
            __syncthreads();
            const uint64_t last = lo + (((uint64_t)bin + 1) << shift) - 1;
            top = last < hi ? last : hi;
            take = below + before + in;
            if (take <= a.cap) break;
            if (shift == 0) {  // one key, more often than the buffer takes
                eq_want = rank - before;
                take = below + before + eq_want;
                break;
            }
            below += before;
            rank -= before;
            lo += (uint64_t)bin << shift;
            hi = top;
        }
    }
    each([&](uint64_t v) {
        if (v < top || (v == top && (eq_want == INT_MAX || atomicAdd(&s_eq, 1) < eq_want)))
            buf[atomicAdd(&s_fill, 1)] = v;
    });
    __syncthreads();
    int p2 = 2;
    while (p2 < take) p2 <<= 1;  // <= cap
    for (int t = take + tid; t < p2; t += kSelThreads) buf[t] = kNoKey;
    __syncthreads();
    sort_keys_block(buf, p2);
    if (a.outk) {
        uint64_t *o = a.outk + ((int64_t)q * a.nseg + seg) * a.k;
        for (int64_t t = tid; t < a.k; t += kSelThreads) o[t] = t < take ? buf[t] : kNoKey;
        return;
    }
    if (flag) return;
    for (int64_t t = tid; t < a.k; t += kSelThreads) {
        const bool ok = t < take;
        const uint64_t v = ok ? buf[t] : 0;
        const float key = dec_order((uint32_t)(v >> 32));
        a.D[q * a.k + t] = ok ? (a.metric == 0 ? key : -key) : (a.metric == 0 ? VS_INF : -VS_INF);
        a.I[q * a.k + t] = ok ? (int32_t)(uint32_t)v : -1;
    }
}

// keys the LDS buffer holds for this k, 0 beyond what a workgroup can sort
int select_keys_cap(int64_t k) {
    if (k > kSelectMaxK) return 0;
    int cap = 64;
    while (cap < 2 * k) cap <<= 1;
    return cap;
}

static hipError_t launch_select_pass(const SelectKeysArgs &a, int64_t blocks, hipStream_t st) {
    void (*fn)(SelectKeysArgs) = !a.off && a.seglen <= kSelRegKeys * kSelThreads ? select_keys_kernel<true>
                                                                       : select_keys_kernel<false>;
    const size_t lds = (size_t)a.cap * 8 + kSelBins * 4;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)fn,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(kSelThreads), lds, st, a);
    return hipGetLastError();
}

// Segments per query: one workgroup reads a segment at a few tens of GB/s,
// so a few queries over many rows are cut into segments of at least 32,768
// keys (and 8 k) whose k best a second pass merges.
int select_keys_segments(int64_t nq, int64_t n, int64_t k, int num_cu) {
    const int64_t by_cu = std::max<int64_t>(1, 2 * (int64_t)num_cu / std::max<int64_t>(1, nq));
    const int64_t by_len = n / std::max<int64_t>(32768, 8 * k);
    // (one workgroup counts its segment's keys in 32 bits)
    const int64_t need = (n + ((int64_t)1 << 30) - 1) >> 30;
    return (int)std::max<int64_t>(need, std::max<int64_t>(1, std::min<int64_t>({by_cu, by_len, 64})));
}

hipError_t launch_select_keys(const uint64_t *keys, int64_t nq, int64_t n, int64_t kstride,
                              int64_t k, int metric, int nseg, uint64_t *part, float *D, int32_t *I,
                              const uint32_t *rowflags, int64_t nflags, uint32_t *hflags,
                              hipStream_t st) {
    if (nq <= 0) return hipSuccess;
    const int cap = select_keys_cap(k);
    if (!cap || k < 1 || nseg < 1 || nq * nseg > INT32_MAX || (nseg > 1 && !part))
        return hipErrorInvalidValue;
    SelectKeysArgs a{};
    a.keys = keys;
    a.n = n;
    a.kstride = kstride;
    a.k = k;
    a.cap = cap;
    a.metric = metric;
    if (nseg > 1) {
        SelectKeysArgs p = a;
        p.seglen = (n + nseg - 1) / nseg;
        p.nseg = nseg;
        p.outk = part;
        if (hipError_t e = launch_select_pass(p, nq * nseg, st)) return e;
        a.keys = part;
        a.n = a.kstride = (int64_t)nseg * k;
    }
    a.seglen = a.n;
    a.nseg = 1;
    a.D = D;
    a.I = I;
    a.rowflags = rowflags;
    a.nflags = nflags;
    a.hflags = hflags;
    return launch_select_pass(a, nq, st);
}

hipError_t launch_select_groups(const uint64_t *keys, const int32_t *off, const int32_t *cnt,
                                int64_t nq, int64_t k, int metric, float *D, int32_t *I,
                                uint32_t *flags, hipStream_t st) {
    if (nq <= 0) return hipSuccess;
    const int cap = select_keys_cap(k);
    if (!cap || k < 1 || nq > INT32_MAX || !off || !cnt) return hipErrorInvalidValue;
    SelectKeysArgs a{};
    a.keys = keys;
    a.k = k;
    a.cap = cap;
    a.metric = metric;
    a.nseg = 1;
    a.off = off;
    a.cnt = cnt;
    a.short_flag = flags;
    a.D = D;
    a.I = I;
    return launch_select_pass(a, nq, st);
}

__global__ __launch_bounds__(256) void count_pairs_kernel(const int32_t *__restrict__ cq, int64_t m,
                                                          int64_t nq, int32_t *__restrict__ cnt) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= m) return;
    const int32_t q = cq[t];
    if (q >= 0 && q < nq) atomicAdd(&cnt[q], 1);
}

hipError_t launch_count_pairs(const int32_t *cq, int64_t m, int64_t nq, int32_t *cnt,
                              hipStream_t st) {
    if (m <= 0) return hipSuccess;
    count_pairs_kernel<<<dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st>>>(cq, m, nq, cnt);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Exact scores of (query, row) pairs in any order.  A lane sums one pair in
// dimension order; a wave's 64 rows and 64 query rows come through LDS in
// 32-element chunks, eight lanes reading 128 contiguous bytes of each, with
// the next chunk's loads in flight while one is summed.  (A lane reading its
// own row touches 64 cache lines per load.)  One wave per workgroup: waves
// share nothing, and 18 KB of LDS leave eight on a CU.
// ---------------------------------------------------------------------------
constexpr int kPairK = 32, kPairLd = kPairK + 4;

template <int ST, int METRIC, typename Done>
__device__ __forceinline__ void exact_pairs_wave(const void *xb, int64_t ld, int64_t d,
                                                 const float *qf, const int32_t *cq,
                                                 const int32_t *ci, int64_t m, int64_t nq,
                                                 int64_t n, uint32_t *flags, Done &&done) {
    __shared__ __align__(16) float xs[64][kPairLd];
    __shared__ __align__(16) float qs[64][kPairLd];
    __shared__ int s_q[64], s_id[64];
    const int lane = threadIdx.x;
    const int64_t t = (int64_t)blockIdx.x * 64 + lane;
    bool ok = t < m;
    int32_t q = ok ? cq[t] : 0, id = ok ? ci[t] : 0;
    if (ok && (q < 0 || q >= nq || id < 0 || id >= n)) {
        atomicOr(flags, kFlagBadId);
        ok = false;
        q = id = 0;
    }
    s_q[lane] = q;
    s_id[lane] = id;
    __syncthreads();
    // rows: pieces of 16 bytes; queries: rows of d floats without alignment,
    // so element by element where d is not a multiple of four
    constexpr int PE = ST == 1 ? 8 : 4, TPR = kPairK / PE, NPR = 64 * TPR / 64;
    u32x4_t xr[NPR];
    float4 qr[8];
    const bool q4 = (d & 3) == 0;
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < NPR; ++i) {
            const int r = i * (64 / TPR) + lane / TPR, c = (lane % TPR) * PE;
            const int64_t e = (int64_t)s_id[r] * ld + k0 + c;
            xr[i] = *(const u32x4_t *)((const char *)xb + e * (ST == 1 ? 2 : 4));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = i * 8 + lane / 8;
            const int64_t j = k0 + (lane % 8) * 4;
            const float *p = qf + (int64_t)s_q[r] * d + j;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q4) {
                if (j < d) v = *(const float4 *)p;
            } else {
                if (j < d) v.x = p[0];
                if (j + 1 < d) v.y = p[1];
                if (j + 2 < d) v.z = p[2];
                if (j + 3 < d) v.w = p[3];
            }
            qr[i] = v;
        }
    };
    double s = 0.0;
    load(0);
    for (int64_t k0 = 0; k0 < d; k0 += kPairK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NPR; ++i) {
            const int r = i * (64 / TPR) + lane / TPR, c = (lane % TPR) * PE;
            const u32x4_t p = xr[i];
            if constexpr (ST == 1) {
                const u32x4_t lo = {p.x << 16, p.x & 0xFFFF0000u, p.y << 16, p.y & 0xFFFF0000u};
                const u32x4_t hi = {p.z << 16, p.z & 0xFFFF0000u, p.w << 16, p.w & 0xFFFF0000u};
                *(u32x4_t *)&xs[r][c] = lo;
                *(u32x4_t *)&xs[r][c + 4] = hi;
            } else {
                *(u32x4_t *)&xs[r][c] = p;
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) *(float4 *)&qs[i * 8 + lane / 8][(lane % 8) * 4] = qr[i];
        __syncthreads();
        if (k0 + kPairK < d) load(k0 + kPairK);
        // (elements past d are zero on both sides: their terms add +0)
#pragma unroll
        for (int j = 0; j < kPairK; j += 4) {
            const float4 xv = *(const float4 *)&xs[lane][j], qv = *(const float4 *)&qs[lane][j];
            const float xa[4] = {xv.x, xv.y, xv.z, xv.w}, qa[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if constexpr (METRIC == 0) {
                    const double diff = (double)qa[c] - (double)xa[c];
                    s = s + diff * diff;
                } else {
                    s = __builtin_fma((double)qa[c], (double)xa[c], s);
                }
            }
        }
    }
    if (t < m) done(t, q, id, ok, s);
}

template <int ST, int METRIC>
__global__ __launch_bounds__(64) void exact_pair_keys_kernel(
    const void *xb, int64_t ld, int64_t d, const float *qf, const int32_t *cq, const int32_t *ci,
    int64_t m, int64_t nq, int64_t n, const int32_t *off, int32_t *fill, uint64_t *keys,
    uint32_t *flags) {
    exact_pairs_wave<ST, METRIC>(
        xb, ld, d, qf, cq, ci, m, nq, n, flags,
        [&](int64_t, int32_t q, int32_t id, bool ok, double s) {
            if (!ok) return;
            const float key = METRIC == 0 ? (float)s : -(float)s;
            keys[(int64_t)off[q] + atomicAdd(&fill[q], 1)] =
                ((uint64_t)enc_order(key) << 32) | (uint32_t)id;
        });
}

hipError_t launch_exact_pair_keys(const void *xb, int storage, int64_t ld, int64_t d, int metric,
                                  const float *qf, const int32_t *cq, const int32_t *ci, int64_t m,
                                  int64_t nq, int64_t n, const int32_t *off, int32_t *fill,
                                  uint64_t *keys, uint32_t *flags, hipStream_t st) {
    if (m <= 0) return hipSuccess;
    if ((m + 63) / 64 > INT32_MAX) return hipErrorInvalidValue;
    auto fn = storage == 1 ? (metric == 0 ? exact_pair_keys_kernel<1, 0> : exact_pair_keys_kernel<1, 1>)
                           : (metric == 0 ? exact_pair_keys_kernel<0, 0> : exact_pair_keys_kernel<0, 1>);
    hipLaunchKernelGGL(fn, dim3((unsigned)((m + 63) / 64)), dim3(64), 0, st, xb, ld, d, qf, cq, ci,
                       m, nq, n, off, fill, keys, flags);
    return hipGetLastError();
}

// Range candidates: score, sort key and test of each pair.
template <int ST, int METRIC>
__global__ __launch_bounds__(64) void range_keys_kernel(
    const void *xb, int64_t ld, int64_t d, const float *qf, const int32_t *cq, const int32_t *ci,
    int64_t m, double radius, int idbits, uint64_t *keys, float *score, unsigned long long *kept,
    int64_t n, int64_t nq, uint32_t *flags) {
    exact_pairs_wave<ST, METRIC>(
        xb, ld, d, qf, cq, ci, m, nq, n, flags,
        [&](int64_t t, int32_t q, int32_t id, bool ok, double s) {
            const bool hit = ok && (METRIC == 0 ? s <= radius : s >= radius);
            keys[t] = hit ? (uint64_t)q << idbits | (uint32_t)id : ~0ull;
            score[t] = (float)s;
            const uint64_t hits = __ballot(hit);
            if (hits && (int)threadIdx.x == __builtin_ctzll(hits))
                atomicAdd(kept, (unsigned long long)__builtin_popcountll(hits));
        });
}

hipError_t launch_range_keys(const void *xb, int storage, int64_t ld, int64_t d, int metric,
                             const float *qf, const int32_t *cq, const int32_t *ci, int64_t m,
                             double radius, int idbits, uint64_t *keys, float *score,
                             unsigned long long *kept, int64_t n, int64_t nq, uint32_t *flags,
                             hipStream_t st) {
    if (m <= 0) return hipSuccess;
    if ((m + 63) / 64 > INT32_MAX) return hipErrorInvalidValue;
    auto fn = storage == 1 ? (metric == 0 ? range_keys_kernel<1, 0> : range_keys_kernel<1, 1>)
                           : (metric == 0 ? range_keys_kernel<0, 0> : range_keys_kernel<0, 1>);
    hipLaunchKernelGGL(fn, dim3((unsigned)((m + 63) / 64)), dim3(64), 0, st, xb, ld, d, qf, cq, ci,
                       m, radius, idbits, keys, score, kept, n, nq, flags);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void range_unpack_kernel(const uint64_t *__restrict__ sorted,
                                                           int64_t m, int idbits,
                                                           int32_t *__restrict__ q,
                                                           int32_t *__restrict__ id, int64_t nlims,
                                                           int64_t *__restrict__ lims) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < m) {
        const uint64_t k = sorted[t];
        q[t] = (int32_t)(k >> idbits);
        id[t] = (int32_t)(k & (((uint64_t)1 << idbits) - 1));
    }
    if (t < nlims) {  // the first key of query t or a later one
        const uint64_t key = (uint64_t)t << idbits;
        int64_t lo = 0, hi = m;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (sorted[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        lims[t] = lo;
    }
}

hipError_t launch_range_unpack(const uint64_t *sorted, int64_t m, int idbits, int32_t *q,
                               int32_t *id, int64_t nlims, int64_t *lims, hipStream_t st) {
    const int64_t t = std::max(m, nlims);
    if (t <= 0) return hipSuccess;
    range_unpack_kernel<<<dim3((unsigned)((t + 255) / 256)), dim3(256), 0, st>>>(sorted, m, idbits,
                                                                               q, id, nlims, lims);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Exact keys of row subsets: pair p = (query p / nseg, segment p % nseg) names
// the rows ids[seg_off[p] .. + seg_len[p]); its keys go to keys[koff[p] ..).
// A workgroup takes `group` pairs: each wave takes 64 rows at a time through
// its own LDS buffer in 32-element chunks (eight lanes read 128 contiguous
// bytes of a row, the next chunk in flight), a lane sums one row, and the
// queries' values come through scalar loads as in exact_tile_kernel.
//
// Bound by the row reads from L2 (one pair at a time: 7.8 TB/s), so `perm`
// (or null) walks the pairs in the order of their segments, each XCD a
// contiguous part of it, and four pairs of one segment (an inverted list that
// many queries probe) share each row read.  1,000 queries x 16 of 256 lists of
// 200,000 x 128 rows, 5.2e7 rows in all: one thread per row 4.2 ms, one pair
// at a time 3.3 ms, four 2.2 ms.
// ---------------------------------------------------------------------------
struct SubsetKArgs {
    const void *xb;
    int64_t ld, d, ldd, n;
    const double *qd;
    const int32_t *ids;
    const int64_t *seg_off, *seg_len, *koff;
    const int32_t *perm;
    int64_t nseg, npairs;
    int group;
    uint64_t *keys;
    uint32_t *flags;
};
constexpr int kSubsetGroup = 4;

// The keys of QT pairs of one segment.
template <int ST, int METRIC, int QT>
__device__ __forceinline__ void subset_keys_run(const SubsetKArgs &a, const int64_t *pair,
                                                float (*xs)[kPairLd], int wave, int lane) {
    const int64_t len = a.seg_len[pair[0]], i0 = a.seg_off[pair[0]];
    const_f64_t q[QT];
    uint64_t *out[QT];
#pragma unroll
    for (int u = 0; u < QT; ++u) {
        q[u] = (const_f64_t)(uintptr_t)(a.qd + pair[u] / a.nseg * a.ldd);
        out[u] = a.keys + a.koff[pair[u]];
    }
    constexpr int PE = ST == 1 ? 8 : 4, TPR = kPairK / PE, NPR = TPR;
    for (int64_t base = wave * 64; base < len; base += 256) {
        const bool in = base + lane < len;
        int32_t id = in ? a.ids[i0 + base + lane] : 0;
        bool ok = in;
        if (id < 0 || id >= a.n) {
            atomicOr(a.flags, kFlagBadId);
            ok = false;
            id = 0;
        }
        u32x4_t xr[NPR];
        auto load = [&](int64_t k0) {
#pragma unroll
            for (int i = 0; i < NPR; ++i) {
                const int r = i * (64 / TPR) + lane / TPR;
                const int64_t e = (int64_t)__shfl(id, r) * a.ld + k0 + (lane % TPR) * PE;
                xr[i] = *(const u32x4_t *)((const char *)a.xb + e * (ST == 1 ? 2 : 4));
            }
        };
        double s[QT];
#pragma unroll
        for (int u = 0; u < QT; ++u) s[u] = 0.0;
        load(0);
        for (int64_t k0 = 0; k0 < a.d; k0 += kPairK) {
            lds_wave_sync();
#pragma unroll
            for (int i = 0; i < NPR; ++i) {
                float *dst = &xs[i * (64 / TPR) + lane / TPR][(lane % TPR) * PE];
                const u32x4_t v = xr[i];
                if constexpr (ST == 1) {
                    *(u32x4_t *)dst = u32x4_t{v.x << 16, v.x & 0xFFFF0000u, v.y << 16, v.y & 0xFFFF0000u};
                    *(u32x4_t *)(dst + 4) = u32x4_t{v.z << 16, v.z & 0xFFFF0000u, v.w << 16, v.w & 0xFFFF0000u};
                } else {
                    *(u32x4_t *)dst = v;
                }
            }
            lds_wave_sync();
            if (k0 + kPairK < a.d) load(k0 + kPairK);
            // (elements past d are zero on both sides: their terms add +0)
#pragma unroll 2
            for (int j = 0; j < kPairK; j += 4) {
                const float4 x4 = *(const float4 *)&xs[lane][j];
                const double x[4] = {(double)x4.x, (double)x4.y, (double)x4.z, (double)x4.w};
#pragma unroll
                for (int u = 0; u < QT; ++u) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const double qv = q[u][k0 + j + c];
                        if constexpr (METRIC == 0) {
                            const double diff = qv - x[c];
                            s[u] = s[u] + diff * diff;
                        } else {
                            s[u] = __builtin_fma(qv, x[c], s[u]);
                        }
                    }
                }
            }
        }
        if (in) {
#pragma unroll
            for (int u = 0; u < QT; ++u) {
                const float key = METRIC == 0 ? (float)s[u] : -(float)s[u];
                out[u][base + lane] = ok ? ((uint64_t)enc_order(key) << 32) | (uint32_t)id : kNoKey;
            }
        }
    }
}

template <int ST, int METRIC>
__global__ __launch_bounds__(256) void subset_keys_kernel(SubsetKArgs a) {
    __shared__ __align__(16) float xsh[4][64][kPairLd];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t groups = (a.npairs + a.group - 1) / a.group, per = (groups + 7) / 8;
    const int64_t w = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int64_t)(blockIdx.x >> 3) >= per || w >= groups) return;
    const int64_t p0 = w * a.group, np = min((int64_t)a.group, a.npairs - p0);
    int64_t pair[kSubsetGroup];
    bool same = np == kSubsetGroup;
    for (int u = 0; u < kSubsetGroup; ++u) {
        const int64_t t = p0 + min((int64_t)u, np - 1);
        pair[u] = a.perm ? (int64_t)a.perm[t] : t;
        same = same && a.seg_off[pair[u]] == a.seg_off[pair[0]] &&
               a.seg_len[pair[u]] == a.seg_len[pair[0]];
    }
    if (same) {
        subset_keys_run<ST, METRIC, kSubsetGroup>(a, pair, xsh[wave], wave, lane);
    } else {
        for (int u = 0; u < np; ++u) subset_keys_run<ST, METRIC, 1>(a, pair + u, xsh[wave], wave, lane);
    }
}

hipError_t launch_subset_keys(const void *xb, int storage, int64_t ld, int64_t d, int metric,
                              const double *qd, int64_t nq, int64_t n, const int32_t *ids,
                              const int64_t *seg_off, const int64_t *seg_len, const int64_t *koff,
                              const int32_t *perm, int64_t nseg, uint64_t *keys, uint32_t *flags,
                              hipStream_t st) {
    if (nq <= 0 || nseg <= 0) return hipSuccess;
    SubsetKArgs a{xb,   ld,   d,    exact_ldd(d), n,    qd,   ids, seg_off, seg_len, koff,
                  perm, nseg, nq * nseg, perm ? kSubsetGroup : 1, keys, flags};
    const int64_t groups = (a.npairs + a.group - 1) / a.group, grid = (groups + 7) / 8 * 8;
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    auto fn = storage == 1 ? (metric == 0 ? subset_keys_kernel<1, 0> : subset_keys_kernel<1, 1>)
                           : (metric == 0 ? subset_keys_kernel<0, 0> : subset_keys_kernel<0, 1>);
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace vs
