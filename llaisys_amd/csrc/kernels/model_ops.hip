// Elementwise / normalisation / indexing kernels of the reference's model ops
// (README.md:157-292; formulas test/ops/{add,argmax,embedding,rms_norm,rope,
// swiglu}.py), for the Qwen2 decode step built on the paged KV path. All math
// is fp32; results are rounded once to the tensor dtype.
#include "launch.hpp"
#include "step_common.hpp"

#include "../device/hip_check.hpp"

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <initializer_list>

namespace llaisys::kernels {

namespace {

template <typename T> __device__ __forceinline__ float ld(const T *p, size_t i);
template <> __device__ __forceinline__ float ld<float>(const float *p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float ld<__half>(const __half *p, size_t i) { return __half2float(p[i]); }
template <> __device__ __forceinline__ float ld<__hip_bfloat16>(const __hip_bfloat16 *p, size_t i) {
    return __bfloat162float(p[i]);
}
template <typename T> __device__ __forceinline__ void st(T *p, size_t i, float v);
template <> __device__ __forceinline__ void st<float>(float *p, size_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void st<__half>(__half *p, size_t i, float v) { p[i] = __float2half_rn(v); }
template <> __device__ __forceinline__ void st<__hip_bfloat16>(__hip_bfloat16 *p, size_t i, float v) {
    p[i] = __float2bfloat16(v);
}

constexpr int kThreads = 256;

// 16 B of a tensor as floats.
template <typename T> struct Vec {
    static constexpr int N = 16 / sizeof(T);
    float f[N];
    __device__ __forceinline__ void load(const T *p) { widen(*reinterpret_cast<const uint4 *>(p)); }
    __device__ __forceinline__ void widen(const uint4 &w) {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            if constexpr (sizeof(T) == 4) {
                f[e] = __uint_as_float((&w.x)[e]);
            } else {
                const uint16_t h = uint16_t((&w.x)[e >> 1] >> ((e & 1) * 16));
                f[e] = ld(reinterpret_cast<const T *>(&h), 0);
            }
        }
    }
    __device__ __forceinline__ void store(T *p) const {
        uint4 w;
        T *t = reinterpret_cast<T *>(&w);
#pragma unroll
        for (int e = 0; e < N; ++e) st(t, e, f[e]);
        *reinterpret_cast<uint4 *>(p) = w;
    }
};

__device__ __forceinline__ float addOf(float a, float b) { return a + b; }
// up * gate / (1 + exp(-gate))
__device__ __forceinline__ float swigluOf(float gate, float up) { return up * gate / (1.f + expf(-gate)); }

// out[i] = F(a[i], b[i]): 16 B a thread and operand where all three are 16 B
// aligned (VEC), the last n % (elements of 16 B) one by one. HBM bytes bound
// it; element by element the loads were 2 B a lane: swiglu of 777 x 8960 bf16
// (42 MB) 12.4 -> 8.2 us, of 8192 x 8960 128 -> 75 us (5.9 TB/s).
template <typename T, bool VEC, float (*F)(float, float)>
__global__ void __launch_bounds__(kThreads) binaryKernel(T *out, const T *a, const T *b, size_t n) {
    const size_t t = blockIdx.x * size_t(kThreads) + threadIdx.x, step = size_t(gridDim.x) * kThreads;
    size_t done = 0;
    if constexpr (VEC) {
        constexpr int N = Vec<T>::N;
        done = n / N * N;
        for (size_t i = t * N; i < done; i += step * N) {
            Vec<T> x, y;
            x.load(a + i);
            y.load(b + i);
#pragma unroll
            for (int e = 0; e < N; ++e) x.f[e] = F(x.f[e], y.f[e]);
            x.store(out + i);
        }
    }
    for (size_t i = done + t; i < n; i += step) st(out, i, F(ld(a, i), ld(b, i)));
}

// out[r, c] = x[r, c] + bias[c]
template <typename T> __global__ void biasKernel(T *x, const T *bias, size_t rows, size_t cols) {
    const size_t n = rows * cols;
    for (size_t i = blockIdx.x * size_t(kThreads) + threadIdx.x; i < n; i += size_t(gridDim.x) * kThreads)
        st(x, i, ld(x, i) + ld(bias, i % cols));
}

template <typename T> __global__ void fillRowsKernel(T *x, const T *row, size_t rows, size_t cols) {
    const size_t n = rows * cols;
    for (size_t i = blockIdx.x * size_t(kThreads) + threadIdx.x; i < n; i += size_t(gridDim.x) * kThreads)
        x[i] = row[i % cols];
}

__device__ float blockSum(float v, float *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.f;
    for (int w = 0; w < kThreads / 64; ++w) s += red[w];
    __syncthreads();
    return s;
}

// One block per row: y = x * w / sqrt(mean(x^2) + eps); 16 B pieces (VEC)
// where d is whole pieces and the tensors are aligned.
template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads) rmsNormKernel(T *out, const T *x, const T *w, int d, float eps) {
    __shared__ float red[kThreads / 64];
    const size_t row = blockIdx.x;
    constexpr int N = VEC ? Vec<T>::N : 1;
    float ss = 0.f;
    for (int c = threadIdx.x * N; c < d; c += kThreads * N) {
        if constexpr (VEC) {
            Vec<T> v;
            v.load(x + row * d + c);
#pragma unroll
            for (int e = 0; e < N; ++e) ss += v.f[e] * v.f[e];
        } else {
            const float v = ld(x, row * d + c);
            ss += v * v;
        }
    }
    const float inv = rsqrtf(blockSum(ss, red) / float(d) + eps);
    for (int c = threadIdx.x * N; c < d; c += kThreads * N) {
        if constexpr (VEC) {
            Vec<T> v, g;
            v.load(x + row * d + c);
            g.load(w + c);
#pragma unroll
            for (int e = 0; e < N; ++e) v.f[e] = v.f[e] * inv * g.f[e];
            v.store(out + row * d + c);
        } else {
            st(out, row * d + c, ld(x, row * d + c) * inv * ld(w, c));
        }
    }
}

// The same for rows of whole 16 B pieces, at most 64 NV of them: a wave per
// row, which stays in registers between the sum and the result (w is on its
// way beside it), and no barrier. 8192 rows of 1536 bf16: 9.9 -> 8.6 us.
template <typename T, int NV>
__global__ void __launch_bounds__(kThreads) rmsNormRowKernel(T *out, const T *x, const T *w, size_t rows, int d, float eps) {
    const size_t row = blockIdx.x * size_t(kThreads / 64) + (threadIdx.x >> 6);
    if (row >= rows) return;
    constexpr int N = Vec<T>::N;
    const int lane = threadIdx.x & 63, nv = d / N;
    // Every piece is requested at once: lanes past the row's end repeat its
    // last piece, which then counts for nothing (a load under a condition
    // would be waited for before the next).
    uint4 v[NV], g[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = reinterpret_cast<const uint4 *>(x + row * d)[min(lane + 64 * i, nv - 1)];
#pragma unroll
    for (int i = 0; i < NV; ++i) g[i] = reinterpret_cast<const uint4 *>(w)[min(lane + 64 * i, nv - 1)];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        Vec<T> a;
        a.widen(v[i]);
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < N; ++e) sum += a.f[e] * a.f[e];
        ss += lane + 64 * i < nv ? sum : 0.f;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float inv = rsqrtf(ss / float(d) + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        Vec<T> a, b;
        a.widen(v[i]);
        b.widen(g[i]);
#pragma unroll
        for (int e = 0; e < N; ++e) a.f[e] = a.f[e] * inv * b.f[e];
        if (lane + 64 * i < nv) a.store(out + row * d + size_t(lane + 64 * i) * N);
    }
}

// Rotate halves: for j < d/2, phi = pos / theta^(2j/d) computed in fp32 as the
// reference formula does; a' = a cos - b sin, b' = b cos + a sin.
// The block's token has one angle per j, whatever the head. kShared: they are
// worked out once (powf, a division and sincosf each) and shared through LDS;
// kPieces: and the rows move in 16 B pieces, where half a head is whole pieces
// and the tensors are aligned. 4096 tokens x 12 heads of 128 bf16: 19.7 -> 6.6
// us. kOwn: every element works its own out, the shorter way where no more than
// one wave has something to do or one head shares with none (us, kOwn / kPieces:
// 5000 tokens x 2 heads of 16 3.9 / 5.1, 3000 x 1 of 256 4.4 / 4.7; 4096 x 2 of
// 128 5.3 / 4.7), and for heads too large for the LDS.
constexpr int kRopeHalf = 512; // angles kept in LDS
enum RopeMode { kOwn, kShared, kPieces };

__device__ __forceinline__ float2 ropeAngle(float p, int j, int d, float theta) {
    float s, c;
    sincosf(p / powf(theta, float(2 * j) / float(d)), &s, &c);
    return make_float2(s, c);
}

template <typename T, RopeMode MODE>
__global__ void __launch_bounds__(kThreads) ropeKernel(T *out, const T *in, const int64_t *pos, int nhead, int d, float theta) {
    __shared__ float2 trig[MODE == kOwn ? 1 : kRopeHalf];
    constexpr bool VEC = MODE == kPieces;
    const size_t tok = blockIdx.x;
    const int half = d / 2;
    const float p = float(pos[tok]);
    if constexpr (MODE != kOwn) {
        for (int j = threadIdx.x; j < half; j += kThreads) trig[j] = ropeAngle(p, j, d, theta);
        __syncthreads();
    }
    constexpr int N = VEC ? Vec<T>::N : 1;
    const int pieces = half / N;
    for (int t = threadIdx.x; t < nhead * pieces; t += kThreads) {
        const int h = t / pieces, j = (t - h * pieces) * N;
        const size_t base = (tok * nhead + h) * size_t(d) + j;
        if constexpr (VEC) {
            Vec<T> a, b, ra, rb;
            a.load(in + base);
            b.load(in + base + half);
#pragma unroll
            for (int e = 0; e < N; ++e) {
                const float2 sc = trig[j + e];
                ra.f[e] = a.f[e] * sc.y - b.f[e] * sc.x;
                rb.f[e] = b.f[e] * sc.y + a.f[e] * sc.x;
            }
            ra.store(out + base);
            rb.store(out + base + half);
        } else {
            const float2 sc = MODE == kShared ? trig[j] : ropeAngle(p, j, d, theta);
            const float a = ld(in, base), b = ld(in, base + half);
            st(out, base, a * sc.y - b * sc.x);
            st(out, base + half, b * sc.y + a * sc.x);
        }
    }
}

template <typename T>
__global__ void embeddingKernel(T *out, const int64_t *idx, const T *weight, int64_t vocab, int d, int *err) {
    const size_t r = blockIdx.x;
    const int64_t i = idx[r];
    if (i < 0 || i >= vocab) {
        if (threadIdx.x == 0) atomicOr(err, 4);
        return;
    }
    for (int c = threadIdx.x; c < d; c += kThreads) out[r * d + c] = weight[size_t(i) * d + c];
}

// argmax over the last dim, split over columns: stage 1 reduces chunks of
// kArgmaxChunk columns of one row to a 64-bit key, stage 2 reduces a row's
// chunk keys. key = order-preserving bits of the value (NaN above +inf, as
// torch.max propagates NaN) << 32 | ~column, so the maximum key is the
// largest value at its first column.
constexpr int kArgmaxChunk = 4096;


__device__ __forceinline__ uint64_t waveMax(uint64_t k) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint64_t o = __shfl_xor(k, off);
        k = o > k ? o : k;
    }
    return k;
}

// grid (chunks, rows): keys[row * chunks + chunk]. vec: 2-byte values, n % 8
// == 0 and a 16 B aligned base, read as 16 B vectors (8 columns) per load.
template <typename T>
__global__ void __launch_bounds__(kThreads) argmaxChunkKernel(uint64_t *keys, const T *vals, int64_t n, int chunks,
                                                              int vec) {
    __shared__ uint64_t red[kThreads / 64];
    const size_t row = blockIdx.y;
    const int64_t c0 = int64_t(blockIdx.x) * kArgmaxChunk;
    const int64_t c1 = min(n, c0 + kArgmaxChunk);
    uint64_t best = 0;
    if (vec) {
        const uint4 *v = reinterpret_cast<const uint4 *>(vals + row * n);
        for (int64_t c = c0 + 8 * threadIdx.x; c < c1; c += 8 * kThreads) {
            const uint4 u = v[c / 8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint16_t bits = uint16_t((&u.x)[e >> 1] >> ((e & 1) * 16));
                const uint64_t k = argmaxKey(ld(reinterpret_cast<const T *>(&bits), 0), c + e);
                best = k > best ? k : best;
            }
        }
    } else {
        for (int64_t c = c0 + threadIdx.x; c < c1; c += kThreads) {
            const uint64_t k = argmaxKey(ld(vals, row * n + c), c);
            best = k > best ? k : best;
        }
    }
    best = waveMax(best);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) best = red[w] > best ? red[w] : best;
        keys[row * chunks + blockIdx.x] = best;
    }
}

// one wave per row
template <typename T>
__global__ void __launch_bounds__(64) argmaxFinishKernel(int64_t *idx, T *val, const uint64_t *keys, const T *vals,
                                                        int64_t n, int chunks) {
    const size_t row = blockIdx.x;
    uint64_t best = 0;
    for (int c = threadIdx.x; c < chunks; c += 64) best = keys[row * chunks + c] > best ? keys[row * chunks + c] : best;
    best = waveMax(best);
    if (threadIdx.x == 0) {
        const int64_t col = int64_t(~uint32_t(best & 0xffffffffu));
        idx[row] = col;
        if (val) val[row] = vals[row * n + col];
    }
}

// Strided copy of equal-shaped tensors (up to kMaxDims dims), element size esz.
struct StridedDesc {
    int ndim;
    int64_t shape[kMaxDims];
    int64_t out_stride[kMaxDims];
    int64_t in_stride[kMaxDims];
};

template <typename E> __global__ void rearrangeKernel(E *out, const E *in, StridedDesc d, size_t n) {
    for (size_t i = blockIdx.x * size_t(kThreads) + threadIdx.x; i < n; i += size_t(gridDim.x) * kThreads) {
        size_t rem = i;
        int64_t oo = 0, io = 0;
        for (int k = d.ndim - 1; k >= 0; --k) {
            const int64_t c = int64_t(rem % size_t(d.shape[k]));
            rem /= size_t(d.shape[k]);
            oo += c * d.out_stride[k];
            io += c * d.in_stride[k];
        }
        out[oo] = in[io];
    }
}

unsigned gridFor(size_t n) { return unsigned(std::min<size_t>((n + kThreads - 1) / kThreads, 65536)); }

template <template <typename> class F, typename... Args> void byType(ElemType t, Args &&...args) {
    switch (t) {
    case ElemType::F32: return F<float>::run(args...);
    case ElemType::F16: return F<__half>::run(args...);
    case ElemType::BF16: return F<__hip_bfloat16>::run(args...);
    }
}

bool aligned16(std::initializer_list<const void *> ps) {
    uintptr_t all = 0;
    for (const void *p : ps) all |= reinterpret_cast<uintptr_t>(p);
    return all % 16 == 0;
}

template <typename T, float (*F)(float, float)>
void launchBinary(void *o, const void *a, const void *b, size_t n, hipStream_t s) {
    if (!n) return;
    if (aligned16({o, a, b})) {
        const size_t pieces = (n + Vec<T>::N - 1) / Vec<T>::N;
        hipLaunchKernelGGL((binaryKernel<T, true, F>), dim3(gridFor(pieces)), dim3(kThreads), 0, s, (T *)o, (const T *)a, (const T *)b, n);
    } else {
        hipLaunchKernelGGL((binaryKernel<T, false, F>), dim3(gridFor(n)), dim3(kThreads), 0, s, (T *)o, (const T *)a, (const T *)b, n);
    }
}
template <typename T> struct AddL {
    static void run(void *c, const void *a, const void *b, size_t n, hipStream_t s) { launchBinary<T, addOf>(c, a, b, n, s); }
};
template <typename T> struct SwigluL {
    static void run(void *o, const void *g, const void *u, size_t n, hipStream_t s) { launchBinary<T, swigluOf>(o, g, u, n, s); }
};
template <typename T> struct BiasL {
    static void run(void *x, const void *b, size_t rows, size_t cols, hipStream_t s) {
        if (rows * cols)
            hipLaunchKernelGGL(biasKernel<T>, dim3(gridFor(rows * cols)), dim3(kThreads), 0, s, (T *)x, (const T *)b, rows, cols);
    }
};
template <typename T> struct FillRowsL {
    static void run(void *x, const void *r, size_t rows, size_t cols, hipStream_t s) {
        if (rows * cols)
            hipLaunchKernelGGL(fillRowsKernel<T>, dim3(gridFor(rows * cols)), dim3(kThreads), 0, s, (T *)x, (const T *)r, rows, cols);
    }
};
template <typename T> struct RmsL {
    static void run(void *o, const void *x, const void *w, size_t rows, int d, float eps, hipStream_t s) {
        if (!rows) return;
        constexpr int N = Vec<T>::N;
        const bool vec = d % N == 0 && aligned16({o, x, w});
        const dim3 grid(unsigned((rows + kThreads / 64 - 1) / (kThreads / 64)));
        // A block per row spreads few rows over more waves: 2048 x 4096 in 16 bits
        // 5.4 us and 5.9 with a wave per row, 1025 x 4096 4.1 and 4.2; rows past
        // four pieces a lane need more of them (2100 x 4096 6.1 / 6.8, 3000 8.7 /
        // 8.6, 4096 11.9 / 11.0) than shorter ones (3000 x 1536 4.8 / 4.4).
        const bool many = rows > (d <= 64 * 4 * N ? 2048 : 3072);
        if (many && vec && d <= 64 * 4 * N)
            hipLaunchKernelGGL((rmsNormRowKernel<T, 4>), grid, dim3(kThreads), 0, s, (T *)o, (const T *)x, (const T *)w, rows, d, eps);
        else if (many && vec && d <= 64 * 8 * N)
            hipLaunchKernelGGL((rmsNormRowKernel<T, 8>), grid, dim3(kThreads), 0, s, (T *)o, (const T *)x, (const T *)w, rows, d, eps);
        else if (vec)
            hipLaunchKernelGGL((rmsNormKernel<T, true>), dim3(rows), dim3(kThreads), 0, s, (T *)o, (const T *)x, (const T *)w, d, eps);
        else
            hipLaunchKernelGGL((rmsNormKernel<T, false>), dim3(rows), dim3(kThreads), 0, s, (T *)o, (const T *)x, (const T *)w, d, eps);
    }
};
template <typename T> struct RopeL {
    static void run(void *o, const void *x, const int64_t *pos, size_t ntok, int nhead, int d, float theta, hipStream_t s) {
        if (!ntok) return;
        const int half = d / 2;
        if (half > kRopeHalf || nhead == 1 || nhead * half <= 64)
            hipLaunchKernelGGL((ropeKernel<T, kOwn>), dim3(ntok), dim3(kThreads), 0, s, (T *)o, (const T *)x, pos, nhead, d, theta);
        else if (half % Vec<T>::N == 0 && aligned16({o, x}))
            hipLaunchKernelGGL((ropeKernel<T, kPieces>), dim3(ntok), dim3(kThreads), 0, s, (T *)o, (const T *)x, pos, nhead, d, theta);
        else
            hipLaunchKernelGGL((ropeKernel<T, kShared>), dim3(ntok), dim3(kThreads), 0, s, (T *)o, (const T *)x, pos, nhead, d, theta);
    }
};
template <typename T> struct EmbL {
    static void run(void *o, const int64_t *idx, const void *w, size_t rows, int64_t vocab, int d, int *err, hipStream_t s) {
        if (rows) hipLaunchKernelGGL(embeddingKernel<T>, dim3(rows), dim3(kThreads), 0, s, (T *)o, idx, (const T *)w, vocab, d, err);
    }
};
template <typename T> struct ArgmaxL {
    static void run(int64_t *idx, void *val, const void *vals, size_t rows, int64_t n, uint64_t *keys, hipStream_t s) {
        if (!rows) return;
        const int chunks = int((n + kArgmaxChunk - 1) / kArgmaxChunk);
        const int vec = sizeof(T) == 2 && n % 8 == 0 && reinterpret_cast<uintptr_t>(vals) % 16 == 0;
        hipLaunchKernelGGL(argmaxChunkKernel<T>, dim3(chunks, unsigned(rows)), dim3(kThreads), 0, s, keys, (const T *)vals, n,
                           chunks, vec);
        hipLaunchKernelGGL(argmaxFinishKernel<T>, dim3(unsigned(rows)), dim3(64), 0, s, idx, (T *)val, keys, (const T *)vals, n, chunks);
    }
};

} // namespace

void add(void *c, const void *a, const void *b, ElemType t, size_t n, void *stream) {
    byType<AddL>(t, c, a, b, n, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void swiglu(void *out, const void *gate, const void *up, ElemType t, size_t n, void *stream) {
    byType<SwigluL>(t, out, gate, up, n, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void addBias(void *x, const void *bias, ElemType t, size_t rows, size_t cols, void *stream) {
    byType<BiasL>(t, x, bias, rows, cols, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void fillRows(void *x, const void *row, ElemType t, size_t rows, size_t cols, void *stream) {
    byType<FillRowsL>(t, x, row, rows, cols, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void rmsNorm(void *out, const void *x, const void *w, ElemType t, size_t rows, int d, float eps, void *stream) {
    byType<RmsL>(t, out, x, w, rows, d, eps, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void rope(void *out, const void *in, const int64_t *pos, ElemType t, size_t ntok, int nhead, int d, float theta,
          void *stream) {
    byType<RopeL>(t, out, in, pos, ntok, nhead, d, theta, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void embedding(void *out, const int64_t *idx, const void *weight, ElemType t, size_t rows, int64_t vocab, int d,
               int *err, void *stream) {
    byType<EmbL>(t, out, idx, weight, rows, vocab, d, err, static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void argmaxFinishKeys(int64_t *idx, const uint64_t *keys, size_t rows, int chunks, void *stream) {
    if (!rows) return;
    hipLaunchKernelGGL(argmaxFinishKernel<__hip_bfloat16>, dim3(unsigned(rows)), dim3(64), 0,
                       static_cast<hipStream_t>(stream), idx, nullptr, keys, nullptr, int64_t(0), chunks);
    HIP_CHECK(hipGetLastError());
}

size_t argmaxWorkspaceBytes(size_t rows, int64_t n) {
    return rows * size_t((n + kArgmaxChunk - 1) / kArgmaxChunk) * sizeof(uint64_t);
}
void argmax(int64_t *idx, void *val, const void *vals, ElemType t, size_t rows, int64_t n, void *workspace,
            void *stream) {
    byType<ArgmaxL>(t, idx, val, vals, rows, n, static_cast<uint64_t *>(workspace), static_cast<hipStream_t>(stream));
    HIP_CHECK(hipGetLastError());
}
void rearrange(void *out, const void *in, size_t esz, int ndim, const int64_t *shape, const int64_t *out_strides,
               const int64_t *in_strides, void *stream) {
    LLAISYS_CHECK(ndim >= 0 && ndim <= kMaxDims, "rearrange: at most " << kMaxDims << " dims");
    StridedDesc d{};
    d.ndim = ndim;
    size_t n = 1;
    for (int k = 0; k < ndim; ++k) {
        d.shape[k] = shape[k];
        d.out_stride[k] = out_strides[k];
        d.in_stride[k] = in_strides[k];
        n *= size_t(shape[k]);
    }
    if (!n) return;
    auto s = static_cast<hipStream_t>(stream);
    switch (esz) {
    case 1: hipLaunchKernelGGL(rearrangeKernel<uint8_t>, dim3(gridFor(n)), dim3(kThreads), 0, s, (uint8_t *)out, (const uint8_t *)in, d, n); break;
    case 2: hipLaunchKernelGGL(rearrangeKernel<uint16_t>, dim3(gridFor(n)), dim3(kThreads), 0, s, (uint16_t *)out, (const uint16_t *)in, d, n); break;
    case 4: hipLaunchKernelGGL(rearrangeKernel<uint32_t>, dim3(gridFor(n)), dim3(kThreads), 0, s, (uint32_t *)out, (const uint32_t *)in, d, n); break;
    case 8: hipLaunchKernelGGL(rearrangeKernel<uint64_t>, dim3(gridFor(n)), dim3(kThreads), 0, s, (uint64_t *)out, (const uint64_t *)in, d, n); break;
    default: LLAISYS_RAISE("rearrange: element size " << esz << " not supported");
    }
    HIP_CHECK(hipGetLastError());
}

} // namespace llaisys::kernels
