// Contiguous causal GQA attention on the matrix cores: self_attention for
// head dims d == dv of 64 or 128 (self_attention.hip has the general kernel,
// the formula and the dispatch).
//
// A "column" is a (query, query head of the kv head) pair, query-major:
// column c = query c / G, head c % G of the group, so the G heads that share
// a kv head share its K and V. A workgroup of WC x WK waves takes one kv
// head's tile of 16 CT WC columns; in every stage of 32 KU WK keys, wave
// (wc, wk) takes columns 16 CT wc .. and the stage's keys 32 KU wk ..:
//   S^T[32 keys x 16 cols] = K . Q^T   (accumulator: lane's column, keys 4 grp + i)
//   O^T[D x 16 cols] += V^T . P^T      (the accumulator's keys are the B operand's)
// so nothing but the running max crosses lanes, and the WK partial states of
// a column meet in LDS once, after the last stage.
//
// Bound: for prompts the MFMAs (a third of them the weights' low halves) and
// the softmax beside them, 41 % and 55 % of a busy CU's time at 4096 x 4096;
// for single tokens latency. A wave per (query, head) in plain FMAs, the
// kernel that took every shape before, walked K and V again for every query
// and head: 488 us (6 TFLOP/s) for 1000 x 1000, 12:2 heads of 128 in bf16,
// against 18.5 us now (166 TFLOP/s); 777 x 777 324 -> 14 us, one f32 token
// against 513 keys 12.8 -> 9.9 us.
//
// K and V stages go to LDS as rows by buffer_load ... lds (16 B a lane; rows
// past S come back as zeros), piece p of row r at slot p ^ key(r), so that
// the fragment reads hit every bank evenly: K as 16 B pieces of 16 rows, V
// of 16-bit types by ds_read_b64_tr_b16, which hands each lane 4 keys of its
// own dim, V of f32 as 16 B pieces (4 dims of a key; the dim blocks of the
// product are then every fourth dim).
//
// 32-bit weights: P enters the 16-bit product as hi + lo (two MFMAs), f32
// runs on the f32 MFMA. Two halves hold a weight to 2^-17 or better as long
// as neither leaves the type's range: always for bf16; f16 takes weights
// below 2^-15 of a column's largest in passes of their own, scaled up (a
// weight below 2^-25 is nothing in f16, and thousands of them can outweigh
// the rest where their values are large). What that takes where no weight is
// small: 1000 x 1000 19.5 -> 20.4 us, 512 x 1536 17.4 -> 19.2.
//
// The f32 MFMAs add their four products to one running sum, so a long chain
// of them rounds as often as it is long. The scores take four chains and the
// values a fresh one every stage: error against 64 bits (2-norm) at 512 x 1536
// 5.2e-7 -> 2.2e-7, 1 x 513 4.2e-7 -> 2.2e-7 (4.3e-7 and 4.0e-7 by plain FMAs),
// for 65.1 us instead of 60.5 and 10.0 instead of 9.7.
//
// A weight of zero times a non-finite V is NaN, and a column must not see
// keys past its own; nor may the lazy max's larger weights overflow a sum. A
// tile whose result is not finite is worked out again with weights of at most
// one: rows of V that hold a huge value are zeros to the MFMAs and go to the
// columns that see them in plain FMAs, and only the columns in question are
// written. An inf in the first of 1000 x 1000 keys: 46 us (those columns one
// by one over their keys: 670, and the general kernel 490); 1 x 513: 21 us
// (92, and 15).
#include "lanes.hpp"
#include "launch.hpp"
#include "self_attention.hpp"

#include "../device/hip_check.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

namespace llaisys::kernels {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr uint32_t kRsrcWord3 = 0x00020000u; // raw buffer, 32-bit dwords (gfx9 family)

struct AttnArgs {
    void *out;
    const void *q, *k, *v;
    float *part;
    int L, S, nh, nkvh, G, NS;
    float scale_log2;
};

template <typename T> struct Piece; // 16-bit types: 8 elements of 16 B
template <> struct Piece<__bf16> {
    typedef bf16x8 type;
    __device__ __forceinline__ static f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Piece<_Float16> {
    typedef f16x8 type;
    __device__ __forceinline__ static f32x4 mfma(f16x8 a, f16x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// Rows of PPR 16 B pieces in LDS: piece p of row r at slot p ^ rowKey(r).
// 16 rows of one piece (a K read) and 16 rows of a piece pair (a V read)
// then spread evenly over the banks.
template <int PPR> __device__ __forceinline__ int rowKey(int r) { return PPR >= 16 ? r & 15 : (r >> 1) & (PPR - 1); }

// Four dim blocks of V: at[i] and NEXT bytes on (the second 16 keys). As
// assembly with its wait: before the builtin of this read the compiler waits
// for every LDS load in flight, the next stage's among them.
template <int NEXT> __device__ __forceinline__ void readV4(u32x2 (&w)[8], const uint32_t (&at)[4]) {
    asm volatile("ds_read_b64_tr_b16 %0, %8\n\t"
                 "ds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %2, %9\n\t"
                 "ds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %4, %10\n\t"
                 "ds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %6, %11\n\t"
                 "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]),
                   "=&v"(w[7])
                 : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(NEXT));
}

__device__ __forceinline__ bool finite(float x) { return __builtin_fabsf(x) <= 3.402823466e38f; }

// Whether a 16 B piece of V holds a value whose products could leave the range
// of the sums: inf, NaN, and of the types with f32's exponents 2^100 and more.
template <typename T> __device__ __forceinline__ bool holdsHuge(const u32x4 &w) {
    bool huge = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (sizeof(T) == 4) {
            huge |= (w[e] & 0x7fffffffu) >= 0x71800000u;
        } else {
            constexpr uint32_t kFrom = std::is_same<T, _Float16>::value ? 0x7c00u : 0x7180u;
            huge |= (w[e] & 0x7fffu) >= kFrom || ((w[e] >> 16) & 0x7fffu) >= kFrom;
        }
    }
    return huge;
}

template <typename T, int D, int CT, int WC, int WK, int KU>
__global__ void __launch_bounds__(64 * WC * WK) selfAttentionMfmaKernel(AttnArgs a) {
    constexpr int ES = sizeof(T), NW = WC * WK;
    constexpr bool F32 = ES == 4, F16 = std::is_same<T, _Float16>::value;
    constexpr int PPR = D * ES / 16;        // 16 B pieces of a row
    constexpr int KW = 32 * KU;             // keys of a wave and stage
    constexpr int KS = KW * WK;             // keys of a stage
    constexpr int COLS = 16 * CT * WC;      // columns of the workgroup
    constexpr int RPI = 64 / PPR;           // rows per load instruction
    constexpr bool PRIV = WC == 1;          // the waves share no keys
    constexpr int STAGE = 2 * KS * PPR;     // pieces of a stage: K rows, V rows
    constexpr int OP = D + 4;               // pitch of a column of partial O
    static_assert(KW % RPI == 0 && (PRIV || KS % (RPI * NW) == 0), "every wave issues the same loads");
    extern __shared__ u32x4 lds[]; // NB stages; afterwards the waves' partial states
    __shared__ int bad[COLS];

    int lane = threadIdx.x & 63, n = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wc = wave % WC, wk = wave / WC;
    // Tiles from the last (most keys) to the first; neighbouring workgroups
    // take different kv heads, so an XCD's L2 holds few of them.
    const int cols = a.L * a.G;
    const int kh = int(blockIdx.x) % a.nkvh, rest = int(blockIdx.x) / a.nkvh;
    const int z = rest % a.NS;
    const int tile = (cols + COLS - 1) / COLS - 1 - rest / a.NS;
    const int col0 = tile * COLS;
    const int shift = a.S - a.L; // query i sees keys <= i + shift
    const int keys = min(cols - 1, col0 + COLS - 1) / a.G + shift + 1;
    const int stages = (keys + KS - 1) / KS;
    const int s0 = z * stages / a.NS, s1 = (z + 1) * stages / a.NS;

    // The wave's columns and what they may see.
    const int cw = col0 + wc * CT * 16;
    int limit[CT];
    int lim_lo = -1, lim_hi = -1; // over the wave's columns
    if (cw < cols) {
        lim_lo = cw / a.G + shift;
        lim_hi = min(cols - 1, cw + CT * 16 - 1) / a.G + shift;
    }
    const T *qp = static_cast<const T *>(a.q);
    u32x4 qop[CT][F32 ? D / 16 : D / 32];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c = cw + ct * 16 + n;
        const bool ok = c < cols;
        const int cc = ok ? c : cols - 1, qi = cc / a.G;
        limit[ct] = ok ? qi + shift : -1;
        const T *qr = qp + (size_t(qi) * a.nh + kh * a.G + (cc - qi * a.G)) * D + grp * (16 / ES);
#pragma unroll
        for (int s = 0; s < (F32 ? D / 16 : D / 32); ++s)
            qop[ct][s] = *reinterpret_cast<const u32x4 *>(qr + s * (64 / ES));
    }

    const uint32_t row_bytes = uint32_t(a.nkvh) * D * ES;
    const __amdgpu_buffer_rsrc_t kr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.k), (short)0, int(a.S * row_bytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t vr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.v), (short)0, int(a.S * row_bytes), kRsrcWord3);
    // K (V) rows of a stage to dst: the load instructions first, first +
    // step, ... < KS / RPI, RPI rows each.
    auto load = [&](const __amdgpu_buffer_rsrc_t &rsrc, u32x4 *dst, int stage, int first, auto step, auto count) {
#pragma unroll
        for (int b = 0; b < decltype(count)::value; ++b) {
            const int blk = first + decltype(step)::value * b, r = blk * RPI + lane / PPR;
            const uint32_t off = uint32_t(stage * KS + r) * row_bytes + kh * (D * ES) +
                                 16 * ((lane % PPR) ^ rowKey<PPR>(r));
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void *)(dst + blk * 64), 16, int(off), 0, 0, 0);
        }
    };

    // O^T blocks: 16-bit, block i: dims 16 i + 4 grp + e; f32, block
    // 4 b + j: dims 64 b + 16 grp + 4 e + j.
    f32x4 acc[CT][D / 16];
    float m[CT], l[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        m[ct] = -INFINITY;
        l[ct] = 0.f;
#pragma unroll
        for (int i = 0; i < D / 16; ++i) acc[ct][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // S^T of the wave's keys from LDS, those a column may not see at -inf.
    auto scores = [&](const u32x4 *ks, int key0, f32x4 (&sc)[2 * KU][CT]) {
        constexpr int CH = F32 ? 4 : 1; // chains of a sum
        f32x4 part[CH][2 * KU][CT];
#pragma unroll
        for (int e = 0; e < CH; ++e)
#pragma unroll
            for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) part[e][kt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < (F32 ? D / 16 : D / 32); ++s) {
            u32x4 kf[2 * KU];
#pragma unroll
            for (int kt = 0; kt < 2 * KU; ++kt) kf[kt] = ks[(kt * 16 + n) * PPR + ((4 * s + grp) ^ rowKey<PPR>(n))];
            if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct)
                            part[e][kt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                __uint_as_float(kf[kt][e]), __uint_as_float(qop[ct][s][e]), part[e][kt][ct], 0, 0, 0);
            } else {
                using P = Piece<T>;
#pragma unroll
                for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        part[0][kt][ct] = P::mfma(__builtin_bit_cast(typename P::type, kf[kt]),
                                                  __builtin_bit_cast(typename P::type, qop[ct][s]), part[0][kt][ct]);
            }
        }
#pragma unroll
        for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                sc[kt][ct] = part[0][kt][ct];
                if constexpr (F32) sc[kt][ct] = (sc[kt][ct] + part[1][kt][ct]) + (part[2][kt][ct] + part[3][kt][ct]);
            }
        if (key0 + KW - 1 > lim_lo) {
#pragma unroll
            for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        sc[kt][ct][i] = key0 + kt * 16 + 4 * grp + i <= limit[ct] ? sc[kt][ct][i] : -INFINITY;
        }
    };
    // The scores' weights in their place: online softmax in base 2, per
    // column. The running max moves (and O and l are rescaled) only when a column's
    // scores exceed it by more than 2^lazy; the normalised result is the same. f16:
    // 2^7 higher, weights up to 2^15, which leaves the type's range to the small ones.
    constexpr float kLazy = 8.f, kUp = F16 ? 7.f : 0.f;
    auto softmax = [&](f32x4 (&sc)[2 * KU][CT], float lazy) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float mx = sc[0][ct][0];
#pragma unroll
            for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[kt][ct][i]);
            mx = maxOverGroups(mx) * a.scale_log2 - kUp; // (the scale is positive)
            const float m_true = fmaxf(m[ct], mx);
            if (__builtin_amdgcn_ballot_w64(m_true > m[ct] + lazy) != 0) {
                const float alpha = __builtin_amdgcn_exp2f(m[ct] - (m_true == -INFINITY ? 0.f : m_true));
                l[ct] *= alpha;
#pragma unroll
                for (int i = 0; i < D / 16; ++i) acc[ct][i] *= alpha;
                m[ct] = m_true;
            }
            const float mu = m[ct] == -INFINITY ? 0.f : m[ct];
            float sum = 0.f;
#pragma unroll
            for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sc[kt][ct][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kt][ct][i], a.scale_log2, -mu));
                    sum += sc[kt][ct][i];
                }
            l[ct] += sum;
        }
    };
    auto addValues = [&](const u32x4 *vs, const f32x4 (&sc)[2 * KU][CT]) {
        if constexpr (F32) {
#pragma unroll
            for (int b = 0; b < D / 64; ++b) {
                f32x4 sum[4][CT];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) sum[j][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = kt * 16 + 4 * grp + i;
                        const u32x4 vf = vs[r * PPR + ((16 * b + n) ^ rowKey<PPR>(r))];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int ct = 0; ct < CT; ++ct)
                                sum[j][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vf[j]), sc[kt][ct][i],
                                                                                  sum[j][ct], 0, 0, 0);
                    }
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) acc[ct][4 * b + j] += sum[j][ct];
            }
        } else {
            using P = Piece<T>;
            const int r = 4 * grp + (n >> 2); // the lane's row of a 16-key V read
            const uint32_t vbase = uint32_t(uintptr_t((lds_void *)vs)) + 16 * PPR * r + 8 * (n & 1);
            const int half = (n >> 1) & 1;
            // One pass: the weights that are at least kSmall when scaled by `up`
            // (a power of two; bf16: all of them); whether a lane has smaller ones.
            constexpr float kSmall = 0x1p-8f, kStep = 0x1p23f;
            auto pass = [&](auto first, float up) {
                constexpr bool FIRST = decltype(first)::value;
                bool rest = false;
#pragma unroll
                for (int u = 0; u < KU; ++u) {
                    typename P::type hi[CT], lo[CT];
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            float p = sc[2 * u + (e >> 2)][ct][e & 3];
                            if constexpr (F16) {
                                if (!FIRST) p = p * up < kSmall * kStep ? p * up : 0.f;
                                rest |= p > 0.f && p < kSmall;
                                p = p < kSmall ? 0.f : p;
                            }
                            hi[ct][e] = T(p);
                            lo[ct][e] = T(p - float(hi[ct][e]));
                        }
#pragma unroll
                    for (int i0 = 0; i0 < D / 16; i0 += 4) {
                        uint32_t at[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            at[i] = vbase + u * 32 * PPR * 16 + 16 * ((2 * (i0 + i) + half) ^ rowKey<PPR>(r));
                        u32x2 w[8];
                        readV4<16 * PPR * 16>(w, at);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const auto vf = __builtin_bit_cast(
                                typename P::type, u32x4{w[2 * i][0], w[2 * i][1], w[2 * i + 1][0], w[2 * i + 1][1]});
#pragma unroll
                            for (int ct = 0; ct < CT; ++ct) {
                                f32x4 &o = acc[ct][i0 + i];
                                if constexpr (FIRST)
                                    o = P::mfma(vf, lo[ct], P::mfma(vf, hi[ct], o));
                                else
                                    o += P::mfma(vf, lo[ct], P::mfma(vf, hi[ct], f32x4{0.f, 0.f, 0.f, 0.f})) * (1.f / up);
                            }
                        }
                    }
                }
                return __builtin_amdgcn_ballot_w64(rest) != 0;
            };
            bool rest = pass(std::true_type(), 1.f);
            if constexpr (F16)
                for (float up = kStep; rest && up < INFINITY; up *= kStep) rest = pass(std::false_type(), up);
        }
    };

    // The scores, weights and values of stages [s0, s1).
    auto run = [&]() {
        if constexpr (PRIV) {
            // One column group: a wave shares its keys with no other, so each runs
            // its own pair of buffers without barriers: the next keys' K is on its
            // way while the weights and the values of these are worked out, their
            // V during the next scores. (Past the end rows of zeros, or unused.)
            u32x4 *kb = lds + 2 * wave * KW * PPR, *vb = kb + KW * PPR;
            constexpr int LW = KW / RPI;
            const std::integral_constant<int, 1> one;
            const std::integral_constant<int, LW> lw;
            auto issue = [&](const __amdgpu_buffer_rsrc_t &rsrc, u32x4 *dst, int st) {
                load(rsrc, dst - wk * KW * PPR, st, wk * LW, one, lw);
            };
            const int n_st = min(s1, lim_hi < wk * KW ? 0 : (lim_hi - wk * KW) / KS + 1); // the wave's last stage + 1
            if (s0 < n_st) {
                issue(kr, kb, s0);
                issue(vr, vb, s0);
            }
            for (int st = s0; st < n_st; ++st) {
                f32x4 sc[2 * KU][CT];
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LW) : "memory");
                scores(kb, st * KS + wk * KW, sc);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                issue(kr, kb, st + 1);
                softmax(sc, kLazy);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LW) : "memory");
                addValues(vb, sc);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                issue(vr, vb, st + 1);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {
            const std::integral_constant<int, NW> step;
            const std::integral_constant<int, KS / RPI / NW> count;
            auto issue = [&](int st, int buf) {
                load(kr, lds + buf * STAGE, st, wave, step, count);
                load(vr, lds + buf * STAGE + KS * PPR, st, wave, step, count);
            };
            if (s0 < s1) issue(s0, 0);
            for (int st = s0; st < s1; ++st) {
                const int buf = (st - s0) & 1;
                // This stage has landed, and everyone has read the one whose buffer the next takes.
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (st + 1 < s1) issue(st + 1, buf ^ 1);
                const int key0 = st * KS + wk * KW;
                if (key0 > lim_hi) continue; // none of the wave's columns sees these keys
                const u32x4 *ks = lds + buf * STAGE + wk * KW * PPR;
                f32x4 sc[2 * KU][CT];
                scores(ks, key0, sc);
                softmax(sc, kLazy);
                addValues(ks + KS * PPR, sc);
            }
        }
    };
    // The same with one buffer, weights of at most one and the huge rows apart.
    auto runAgain = [&]() {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            m[ct] = -INFINITY;
            l[ct] = 0.f;
#pragma unroll
            for (int i = 0; i < D / 16; ++i) acc[ct][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const std::integral_constant<int, NW> step;
        const std::integral_constant<int, KS / RPI / NW> count;
        const u32x4 *ks = lds + wk * KW * PPR;
        u32x4 *vs = lds + (KS + wk * KW) * PPR;
        for (int st = s0; st < s1; ++st) {
            __syncthreads(); // everyone has read the stage before
            load(kr, lds, st, wave, step, count);
            load(vr, lds + KS * PPR, st, wave, step, count);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            uint64_t huge = 0; // of the wave's keys
            for (int b = 0; b < KW / RPI; ++b) {
                const uint64_t pieces = __builtin_amdgcn_ballot_w64(holdsHuge<T>(vs[b * 64 + lane]));
                for (int r = 0; r < RPI; ++r)
                    if ((pieces >> (r * PPR)) & ((1ull << PPR) - 1)) huge |= 1ull << (b * RPI + r);
            }
            __syncthreads(); // (the waves of other columns share these rows)
            for (int b = 0; b < KW / RPI; ++b)
                if ((huge >> (b * RPI + lane / PPR)) & 1) vs[b * 64 + lane] = u32x4{0, 0, 0, 0};
            __syncthreads();
            const int key0 = st * KS + wk * KW;
            if (key0 > lim_hi) continue;
            f32x4 sc[2 * KU][CT];
            scores(ks, key0, sc);
            softmax(sc, 0.f);
            addValues(vs, sc);
            for (; huge; huge &= huge - 1) {
                const int j = __builtin_ctzll(huge), key = key0 + j;
                const T *vrow = static_cast<const T *>(a.v) + (size_t(key) * a.nkvh + kh) * D;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    // Key 16 kt + 4 g + i of the wave's is element i of lane group g.
                    float p = 0.f;
#pragma unroll
                    for (int kt = 0; kt < 2 * KU; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (j / 16 == kt && j % 4 == i) p = sc[kt][ct][i];
                    p = __shfl(p, (j / 4 % 4) * 16 + n);
#pragma unroll
                    for (int i = 0; i < D / 16; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int dim = F32 ? 64 * (i / 4) + 16 * grp + 4 * e + i % 4 : 16 * i + 4 * grp + e;
                            const float sum = fmaf(p, float(vrow[dim]), acc[ct][i][e]);
                            acc[ct][i][e] = key <= limit[ct] ? sum : acc[ct][i][e];
                            asm volatile("" ::: "memory"); // (a load at a time: registers)
                        }
                }
            }
        }
    };

    // The waves' states to the results; AGAIN: of the columns in bad, else
    // filling bad. Whether some column is.
    auto finish = [&](auto second) {
        constexpr bool AGAIN = decltype(second)::value;
        // The waves' states into LDS (every stage has been read), column-major.
        float *po = reinterpret_cast<float *>(lds), *pml = po + NW * CT * 16 * OP;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const float lt = sumOverGroups(l[ct]);
            const int c = (wave * CT + ct) * 16 + n;
            if (grp == 0) *reinterpret_cast<f32x2 *>(pml + 2 * c) = f32x2{m[ct], lt};
#pragma unroll
            for (int i = 0; i < D / 16; ++i) {
                if constexpr (F32) {
                    const int b = i / 4, e = i % 4;
                    *reinterpret_cast<f32x4 *>(po + c * OP + 64 * b + 16 * grp + 4 * e) =
                        f32x4{acc[ct][4 * b][e], acc[ct][4 * b + 1][e], acc[ct][4 * b + 2][e], acc[ct][4 * b + 3][e]};
                } else {
                    *reinterpret_cast<f32x4 *>(po + c * OP + 16 * i + 4 * grp) = acc[ct][i];
                }
            }
        }
        if (!AGAIN)
            for (int c = threadIdx.x; c < COLS; c += 64 * NW) bad[c] = 0;
        __syncthreads();
        // Column c's WK states are those of waves wc + WC k; 4 dims a thread.
        auto put = [&](int c, int d0, f32x4 o, float M, float Ls) {
            const int cc = col0 + c, qi = cc / a.G;
            const size_t row = size_t(qi) * a.nh + kh * a.G + (cc - qi * a.G);
            if (a.NS > 1) {
                float *rec = a.part + (row * a.NS + z) * (D + 2);
                if (d0 == 0) *reinterpret_cast<f32x2 *>(rec) = f32x2{M, Ls};
                *reinterpret_cast<f32x2 *>(rec + 2 + d0) = f32x2{o[0], o[1]};
                *reinterpret_cast<f32x2 *>(rec + 4 + d0) = f32x2{o[2], o[3]};
                return;
            }
            typedef T t4 __attribute__((ext_vector_type(4)));
            const float inv = 1.f / Ls;
            *reinterpret_cast<t4 *>(static_cast<T *>(a.out) + row * D + d0) =
                t4{T(o[0] * inv), T(o[1] * inv), T(o[2] * inv), T(o[3] * inv)};
        };
        int any_bad = 0;
        for (int i = threadIdx.x; i < COLS * (D / 4); i += 64 * NW) {
            const int c = i / (D / 4), d0 = 4 * (i % (D / 4));
            if (col0 + c >= cols) break;
            if (AGAIN && !bad[c]) continue;
            const int w0 = c / (CT * 16), cl = c % (CT * 16);
            float M = -INFINITY;
#pragma unroll
            for (int k = 0; k < WK; ++k) M = fmaxf(M, pml[2 * ((w0 + WC * k) * CT * 16 + cl)]);
            float Ls = 0.f;
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
            const float Mu = M == -INFINITY ? 0.f : M; // no key of this split seen: weights 0
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const int x = (w0 + WC * k) * CT * 16 + cl;
                const float w = __builtin_amdgcn_exp2f(pml[2 * x] - Mu);
                Ls += pml[2 * x + 1] * w;
                o += *reinterpret_cast<const f32x4 *>(po + x * OP + d0) * w;
            }
            const bool fine = finite(o[0]) && finite(o[1]) && finite(o[2]) && finite(o[3]) && finite(Ls);
            if (!AGAIN && !fine) {
                bad[c] = 1;
                any_bad = 1;
            }
            put(c, d0, o, M, Ls);
        }
        return !AGAIN && __syncthreads_or(any_bad) != 0;
    };

    run();
    if (!finish(std::false_type())) return;
    // (Addresses worked out from here on, not kept from before: registers.)
    asm volatile("" : "+v"(lane), "+v"(n), "+v"(grp));
    runAgain();
    finish(std::true_type());
}

template <typename T, int D, int CT, int WC, int WK, int KU>
void launchMfma(const AttnArgs &a, hipStream_t s) {
    constexpr int COLS = 16 * CT * WC, NW = WC * WK;
    constexpr size_t stage = size_t(WC > 1 ? 2 : 1) * 2 * 32 * KU * WK * D * sizeof(T);
    constexpr size_t merge = size_t(NW) * CT * 16 * (D + 6) * sizeof(float);
    constexpr size_t lds = stage > merge ? stage : merge;
    static_assert(lds + COLS * sizeof(int) <= 160 * 1024, "one workgroup's LDS");
    auto *kernel = selfAttentionMfmaKernel<T, D, CT, WC, WK, KU>;
    // More than 64 KB of LDS has to be asked for, once per device.
    static std::mutex mu;
    static std::vector<bool> raised;
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lock(mu);
        if (size_t(dev) >= raised.size()) raised.resize(dev + 1, false);
        if (!raised[dev]) {
            HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
            raised[dev] = true;
        }
    }
    const unsigned tiles = unsigned((size_t(a.L) * a.G + COLS - 1) / COLS);
    hipLaunchKernelGGL(kernel, dim3(tiles * unsigned(a.NS) * unsigned(a.nkvh)), dim3(64 * NW), lds, s, a);
    HIP_CHECK(hipGetLastError());
}

// Workgroup shapes: columns of a tile, keys of a stage.
struct Shape {
    int cols, keys;
};
constexpr Shape kShapes16[] = {{16, 256}, {32, 256}, {64, 128}, {128, 128}};
constexpr Shape kShapes32[] = {{16, 128}, {32, 128}};

template <typename T, int D> void launchShape(int shape, const AttnArgs &a, hipStream_t s) {
    if constexpr (sizeof(T) == 4) {
        switch (shape) {
        case 0: return launchMfma<T, D, 1, 1, 4, 1>(a, s);
        default: return launchMfma<T, D, 2, 1, 4, 1>(a, s);
        }
    } else {
        switch (shape) {
        case 0: return launchMfma<T, D, 1, 1, 8, 1>(a, s);
        case 1: return launchMfma<T, D, 2, 1, 8, 1>(a, s);
        case 2: return launchMfma<T, D, 2, 2, 4, 1>(a, s);
        default: return launchMfma<T, D, 2, 4, 2, 2>(a, s);
        }
    }
}

} // namespace

bool selfAttentionMfmaTakes(ElemType type, int L, int S, int nkvh, int d, int dv, float scale) {
    const size_t es = type == ElemType::F32 ? 4 : 2;
    // (32-bit buffer offsets; a masked score times the scale has to stay -inf)
    return d == dv && (d == 64 || d == 128) && scale > 0.f && scale < INFINITY &&
           (size_t(S) + 256) * nkvh * d * es < (size_t(1) << 31) && L > 0;
}

// Tiles of 16 columns while they fit the CUs in one round, then the widest
// that gives every CU about two or fewer: the narrow ones finish sooner, the
// wide ones read K and V less often. 16-bit, 12:2 heads of 128, by tile of
// 16 / 32 / 64 / 128 columns (us):
//   q x keys      200 x 1000   512 x 1536   1000 x 1000   2048 x 2048   4096 x 4096
//   16               9.8          19.9         20.3          53.7          174
//   32              13.0          16.2         18.4          43.7          126
//   64              16.7          26.8         21.3          37.7          123
//   128             19.8          28.8         29.7          52.3          107
// f32 (rate of its MFMA, a 16th): 16 / 32 columns 13.4 / 20.7 us at 300 x
// 300, 51.6 / 45.1 at 1000 x 1000; wider tiles were slower everywhere.
// Key splits cost a merge launch, 2.5 us, three stages of the 16-bit kernel:
// 1 x 1000 keys (4 stages) 8.3 us whole and 8.5 split, 1 x 2000 9.9 us in
// four splits and 8.6 in eight.
// An f32 stage takes longer: 1 x 513 (5 stages) 9.9 us in five, 11.9 in four.
SelfAttentionPlan planSelfAttentionMfma(ElemType type, int L, int S, int nh, int nkvh, int cus) {
    const bool f32 = type == ElemType::F32;
    const Shape *shapes = f32 ? kShapes32 : kShapes16;
    const int n_shapes = f32 ? 2 : 4;
    const long cols = long(L) * (nh / nkvh);
    auto groups = [&](int s) { return (cols + shapes[s].cols - 1) / shapes[s].cols * nkvh; };
    SelfAttentionPlan p{0, 1};
    if (groups(0) > cus)
        for (p.shape = 1; p.shape < n_shapes - 1 && groups(p.shape) > 2L * cus;) ++p.shape;
    const int stages = (S + shapes[p.shape].keys - 1) / shapes[p.shape].keys;
    const long most = std::min<long>(kSelfAttentionMaxSplits, cus / groups(p.shape));
    if (stages > (f32 ? 2 : 4)) p.splits = int(std::max<long>(1, std::min<long>(stages, most)));
    return p;
}

void selfAttentionMfma(void *out, const void *q, const void *k, const void *v, ElemType type, int L, int S, int nh,
                       int nkvh, int d, float scale, const SelfAttentionPlan &plan, float *part, void *stream) {
    AttnArgs a;
    a.out = out;
    a.q = q;
    a.k = k;
    a.v = v;
    a.part = part;
    a.L = L;
    a.S = S;
    a.nh = nh;
    a.nkvh = nkvh;
    a.G = nh / nkvh;
    a.NS = plan.splits;
    a.scale_log2 = scale * 1.4426950408889634f;
    auto s = static_cast<hipStream_t>(stream);
    auto byDim = [&](auto zero) {
        using T = decltype(zero);
        if (d == 64)
            launchShape<T, 64>(plan.shape, a, s);
        else
            launchShape<T, 128>(plan.shape, a, s);
    };
    switch (type) {
    case ElemType::F32: return byDim(float(0));
    case ElemType::F16: return byDim(_Float16(0));
    case ElemType::BF16: return byDim(__bf16(0));
    }
}

} // namespace llaisys::kernels
