// Shared device helpers for the gfx950 multiprecision kernels.
//
// Multiword integers are read through small accessor functors `src(i) -> u32 word i` so the same
// streaming routines serve limb planes in HBM, per-thread words in LDS and values being
// reconstructed. Every routine runs over a run-time word count: no per-L template instances.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/sdpvibe_hip.h"

typedef uint32_t u32;
typedef uint64_t u64;
typedef int64_t i64;
typedef int32_t i32;
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

#define EZV (-(1LL << 40))

// Dynamic LDS of a kernel (the host emulator in tests/emu supplies its own definition).
#ifndef SDPV_DYNAMIC_LDS
#define SDPV_DYNAMIC_LDS(type, name) extern __shared__ __align__(16) type name[]
#endif
// 16 bytes per lane from global memory straight into LDS at ldsbase + 16 * lane (gfx950 direct
// load; ldsbase uniform across the wave), and a wait until at most n vector-memory operations of
// this wave are outstanding (s_waitcnt immediate: vmcnt split over bits 3:0 and 15:14).
#ifndef SDPV_LDS_DMA16
#define SDPV_LDS_DMA16(gptr, ldsbase)                                                            \
    __builtin_amdgcn_global_load_lds((const void*)(gptr),                                        \
                                     (__attribute__((address_space(3))) void*)(ldsbase), 16, 0, 0)
#define SDPV_WAIT_VMCNT(n) \
    __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14))
#endif
// Four multiply-adds into 96-bit accumulators acc + ov 2^64: v_mad_u64_u32 with its carry out taken by one
// addition (the compiler forms the product with a zero addend and adds it in 64 bits twice). The four
// multiplies go first, so that three instructions lie between a carry's write and its read (a VALU read of
// an SGPR that a VALU wrote needs two wait states). CHAIN4: four terms a[u] b[u] of one sum; COLS4: one
// factor x times y[u] into four sums; MAC96: one term alone. The sums are early clobbers: the first multiply
// writes a sum while later ones still read their factors, and a factor equal to a sum's start value (zero, or
// half of it) would otherwise get its register. SETTLE(v, w): the wait states that a lane move of v or w needs
// after such a block (the compiler does not see the block's instructions).
#ifndef SDPV_MAC96_CHAIN4
#define SDPV_MAC96_CHAIN4(acc, ov, a, b)                                                          \
    do {                                                                                          \
        u64 m0_, m1_, m2_, m3_;                                                                   \
        asm("v_mad_u64_u32 %0, %2, %6, %10, %0\n\tv_mad_u64_u32 %0, %3, %7, %11, %0\n\t"          \
            "v_mad_u64_u32 %0, %4, %8, %12, %0\n\tv_mad_u64_u32 %0, %5, %9, %13, %0\n\t"          \
            "v_addc_co_u32 %1, %2, 0, %1, %2\n\tv_addc_co_u32 %1, %3, 0, %1, %3\n\t"              \
            "v_addc_co_u32 %1, %4, 0, %1, %4\n\tv_addc_co_u32 %1, %5, 0, %1, %5"                  \
            : "+&v"(acc), "+&v"(ov), "=&s"(m0_), "=&s"(m1_), "=&s"(m2_), "=&s"(m3_)               \
            : "v"((a)[0]), "v"((a)[1]), "v"((a)[2]), "v"((a)[3]), "v"((b)[0]), "v"((b)[1]),       \
              "v"((b)[2]), "v"((b)[3]));                                                          \
    } while (0)
#define SDPV_MAC96_COLS4(acc, ov, x, y)                                                           \
    do {                                                                                          \
        u64 m0_, m1_, m2_, m3_;                                                                   \
        asm("v_mad_u64_u32 %0, %8, %12, %13, %0\n\tv_mad_u64_u32 %1, %9, %12, %14, %1\n\t"        \
            "v_mad_u64_u32 %2, %10, %12, %15, %2\n\tv_mad_u64_u32 %3, %11, %12, %16, %3\n\t"      \
            "v_addc_co_u32 %4, %8, 0, %4, %8\n\tv_addc_co_u32 %5, %9, 0, %5, %9\n\t"              \
            "v_addc_co_u32 %6, %10, 0, %6, %10\n\tv_addc_co_u32 %7, %11, 0, %7, %11"              \
            : "+&v"((acc)[0]), "+&v"((acc)[1]), "+&v"((acc)[2]), "+&v"((acc)[3]), "+&v"((ov)[0]), \
              "+&v"((ov)[1]), "+&v"((ov)[2]), "+&v"((ov)[3]), "=&s"(m0_), "=&s"(m1_),             \
              "=&s"(m2_), "=&s"(m3_)                                                              \
            : "v"(x), "v"((y)[0]), "v"((y)[1]), "v"((y)[2]), "v"((y)[3]));                        \
    } while (0)
#define SDPV_MAC96(acc, ov, a, b)                                                                 \
    do {                                                                                          \
        u64 m0_;                                                                                  \
        asm("v_mad_u64_u32 %0, %2, %3, %4, %0\n\ts_nop 1\n\tv_addc_co_u32 %1, %2, 0, %1, %2"       \
            : "+&v"(acc), "+&v"(ov), "=&s"(m0_)                                                   \
            : "v"(a), "v"(b));                                                                    \
    } while (0)
#define SDPV_SETTLE(v, w) asm("s_nop 1" : "+v"(v), "+v"(w))
#endif
#define SDPV_TRY_LAUNCH()                                   \
    do {                                                    \
        hipError_t err__ = hipGetLastError();               \
        if (err__ != hipSuccess) return SDPV_ELAUNCH;       \
    } while (0)

static inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Orders LDS writes of a wave before later reads by other lanes of the same wave.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exchanges lanes 32-63 of x with lanes 0-31 of y (v_permlane32_swap). Writing a register as
// (lanes 0-31, lanes 32-63): (x_lo, x_hi), (y_lo, y_hi) become x = (x_lo, y_lo), y = (x_hi, y_hi).
__device__ __forceinline__ void swap_halves(u32& x, u32& y) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}

// The value of the lane below (lane 0: zero) and of the lane above (lane 63: zero) of the wave: one
// data-parallel move each, no LDS crossbar.
__device__ __forceinline__ u32 lane_below(u32 v) {
    return (u32)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xf, 0xf, true);   // wave_shr:1
}
__device__ __forceinline__ u32 lane_above(u32 v) {
    return (u32)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xf, 0xf, true);   // wave_shl:1
}
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
// the value of lane src (uniform)
__device__ __forceinline__ u32 lane_read(u32 v, int src) { return (u32)__builtin_amdgcn_readlane((int)v, src); }
__device__ __forceinline__ u64 ballot64(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// 1 in the lanes of the mask m (uniform)
__device__ __forceinline__ u32 mask_bit(u64 m) { return __builtin_amdgcn_inverse_ballot_w64(m) ? 1u : 0u; }

__device__ __forceinline__ int clz32(u32 x) { return __clz((int)x); }

// Word i of the infinite two's-complement extension of an ns-word value (sdpvibe/limbops.py:22-28).
template <class Src>
__device__ __forceinline__ u32 ext_word(const Src& src, int ns, u32 ext, i64 i) {
    if (i < 0) return 0u;
    if (i >= ns) return ext;
    return src((int)i);
}

// Streaming rounding shift, the semantics of limbops._shift_round_kernel (sdpvibe/limbops.py:32-62):
// out word k (k < Lout) of round_half_up(x / 2^s) = floor((x + 2^(s-1)) / 2^s) for s > 0, exact
// left shift for s <= 0, x two's complement of ns words. Returns 1 when word Lout of the rounded
// value differs from the sign extension of word Lout-1 (the reference's overflow test).
template <class Src, class Out>
__device__ __forceinline__ int shr_round(const Src& src, int ns, i64 s, int Lout, Out out) {
    const u32 ext = (src(ns - 1) >> 31) ? 0xffffffffu : 0u;
    const i64 q = s >> 5;
    const int r = (int)(s & 31);
    u64 carry = 0;
    if (s >= 1) {
        const i64 sb = s - 1;
        carry = (ext_word(src, ns, ext, sb >> 5) >> (int)(sb & 31)) & 1u;
    }
    u32 prev = 0;
    u64 lo = ext_word(src, ns, ext, q);
    for (int k = 0; k <= Lout; k++) {
        const u64 hi = ext_word(src, ns, ext, q + k + 1);   // each source word is read once
        const u64 v = (((lo | (hi << 32)) >> r) & 0xffffffffull) + carry;
        lo = hi;
        carry = v >> 32;
        const u32 w = (u32)v;
        if (k < Lout) {
            out(k, w);
            prev = w;
        } else {
            const u32 want = (prev >> 31) ? 0xffffffffu : 0u;
            return w != want;
        }
    }
    return 0;
}

// Words k < Lout of floor(v / 2^s) + c (s < 0: exact left shift), v the two's complement value
// of ns words read through src (zero below word 0, sign words above ns - 1), in batches of 8
// independent reads; returns word Lout of that sum. |s| is clamped to where the words no longer
// change (beyond the value, or beyond the output).
template <class Src, class Out>
__device__ __forceinline__ u32 shift_words(const Src& src, int ns, u32 ext, i64 s, u32 c, int Lout, Out out) {
    const i64 smax = 32 * (i64)ns + 32, smin = -32 * ((i64)Lout + 2);
    s = s > smax ? smax : (s < smin ? smin : s);
    auto wd = [&](int t) -> u32 {
        const u32 v = src(t < 0 ? 0 : (t >= ns ? ns - 1 : t));
        return t < 0 ? 0u : (t >= ns ? ext : v);
    };
    const int qs = (int)(s >> 5), r = (int)(s & 31);
    for (int k0 = 0; k0 < Lout; k0 += 8) {
        u32 x[9];
#pragma unroll
        for (int u = 0; u < 9; u++) x[u] = wd(qs + k0 + u);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            if (k0 + u < Lout) {
                const u32 d = (u32)((((u64)x[u + 1] << 32) | x[u]) >> r);
                const u32 t = d + c;
                c = t < d ? 1u : 0u;
                out(k0 + u, t);
            }
        }
    }
    return (u32)((((u64)wd(qs + Lout + 1) << 32) | wd(qs + Lout)) >> r) + c;
}

// shr_round with the source read in batches (shift_words): same words, same return value.
template <class Src, class Out>
__device__ __forceinline__ int shr_round_batched(const Src& src, int ns, i64 s, int Lout, Out out) {
    const u32 ext = (src(ns - 1) >> 31) ? 0xffffffffu : 0u;
    u32 c = 0;
    if (s >= 1) {
        const i64 sb = s - 1;
        c = (sb >> 5) >= ns ? (ext & 1u) : (src((int)(sb >> 5)) >> (int)(sb & 31)) & 1u;
    }
    u32 prev = 0;
    const u32 top = shift_words(src, ns, ext, s, c, Lout, [&](int k, u32 v) {
        out(k, v);
        prev = v;
    });
    return top != ((prev >> 31) ? 0xffffffffu : 0u);
}

// Bit length of v (of ~v when v < 0), limbops._bitlen_kernel (sdpvibe/limbops.py:197-210).
template <class Src>
__device__ __forceinline__ int bitlen_tc(const Src& src, int n) {
    const u32 ext = (src(n - 1) >> 31) ? 0xffffffffu : 0u;
    for (int k = n - 1; k >= 0; k--) {
        const u32 x = src(k) ^ ext;
        if (x) return 32 * k + 32 - clz32(x);
    }
    return 0;
}

// Magnitude view of an n-word two's-complement value: |x| word i, computed on the fly.
// For negative x with lowest nonzero word z: words below z are 0, word z is -x_z, above ~x_i.
template <class Src>
struct MagView {
    Src src;
    int n;
    bool neg;
    int z;
    __device__ __forceinline__ MagView(const Src& s, int n_) : src(s), n(n_) {
        neg = (src(n - 1) >> 31) != 0;
        z = 0;
        if (neg) {
            while (z < n - 1 && src(z) == 0u) z++;
        }
    }
    __device__ __forceinline__ u32 operator()(int i) const {
        if (!neg) return src(i);
        if (i < z) return 0u;
        const u32 v = src(i);
        return i == z ? (u32)(0u - v) : ~v;
    }
};

// Plain bit length of a magnitude (mpf.py:32-35 `bitlen`).
template <class Src>
__device__ __forceinline__ int bitlen_mag(const Src& src, int n) {
    for (int k = n - 1; k >= 0; k--) {
        const u32 x = src(k);
        if (x) return 32 * k + 32 - clz32(x);
    }
    return 0;
}

// shift_mag of sdpvibe/mpf.py:36-56: dst[0..nd) = round_half_up(|src| / 2^s) (s > 0, magnitude
// half up, carry out of the top word dropped) or |src| * 2^-s (s <= 0, bits above nd dropped).
template <class Src, class Out>
__device__ __forceinline__ void shift_mag(const Src& src, int ns, i64 s, int nd, Out out) {
    if (s > 0) {
        const i64 q = s >> 5;
        const int r = (int)(s & 31);
        const i64 sb = s - 1, qb = sb >> 5;
        const int rb = (int)(sb & 31);
        u64 c = (qb < ns) ? ((src((int)qb) >> rb) & 1u) : 0u;
        for (int k = 0; k < nd; k++) {
            const i64 i0 = q + k, i1 = q + k + 1;
            const u32 lo = i0 < ns ? src((int)i0) : 0u;
            const u32 hi = i1 < ns ? src((int)i1) : 0u;
            const u32 d = r ? ((lo >> r) | (hi << (32 - r))) : lo;
            const u64 t = (u64)d + c;
            c = t >> 32;
            out(k, (u32)t);
        }
    } else {
        const i64 t = -s, q = t >> 5;
        const int r = (int)(t & 31);
        for (int k = 0; k < nd; k++) {
            const i64 i0 = k - q, i1 = k - q - 1;
            const u32 lo = (i0 >= 0 && i0 < ns) ? src((int)i0) : 0u;
            const u32 lo2 = (i1 >= 0 && i1 < ns) ? src((int)i1) : 0u;
            out(k, r ? ((lo << r) | (lo2 >> (32 - r))) : lo);
        }
    }
}

// Streaming two's-complement negation of words produced in increasing order.
struct NegStream {
    bool neg;
    u64 c;
    __device__ __forceinline__ explicit NegStream(bool n) : neg(n), c(1) {}
    __device__ __forceinline__ u32 operator()(u32 v) {
        if (!neg) return v;
        const u64 t = (u64)(~v) + c;
        c = t >> 32;
        return (u32)t;
    }
};

// Exact residue of a signed 32-bit integer modulo m (< 2^15) in [0, m), via a double reciprocal
// and one correction each way (|x| < 2^31 keeps the quotient estimate within 1).
__device__ __forceinline__ int mod_m(int x, int m, double minv) {
    const int q = (int)floor((double)x * minv);
    int r = x - q * m;
    if (r < 0) r += m;
    if (r >= m) r -= m;
    return r;
}

// Centred residue in [-(m-1)/2, (m-1)/2] split into 128*hi + lo, lo in [-64, 63].
__device__ __forceinline__ void split_centred(int r, int m, int& hi, int& lo) {
    if (r > (m >> 1)) r -= m;
    lo = ((r + 64) & 127) - 64;
    hi = (r - lo) >> 7;
}

// acc + ov 2^64 = sum of x[i] y[K - i] over the static column K of two N-word magnitudes
template <int N, int K>
__device__ __forceinline__ void column_sum(const u32* x, const u32* y, u64& acc, u32& ov) {
    constexpr int I0 = K - (N - 1) > 0 ? K - (N - 1) : 0, I1 = K < N - 1 ? K : N - 1, NT = I1 - I0 + 1;
    acc = 0;
    ov = 0;
#pragma unroll
    for (int q = 0; q < NT / 4; q++) {
        const u32 yv[4] = {y[K - I0 - 4 * q], y[K - I0 - 4 * q - 1], y[K - I0 - 4 * q - 2], y[K - I0 - 4 * q - 3]};
        SDPV_MAC96_CHAIN4(acc, ov, x + I0 + 4 * q, yv);
    }
#pragma unroll
    for (int i = I0 + NT / 4 * 4; i <= I1; i++) SDPV_MAC96(acc, ov, x[i], y[K - i]);
}
// x (NW words, L of them given, the others the sign) <- the words of round_half_up(x / 2^s), s >= 0 per lane, and
// `ext` the word that extends them. The rounding bit is added first; then every word is a funnel shift of two
// neighbours, and whole words move by 1 and 2 in registers and by multiples of 4 through the lane's 16-byte
// aligned slot (aligned accesses have no bank conflicts; only when some lane of the wave needs it).
template <int NW>
__device__ __forceinline__ void round_words(u32* x, int L, i64 s, u32& ext, v4i* slot) {
    ext = 0;
#pragma unroll
    for (int w = 0; w < NW; w++)
        if (w == L - 1) ext = (x[w] >> 31) ? ~0u : 0u;
#pragma unroll
    for (int w = NW - 8 > 0 ? NW - 8 : 0; w < NW; w++)
        if (w >= L) x[w] = ext;
    const int sc = s > 32 * NW ? 32 * NW : (int)s, hb = sc - 1;
    const u32 half = sc > 0 ? 1u << (hb & 31) : 0u;
    const int hw = hb >> 5;
    u32 c = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const u64 t = (u64)x[w] + (w == hw ? half : 0u) + c;
        x[w] = (u32)t;
        c = (u32)(t >> 32);
    }
    ext += c;
    const int r = sc & 31, q = sc >> 5;
#pragma unroll
    for (int w = 0; w < NW; w++) x[w] = (u32)((((u64)(w + 1 < NW ? x[w + 1] : ext) << 32) | x[w]) >> r);
#pragma unroll
    for (int w = 0; w < NW; w++) x[w] = (q & 1) ? (w + 1 < NW ? x[w + 1] : ext) : x[w];
#pragma unroll
    for (int w = 0; w < NW; w++) x[w] = (q & 2) ? (w + 2 < NW ? x[w + 2] : ext) : x[w];
    if (ballot64(q >= 4)) {
        const int q4 = q >> 2;
#pragma unroll
        for (int g = 0; g < NW / 4; g++)
            slot[g] = v4i{(int)x[4 * g], (int)x[4 * g + 1], (int)x[4 * g + 2], (int)x[4 * g + 3]};
#pragma unroll
        for (int g = 0; g < NW / 4; g++) {
            const bool in = g + q4 < NW / 4;
            const v4i v = slot[in ? g + q4 : 0];
#pragma unroll
            for (int u = 0; u < 4; u++) x[4 * g + u] = in ? (u32)v[u] : ext;
        }
    }
}

// Bytewise a + b of packed int8 lanes (no carries between bytes); exact when each byte sum
// stays in [-128, 127].
__device__ __forceinline__ u32 add_bytes(u32 a, u32 b) {
    return ((a & 0x7f7f7f7fu) + (b & 0x7f7f7f7fu)) ^ ((a ^ b) & 0x80808080u);
}

// XCD-aware workgroup order: the hardware deals workgroups round-robin over the 8 XCDs; this
// maps them so that each XCD receives a contiguous range of logical ids (shared operands stay in
// one L2). Bijective on [0, total).
__device__ __forceinline__ i64 xcd_remap(i64 h, i64 total) {
    const i64 nfull = total - (total & 7);
    if (h >= nfull) return h;
    return (h & 7) * (nfull >> 3) + (h >> 3);
}
