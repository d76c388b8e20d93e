// Limb-level bookkeeping and per-entry multiprecision floats on gfx950.
// One thread per entry; words are streamed straight from the limb planes (coalesced across
// entries) or kept in per-thread LDS slices, so a single kernel serves every limb count.
#include "common.hpp"

namespace {

struct PlaneSrc {  // limbs of one entry in limb-plane layout
    const i32* p;
    i64 stride;
    __device__ __forceinline__ u32 operator()(int k) const { return (u32)p[(i64)k * stride]; }
};

struct LdsSrc {  // per-thread words in LDS, thread-strided (bank-conflict free)
    const u32* p;
    int stride;
    __device__ __forceinline__ u32 operator()(int k) const { return p[k * stride]; }
};

constexpr int TPB = 256;

// ------------------------------------------------------------------ shift_round
__global__ void __launch_bounds__(TPB) k_shift_round(const i32* __restrict__ X, i64 B, int Lin,
                                                     const i64* __restrict__ S, i32* __restrict__ O,
                                                     int Lout, i32* __restrict__ flag, int per_entry) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x;
    if (e >= B) return;
    PlaneSrc src{X + e, B};
    const int bad = shr_round(src, Lin, S[e], Lout, [&](int k, u32 w) { O[(i64)k * B + e] = (i32)w; });
    if (per_entry) {
        flag[e] = bad;
    } else if (bad) {
        atomicOr(flag, 1);
    }
}

// ------------------------------------------------------------------ add_same
__global__ void __launch_bounds__(TPB) k_add_same(const i32* __restrict__ A, const i32* __restrict__ Bm,
                                                  i32* __restrict__ O, int L, i64 B, int sub) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x;
    if (e >= B) return;
    u64 c = sub ? 1u : 0u;
    for (int k = 0; k < L; k++) {
        const u32 a = (u32)A[(i64)k * B + e];
        u32 b = (u32)Bm[(i64)k * B + e];
        if (sub) b = ~b;
        const u64 t = (u64)a + b + c;
        c = t >> 32;
        O[(i64)k * B + e] = (i32)(u32)t;
    }
}

// ------------------------------------------------------------------ bitlen / top
__global__ void __launch_bounds__(TPB) k_bitlen(const i32* __restrict__ X, int L, i64 B, i64* __restrict__ out) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x;
    if (e >= B) return;
    out[e] = bitlen_tc(PlaneSrc{X + e, B}, L);
}

__global__ void __launch_bounds__(TPB) k_mpf_top(const i32* __restrict__ m, const i64* __restrict__ ev, int L,
                                                 i64 n, i64* __restrict__ top) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x;
    if (e >= n) return;
    const i64 ex = ev[e];
    top[e] = (ex == EZV) ? EZV : ex + bitlen_tc(PlaneSrc{m + e, n}, L);
}

// ------------------------------------------------------------------ batched aligned add
// batched.py:56-79: both operands shift right by >= 1 bit (round half up), then add (wraps).
__global__ void __launch_bounds__(TPB) k_badd_align(const i32* __restrict__ A, const i32* __restrict__ Bm,
                                                    const i64* __restrict__ EA, const i64* __restrict__ EB,
                                                    i32* __restrict__ O, i64* __restrict__ EO, int L,
                                                    i64 entries, i64 rows, i64 cols, int sub) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x;
    if (e >= entries) return;
    const i64 col = (e / (rows * cols)) * cols + e % cols;
    const i64 ea = EA[col], eb = EB[col];
    const i64 ex = (ea > eb ? ea : eb) + 1;
    PlaneSrc sa{A + e, entries}, sb{Bm + e, entries};
    // Stream both rounded operands word by word and add them with a running carry.
    // Each rounded operand fits L words (a right shift of at least one bit).
    const u32 exta = (sa(L - 1) >> 31) ? 0xffffffffu : 0u;
    const u32 extb = (sb(L - 1) >> 31) ? 0xffffffffu : 0u;
    const i64 s_a = ex - ea, s_b = ex - eb;
    const i64 qa = s_a >> 5, qb = s_b >> 5;
    const int ra = (int)(s_a & 31), rb = (int)(s_b & 31);
    u64 ca = (ext_word(sa, L, exta, (s_a - 1) >> 5) >> (int)((s_a - 1) & 31)) & 1u;
    u64 cb = (ext_word(sb, L, extb, (s_b - 1) >> 5) >> (int)((s_b - 1) & 31)) & 1u;
    u64 c = sub ? 1u : 0u;
    for (int k = 0; k < L; k++) {
        const u64 a = ((((u64)ext_word(sa, L, exta, qa + k)) | ((u64)ext_word(sa, L, exta, qa + k + 1) << 32)) >> ra & 0xffffffffull) + ca;
        const u64 b = ((((u64)ext_word(sb, L, extb, qb + k)) | ((u64)ext_word(sb, L, extb, qb + k + 1) << 32)) >> rb & 0xffffffffull) + cb;
        ca = a >> 32;
        cb = b >> 32;
        u32 bw = (u32)b;
        if (sub) bw = ~bw;
        const u64 t = (u64)(u32)a + bw + c;
        c = t >> 32;
        O[(i64)k * entries + e] = (i32)(u32)t;
    }
    if ((e / cols) % rows == 0) EO[col] = ex;
}

// blocks of uneven dimension to and from a stack: up to 32 per launch, their places passed with the launch
// (no table to copy, none to keep). One workgroup row of grid.y per block, 8 limb planes per grid.z. Two copies
// per block and array before: factoring and solving 400 uneven blocks
// took 2623 launches and 23.4 ms, now 567 and 14.3.
constexpr int BLOCKS = 32;
struct BlockList {
    sdpv_block b[BLOCKS];
};
__global__ void __launch_bounds__(TPB) k_copy_blocks(BlockList list, i32* __restrict__ m, i64* __restrict__ e, int L,
                                                     i64 count, i64 j0, i64 rows, i64 cols, int to_stack) {
    const sdpv_block& b = list.b[blockIdx.y];
    const i64 n = rows * cols, x = blockIdx.x * (i64)TPB + threadIdx.x;
    if (x >= n) return;
    const i64 i = (u32)x / (u32)cols, j = x - i * cols;
    const bool in = i < b.rows && j < b.cols;
    if (!in && !to_stack) return;
    const int k0 = 8 * blockIdx.z, kn = min(L - k0, 8);
    i32* s = m + ((i64)k0 * count + j0 + blockIdx.y) * n + x;
    i32* p = in ? b.m + k0 * b.mp + i * b.mr + j * b.mc : nullptr;
    i32 v[8];
#pragma unroll
    for (int u = 0; u < 8; u++)
        if (u < kn) v[u] = !to_stack ? s[u * count * n] : in ? p[u * b.mp] : 0;
#pragma unroll
    for (int u = 0; u < 8; u++)
        if (u < kn) (to_stack ? s[u * count * n] : p[u * b.mp]) = v[u];
    if (k0 == 0) {
        i64* se = e + (j0 + blockIdx.y) * n + x;
        if (to_stack) *se = in ? b.e[i * b.er + j * b.ec] : EZV;
        else b.e[i * b.er + j * b.ec] = *se;
    }
}

// both parts of a stacked solve re-rounded to their columns' larger exponent and joined, one pass (a
// rounding each, a broadcast shift per entry and a concatenation took seven launches)
__global__ void __launch_bounds__(TPB) k_stack_common(const i32* __restrict__ P1, const i64* __restrict__ E1,
                                                      const i32* __restrict__ P2, const i64* __restrict__ E2,
                                                      i32* __restrict__ O, i64* __restrict__ EO, int L, i64 nb, i64 R1,
                                                      i64 R2, i64 C, i32* __restrict__ flag) {
    const i64 e = blockIdx.x * (i64)TPB + threadIdx.x, R = R1 + R2, n = nb * R * C;
    if (e >= n) return;
    const i64 c = e % C, r = e / C % R, b = e / (C * R), col = b * C + c;
    const i64 ea = E1[col], eb = E2[col], ex = ea > eb ? ea : eb;
    const bool up = r < R1;
    const i64 n1 = nb * R1 * C, n2 = nb * R2 * C;
    const PlaneSrc src = up ? PlaneSrc{P1 + (b * R1 + r) * C + c, n1} : PlaneSrc{P2 + (b * R2 + r - R1) * C + c, n2};
    const int bad = shr_round_batched(src, L, ex - (up ? ea : eb), L, [&](int k, u32 w) { O[(i64)k * n + e] = (i32)w; });
    if (bad && flag) atomicOr(flag, 1);
    if (r == 0) EO[col] = ex;
}

// ------------------------------------------------------------------ mpf_norm (mpf.py:127-140)
__global__ void __launch_bounds__(TPB) k_mpf_norm(const i32* __restrict__ X, const i64* __restrict__ eI, int LI,
                                                  i32* __restrict__ O, i64* __restrict__ eO, int L, i64 n) {
    const i64 i = blockIdx.x * (i64)TPB + threadIdx.x;
    if (i >= n) return;
    const int NB = 32 * L - 2;
    PlaneSrc x{X + i, n};
    MagView<PlaneSrc> mag(x, LI);
    const int bl = bitlen_mag(mag, LI);
    if (bl == 0) {
        for (int k = 0; k < L; k++) O[(i64)k * n + i] = 0;
        eO[i] = EZV;
        return;
    }
    const int s = bl - NB;
    NegStream ng(mag.neg);
    shift_mag(mag, LI, s, L, [&](int k, u32 w) { O[(i64)k * n + i] = (i32)ng(w); });
    eO[i] = eI[i] + s;
}

// ------------------------------------------------------------------ products and sums in registers
// Up to 40 limbs both operands of an entry live in registers, in arrays of N >= L words with static indexes
// (N = 8, 16, 24, 28, 32, 36 or 40). Bound: reading two operands and writing one; a product's N^2
// multiply-adds take about as long.

// magnitude of the two's complement words x (zero above the sign's word), its sign returned
template <int N>
__device__ __forceinline__ bool to_magnitude(u32* x, u32 top) {
    const bool neg = (top >> 31) != 0;
    const u32 f = neg ? ~0u : 0u;
    u32 c = neg ? 1u : 0u;
#pragma unroll
    for (int w = 0; w < N; w++) {
        const u64 t = (u64)(x[w] ^ f) + c;
        x[w] = (u32)t;
        c = (u32)(t >> 32);
    }
    return neg;
}

// words of a product from column K on into p[K - (N - 1)] for K >= N - 1 (the lower ones carry only)
template <int N, int K>
struct MulColumns {
    static __device__ __forceinline__ void run(const u32* x, const u32* y, u64& carry, u32* p) {
        u64 acc;
        u32 ov;
        column_sum<N, K>(x, y, acc, ov);
        const u64 sm = acc + carry;
        carry = (sm >> 32) | ((u64)(ov + (sm < carry ? 1u : 0u)) << 32);
        if (K >= N - 1) p[K >= N - 1 ? K - (N - 1) : 0] = (u32)sm;
        if constexpr (K < 2 * N - 2) MulColumns<N, K + 1>::run(x, y, carry, p);
        else p[N] = (u32)carry;
    }
};

// any product (operands that are not normalised): columns from memory, once for the length, once rounded
__device__ void mul_any(const PlaneSrc& xa, const PlaneSrc& xb, int L, i64 n, i64 i, i32* O, i64* eO, i64 e) {
    MagView<PlaneSrc> ma(xa, L), mb(xb, L);
    int bl = 0, s = 0;
    i64 q1 = 0;
    u32 prev = 0, c = 0;
    NegStream ng(ma.neg != mb.neg);
    for (int pass = 0; pass < 2; pass++) {
        u64 carry = 0, hprev = 0;
        for (int k = 0; k < 2 * L + 1; k++) {
            u64 lo = 0, hi = 0;
            const int first = k - L + 1 > 0 ? k - L + 1 : 0, last = k < L - 1 ? k : L - 1;
            for (int x = first; x <= last; x++) {
                const u64 pr = (u64)ma(x) * mb(k - x);
                lo += (u32)pr;
                hi += pr >> 32;
            }
            const u64 sum = lo + hprev + carry;
            const u32 w = (u32)sum;
            carry = sum >> 32;
            hprev = hi;
            if (pass == 0) {
                if (w) bl = 32 * k + 32 - clz32(w);
                continue;
            }
            if (s > 0) {                                  // word k of the product completes output word k - 1 - q1
                if (k == q1) c = (w >> ((s - 1) & 31)) & 1u;
                if (k > q1 && k - 1 - q1 < L) {
                    const u64 d = ((((u64)w << 32) | prev) >> (((s - 1) & 31) + 1)) & 0xffffffffull;
                    const u64 t = d + c;
                    c = (u32)(t >> 32);
                    O[(k - 1 - q1) * n + i] = (i32)ng((u32)t);
                }
            } else {                                      // left shift by whole words and bits: words below stay zero
                const int t = -s, q = t >> 5, r = t & 31;
                if (k == 0)
                    for (int z = 0; z < q && z < L; z++) O[(i64)z * n + i] = (i32)ng(0u);
                if (k + q < L) O[(i64)(k + q) * n + i] = (i32)ng(r ? (w << r) | (prev >> (32 - r)) : w);
            }
            prev = w;
        }
        s = bl - (32 * L - 2);
        q1 = s > 0 ? (s - 1) >> 5 : 0;
    }
    eO[i] = e + s;
}

// one entry per thread. Limbs sit in the upper L of N words, so the product of two normalised entries has
// its rounded words at static places whatever L is. 787 320 products at L = 24 on one MI355X:
// 0.061 ms, 4.0 TB/s (operands in LDS slices, word by word: 0.511 ms); one after the other on the same operands,
// as they stay in the caches, L = 14 / 24 / 32 / 40 0.033 / 0.052 / 0.081 / 0.114 ms (0.128 / 0.420 / 1.04 / 1.48).
template <int N>
__global__ void __launch_bounds__(256) k_mul_regs(const i32* __restrict__ A, const i64* __restrict__ eA,
                                                  const i32* __restrict__ Bm, const i64* __restrict__ eB,
                                                  i32* __restrict__ O, i64* __restrict__ eO, int L, i64 n, int bscalar) {
    const i64 i = blockIdx.x * (i64)256 + threadIdx.x;
    if (i >= n) return;
    const i64 ib = bscalar ? 0 : i, nb = bscalar ? 1 : n;
    const int d = N - L;
    u32 x[N], y[N];
#pragma unroll
    for (int w = 0; w < N; w++) {
        x[w] = w >= d ? (u32)A[(i64)(w - d) * n + i] : 0u;
        y[w] = w >= d ? (u32)Bm[(i64)(w - d) * nb + ib] : 0u;
    }
    const i64 e = eA[i] + eB[ib];
    const bool neg = to_magnitude<N>(x, x[N - 1]) != to_magnitude<N>(y, y[N - 1]);
    u32 za = 0, zb = 0;
#pragma unroll
    for (int w = 0; w < N; w++) {
        za |= x[w];
        zb |= y[w];
    }
    if (za == 0u || zb == 0u) {
        for (int k = 0; k < L; k++) O[(i64)k * n + i] = 0;
        eO[i] = EZV;
        return;
    }
    u32 p[N + 1];                                         // words N - 1 .. 2N - 1 of the product
    u64 carry = 0;
    MulColumns<N, 0>::run(x, y, carry, p);
    // bit length from the two top words; the shift to 32 L - 2 bits must start in word 2N - L - 1
    const int bl = 32 * (2 * L - 2) + (p[N] ? 64 - clz32(p[N]) : 32 - clz32(p[N - 1]));
    const int s = bl - (32 * L - 2);
    if ((p[N] | p[N - 1]) == 0u || (s - 1) >> 5 != L - 1) {
        mul_any(PlaneSrc{A + i, n}, PlaneSrc{Bm + ib, nb}, L, n, i, O, eO, e);
        return;
    }
    const int r = (s - 1) & 31, q = N - L;                // p[q]: the word with the rounding bit
    u32 c = 0, nc = neg ? 1u : 0u;
    const u32 f = neg ? ~0u : 0u;
#pragma unroll
    for (int w = 0; w < N; w++) {
        if (w == q) c = (p[w] >> r) & 1u;
        const u64 t = (((((u64)p[w + 1] << 32) | p[w]) >> r >> 1) & 0xffffffffull) + c;
        c = (u32)(t >> 32);
        if (w >= q) {
            const u64 u = (u64)((u32)t ^ f) + nc;
            nc = (u32)(u >> 32);
            O[(i64)(w - q) * n + i] = (i32)(u32)u;
        }
    }
    eO[i] = e + s;
}

// x >>= 32 q words in registers (0 <= q < 64), words moved in steps that some lane of the wave needs
template <int N>
__device__ __forceinline__ void words_down(u32* x, int q) {
#pragma unroll
    for (int st = 1; st < 64; st <<= 1) {
        if (st < N ? ballot64(q & st) != 0 : false) {
#pragma unroll
            for (int w = 0; w < N; w++) x[w] = (q & st) ? (w + st < N ? x[w + st] : 0u) : x[w];
        } else if (st >= N) {
#pragma unroll
            for (int w = 0; w < N; w++) x[w] = (q & st) ? 0u : x[w];
        }
    }
}
template <int N>
__device__ __forceinline__ void words_up(u32* x, int q) {
#pragma unroll
    for (int st = 1; st < 64; st <<= 1) {
        if (st < N ? ballot64(q & st) != 0 : false) {
#pragma unroll
            for (int w = N - 1; w >= 0; w--) x[w] = (q & st) ? (w >= st ? x[w - st] : 0u) : x[w];
        } else if (st >= N) {
#pragma unroll
            for (int w = 0; w < N; w++) x[w] = (q & st) ? 0u : x[w];
        }
    }
}
// x <- round_half_up(x / 2^s), s >= 1 (x, N words, unsigned); lanes with s < 1 keep x
template <int N>
__device__ __forceinline__ void round_down(u32* x, i64 s) {
    const bool on = s >= 1;
    const int t = on ? (int)(s > 32 * N + 1 ? 32 * N + 1 : s) - 1 : 0, r = t & 31;
    words_down<N>(x, t >> 5);
    u32 c = (x[0] >> r) & 1u;
#pragma unroll
    for (int w = 0; w < N; w++) {
        const u64 v = (((((u64)(w + 1 < N ? x[w + 1] : 0u) << 32) | x[w]) >> r >> 1) & 0xffffffffull) + c;
        c = (u32)(v >> 32);
        x[w] = on ? (u32)v : x[w];
    }
}

// A + sgn B (mpf.py:92-124): the operand with the larger exponent one word up, the other rounded to the same
// place, magnitudes added or subtracted, the result normalised. 787 320 sums at L = 24 on one
// MI355X: 0.079 ms, 3.1 TB/s (operands read word by word at every use, sums in LDS: 0.344 ms); one after the
// other on the same operands, L = 14 / 24 / 32 / 40 0.037 / 0.053 / 0.105 / 0.149 ms (0.090 / 0.189 / 0.319 / 0.472):
// above 24 limbs the registers hold three waves per SIMD, above 32 two.
template <int N>
__global__ void __launch_bounds__(256) k_add_regs(const i32* __restrict__ A, const i64* __restrict__ eA,
                                                  const i32* __restrict__ Bm, const i64* __restrict__ eB,
                                                  i32* __restrict__ O, i64* __restrict__ eO, int L, i64 n, int sgn) {
    constexpr int W = N + 2;
    const i64 i0 = blockIdx.x * (i64)256 + threadIdx.x, i = i0 < n ? i0 : n - 1;   // every lane takes part in ballots
    u32 x[W], y[W];                                       // one word up
    x[0] = y[0] = x[W - 1] = y[W - 1] = 0u;
#pragma unroll
    for (int w = 0; w < N; w++) {
        x[w + 1] = w < L ? (u32)A[(i64)w * n + i] : 0u;
        y[w + 1] = w < L ? (u32)Bm[(i64)w * n + i] : 0u;
    }
    i64 ea = eA[i], eb = eB[i];
    auto magnitude = [&](u32* v) {                        // of the L words from v[1] on
        u32 top = 0;
#pragma unroll
        for (int w = 1; w <= N; w++) top = w == L ? v[w] : top;
        const bool neg = (top >> 31) != 0;
        const u32 f = neg ? ~0u : 0u;
        u32 c = neg ? 1u : 0u;
#pragma unroll
        for (int w = 1; w <= N; w++) {
            const u64 t = (u64)(w <= L ? v[w] ^ f : 0u) + c;
            v[w] = w <= L ? (u32)t : 0u;
            c = (u32)(t >> 32);
        }
        return neg;
    };
    bool na = magnitude(x), nbg = magnitude(y) != (sgn < 0);
    u32 za = 0, zb = 0;
#pragma unroll
    for (int w = 1; w <= N; w++) {
        za |= x[w];
        zb |= y[w];
    }
    if (za == 0u) ea = EZV;
    if (zb == 0u) eb = EZV;
    const bool zero = ea == EZV && eb == EZV;
    if (ea == EZV || eb == EZV) {                         // a zero operand adds nothing
#pragma unroll
        for (int w = 0; w < W; w++) {
            x[w] = ea == EZV ? 0u : x[w];
            y[w] = eb == EZV ? 0u : y[w];
        }
    }
    const bool sw = eb > ea;                              // x: the larger exponent
#pragma unroll
    for (int w = 0; w < W; w++) {
        const u32 t = x[w];
        x[w] = sw ? y[w] : t;
        y[w] = sw ? t : y[w];
    }
    const bool nx = sw ? nbg : na, ny = sw ? na : nbg;
    const i64 et = (sw ? eb : ea) - 32, dist = sw ? eb - ea : ea - eb;
    round_down<W>(y, dist);
    // magnitudes: x + y, or x - y with the sign of the larger
    const bool sub = nx != ny;
    const u32 fy = sub ? ~0u : 0u;
    u32 c = sub ? 1u : 0u;
#pragma unroll
    for (int w = 0; w < W; w++) {
        const u64 t = (u64)x[w] + (y[w] ^ fy) + c;
        x[w] = (u32)t;
        c = (u32)(t >> 32);
    }
    const bool flip = sub && c == 0u;                     // y was larger
    const bool neg = nx != flip;
    if (ballot64(flip)) {
        const u32 ff = flip ? ~0u : 0u;
        c = flip ? 1u : 0u;
#pragma unroll
        for (int w = 0; w < W; w++) {
            const u64 t = (u64)(x[w] ^ ff) + c;
            x[w] = (u32)t;
            c = (u32)(t >> 32);
        }
    }
    int bl = 0;
#pragma unroll
    for (int w = 0; w < W; w++) bl = x[w] ? 32 * w + 32 - clz32(x[w]) : bl;
    const int s = bl == 0 ? 0 : bl - (32 * L - 2);
    if (ballot64(s < 0)) {                                // cancellation: left
        const int t = s < 0 ? -s : 0, r = t & 31;
        words_up<W>(x, t >> 5);
#pragma unroll
        for (int w = W - 1; w >= 0; w--) x[w] = (u32)(((((u64)x[w] << 32) | (w > 0 ? x[w - 1] : 0u)) << r) >> 32);
    }
    round_down<W>(x, s);
    if (i0 >= n) return;
    const bool none = zero || bl == 0;
    const u32 f = neg ? ~0u : 0u;
    c = neg ? 1u : 0u;
#pragma unroll
    for (int w = 0; w < N; w++) {
        const u64 t = (u64)(x[w] ^ f) + c;
        c = (u32)(t >> 32);
        if (w < L) O[(i64)w * n + i] = none ? 0 : (i32)(u32)t;
    }
    eO[i] = none ? EZV : et + s;
}

// ------------------------------------------------------------------ mpf_mul (mpf.py:58-89), more than 40 limbs
// Magnitudes staged in per-thread LDS slices; product scanning over runtime L.
constexpr int MUL_TPB = 64;
__global__ void __launch_bounds__(MUL_TPB) k_mpf_mul(const i32* __restrict__ A, const i64* __restrict__ eA,
                                                     const i32* __restrict__ Bm, const i64* __restrict__ eB,
                                                     i32* __restrict__ O, i64* __restrict__ eO, int L, i64 n,
                                                     int bscalar) {
    SDPV_DYNAMIC_LDS(u32, lds);
    const int t = threadIdx.x;
    const i64 i = blockIdx.x * (i64)MUL_TPB + t;
    if (i >= n) return;
    const i64 ib = bscalar ? 0 : i, nb = bscalar ? 1 : n;
    u32* a = lds + t;                    // a[k * MUL_TPB]
    u32* b = lds + L * MUL_TPB + t;      // b[k * MUL_TPB]
    u32* p = lds + 2 * L * MUL_TPB + t;  // p[k * MUL_TPB], 2L words
    PlaneSrc xa{A + i, n}, xb{Bm + ib, nb};
    MagView<PlaneSrc> ma(xa, L), mb(xb, L);
    for (int k = 0; k < L; k++) {
        a[k * MUL_TPB] = ma(k);
        b[k * MUL_TPB] = mb(k);
    }
    LdsSrc la{a, MUL_TPB}, lb{b, MUL_TPB};
    if (bitlen_mag(la, L) == 0 || bitlen_mag(lb, L) == 0) {
        for (int k = 0; k < L; k++) O[(i64)k * n + i] = 0;
        eO[i] = EZV;
        return;
    }
    u64 carry = 0, hprev = 0;
    for (int k = 0; k < 2 * L - 1; k++) {
        u64 lo = 0, hi = 0;
        const int first = k - L + 1 > 0 ? k - L + 1 : 0, last = k < L - 1 ? k : L - 1;
        for (int x = first; x <= last; x++) {
            const u64 pr = (u64)a[x * MUL_TPB] * b[(k - x) * MUL_TPB];
            lo += (u32)pr;
            hi += pr >> 32;
        }
        const u64 sum = lo + hprev + carry;
        p[k * MUL_TPB] = (u32)sum;
        carry = sum >> 32;
        hprev = hi;
    }
    p[(2 * L - 1) * MUL_TPB] = (u32)(hprev + carry);
    LdsSrc lp{p, MUL_TPB};
    const int NB = 32 * L - 2;
    const int s = bitlen_mag(lp, 2 * L) - NB;
    NegStream ng(ma.neg != mb.neg);
    shift_mag(lp, 2 * L, s, L, [&](int k, u32 w) { O[(i64)k * n + i] = (i32)ng(w); });
    eO[i] = eA[i] + eB[ib] + s;
}

// ------------------------------------------------------------------ mpf_add (mpf.py:92-124), more than 40 limbs
constexpr int ADD_TPB = 64;
__global__ void __launch_bounds__(ADD_TPB) k_mpf_add(const i32* __restrict__ A, const i64* __restrict__ eA,
                                                     const i32* __restrict__ Bm, const i64* __restrict__ eB,
                                                     i32* __restrict__ O, i64* __restrict__ eO, int L, i64 n,
                                                     int sgn) {
    SDPV_DYNAMIC_LDS(u32, lds);
    const int t = threadIdx.x;
    const i64 i = blockIdx.x * (i64)ADD_TPB + t;
    if (i >= n) return;
    const int W = L + 2;
    u32* wa = lds + t;            // wa[k * ADD_TPB], W words
    PlaneSrc xa{A + i, n}, xb{Bm + i, n};
    MagView<PlaneSrc> ma(xa, L), mb(xb, L);
    const bool na = ma.neg, nbg = mb.neg ^ (sgn < 0);
    i64 ea = eA[i], eb = eB[i];
    const int la = bitlen_mag(ma, L), lb = bitlen_mag(mb, L);
    if (la == 0) ea = EZV;
    if (lb == 0) eb = EZV;
    if (ea == EZV && eb == EZV) {
        for (int k = 0; k < L; k++) O[(i64)k * n + i] = 0;
        eO[i] = EZV;
        return;
    }
    const i64 tt = (ea > eb ? ea : eb) - 32;
    const i64 da = ea - tt, db = eb - tt;
    const i64 clampv = 32 * (i64)(L + 3);
    const i64 sa = da < -clampv ? clampv : -da;
    const i64 sb = db < -clampv ? clampv : -db;
    // wa = +-round(|a| / 2^sa) in W words
    {
        NegStream ng(na);
        if (ea == EZV) {
            for (int k = 0; k < W; k++) wa[k * ADD_TPB] = 0;
        } else {
            shift_mag(ma, L, sa, W, [&](int k, u32 w) { wa[k * ADD_TPB] = ng(w); });
        }
    }
    // wa += +-round(|b| / 2^sb), streamed
    if (eb != EZV) {
        NegStream ng(nbg);
        u64 c = 0;
        shift_mag(mb, L, sb, W, [&](int k, u32 w) {
            const u64 v = (u64)wa[k * ADD_TPB] + ng(w) + c;
            wa[k * ADD_TPB] = (u32)v;
            c = v >> 32;
        });
    }
    LdsSrc sw{wa, ADD_TPB};
    MagView<LdsSrc> mw(sw, W);
    const int bl = bitlen_mag(mw, W);
    if (bl == 0) {
        for (int k = 0; k < L; k++) O[(i64)k * n + i] = 0;
        eO[i] = EZV;
        return;
    }
    const int NB = 32 * L - 2;
    const int s = bl - NB;
    NegStream ng(mw.neg);
    shift_mag(mw, W, s, L, [&](int k, u32 w) { O[(i64)k * n + i] = (i32)ng(w); });
    eO[i] = tt + s;
}

// ------------------------------------------------------------------ row alignment exponents
// Erow = max_k top(entry) - NB over entries with e != EZ (mpf.py:390-395), computed as a K-split
// reduction: a fill pass, then blocks over (rows, k slices) combine with 64-bit atomicMax.
// Rows without such entries keep SDPV_EZ (the reference then uses exponent 0; no product
// depends on it because every entry of such a row is zero).
__device__ __forceinline__ i64 entry_top(const i32* X, const i64* e, int L, i64 plane, i64 off) {
    const i64 ex = e[off];
    if (ex == EZV) return EZV;
    return ex + bitlen_tc(PlaneSrc{X + off, plane}, L);
}

// top of an entry when its exponent is known and its top limb is neither 0 nor -1 (normalised
// MPF); otherwise the full scan
__device__ __forceinline__ i64 entry_top_fast(const i32* X, i64 plane, int L, i64 off, i64 ex, u32 topw) {
    if (ex == EZV) return EZV;
    if (topw != 0u && topw != 0xffffffffu) {
        const u32 x = topw ^ ((topw >> 31) ? 0xffffffffu : 0u);
        return ex + 32 * (i64)(L - 1) + 32 - clz32(x);
    }
    return ex + bitlen_tc(PlaneSrc{X + off, plane}, L);
}

__device__ __forceinline__ i64 row_exp_of(i64 mx, int L) { return mx == EZV ? EZV : mx - (32 * (i64)L - 2); }

// rows contiguous in k (ldk == 1): one wave per row, 8 entries per lane in flight
__global__ void __launch_bounds__(256) k_row_exp_wave(const i32* __restrict__ X, const i64* __restrict__ e, int L,
                                                      i64 plane, i64 nrows, i64 rows, i64 K, i64 ldb, i64 ldr,
                                                      i64* __restrict__ Erow) {
    const i64 R = blockIdx.x * (i64)4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (R >= nrows) return;
    const i64 b = R / rows, r = R % rows;
    const i64 base = b * ldb + r * ldr;
    const i32* top = X + (i64)(L - 1) * plane;
    i64 mx = EZV;
    for (i64 k0 = 0; k0 < K; k0 += 8 * 64) {
        i64 ex[8];
        u32 tw[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const i64 k = k0 + u * 64 + lane;
            ex[u] = k < K ? e[base + k] : EZV;
            tw[u] = k < K ? (u32)top[base + k] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const i64 t = entry_top_fast(X, plane, L, base + k0 + u * 64 + lane, ex[u], tw[u]);
            mx = t > mx ? t : mx;
        }
    }
    for (int o = 32; o >= 1; o >>= 1) {
        const i64 v = __shfl_xor(mx, o, 64);
        mx = v > mx ? v : mx;
    }
    if (lane == 0) Erow[R] = row_exp_of(mx, L);
}

// other layouts: 64 rows (lanes) per block of 16 waves, wave w takes k = w, w + 16, ... of the
// block's k range (blockIdx.y: one of gridDim.y parts of kchunk); the 16 partial maxima per row
// meet in LDS. With several k parts the rows meet by an atomic maximum over a filled Erow.
__global__ void __launch_bounds__(1024) k_row_exp_cols(const i32* __restrict__ X, const i64* __restrict__ e, int L,
                                                       i64 plane, i64 nrows, i64 rows, i64 K, i64 ldb, i64 ldr,
                                                       i64 ldk, i64 kchunk, i64* __restrict__ Erow) {
    __shared__ i64 part[16][64];
    const int lane = threadIdx.x & 63, kg = threadIdx.x >> 6;
    const i64 R = blockIdx.x * (i64)64 + lane;
    const i64 kb = (i64)blockIdx.y * kchunk, ke = kb + kchunk < K ? kb + kchunk : K;
    i64 mx = EZV;
    if (R < nrows) {
        const i64 b = R / rows, r = R % rows;
        const i64 base = b * ldb + r * ldr;
        const i32* top = X + (i64)(L - 1) * plane;
        for (i64 k0 = kb + kg; k0 < ke; k0 += 8 * 16) {
            i64 ex[8];
            u32 tw[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const i64 k = k0 + u * 16;
                ex[u] = k < ke ? e[base + k * ldk] : EZV;
                tw[u] = k < ke ? (u32)top[base + k * ldk] : 0u;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const i64 t = entry_top_fast(X, plane, L, base + (k0 + u * 16) * ldk, ex[u], tw[u]);
                mx = t > mx ? t : mx;
            }
        }
    }
    part[kg][lane] = mx;
    __syncthreads();
    if (kg == 0 && R < nrows) {
        for (int q = 1; q < 16; q++) mx = part[q][lane] > mx ? part[q][lane] : mx;
        const i64 v = row_exp_of(mx, L);               // monotone in mx: the maximum commutes
        if (gridDim.y == 1) Erow[R] = v;
        else if (v != EZV) atomicMax((long long*)&Erow[R], (long long)v);
    }
}

// strided rows, few of them: 16 rows per block (lane = 16 rows x 4 k), its 16 waves over k, so that
// few rows still give enough blocks without splitting k (no fill, no atomics); the 64 k partial
// maxima of a row meet by lane exchange within the wave and in LDS across the waves
__global__ void __launch_bounds__(1024) k_row_exp_cols16(const i32* __restrict__ X, const i64* __restrict__ e, int L,
                                                         i64 plane, i64 nrows, i64 rows, i64 K, i64 ldb, i64 ldr,
                                                         i64 ldk, i64* __restrict__ Erow) {
    __shared__ i64 part[16][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rl = lane & 15, kq = lane >> 4;
    const i64 R = blockIdx.x * (i64)16 + rl;
    i64 mx = EZV;
    if (R < nrows) {
        const i64 b = R / rows, r = R % rows;
        const i64 base = b * ldb + r * ldr;
        const i32* top = X + (i64)(L - 1) * plane;
        for (i64 k0 = wave * 4 + kq; k0 < K; k0 += 8 * 64) {
            i64 ex[8];
            u32 tw[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const i64 k = k0 + u * 64;
                ex[u] = k < K ? e[base + k * ldk] : EZV;
                tw[u] = k < K ? (u32)top[base + k * ldk] : 0u;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const i64 t = entry_top_fast(X, plane, L, base + (k0 + u * 64) * ldk, ex[u], tw[u]);
                mx = t > mx ? t : mx;
            }
        }
    }
    for (int o = 16; o <= 32; o <<= 1) {                  // the 4 k lanes of a row within the wave
        const i64 v = __shfl_xor(mx, o, 64);
        mx = v > mx ? v : mx;
    }
    if (kq == 0) part[wave][rl] = mx;
    __syncthreads();
    if (wave == 0 && kq == 0 && R < nrows) {
        for (int q = 1; q < 16; q++) mx = part[q][rl] > mx ? part[q][rl] : mx;
        Erow[R] = row_exp_of(mx, L);
    }
}

__global__ void __launch_bounds__(256) k_fill_i64(i64* __restrict__ p, i64 n, i64 v) {
    const i64 i = blockIdx.x * (i64)256 + threadIdx.x;
    if (i < n) p[i] = v;
}

inline unsigned nblocks(i64 n, int tpb) { return (unsigned)((n + tpb - 1) / tpb); }

}  // namespace

extern "C" {

int sdpv_version(void) { return 1; }

#ifndef SDPV_SOURCE_HASH
#error "build with -DSDPV_SOURCE_HASH=<hash of the sources> (sdpvibe_amd/build.py does)"
#endif
uint64_t sdpv_source_hash(void) { return (uint64_t)SDPV_SOURCE_HASH; }

void* sdpv_host_alloc(int64_t bytes) {
    if (bytes <= 0) return nullptr;
    void* p = nullptr;
    if (hipHostMalloc(&p, (size_t)bytes, hipHostMallocDefault) != hipSuccess) return nullptr;
    return p;
}

int sdpv_host_free(void* p) {
    if (!p) return SDPV_OK;
    return hipHostFree(p) == hipSuccess ? SDPV_OK : SDPV_EARG;
}

int sdpv_shift_round(const int32_t* X, int64_t Lin, int64_t B, const int64_t* s, int32_t* out, int64_t Lout,
                     int32_t* flag, int32_t per_entry, void* stream) {
    if (B < 0 || Lin < 1 || Lout < 1) return SDPV_EARG;
    if (B == 0) return SDPV_OK;
    if (!X || !s || !out || !flag) return SDPV_EARG;
    hipLaunchKernelGGL(k_shift_round, dim3(nblocks(B, TPB)), dim3(TPB), 0, as_stream(stream), X, (i64)B, (int)Lin,
                       s, out, (int)Lout, flag, (int)per_entry);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_add_same(const int32_t* A, const int32_t* Bm, int32_t* out, int64_t L, int64_t B, int32_t sgn,
                  void* stream) {
    if (B < 0 || L < 1 || (sgn != 1 && sgn != -1)) return SDPV_EARG;
    if (B == 0) return SDPV_OK;
    if (!A || !Bm || !out) return SDPV_EARG;
    hipLaunchKernelGGL(k_add_same, dim3(nblocks(B, TPB)), dim3(TPB), 0, as_stream(stream), A, Bm, out, (int)L,
                       (i64)B, (int)(sgn < 0));
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_bitlen(const int32_t* X, int64_t L, int64_t B, int64_t* out, void* stream) {
    if (B < 0 || L < 1) return SDPV_EARG;
    if (B == 0) return SDPV_OK;
    if (!X || !out) return SDPV_EARG;
    hipLaunchKernelGGL(k_bitlen, dim3(nblocks(B, TPB)), dim3(TPB), 0, as_stream(stream), X, (int)L, (i64)B, out);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_mpf_top(const int32_t* m, const int64_t* e, int64_t L, int64_t n, int64_t* top, void* stream) {
    if (n < 0 || L < 1) return SDPV_EARG;
    if (n == 0) return SDPV_OK;
    if (!m || !e || !top) return SDPV_EARG;
    hipLaunchKernelGGL(k_mpf_top, dim3(nblocks(n, TPB)), dim3(TPB), 0, as_stream(stream), m, e, (int)L, (i64)n, top);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_badd_align(const int32_t* A, const int32_t* Bm, const int64_t* EA, const int64_t* EB, int32_t* out,
                    int64_t* EO, int64_t L, int64_t nb, int64_t rows, int64_t cols, int32_t sgn, void* stream) {
    if (L < 1 || nb < 0 || rows < 0 || cols < 0 || (sgn != 1 && sgn != -1)) return SDPV_EARG;
    const i64 entries = nb * rows * cols;
    if (entries == 0) return SDPV_OK;
    if (!A || !Bm || !EA || !EB || !out || !EO) return SDPV_EARG;
    hipLaunchKernelGGL(k_badd_align, dim3(nblocks(entries, TPB)), dim3(TPB), 0, as_stream(stream), A, Bm, EA, EB,
                       out, EO, (int)L, entries, (i64)rows, (i64)cols, (int)(sgn < 0));
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_copy_blocks(const sdpv_block* blocks, int64_t count, int32_t* m, int64_t* e, int64_t L, int64_t rows,
                     int64_t cols, int32_t to_stack, void* stream) {
    if (count < 0 || L < 1 || rows < 0 || cols < 0) return SDPV_EARG;
    const i64 n = rows * cols;
    if (count == 0 || n == 0) return SDPV_OK;
    if (!blocks || !m || !e) return SDPV_EARG;
    if (n > (1LL << 32) - TPB || L > 8 * 65535) return SDPV_ESIZE;   // 32-bit places, a launch's threads
    for (i64 j = 0; j < count; j++) {
        const sdpv_block& b = blocks[j];
        if (b.rows < 0 || b.cols < 0 || b.rows > rows || b.cols > cols) return SDPV_EARG;
        if (b.rows && b.cols && (!b.m || !b.e)) return SDPV_EARG;
    }
    for (i64 j0 = 0; j0 < count; j0 += BLOCKS) {
        BlockList list;
        const int c = (int)(count - j0 < BLOCKS ? count - j0 : BLOCKS);
        for (int j = 0; j < c; j++) list.b[j] = blocks[j0 + j];
        hipLaunchKernelGGL(k_copy_blocks, dim3(nblocks(n, TPB), (unsigned)c, (unsigned)((L + 7) / 8)), dim3(TPB), 0,
                           as_stream(stream), list, m, e, (int)L, (i64)count, (i64)j0, (i64)rows, (i64)cols, (int)to_stack);
        SDPV_TRY_LAUNCH();
    }
    return SDPV_OK;
}

int sdpv_stack_common(const int32_t* P1, const int64_t* e1, const int32_t* P2, const int64_t* e2, int32_t* out,
                      int64_t* EO, int64_t L, int64_t nb, int64_t R1, int64_t R2, int64_t C, int32_t* flag,
                      void* stream) {
    if (L < 1 || nb < 0 || R1 < 1 || R2 < 1 || C < 0) return SDPV_EARG;
    const i64 n = nb * (R1 + R2) * C;
    if (n == 0) return SDPV_OK;
    if (!P1 || !P2 || !e1 || !e2 || !out || !EO) return SDPV_EARG;
    hipLaunchKernelGGL(k_stack_common, dim3(nblocks(n, TPB)), dim3(TPB), 0, as_stream(stream), P1, e1, P2, e2, out, EO,
                       (int)L, (i64)nb, (i64)R1, (i64)R2, (i64)C, flag);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_mpf_norm(const int32_t* X, const int64_t* eI, int64_t LI, int32_t* O, int64_t* eO, int64_t L, int64_t n,
                  void* stream) {
    if (n < 0 || L < 1 || LI < 1) return SDPV_EARG;
    if (n == 0) return SDPV_OK;
    if (!X || !eI || !O || !eO) return SDPV_EARG;
    hipLaunchKernelGGL(k_mpf_norm, dim3(nblocks(n, TPB)), dim3(TPB), 0, as_stream(stream), X, eI, (int)LI, O, eO,
                       (int)L, (i64)n);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_mpf_mul(const int32_t* A, const int64_t* eA, const int32_t* Bm, const int64_t* eB, int32_t* O,
                 int64_t* eO, int64_t L, int64_t n, int32_t bscalar, void* stream) {
    if (n < 0 || L < 1) return SDPV_EARG;
    if (L > 128) return SDPV_ESIZE;
    if (n == 0) return SDPV_OK;
    if (!A || !eA || !Bm || !eB || !O || !eO) return SDPV_EARG;
#define SDPV_MUL(N)                                                                                              \
    if (L <= N) {                                                                                                \
        hipLaunchKernelGGL(k_mul_regs<N>, dim3(nblocks(n, 256)), dim3(256), 0, as_stream(stream), A, eA, Bm, eB, O, \
                           eO, (int)L, (i64)n, (int)(bscalar != 0));                                             \
        SDPV_TRY_LAUNCH();                                                                                       \
        return SDPV_OK;                                                                                          \
    }
    SDPV_MUL(8) SDPV_MUL(16) SDPV_MUL(24) SDPV_MUL(28) SDPV_MUL(32) SDPV_MUL(36) SDPV_MUL(40)
#undef SDPV_MUL
    const size_t lds = (size_t)4 * L * MUL_TPB * sizeof(u32);
    hipLaunchKernelGGL(k_mpf_mul, dim3(nblocks(n, MUL_TPB)), dim3(MUL_TPB), lds, as_stream(stream), A, eA, Bm, eB,
                       O, eO, (int)L, (i64)n, (int)(bscalar != 0));
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_mpf_add(const int32_t* A, const int64_t* eA, const int32_t* Bm, const int64_t* eB, int32_t* O,
                 int64_t* eO, int64_t L, int64_t n, int32_t sgn, void* stream) {
    if (n < 0 || L < 1 || (sgn != 1 && sgn != -1)) return SDPV_EARG;
    if (L > 256) return SDPV_ESIZE;
    if (n == 0) return SDPV_OK;
    if (!A || !eA || !Bm || !eB || !O || !eO) return SDPV_EARG;
#define SDPV_ADD(N)                                                                                              \
    if (L <= N) {                                                                                                \
        hipLaunchKernelGGL(k_add_regs<N>, dim3(nblocks(n, 256)), dim3(256), 0, as_stream(stream), A, eA, Bm, eB, O, \
                           eO, (int)L, (i64)n, (int)sgn);                                                        \
        SDPV_TRY_LAUNCH();                                                                                       \
        return SDPV_OK;                                                                                          \
    }
    SDPV_ADD(8) SDPV_ADD(16) SDPV_ADD(24) SDPV_ADD(28) SDPV_ADD(32) SDPV_ADD(36) SDPV_ADD(40)
#undef SDPV_ADD
    const size_t lds = (size_t)(L + 2) * ADD_TPB * sizeof(u32);
    hipLaunchKernelGGL(k_mpf_add, dim3(nblocks(n, ADD_TPB)), dim3(ADD_TPB), lds, as_stream(stream), A, eA, Bm, eB,
                       O, eO, (int)L, (i64)n, (int)sgn);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

int sdpv_row_exp(const int32_t* X, const int64_t* e, int64_t L, int64_t plane, int64_t nb, int64_t rows, int64_t K,
                 int64_t ldb, int64_t ldr, int64_t ldk, int64_t* Erow, void* stream) {
    if (L < 1 || nb < 0 || rows < 0 || K < 0) return SDPV_EARG;
    const i64 nrows = nb * rows;
    if (nrows == 0) return SDPV_OK;
    if (!X || !e || !Erow) return SDPV_EARG;
    hipStream_t st = as_stream(stream);
    if (ldk == 1) {
        hipLaunchKernelGGL(k_row_exp_wave, dim3(nblocks(nrows, 4)), dim3(256), 0, st, X, e, (int)L, (i64)plane, nrows,
                           (i64)rows, (i64)K, (i64)ldb, (i64)ldr, Erow);
    } else {
        // few row groups of 64: 16-row blocks when they are enough (32 or more, or a short k),
        // else split k as well, so that the launch fills the device
        const i64 groups = (nrows + 63) / 64;
        if (groups < 128 && K > 256 && ((nrows + 15) / 16 >= 32 || K <= 4096)) {
            hipLaunchKernelGGL(k_row_exp_cols16, dim3(nblocks(nrows, 16)), dim3(1024), 0, st, X, e, (int)L,
                               (i64)plane, nrows, (i64)rows, (i64)K, (i64)ldb, (i64)ldr, (i64)ldk, Erow);
            SDPV_TRY_LAUNCH();
            return SDPV_OK;
        }
        i64 parts = 1;
        if (groups < 128 && K > 256) {
            parts = (256 + groups - 1) / groups;
            const i64 kmax = (K + 127) / 128;
            parts = parts < kmax ? parts : kmax;
            if (parts > 65535) parts = 65535;
        }
        const i64 kchunk = (K + parts - 1) / parts;
        if (parts > 1)
            hipLaunchKernelGGL(k_fill_i64, dim3(nblocks(nrows, 256)), dim3(256), 0, st, Erow, nrows, (i64)EZV);
        hipLaunchKernelGGL(k_row_exp_cols, dim3((unsigned)groups, (unsigned)parts), dim3(1024), 0, st, X, e, (int)L,
                           (i64)plane, nrows, (i64)rows, (i64)K, (i64)ldb, (i64)ldr, (i64)ldk, kchunk, Erow);
    }
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

}  // extern "C"
