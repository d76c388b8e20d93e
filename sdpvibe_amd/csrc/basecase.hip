// Tile base case on gfx950: batched multiprecision Cholesky and triangular inverse of BT x BT
// tiles in wide fixed point (WL = L + 24 words, F = 32 L fractional bits), the arithmetic of the
// reference's chol_tiles / trinv_tiles (sdpvibe/basecase.py:13-246).
//
// Every product is the reference's truncated product mulfx (columns below LF - 2 dropped, signs
// applied to magnitudes), so results are bit-identical. Two forms of the product: one thread
// streams it word by word from LDS operands into its consumer (store, subtract, accumulate), or
// one wave holds a word per lane, sums the columns on the lanes and normalises them with shuffles
// and ballot carry-lookahead (lane_mul). When the tile's lower triangle fits in LDS
// (k_tile_chol_lds) the factorisation runs there and the inverse is built column-parallel
// (k_tile_inverse); otherwise k_tile_factor works on the tile in HBM.
#include <cstdlib>

#include "common.hpp"

namespace {

constexpr int TT = 256;  // threads per workgroup of k_tile_factor and k_tile_trsv

struct Slot {  // thread-strided word array in LDS
    u32* p;
    __device__ __forceinline__ u32& operator[](int k) const { return p[k * TT]; }
};

// copy |v| into slot s (WL words), return the sign of v
template <class Src>
__device__ __forceinline__ bool load_mag(Slot s, const Src& v, int WL) {
    const bool neg = (v(WL - 1) >> 31) != 0;
    u64 c = 1;
    for (int k = 0; k < WL; k++) {
        u32 w = v(k);
        if (neg) {
            const u64 t = (u64)(~w) + c;
            w = (u32)t;
            c = t >> 32;
        }
        s[k] = w;
    }
    return neg;
}

template <class S>
__device__ __forceinline__ int topl_slot(const S& s, int WL) {
    for (int i = WL - 1; i > 0; i--)
        if (s[i]) return i;
    return 0;
}

// column sum sum_{i=i0}^{i1} x[i] y[k - i] as 32-bit halves (lo: low words, hi: high words), eight
// terms at a time so that sixteen LDS reads are in flight before the multiplies use them
template <class X, class Y>
__device__ __forceinline__ void col_sum(const X& x, const Y& y, int k, int i0, int i1, u64& lo, u64& hi) {
    int i = i0;
    for (; i + 7 <= i1; i += 8) {
        u32 a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            a[u] = x[i + u];
            b[u] = y[k - i - u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const u64 p = (u64)a[u] * b[u];
            lo += (u32)p;
            hi += p >> 32;
        }
    }
    for (; i <= i1; i++) {
        const u64 p = (u64)x[i] * y[k - i];
        lo += (u32)p;
        hi += p >> 32;
    }
}

// Streams the magnitude words j = 0..WL-1 of mulfx(a, b, t) (sdpvibe/basecase.py:31-53) from the
// magnitudes x = |a|, y = |b| (word accessors x[i], y[i]); out(j, word). Columns kmin..LF-1 only
// feed the carry chain.
template <class X, class Y, class Out>
__device__ __forceinline__ void mulfx_mag(const X& x, const Y& y, int t, int WL, int LF, Out out) {
    const int ta = topl_slot(x, WL), tb = topl_slot(y, WL);
    const int la = t ? max(0, ta - t + 1) : 0, lb = t ? max(0, tb - t + 1) : 0;
    const int kmin = max(LF - 2, la + lb), kmax = ta + tb;
    u64 carry = 0, hprev = 0;
    auto column = [&](int k) -> u64 {
        u64 lo = 0, hi = 0;
        if (k <= kmax) col_sum(x, y, k, max(la, k - tb), min(ta, k - lb), lo, hi);
        const u64 sm = lo + hprev + carry;
        carry = sm >> 32;
        hprev = hi;
        return sm;
    };
    for (int k = kmin; k < LF && k <= kmax + 2; k++) column(k);
    for (int j = 0; j < WL; j++) {
        const int k = LF + j;
        out(j, (k >= kmin && k <= kmax + 2) ? (u32)column(k) : 0u);
    }
}

// the same product with the sign applied: out(j, word j of the two's complement result)
template <class Out>
__device__ __forceinline__ void mulfx_stream(Slot x, Slot y, bool neg, int t, int WL, int LF, Out out) {
    u64 nc = 1;
    mulfx_mag(x, y, t, WL, LF, [&](int j, u32 w) {
        if (neg) {
            const u64 tt = (u64)(~w) + nc;
            w = (u32)tt;
            nc = tt >> 32;
        }
        out(j, w);
    });
}

struct GlobalEntry {  // WL consecutive words in global memory
    const u32* p;
    __device__ __forceinline__ u32 operator()(int k) const { return p[k]; }
};
struct LdsEntry {
    const u32* p;
    __device__ __forceinline__ u32 operator()(int k) const { return p[k]; }
};

// ---------------------------------------------------------------- wave-level pivot arithmetic
// Arrays of WL words in LDS; called by all TT threads (threads >= 64 only meet the barriers).
struct Pivot {
    u32 *d, *r, *t1, *t2, *sx, *sy;
    u64* col;  // 2 * (2 WL + 4)
    int WL, LF;
};

__device__ __forceinline__ bool isneg_w(const u32* a, int WL) { return (a[WL - 1] >> 31) != 0; }

// r = mulfx(a, b, t) with the column sums spread over wave 0, the carry chain on lane 0
__device__ void wave_mul(const Pivot& P, u32* r, const u32* a, const u32* b, int t) {
    const int tid = threadIdx.x, WL = P.WL, LF = P.LF;
    __syncthreads();
    const bool sa = isneg_w(a, WL), sb = isneg_w(b, WL);
    if (tid == 0) {
        u64 ca = 1, cb = 1;
        for (int k = 0; k < WL; k++) {
            u32 x = a[k], y = b[k];
            if (sa) { const u64 q = (u64)(~x) + ca; x = (u32)q; ca = q >> 32; }
            if (sb) { const u64 q = (u64)(~y) + cb; y = (u32)q; cb = q >> 32; }
            P.sx[k] = x;
            P.sy[k] = y;
        }
    }
    __syncthreads();
    int ta = 0, tb = 0;
    for (int i = WL - 1; i > 0; i--)
        if (P.sx[i]) { ta = i; break; }
    for (int i = WL - 1; i > 0; i--)
        if (P.sy[i]) { tb = i; break; }
    const int la = t ? max(0, ta - t + 1) : 0, lb = t ? max(0, tb - t + 1) : 0;
    const int kmin = max(LF - 2, la + lb), kmax = ta + tb;
    if (tid < 64) {
        for (int k = kmin + tid; k <= kmax; k += 64) {
            u64 lo = 0, hi = 0;
            const int i0 = max(la, k - tb), i1 = min(ta, k - lb);
            for (int i = i0; i <= i1; i++) {
                const u64 p = (u64)P.sx[i] * P.sy[k - i];
                lo += (u32)p;
                hi += p >> 32;
            }
            P.col[2 * (k - kmin)] = lo;
            P.col[2 * (k - kmin) + 1] = hi;
        }
    }
    __syncthreads();
    if (tid == 0) {
        for (int j = 0; j < WL; j++) r[j] = 0;
        u64 carry = 0, hprev = 0;
        for (int k = kmin; k <= kmax + 2 && k < LF + WL; k++) {
            u64 lo = 0, hi = 0;
            if (k <= kmax) {
                lo = P.col[2 * (k - kmin)];
                hi = P.col[2 * (k - kmin) + 1];
            }
            const u64 sm = lo + hprev + carry;
            if (k >= LF) r[k - LF] = (u32)sm;
            carry = sm >> 32;
            hprev = hi;
        }
        if (sa ^ sb) {
            u64 c = 1;
            for (int j = 0; j < WL; j++) {
                const u64 q = (u64)(~r[j]) + c;
                r[j] = (u32)q;
                c = q >> 32;
            }
        }
    }
    __syncthreads();
}

__device__ double to_double_w(const u32* a, int WL, int LF) {  // basecase.py:59-68 (one thread)
    const bool s = isneg_w(a, WL);
    auto mag = [&](int k) {  // word k of |a|
        if (!s) return a[k];
        u64 c = 1;
        u32 w = 0;
        for (int q = 0; q <= k; q++) {
            const u64 t = (u64)(~a[q]) + c;
            w = (u32)t;
            c = t >> 32;
        }
        return w;
    };
    int t = 0;
    for (int k = WL - 1; k > 0; k--)
        if (mag(k)) { t = k; break; }
    double v = (double)mag(t);
    if (t >= 1) v = v * 4294967296.0 + (double)mag(t - 1);
    if (t >= 2) v = v * 4294967296.0 + (double)mag(t - 2);
    const int e = 32 * (t - 2 > 0 ? t - 2 : 0) - 32 * LF;
    v = ldexp(v, e);
    return s ? -v : v;
}

__device__ void from_double_w(u32* r, double v, int WL, int LF) {  // basecase.py:69-78
    for (int i = 0; i < WL; i++) r[i] = 0;
    if (!(v > 0.0) || !isfinite(v)) return;  // non-positive pivot: reciprocal 0
    int e;
    const double m = frexp(v, &e);
    u64 mi = (u64)ldexp(m, 53);
    int pos = e - 53 + 32 * LF;
    if (pos < 0) {
        mi = (-pos < 64) ? (mi >> (-pos)) : 0;
        pos = 0;
    }
    const int li = pos / 32, sh = pos % 32;
    u64 lo = mi << sh;
    u64 hi = sh ? (mi >> (64 - sh)) : 0;
    const u32 wds[4] = {(u32)lo, (u32)(lo >> 32), (u32)hi, (u32)(hi >> 32)};
    for (int k = 0; k < 4 && li + k < WL; k++) r[li + k] = wds[k];
}

// r = d^{-1/2}: double seed, Newton r <- r + r (1 - d r^2) / 2 with precision doubling
// (basecase.py:145-156)
__device__ void wave_rsqrt(const Pivot& P) {
    const int tid = threadIdx.x, WL = P.WL, LF = P.LF;
    if (tid == 0) from_double_w(P.r, 1.0 / sqrt(to_double_w(P.d, WL, LF)), WL, LF);
    for (int bits = 100;; bits *= 2) {
        int t = bits / 32 + 2;
        if (t >= WL) t = 0;
        wave_mul(P, P.t1, P.r, P.r, t);
        wave_mul(P, P.t2, P.t1, P.d, t);
        if (tid == 0) {  // t1 = one - t2
            i64 br = 0;
            for (int i = 0; i < WL; i++) {
                const i64 q = (i64)(i == LF ? 1u : 0u) - (i64)P.t2[i] + br;
                P.t1[i] = (u32)q;
                br = q >> 32;
            }
        }
        wave_mul(P, P.t2, P.r, P.t1, t);
        if (tid == 0) {  // r += t2 >> 1 (arithmetic)
            u64 c = 0;
            for (int i = 0; i < WL; i++) {
                const u32 hw = (i < WL - 1) ? ((P.t2[i] >> 1) | (P.t2[i + 1] << 31)) : (u32)(((int)P.t2[i]) >> 1);
                const u64 q = (u64)P.r[i] + hw + c;
                P.r[i] = (u32)q;
                c = q >> 32;
            }
        }
        __syncthreads();
        if (t == 0) break;
    }
}

// ---------------------------------------------------------------- lane-parallel pivot arithmetic
// For WL <= 64 a number is held by one wave with one word per lane (word k in lane k, zero in lanes >= WL):
// carries come from one 64-bit lookahead over ballots, and a product sums its columns on the lanes. The
// results are word for word those of wave_mul / wave_rsqrt above (the same truncated product).
//
// A 32 x 32 tile at L = 24 is bound by the latency of these products: a pivot is a chain of 16 of them. On
// one wave an instruction that depends on the one before costs 8 cycles, a ballot or a lane read whose
// scalar is used at once 30, and an LDS round trip 56 (in-kernel clock, one MI355X); so nothing but
// the operand words goes through LDS, magnitudes, signs and top words are found once per operand and not
// once per product, and the lane lookahead and the products are always inlined (out of line their LDS
// operands turn into flat accesses). The product took 2300 cycles out of line with its lane exchanges
// through the LDS crossbar.
__device__ __forceinline__ u32 lane_get(u32 v, int src) { return (u32)__shfl((int)v, src, 64); }
__device__ __forceinline__ u64 lane_get64(u64 v, int src) {
    return ((u64)lane_get((u32)(v >> 32), src) << 32) | lane_get((u32)v, src);
}
// value of the previous lane (0 in lane 0)
__device__ __forceinline__ u64 from_below64(u64 v) {
    const int l = lane_id();
    const u64 r = lane_get64(v, l > 0 ? l - 1 : 0);
    return l > 0 ? r : 0;
}

// LDS words of one wave's products: the left magnitude with zeros above, the right one with zeros on both
// sides (column c reads word c - i for every term i). Terms are read in groups that reach up to 32 past the
// top word ta <= LF + 23: words up to LF + 55 on the left, LF - 2 - ta - 32 to LF - 2 + 63 on the right
// (LF <= 40)
constexpr int LANE_X = 96, LANE_Y0 = 60, LANE_Y = LANE_Y0 + 104, LANE_LDS = LANE_X + LANE_Y;

// what the lane operations share: sizes, this lane's word mask (ones below WL), the wave's LDS words
struct Lane {
    int WL, LF;
    u32 in;
    u32* buf;
    __device__ __forceinline__ Lane(int wl, int lf, u32* b) : WL(wl), LF(lf), in(lane_id() < wl ? ~0u : 0u), buf(b) {
        for (int q = lane_id(); q < LANE_LDS; q += 64) buf[q] = 0u;
        wave_sync();
    }
};

// top word index of the number (>= 1), else 0 (topl_slot semantics)
__device__ __forceinline__ int lane_top(u32 w) {
    const u64 nz = ballot64(w != 0);
    return nz ? 63 - __builtin_clzll(nz) : 0;
}

// two's complement negation over WL words: ~w + 1, the +1 absorbed by the lowest nonzero word
__device__ __forceinline__ u32 lane_neg(const Lane& Q, u32 w) {
    const u64 nz = ballot64(w != 0);
    const u64 low = nz & (0 - nz);                       // the lowest nonzero word's lane
    return ((__builtin_amdgcn_inverse_ballot_w64(~(low | (low - 1))) ? ~w : 0u) |
            (__builtin_amdgcn_inverse_ballot_w64(low) ? 0u - w : 0u)) & Q.in;
}

// a + b + cin mod 2^(32 WL): generate / propagate masks from two ballots, the carry into every word
// from one 64-bit addition ((G|P) + G + cin) ^ (G|P) ^ G
__device__ __forceinline__ u32 lane_add(const Lane& Q, u32 a, u32 b, unsigned cin) {
    const u32 s = a + b;
    const u64 G = ballot64(s < a), P = ballot64(s == 0xffffffffu);
    const u64 X = G | P;
    return (s + mask_bit((X + G + cin) ^ X ^ G)) & Q.in;
}

// the words of sum_l (w0 + w1 2^32 + w2 2^64) 2^(32 l) over the lanes of `live` (a run of low lanes;
// w2 < 2^30), carries out of it dropped
__device__ __forceinline__ u32 lane_digits(u32 w0, u32 w1, u32 w2, u64 live) {
    const u64 d = (u64)w0 + lane_below(w1) + lane_below(lane_below(w2));
    const u32 d0 = (u32)d, e = d0 + lane_below((u32)(d >> 32));
    const u64 G = ballot64(e < d0) & live, P = ballot64(e == 0xffffffffu) & live;
    const u64 X = G | P;
    return e + mask_bit((X + G) ^ X ^ G);
}

// a number as magnitude, sign and top word
struct LaneMag {
    u32 m;
    int top;
    bool neg;
};
__device__ __forceinline__ LaneMag lane_mag(const Lane& Q, u32 a) {
    LaneMag r;
    r.neg = (lane_read(a, Q.WL - 1) >> 31) != 0;
    r.m = r.neg ? lane_neg(Q, a) : a;
    r.top = lane_top(r.m);
    return r;
}
// lane_mag of a number that has its top bit clear unless it overflowed: the sign is looked at only when
// the top word is set at all
__device__ __forceinline__ LaneMag lane_mag_pos(const Lane& Q, u32 a) {
    LaneMag r{a, lane_top(a), false};
    if (r.top == Q.WL - 1) r = lane_mag(Q, a);
    return r;
}
__device__ __forceinline__ u32 lane_signed(const Lane& Q, u32 w, bool neg) { return neg ? lane_neg(Q, w) : w; }

// Column sums of the magnitudes in Q.buf (x words la..ta, y words with zeros outside their range) as
// 96-bit values: the lane's column is LF - 2 + lane. HALF: the columns fit the lower 32 lanes; the two
// lane halves take the even and the odd terms and both end up with the sums. U terms per lane and
// group, all their words requested before the first multiply (terms past ta are zero): a group costs one
// LDS latency and 14 cycles a term.
template <bool HALF, int U>
__device__ __forceinline__ void lane_columns(const Lane& Q, int la, int ta, u64& s, u32& o) {
    constexpr int ST = HALF ? 2 : 1;                     // terms between two terms of one lane
    const int l = lane_id(), c = HALF ? (l & 31) : l, h = HALF ? (l >> 5) : 0;
    const u32* xp = Q.buf + la + h;
    const u32* yp = Q.buf + LANE_X + LANE_Y0 + Q.LF - 2 + c - la - h;
    s = 0;
    o = 0;
    for (int i = la; i <= ta; i += U * ST) {
        u32 x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            x[u] = xp[ST * u];
            y[u] = yp[-ST * u];
        }
#pragma unroll
        for (int u = 0; u < U; u += 4) SDPV_MAC96_CHAIN4(s, o, x + u, y + u);
        xp += U * ST;
        yp -= U * ST;
    }
    SDPV_SETTLE(s, o);
    if (HALF) {
        u32 a0 = (u32)s, b0 = a0, a1 = (u32)(s >> 32), b1 = a1, a2 = o, b2 = o;
        swap_halves(a0, b0);
        swap_halves(a1, b1);
        swap_halves(a2, b2);
        const u64 p = ((u64)a1 << 32) | a0, q = ((u64)b1 << 32) | b0;
        s = p + q;
        o = a2 + b2 + (s < p ? 1u : 0u);
    }
}

// columns beyond 64 (both operands far above one): two columns per lane, lane exchanges through the crossbar
__device__ __forceinline__ u32 lane_mul_wide(const u32* xs, const u32* ys, int la, int lb, int ta, int tb, int WL, int LF) {
    const int l = lane_id();
    const int kmin = max(LF - 2, la + lb), kmax = ta + tb;
    // column sums of columns kmin + l (h = 0) and kmin + 64 + l (h = 1) as lo / hi 32-bit halves
    u64 lo[2], hi[2];
    for (int h = 0; h < 2; h++) {
        const int k = kmin + l + 64 * h;
        u64 cl = 0, ch = 0;
        if (k <= kmax) col_sum(xs, ys, k, max(la, k - tb), min(ta, k - lb), cl, ch);
        lo[h] = cl;
        hi[h] = ch;
    }
    // V = sum_q (lo_q + hi_{q-1}) 2^(32 q), q = k - kmin over 128 positions (two per lane)
    // (every lane takes part in every shuffle; lane 0 of the upper half takes lane 63 of the lower)
    auto below = [&](u64 v0, u64 v1, u64& b0, u64& b1) {
        const u64 top = lane_get64(v0, 63), p0 = from_below64(v0), p1 = from_below64(v1);
        b0 = p0;
        b1 = l == 0 ? top : p1;
    };
    u64 b0, b1;
    below(hi[0], hi[1], b0, b1);
    const u64 s0 = lo[0] + b0, s1 = lo[1] + b1;
    // digits below 2^32 + 2^7: d_q = (s_q mod 2^32) + (s_{q-1} >> 32)
    below(s0 >> 32, s1 >> 32, b0, b1);
    const u64 d0 = (s0 & 0xffffffffull) + b0, d1 = (s1 & 0xffffffffull) + b1;
    // final digits: (d_q mod 2^32) + (d_{q-1} >> 32) + carry, the carries from a 128-bit lookahead
    below(d0 >> 32, d1 >> 32, b0, b1);
    const u64 e0 = (d0 & 0xffffffffull) + b0, e1 = (d1 & 0xffffffffull) + b1;
    const u64 G0 = __ballot((e0 >> 32) != 0), P0 = __ballot((u32)e0 == 0xffffffffu);
    const u64 G1 = __ballot((e1 >> 32) != 0), P1 = __ballot((u32)e1 == 0xffffffffu);
    const u64 X0 = G0 | P0, X1 = G1 | P1;
    const u64 sum0 = X0 + G0;
    const u64 C0 = sum0 ^ X0 ^ G0;
    const u64 C1 = (X1 + G1 + (sum0 < X0 ? 1u : 0u)) ^ X1 ^ G1;
    const u32 dig0 = (u32)e0 + (u32)((C0 >> l) & 1u), dig1 = (u32)e1 + (u32)((C1 >> l) & 1u);
    // output word j = digit of column LF + j
    const int q = LF + l - kmin;
    const u32 w0 = lane_get(dig0, q & 63), w1 = lane_get(dig1, q & 63);
    const u32 w = (l >= WL || q < 0 || q > kmax + 2 - kmin) ? 0u : (q < 64 ? w0 : w1);
    return w;
}

// magnitude of mulfx(a, b, t): columns from max(LF - 2, la + lb) on of the truncated operands. U: terms per
// lane and group of the half-wave form (2 U terms: 8 hold t <= 8, 16 hold t <= 16, 32 a number below
// one of up to 32 words)
template <int U>
__device__ __forceinline__ u32 lane_mul(const Lane& Q, const LaneMag& a, const LaneMag& b, int t) {
    const int l = lane_id(), ta = a.top, tb = b.top, LF = Q.LF;
    const int la = (t && ta >= t) ? ta - t + 1 : 0, lb = (t && tb >= t) ? tb - t + 1 : 0;
    wave_sync();                                         // earlier readers of the buffer are done
    Q.buf[l] = a.m;
    Q.buf[LANE_X + LANE_Y0 + l] = l >= lb ? b.m : 0u;
    wave_sync();
    // position q = column LF - 2 + q (columns below la + lb are empty), up to column ta + tb + 2
    const int npos = ta + tb - LF + 5;
    u64 s;
    u32 o, dig;
    if (__builtin_expect(npos <= 32, 1)) {
        lane_columns<true, U>(Q, la, ta, s, o);
        dig = lane_digits((u32)s, (u32)(s >> 32), o, 0xffffffffull);
        dig = l < 32 ? dig : 0u;
    } else if (npos <= 64) {
        lane_columns<false, 16>(Q, la, ta, s, o);
        dig = lane_digits((u32)s, (u32)(s >> 32), o, ~0ull);
    } else {
        return lane_mul_wide(Q.buf, Q.buf + LANE_X + LANE_Y0, la, lb, ta, tb, Q.WL, LF);
    }
    return lane_above(lane_above(dig)) & Q.in;           // output word j = digit of column LF + j
}

// mulfx(a, b, t) of two's complement lane numbers
__device__ __forceinline__ u32 lane_mulfx(const Lane& Q, u32 a, u32 b, int t) {
    const LaneMag x = lane_mag(Q, a), y = lane_mag(Q, b);
    return lane_signed(Q, lane_mul<16>(Q, x, y, t), x.neg != y.neg);
}

// basecase.py:59-68 on a lane number, the same value in every lane
__device__ __forceinline__ double lane_to_double(const LaneMag& a, int LF) {
    const int t = a.top;
    const u32 m0 = lane_read(a.m, t), m1 = lane_read(a.m, t >= 1 ? t - 1 : 0), m2 = lane_read(a.m, t >= 2 ? t - 2 : 0);
    double v = (double)m0;
    if (t >= 1) v = v * 4294967296.0 + (double)m1;
    if (t >= 2) v = v * 4294967296.0 + (double)m2;
    v = ldexp(v, 32 * (t - 2 > 0 ? t - 2 : 0) - 32 * LF);
    return a.neg ? -v : v;
}

// basecase.py:69-78: the lane's word of the fixed-point value of v (0 for non-positive v)
__device__ __forceinline__ u32 lane_from_double(double v, int WL, int LF) {
    const int l = lane_id();
    if (!(v > 0.0) || !isfinite(v) || l >= WL) return 0u;
    int e;
    const double m = frexp(v, &e);
    u64 mi = (u64)ldexp(m, 53);
    int pos = e - 53 + 32 * LF;
    if (pos < 0) {
        mi = (-pos < 64) ? (mi >> (-pos)) : 0;
        pos = 0;
    }
    const int li = pos / 32, sh = pos % 32;
    const u64 lo = mi << sh;
    const u64 hi = sh ? (mi >> (64 - sh)) : 0;
    const int k = l - li;
    return k == 0 ? (u32)lo : k == 1 ? (u32)(lo >> 32) : k == 2 ? (u32)hi : k == 3 ? (u32)(hi >> 32) : 0u;
}

// d^-1/2 (basecase.py:145-156): double seed, Newton steps r <- r + r (1 - d r^2) / 2 on t = bits / 32 + 2 words,
// bits = 100, 200, 400, ... (all words once t >= WL)
template <int U>
__device__ __forceinline__ u32 lane_newton(const Lane& Q, const LaneMag& d, u32 r, int t) {
    const int l = lane_id(), WL = Q.WL, LF = Q.LF;
    const LaneMag R = lane_mag_pos(Q, r);
    const LaneMag t1 = lane_mag_pos(Q, lane_mul<U>(Q, R, R, t));
    const u32 t2 = lane_mul<U>(Q, t1, d, t);
    // one - t2, t2 carrying the sign of its product
    const bool t2neg = t1.neg != d.neg;
    const LaneMag e = lane_mag(Q, lane_add(Q, l == LF ? 1u : 0u, (t2neg ? t2 : ~t2) & Q.in, t2neg ? 0u : 1u));
    const u32 h = lane_signed(Q, lane_mul<U>(Q, R, e, t), R.neg != e.neg);
    const u32 above = lane_above(h);                              // word l + 1
    const u32 half = (l < WL - 1) ? ((h >> 1) | (above << 31)) : (u32)(((int)h) >> 1);
    return lane_add(Q, r, half & Q.in, 0u);                       // r += h >> 1 (arithmetic)
}
// the seed and the steps on 5 and 8 words (bits = 100 and 200; WL >= 25)
__device__ __forceinline__ u32 lane_rsqrt_begin(const Lane& Q, const LaneMag& d) {
    u32 r = lane_from_double(1.0 / sqrt(lane_to_double(d, Q.LF)), Q.WL, Q.LF);
    for (int t = 5; t <= 8; t += 3) r = lane_newton<4>(Q, d, r, t);
    return r;
}
__device__ __forceinline__ u32 lane_rsqrt_finish(const Lane& Q, const LaneMag& d, u32 r) {
    r = lane_newton<8>(Q, d, r, 14);                              // bits = 400
    for (int bits = 800;; bits *= 2) {
        const int t = bits / 32 + 2 < Q.WL ? bits / 32 + 2 : 0;
        r = lane_newton<16>(Q, d, r, t);
        if (t == 0) return r;
    }
}

// ---------------------------------------------------------------- the tile kernel
// W, X, S: AoS (nb, BT, BT, WL) words in global memory (W: working copy, factored in place;
// X: L^-1; S: products of the inverse). LDS: 2 operand slots per thread + pivot area + RINV.
__global__ void __launch_bounds__(TT) k_tile_factor(u32* __restrict__ Wg, u32* __restrict__ Xg, u32* __restrict__ Sg,
                                                   u32* __restrict__ Rg, int BT, int WL, int LF) {
    SDPV_DYNAMIC_LDS(u32, lds);
    const int tid = threadIdx.x;
    const i64 tile = blockIdx.x;
    u32* W = Wg + tile * BT * BT * WL;
    u32* X = Xg + tile * BT * BT * WL;
    u32* S = Sg + tile * BT * BT * WL;
    Slot sx{lds + tid}, sy{lds + WL * TT + tid};
    u32* piv = lds + 2 * WL * TT;
    Pivot P;
    P.d = piv;
    P.r = piv + WL;
    P.t1 = piv + 2 * WL;
    P.t2 = piv + 3 * WL;
    P.sx = piv + 4 * WL;
    P.sy = piv + 5 * WL;
    u32* rinv = piv + 6 * WL;                            // BT x WL
    P.col = (u64*)(rinv + BT * WL + ((BT * WL) & 1));    // 2 (2 WL + 4) u64 (8-byte aligned)
    P.WL = WL;
    P.LF = LF;
    auto ent = [&](u32* base, int i, int j) { return base + ((i64)i * BT + j) * WL; };

    for (int k = 0; k < BT; k++) {
        // pivot: d = A_kk, r = d^-1/2, A_kk = d r, RINV_k = r
        if (WL <= 64) {                                   // one word per lane on wave 0
            if (tid < 64) {
                const Lane Q(WL, LF, (u32*)(P.col + 2 * (2 * WL + 4)));
                const u32 d = tid < WL ? ent(W, k, k)[tid] : 0u;
                const LaneMag dm = lane_mag(Q, d);
                const u32 r = lane_rsqrt_finish(Q, dm, lane_rsqrt_begin(Q, dm));
                const u32 dr = lane_mulfx(Q, d, r, 0);
                if (tid < WL) {
                    ent(W, k, k)[tid] = dr;
                    rinv[k * WL + tid] = r;
                    Rg[(tile * BT + k) * WL + tid] = r;
                }
            }
            __syncthreads();
        } else {
            for (int q = tid; q < WL; q += TT) P.d[q] = ent(W, k, k)[q];
            __syncthreads();
            wave_rsqrt(P);
            wave_mul(P, P.t1, P.d, P.r, 0);
            for (int q = tid; q < WL; q += TT) {
                ent(W, k, k)[q] = P.t1[q];
                rinv[k * WL + q] = P.r[q];
                Rg[(tile * BT + k) * WL + q] = P.r[q];
            }
            __syncthreads();
        }
        // column scale: A_ik = mulfx(A_ik, r)
        for (int i = k + 1 + tid; i < BT; i += TT) {
            u32* aik = ent(W, i, k);
            const bool na = load_mag(sx, GlobalEntry{aik}, WL);
            load_mag(sy, LdsEntry{rinv + k * WL}, WL);
            mulfx_stream(sx, sy, na ^ isneg_w(rinv + k * WL, WL), 0, WL, LF, [&](int j, u32 w) { aik[j] = w; });
        }
        __syncthreads();
        // trailing update over lower pairs: A_ij -= mulfx(A_ik, A_jk)
        const int m = BT - k - 1, npairs = m * (m + 1) / 2;
        for (int p = tid; p < npairs; p += TT) {
            int ii = (int)((sqrtf(8.0f * p + 1.0f) - 1.0f) * 0.5f);
            while ((ii + 1) * (ii + 2) / 2 <= p) ii++;
            while (ii * (ii + 1) / 2 > p) ii--;
            const int jj = p - ii * (ii + 1) / 2;
            const int i = k + 1 + ii, j = k + 1 + jj;
            const bool na = load_mag(sx, GlobalEntry{ent(W, i, k)}, WL);
            const bool nb = load_mag(sy, GlobalEntry{ent(W, j, k)}, WL);
            u32* aij = ent(W, i, j);
            i64 br = 0;
            mulfx_stream(sx, sy, na ^ nb, 0, WL, LF, [&](int jw, u32 w) {
                const i64 q = (i64)aij[jw] - (i64)w + br;
                aij[jw] = (u32)q;
                br = q >> 32;
            });
        }
        __syncthreads();
    }
    // clear the upper triangle; X = 0
    for (int e = tid; e < BT * BT; e += TT) {
        const int i = e / BT, j = e % BT;
        for (int q = 0; q < WL; q++) {
            if (j > i) W[(i64)e * WL + q] = 0;
            X[(i64)e * WL + q] = 0;
        }
    }
    __syncthreads();
    // X = L^-1 row by row: x_ii = rinv_i, x_ik = -rinv_i * sum_{j=k}^{i-1} l_ij x_jk
    for (int i = 0; i < BT; i++) {
        const int np = i * (i + 1) / 2;  // pairs k <= j < i
        for (int p = tid; p < np; p += TT) {
            int jj = (int)((sqrtf(8.0f * p + 1.0f) - 1.0f) * 0.5f);
            while ((jj + 1) * (jj + 2) / 2 <= p) jj++;
            while (jj * (jj + 1) / 2 > p) jj--;
            const int kk = p - jj * (jj + 1) / 2, j = jj;
            const bool na = load_mag(sx, GlobalEntry{ent(W, i, j)}, WL);
            const bool nb = load_mag(sy, GlobalEntry{ent(X, j, kk)}, WL);
            u32* s = ent(S, kk, j);
            mulfx_stream(sx, sy, na ^ nb, 0, WL, LF, [&](int jw, u32 w) { s[jw] = w; });
        }
        __syncthreads();
        for (int kk = tid; kk <= i; kk += TT) {
            u32* xik = ent(X, i, kk);
            if (kk == i) {
                for (int q = 0; q < WL; q++) xik[q] = rinv[i * WL + q];
                continue;
            }
            // acc = sum_j S[kk][j] (exact, wrapping) into slot sx, then x_ik = -(acc * rinv_i)
            u64 c = 0;
            for (int q = 0; q < WL; q++) {
                u64 sm = c;
                for (int j = kk; j < i; j++) sm += ent(S, kk, j)[q];
                sy[q] = (u32)sm;  // raw sum words in sy (two's complement)
                c = sm >> 32;
            }
            // magnitude of acc into sx
            const bool na = (sy[WL - 1] >> 31) != 0;
            u64 cc = 1;
            for (int q = 0; q < WL; q++) {
                u32 w = sy[q];
                if (na) { const u64 tq = (u64)(~w) + cc; w = (u32)tq; cc = tq >> 32; }
                sx[q] = w;
            }
            load_mag(sy, LdsEntry{rinv + i * WL}, WL);
            const bool neg = !(na ^ isneg_w(rinv + i * WL, WL));  // negated product
            mulfx_stream(sx, sy, neg, 0, WL, LF, [&](int jw, u32 w) { xik[jw] = w; });
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- LDS-resident factorisation
// For tiles whose lower triangle fits in LDS (WL <= 64 at BT = 32): the same recurrences as
// k_tile_factor, with the working tile in LDS. Products are formed either by one thread (the
// column sums in a loop, operands read from LDS) or by one wave with a word per lane (lane_mulfx);
// both are the truncated product of the magnitudes with the sign applied, so the results are those
// of k_tile_factor bit for bit (A - (-|p|) is A + |p| modulo 2^(32 WL)). The wave form has far
// less latency per product; the thread form does 256 products at once. The inverse is built by
// k_tile_inverse, one workgroup per (tile, column).
struct Row {  // consecutive words in LDS
    u32* p;
    __device__ __forceinline__ u32& operator[](int k) const { return p[k]; }
};

constexpr int TWAVES = TT / 64;

// words of the LDS-resident factorisation for BT, WL and nw waves (entries padded to an odd
// stride WS)
__host__ __device__ inline i64 lds_factor_words(int BT, int WL, int nw) {
    const i64 WS = WL | 1;
    return (i64)BT * (BT + 1) / 2 * WS + (i64)BT * WS + WL + 2 * BT + LANE_LDS * nw;
}

// row i of the packed lower triangle starts at entry i (i + 1) / 2
__device__ __forceinline__ int tri_base(int i) { return i * (i + 1) / 2; }

// index p of the pairs (i, j), 0 <= j <= i, in row order -> (i, j)
__device__ __forceinline__ void tri_pair(int p, int& i, int& j) {
    int r = (int)((sqrtf(8.0f * p + 1.0f) - 1.0f) * 0.5f);
    while ((r + 1) * (r + 2) / 2 <= p) r++;
    while (r * (r + 1) / 2 > p) r--;
    i = r;
    j = p - r * (r + 1) / 2;
}

// A -= s * mulfx(x, y, 0) on LDS words (s = +1, or -1 when `add`), taken where an operand has words above N
// (ta >= N or tb >= N; a factor of an SPD tile never has): x, y magnitudes with top words ta, tb, A a WL-word two's
// complement target. The column sums are formed four columns at a time: x[i] is read once per block and the four operand words y[kb + c - i] sit in a window of registers
// that shifts by one word per i, so a block costs two LDS reads per i instead of eight; the target
// words of a block are read before its columns are summed. The column sums, the carry chain and the
// target words equal those of mulfx_mag and its consumer (terms outside the tops are zero).
__device__ __forceinline__ void trail_update_any(const u32* x, const u32* y, int ta, int tb, int WL, int LF, u32* A,
                                             bool add) {
    const int kmin = max(LF - 2, 0), kmax = ta + tb, kend = LF + WL;
    u64 carry = 0, cy = 0;             // carry into the next column; carry of the addition
    i64 br = 0;                          // borrow of the subtraction
    for (int kb = kmin; kb < kend; kb += 4) {
        u32 tw[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int j = kb + c - LF;
            tw[c] = (j >= 0 && j < WL) ? A[j] : 0u;
        }
        u64 acc[4] = {0, 0, 0, 0};
        u32 ov[4] = {0, 0, 0, 0};
        if (kb <= kmax) {
            const int I0 = max(0, kb - tb), I1 = min(ta, kb + 3);
            u32 w[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int j = kb + c - I0;
                w[c] = j <= tb ? y[j] : 0u;
            }
            for (int i = I0; i <= I1; i += 4) {
                u32 xa[4], yn[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int ii = i + u, jn = kb - ii - 1;
                    xa[u] = ii <= I1 ? x[ii] : 0u;
                    yn[u] = (jn >= 0 && jn <= tb) ? y[jn] : 0u;
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    SDPV_MAC96_COLS4(acc, ov, xa[u], w);
                    w[3] = w[2];
                    w[2] = w[1];
                    w[1] = w[0];
                    w[0] = yn[u];
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int k = kb + c;
            if (k >= kend) break;
            u32 wv = 0u;
            if (k <= kmax + 2) {
                const u64 sm = acc[c] + carry;
                carry = (sm >> 32) | ((u64)(ov[c] + (sm < carry ? 1u : 0u)) << 32);
                wv = (u32)sm;
            }
            if (k >= LF) {
                if (add) {
                    const u64 q = (u64)tw[c] + wv + cy;
                    A[k - LF] = (u32)q;
                    cy = q >> 32;
                } else {
                    const i64 q = (i64)tw[c] - (i64)wv + br;
                    A[k - LF] = (u32)q;
                    br = q >> 32;
                }
            }
        }
    }
}

template <int N, int K>
struct TrailColumns {
    // columns K and up: digit of column k into word k - LF of A
    template <class Put>
    static __device__ __forceinline__ void run(const u32* x, const u32* y, int LF, u64& carry, Put& put) {
        if (K >= LF - 2) {                               // uniform: the first few columns only
            u64 acc;
            u32 ov;
            column_sum<N, K>(x, y, acc, ov);
            const u64 sm = acc + carry;
            carry = (sm >> 32) | ((u64)(ov + (sm < carry ? 1u : 0u)) << 32);
            if (K >= LF) put(K - LF, (u32)sm);
        }
        if constexpr (K < 2 * N - 2) TrailColumns<N, K + 1>::run(x, y, LF, carry, put);
    }
};

// A -= s * mulfx(x, y, 0) on LDS words (s = +1, or -1 when `add`) for magnitudes of at most N words: both
// operands in registers, every column's terms at static indexes, so that a product is its N (N + 1) / 2
// multiply-adds and 2 N LDS reads (6.5 thousand cycles at N = 24; reading the operands term by term from
// LDS took 38 thousand, more than the pivot chain that these updates run beside).
template <int N>
__device__ __forceinline__ void trail_update(const u32* xs, const u32* ys, int ta, int tb, int WL, int LF, u32* A,
                                             bool add) {
    if (ta >= N || tb >= N) {
        trail_update_any(xs, ys, ta, tb, WL, LF, A, add);
        return;
    }
    u32 x[N], y[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        x[i] = xs[i];
        y[i] = ys[i];
    }
    u64 carry = 0;
    u32 c = add ? 0u : 1u;                               // A + w, or A + ~w + 1
    const u32 flip = add ? 0u : ~0u;
    auto put = [&](int j, u32 w) {
        const u64 q = (u64)A[j] + (w ^ flip) + c;
        A[j] = (u32)q;
        c = (u32)(q >> 32);
    };
    constexpr int K0 = N > 8 ? N - 9 : 0;                // N - 8 < LF <= N (LF <= 8: N = 8)
    TrailColumns<N, K0>::run(x, y, LF, carry, put);
    for (int j = 2 * N - 1 - LF; j < WL; j++) {
        put(j, (u32)carry);
        carry >>= 32;
    }
}

// Pivot k: wave 0 computes r = d^-1/2 and d r (lane_rsqrt, lane_mulfx). Column scale: the waves take the
// entries i > k, L_ik = mulfx(A_ik, r), and keep |L_ik|, its top word and its sign for the trailing
// products; wave 0 takes entry k + 1 and updates the next diagonal entry with it, the other waves take
// the rest. Trailing update over the other pairs k < j <= i: wave 0 goes on to pivot k + 1 (look-ahead)
// while the other waves update the pairs, one per thread. Wave 0 runs the pivot's first Newton steps
// while the others scale, so a step is bound by wave 0's chain of products alone (18: one scale, one
// update, 16 for the pivot). N: words that hold every |L_ik| < 1 (N >= LF).
// 1024 threads (four waves per SIMD: 960 for the trailing products), fewer where the tile and the waves'
// operands would not fit in LDS together, or by SDPV_TILE_THREADS. Updates of at most `lane_pairs` pairs run one
// pair per wave instead (SDPV_TILE_LANE_PAIRS, 0 unless set: wave 0's chain hides them either way). One
// 32 x 32 tile at L = 24 on one MI355X: 0.334 ms (0.795 ms with products out of line and trailing operands
// read term by term from LDS); k_tile_inverse 0.088 ms (0.200 ms). DEFAULT: 1024 threads and no such pairs (known to
// the compiler: 2% on one tile, 4% on 400).
template <int N, bool DEFAULT>
__global__ void __launch_bounds__(1024) k_tile_chol_lds(u32* __restrict__ Wg, u32* __restrict__ Rg, int BT, int WL,
                                                       int LF, int lane_pairs) {
    const int NT = DEFAULT ? 1024 : blockDim.x, NW = NT >> 6;
    SDPV_DYNAMIC_LDS(u32, lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const i64 tile = blockIdx.x;
    const int WS = WL | 1;
    const int ne = BT * (BT + 1) / 2;
    u32* T = lds;                  // ne x WS: the lower triangle, row by row
    u32* CL = T + ne * WS;         // BT x WS: |L_ik| of the pivot column
    u32* RK = CL + BT * WS;        // WL: r of the pivot
    u32* SG = RK + WL;             // BT: sign of L_ik
    u32* TP = SG + BT;             // BT: top word of |L_ik|
    u32* PB = TP + BT + LANE_LDS * wave;  // the wave's lane_mulfx operands
    u32* W = Wg + tile * BT * BT * WL;
    auto te = [&](int i, int j) { return T + (i64)(tri_base(i) + j) * WS; };
    const int total = BT * BT * WL;
    const Lane Q(WL, LF, PB);
    // the lower triangle into LDS, 16 independent loads per thread in flight
    for (int base = tid; base < total; base += 16 * NT) {
        u32 v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int idx = base + u * NT;
            v[u] = idx < total ? W[idx] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int idx = base + u * NT;
            if (idx < total) {
                const int e = idx / WL, q = idx - e * WL, i = e / BT, j = e - i * BT;
                if (j <= i) te(i, j)[q] = v[u];
            }
        }
    }
    __syncthreads();
    // pivot k on wave 0, from the (updated) diagonal entry d held one word per lane: r = d^-1/2,
    // A_kk = mulfx(d, r), RINV_k = r; r0: the root after its first steps
    auto pivot = [&](int k, const LaneMag& d, u32 r0) {
        const u32 r = lane_rsqrt_finish(Q, d, r0);
        const LaneMag rm = lane_mag(Q, r);
        const u32 dr = lane_signed(Q, lane_mul<16>(Q, d, rm, 0), d.neg != rm.neg);
        if (lane < WL) {
            te(k, k)[lane] = dr;
            RK[lane] = r;
            Rg[(tile * BT + k) * WL + lane] = r;
        }
    };
    if (wave == 0) {
        const LaneMag d = lane_mag(Q, lane < WL ? te(0, 0)[lane] : 0u);
        pivot(0, d, lane_rsqrt_begin(Q, d));
    }
    __syncthreads();
    for (int k = 0; k < BT; k++) {
        // column scale: entry k + 1 on wave 0, which also updates the next diagonal entry (pair 0 of the
        // trailing update); the other entries on the other waves in turn
        const LaneMag rk = lane_mag(Q, lane < WL ? RK[lane] : 0u);
        auto scale = [&](int i) {
            u32* a = te(i, k);
            const LaneMag x = lane_mag(Q, lane < WL ? a[lane] : 0u);
            const u32 w = lane_mul<16>(Q, x, rk, 0);
            const bool neg = x.neg != rk.neg;
            const u32 lv = lane_signed(Q, w, neg);
            LaneMag v{w, lane_top(w), neg};
            if (v.top == WL - 1) v = lane_mag(Q, lv);    // the top bit of an overflowed product is a sign
            if (lane < WL) {
                a[lane] = lv;
                CL[(i64)i * WS + lane] = v.m;
            }
            if (lane == 0) {
                SG[i] = v.neg;
                TP[i] = v.top;
            }
            return v;
        };
        LaneMag dnext{0u, 0, false};
        u32 rnext = 0u;
        if (wave == 0) {
            if (k + 1 < BT) {
                const LaneMag v = scale(k + 1);
                u32* dk = te(k + 1, k + 1);
                dnext = lane_mag(Q, lane_add(Q, lane < WL ? dk[lane] : 0u, ~lane_mul<16>(Q, v, v, 0) & Q.in, 1u));
                rnext = lane_rsqrt_begin(Q, dnext);
            }
        } else {
            for (int i = k + 1 + wave; i < BT; i += NW - 1) scale(i);
        }
        __syncthreads();
        if (k == BT - 1) break;
        // trailing update over the lower pairs k < j <= i (all but pair 0): A_ij -= L_ik L_jk, while wave 0
        // finishes pivot k + 1
        const int m = BT - k - 1, npairs = m * (m + 1) / 2;
        if (wave == 0) {
            pivot(k + 1, dnext, rnext);
        } else if (!DEFAULT && npairs - 1 <= lane_pairs) {
            for (int p = wave; p < npairs; p += NW - 1) {
                int ii, jj;
                tri_pair(p, ii, jj);
                const int r = k + 1 + ii, c = k + 1 + jj;
                const LaneMag x = lane_mag(Q, lane < WL ? te(r, k)[lane] : 0u), y = lane_mag(Q, lane < WL ? te(c, k)[lane] : 0u);
                const u32 w = lane_signed(Q, lane_mul<16>(Q, x, y, 0), x.neg != y.neg);
                u32* a = te(r, c);
                const u32 v = lane_add(Q, lane < WL ? a[lane] : 0u, ~w & Q.in, 1u);
                if (lane < WL) a[lane] = v;
            }
        } else {
            for (int p = 1 + tid - 64; p < npairs; p += NT - 64) {
                int ii, jj;
                tri_pair(p, ii, jj);
                const int r = k + 1 + ii, c = k + 1 + jj;
                trail_update<N>(CL + (i64)r * WS, CL + (i64)c * WS, TP[r], TP[c], WL, LF, te(r, c), SG[r] != SG[c]);
            }
        }
        __syncthreads();
    }
    // the factor back, zeros above the diagonal
    for (int idx = tid; idx < total; idx += NT) {
        const int e = idx / WL, q = idx - e * WL, i = e / BT, j = e - i * BT;
        W[idx] = j <= i ? te(i, j)[q] : 0u;
    }
}

// words of k_tile_inverse's LDS for BT, WL and nw waves; the row prefetch takes BT WL <= 8 threads
__host__ __device__ inline i64 lds_inverse_words(int BT, int WL, int nw) {
    return 4 * (i64)BT * WL + 2 * (i64)nw * WL + LANE_LDS * nw;
}
constexpr int INV_PRE = 8;  // words of the next row each thread prefetches

// Column k of X = L^-1 for one tile (the recurrences of k_tile_factor's inverse):
// x_kk = rinv_k; for i > k, x_ik = -mulfx(sum_{j=k}^{i-1} mulfx(l_ij, x_jk), rinv_i), every product
// truncated, the sum exact (modulo 2^(32 WL)). Step i: the NT / 64 waves take the products j = k..i-1
// in turn and add them on the lanes, carries left pending; wave 0 adds the waves' sums, propagates the
// carries once and finishes x_ik with one more product. Row i + 1 of L is loaded while step i computes.
// Grid (nb, BT), 512 threads, or 256 or 1024 by SDPV_INV_THREADS. X entries above the diagonal are written as zeros.
template <bool DEFAULT>
__global__ void __launch_bounds__(DEFAULT ? 512 : 1024) k_tile_inverse(const u32* __restrict__ Wg, const u32* __restrict__ Rg,
                                                      u32* __restrict__ Xg, int BT, int WL, int LF) {
    const int NT = DEFAULT ? 512 : blockDim.x, NW = NT >> 6;
    SDPV_DYNAMIC_LDS(u32, lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const i64 tile = blockIdx.x;
    const int k = blockIdx.y;
    u32* XT = lds;                      // BT x WL: x_jk
    u32* RI = XT + BT * WL;             // BT x WL: rinv
    u32* LR = RI + BT * WL;             // 2 x BT x WL: rows of L (slot j holds l_ij), double buffered
    u32* PART = LR + 2 * BT * WL;       // NW x 2 WL: the waves' partial sums (low and high halves of 64 bits)
    const Lane Q(WL, LF, PART + 2 * NW * WL + LANE_LDS * wave);
    const u32* W = Wg + tile * BT * BT * WL;
    const u32* R = Rg + tile * BT * WL;
    u32* X = Xg + tile * BT * BT * WL;
    for (int idx = tid; idx < BT * WL; idx += NT) RI[idx] = R[idx];
    for (int i = 0; i < k; i++)
        for (int q = tid; q < WL; q += NT) X[((i64)i * BT + k) * WL + q] = 0u;
    // row k + 1 into buffer 0 (entries j = k..k, at slot j)
    if (k + 1 < BT)
        for (int idx = tid; idx < WL; idx += NT) LR[(i64)k * WL + idx] = W[((i64)(k + 1) * BT + k) * WL + idx];
    __syncthreads();
    if (wave == 0 && lane < WL) {       // x_kk = r_k
        const u32 r = RI[k * WL + lane];
        X[((i64)k * BT + k) * WL + lane] = r;
        XT[k * WL + lane] = r;
    }
    __syncthreads();
    for (int i = k + 1; i < BT; i++) {
        u32* cur = LR + ((i - k - 1) & 1) * BT * WL;
        u32* nxt = LR + ((i - k) & 1) * BT * WL;
        // prefetch row i + 1: (i + 1 - k) WL words from entry (i + 1, k)
        u32 pre[INV_PRE];
        const int nw = i + 1 < BT ? (i + 1 - k) * WL : 0;
        const u32* src = W + ((i64)(i + 1) * BT + k) * WL;
#pragma unroll
        for (int u = 0; u < INV_PRE; u++) {
            const int idx = tid + u * NT;
            pre[u] = idx < nw ? src[idx] : 0u;
        }
        // this wave's products, summed exactly: words of two's complement numbers in 64 bits per lane, the
        // carries left for the end (a negative product adds its complement and one)
        u64 acc = 0;
        for (int j = k + wave; j < i; j += NW) {
            const LaneMag lij = lane_mag(Q, lane < WL ? cur[j * WL + lane] : 0u);
            const LaneMag xjk = lane_mag(Q, lane < WL ? XT[j * WL + lane] : 0u);
            const u32 w = lane_mul<16>(Q, lij, xjk, 0);
            acc += lij.neg != xjk.neg ? (u64)(~w & Q.in) + (lane == 0 ? 1u : 0u) : (u64)w;
        }
        if (lane < WL) {
            PART[2 * wave * WL + lane] = (u32)acc;
            PART[(2 * wave + 1) * WL + lane] = (u32)(acc >> 32);
        }
#pragma unroll
        for (int u = 0; u < INV_PRE; u++) {
            const int idx = tid + u * NT;
            if (idx < nw) nxt[k * WL + idx] = pre[u];
        }
        __syncthreads();
        if (wave == 0) {
            u64 part = 0;                // at most BT words below 2^33 in all
            for (int w = 0; w < NW; w++)
                if (lane < WL)
                    part += ((u64)PART[(2 * w + 1) * WL + lane] << 32) + PART[2 * w * WL + lane];
            const LaneMag sum = lane_mag(Q, lane_digits((u32)part, (u32)(part >> 32), 0u, ~0ull) & Q.in);
            const LaneMag ri = lane_mag(Q, lane < WL ? RI[i * WL + lane] : 0u);
            const u32 x = lane_signed(Q, lane_mul<16>(Q, sum, ri, 0), sum.neg == ri.neg);
            if (lane < WL) {
                X[((i64)i * BT + k) * WL + lane] = x;
                XT[i * WL + lane] = x;
            }
        }
        __syncthreads();
    }
}

// Forward substitution L y = v for many vectors with one factored tile (the reference's trsv_warp,
// sdpvibe/basecase.py:228-245): 32 lanes per vector, lane i owns v_i (BT <= 32), kept in place in
// V (nvec, BT, WL). Step j: lane j scales y_j = mulfx(v_j, rinv_j); after the barrier every lane
// i > j subtracts mulfx(l_ij, y_j). All threads run every step (barriers), idle lanes included.
__global__ void __launch_bounds__(TT) k_tile_trsv(const u32* __restrict__ Lw, const u32* __restrict__ R,
                                                 u32* __restrict__ V, i64 nvec, int BT, int WL, int LF) {
    SDPV_DYNAMIC_LDS(u32, lds);
    const int tid = threadIdx.x, lane = tid & 31;
    const i64 vec = (i64)blockIdx.x * (TT / 32) + (tid >> 5);
    const bool live = vec < nvec && lane < BT;
    Slot sx{lds + tid}, sy{lds + WL * TT + tid};
    u32* vb = V + vec * BT * WL;
    for (int j = 0; j < BT; j++) {
        if (live && lane == j) {
            u32* vj = vb + (i64)j * WL;
            const u32* rj = R + (i64)j * WL;
            const bool na = load_mag(sx, GlobalEntry{vj}, WL);
            const bool nr = load_mag(sy, GlobalEntry{rj}, WL);
            mulfx_stream(sx, sy, na ^ nr, 0, WL, LF, [&](int q, u32 w) { vj[q] = w; });
        }
        __syncthreads();
        if (live && lane > j) {
            u32* vi = vb + (i64)lane * WL;
            const bool na = load_mag(sx, GlobalEntry{Lw + ((i64)lane * BT + j) * WL}, WL);
            const bool ny = load_mag(sy, GlobalEntry{vb + (i64)j * WL}, WL);
            i64 br = 0;
            mulfx_stream(sx, sy, na ^ ny, 0, WL, LF, [&](int q, u32 w) {
                const i64 d = (i64)vi[q] - (i64)w + br;
                vi[q] = (u32)d;
                br = d >> 32;
            });
        }
        __syncthreads();
    }
}

// The passes before and after the factorisation take one workgroup per tile row: its words are staged in LDS (one
// entry after the other, odd stride) so that both the planes and the entry-major words are read and written
// in runs, and every output word has a thread of its own. (With a thread per entry they were chains of L to
// WL dependent strided accesses: one 32 x 32 tile at L = 24 took 17.8 us to widen, 14.7 to narrow, and 60 for the
// bit lengths, their maximum and the rounding of the inverse; now 4.8, 7.1 and 6.0.)

// planes -> entry-major wide words, 40 more fractional bits; clears the tile's bit length
__global__ void __launch_bounds__(256) k_tile_widen(const i32* __restrict__ A, i64 plane, i64 ldb, i64 ldr, int BT, int L,
                                                    int WL, u32* __restrict__ W, int* __restrict__ top) {
    SDPV_DYNAMIC_LDS(u32, sm);
    const int t = threadIdx.x, S = L | 1;
    const i64 row = blockIdx.x, b = row / BT, i = row % BT;
    const i32* a = A + b * ldb + i * ldr;
    for (int x = t; x < L * BT; x += 256) sm[(x % BT) * S + x / BT] = (u32)a[(i64)(x / BT) * plane + x % BT];
    if (top && i == 0 && t == 0) top[b] = 0;
    __syncthreads();
    for (int x = t; x < WL * BT; x += 256) {
        const u32* v = sm + (x / WL) * S;
        const int k = x % WL;
        const u32 ext = (v[L - 1] >> 31) ? 0xffffffffu : 0u;
        const u32 lo = k < 2 ? 0u : (k - 2 < L ? v[k - 2] : ext), hi = k < 1 ? 0u : (k - 1 < L ? v[k - 1] : ext);
        W[row * BT * WL + x] = (lo >> 24) | (hi << 8);
    }
}

// the largest bit length of a tile's inverse (of ~v for v < 0, as limbops._bitlen_kernel)
__global__ void __launch_bounds__(256) k_tile_top(const u32* __restrict__ X, int BT, int WL, int* __restrict__ top) {
    SDPV_DYNAMIC_LDS(u32, sm);
    __shared__ int best;
    const int t = threadIdx.x, S = WL | 1;
    const i64 row = blockIdx.x;
    if (t == 0) best = 0;
    for (int x = t; x < WL * BT; x += 256) sm[(x / WL) * S + x % WL] = X[row * BT * WL + x];
    __syncthreads();
    int bl = 0;
    for (int x = t; x < WL * BT; x += 256) {
        const u32* v = sm + (x % BT) * S;
        const int k = x / BT;
        const u32 y = v[k] ^ ((v[WL - 1] >> 31) ? 0xffffffffu : 0u);
        if (y) bl = max(bl, 32 * k + 32 - clz32(y));
    }
    if (bl) atomicMax(&best, bl);
    __syncthreads();
    if (t == 0) atomicMax(top + row / BT, best);
}

// word k of round_half_up(v / 2^s) (s <= 0: exact left shift), v of n words: limbops._shift_round_kernel
struct LdsRow {
    const u32* p;
    __device__ __forceinline__ u32 operator()(int k) const { return p[k]; }
};
__device__ __forceinline__ u32 rounded_word(const u32* v, int n, i64 s, int k) {
    const LdsRow src{v};
    const u32 ext = (v[n - 1] >> 31) ? 0xffffffffu : 0u;
    const i64 q = s >> 5;
    const int r = (int)(s & 31);
    auto sh = [&](int j) {
        return (u32)((ext_word(src, n, ext, q + j) | ((u64)ext_word(src, n, ext, q + j + 1) << 32)) >> r);
    };
    u32 c = s < 1 ? 0u : (ext_word(src, n, ext, (s - 1) >> 5) >> (int)((s - 1) & 31)) & 1u;
    for (int j = k - 1; c && j >= 0; j--) c = sh(j) == 0xffffffffu ? 1u : 0u;   // the carry through words of ones
    return sh(k) + c;
}

// entry-major wide words -> planes: the factor rounded by 2^40 into L limbs, and the inverse as WL words
// (top null) or rounded to hb bits below its largest entry in the tile, with that exponent
__global__ void __launch_bounds__(256) k_tile_narrow(const u32* __restrict__ W, const u32* __restrict__ X, int BT, int L,
                                                     int WL, i32* __restrict__ Lout, i32* __restrict__ Xout,
                                                     i64 plane, const int* __restrict__ top, i64 hb,
                                                     i64* __restrict__ Xe, i32* __restrict__ flag) {
    SDPV_DYNAMIC_LDS(u32, sm);
    const int t = threadIdx.x, S = WL | 1;
    const i64 row = blockIdx.x, e0 = row * BT;
    u32* sx = sm + BT * S;
    for (int x = t; x < WL * BT; x += 256) {
        const int o = (x / WL) * S + x % WL;
        sm[o] = W[e0 * WL + x];
        sx[o] = X[e0 * WL + x];
    }
    __syncthreads();
    for (int x = t; x < (L + 1) * BT; x += 256) {
        const int k = x / BT, j = x % BT;
        const u32 w = rounded_word(sm + j * S, WL, 40, k);
        if (k < L) Lout[(i64)k * plane + e0 + j] = (i32)w;
        else if (flag && w != ((rounded_word(sm + j * S, WL, 40, L - 1) >> 31) ? 0xffffffffu : 0u)) atomicOr(flag, 1);
    }
    if (top) {
        const i64 s = top[row / BT] - hb;
        for (int x = t; x < L * BT; x += 256)
            Xout[(i64)(x / BT) * plane + e0 + x % BT] = (i32)rounded_word(sx + (x % BT) * S, WL, s, x / BT);
        if (row % BT == 0 && t < BT) Xe[row + t] = s - 32 * L;
    } else {
        for (int x = t; x < WL * BT; x += 256) Xout[(i64)(x / BT) * plane + e0 + x % BT] = (i32)sx[(x % BT) * S + x / BT];
    }
}

inline unsigned nblk(i64 n, int tpb) { return (unsigned)((n + tpb - 1) / tpb); }

// a setting of the environment, read once
inline int setting(const char* name, int unset) {
    const char* e = getenv(name);
    return e ? atoi(e) : unset;
}
// threads of the factorisation and, per column, of the inverse (see the kernels; the results are the same
// whatever they are)
inline int tile_threads() {
    static const int v = setting("SDPV_TILE_THREADS", 1024);
    return v == 256 || v == 512 ? v : 1024;
}
inline int inverse_threads() {
    static const int v = setting("SDPV_INV_THREADS", 512);
    return v == 256 || v == 1024 ? v : 512;
}
inline int tile_lane_pairs() {
    static const int v = setting("SDPV_TILE_LANE_PAIRS", 0);
    return v;
}

// the factorisation for magnitudes of N words
template <int N, bool DEFAULT>
int launch_factor_form(u32* W, u32* RI, i64 nb, int BT, int WL, int LF, int nt, size_t lds, hipStream_t st) {
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)k_tile_chol_lds<N, DEFAULT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    hipLaunchKernelGGL((k_tile_chol_lds<N, DEFAULT>), dim3((unsigned)nb), dim3(nt), lds, st, W, RI, BT, WL, LF,
                       tile_lane_pairs());
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}
template <int N>
int launch_factor(u32* W, u32* RI, i64 nb, int BT, int WL, int LF, int nt, size_t lds, hipStream_t st) {
    return nt == 1024 && tile_lane_pairs() <= 0 ? launch_factor_form<N, true>(W, RI, nb, BT, WL, LF, nt, lds, st)
                                                : launch_factor_form<N, false>(W, RI, nb, BT, WL, LF, nt, lds, st);
}

// Xe null: the inverse as WL words; else rounded to hb bits, its exponents (nb, BT) to Xe
int tile_run(const i32* A, i64 plane, i64 ldb, i64 ldr, i64 L, i64 nb, i64 BT, i32* Lout, i32* Xout, i64* Xe, i64 hb,
             u32* work, i32* flag, hipStream_t st) {
    if (L < 1 || nb < 0 || BT < 1 || BT > 64) return SDPV_EARG;
    if (nb == 0) return SDPV_OK;
    if (!A || !Lout || !Xout || !work) return SDPV_EARG;
    const int WL = (int)L + 24;
    const size_t lds = (size_t)2 * WL * TT * 4 + (size_t)(6 * WL + BT * WL + 2) * 4 + (size_t)2 * (2 * WL + 4) * 8 +
                       (WL <= 64 ? LANE_LDS * 4 : 0);
    if (lds > 160 * 1024) return SDPV_ESIZE;
    const i64 n = nb * BT * BT;
    u32* W = work;
    u32* X = work + n * WL;
    u32* S = work + 2 * n * WL;
    u32* RI = work + 3 * n * WL;
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)k_tile_factor, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void*)k_tile_widen, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void*)k_tile_top, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
        (void)hipFuncSetAttribute((const void*)k_tile_narrow, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    int* top = Xe ? (int*)(RI + nb * BT * WL) : nullptr;
    const i64 nrow = nb * BT;
    if (nrow > 0x7fffffffLL) return SDPV_ESIZE;
    hipLaunchKernelGGL(k_tile_widen, dim3((unsigned)nrow), dim3(256), (size_t)4 * BT * (L | 1), st, A, plane, ldb, ldr,
                       (int)BT, (int)L, WL, W, top);
    SDPV_TRY_LAUNCH();
    int nt = tile_threads(), ni = inverse_threads();
    auto lds_f = [&] { return (size_t)lds_factor_words((int)BT, WL, nt / 64) * 4; };
    while (nt > 256 && lds_f() > 160 * 1024) nt /= 2;   // a wave's operands take 1 KB: BT = 38 at L = 24 fits with eight
    while (ni < 512 && BT * WL > INV_PRE * ni) ni *= 2;
    const size_t lds_i = (size_t)lds_inverse_words((int)BT, WL, ni / 64) * 4;
    if (WL <= 64 && lds_f() <= 160 * 1024 && BT * WL <= INV_PRE * ni) {
        // the tile stays in LDS; the inverse one workgroup per column
        const int rc = L <= 8 ? launch_factor<8>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                     : L <= 16 ? launch_factor<16>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                     : L <= 24 ? launch_factor<24>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                     : L <= 28 ? launch_factor<28>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                     : L <= 32 ? launch_factor<32>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                     : L <= 36 ? launch_factor<36>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st)
                               : launch_factor<40>(W, RI, nb, (int)BT, WL, (int)L, nt, lds_f(), st);
        if (rc != SDPV_OK) return rc;
        if (ni == 512)
            hipLaunchKernelGGL(k_tile_inverse<true>, dim3((unsigned)nb, (unsigned)BT), dim3(ni), lds_i, st, W, RI, X,
                               (int)BT, WL, (int)L);
        else
            hipLaunchKernelGGL(k_tile_inverse<false>, dim3((unsigned)nb, (unsigned)BT), dim3(ni), lds_i, st, W, RI, X,
                               (int)BT, WL, (int)L);
        SDPV_TRY_LAUNCH();
    } else {
        hipLaunchKernelGGL(k_tile_factor, dim3((unsigned)nb), dim3(TT), lds, st, W, X, S, RI, (int)BT, WL, (int)L);
        SDPV_TRY_LAUNCH();
    }
    const size_t lds_row = (size_t)4 * BT * (WL | 1);
    if (top) {
        hipLaunchKernelGGL(k_tile_top, dim3((unsigned)nrow), dim3(256), lds_row, st, X, (int)BT, WL, top);
        SDPV_TRY_LAUNCH();
    }
    hipLaunchKernelGGL(k_tile_narrow, dim3((unsigned)nrow), dim3(256), 2 * lds_row, st, W, X, (int)BT, (int)L, WL, Lout,
                       Xout, n, top, hb, Xe, flag);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

}  // namespace

extern "C" {

int sdpv_tile_chol(const int32_t* A, int64_t L, int64_t nb, int64_t BT, int32_t* Lout, int32_t* Xw, uint32_t* work,
                   int32_t* flag, void* stream) {
    return tile_run(A, nb * BT * BT, BT * BT, BT, L, nb, BT, Lout, Xw, nullptr, 0, work, flag, as_stream(stream));
}

int sdpv_tile_chol_inv(const int32_t* A, int64_t plane, int64_t ldb, int64_t ldr, int64_t L, int64_t nb, int64_t BT,
                       int32_t* Lout, int32_t* X, int64_t* Xe, int64_t hb, uint32_t* work, int32_t* flag, void* stream) {
    if (nb > 0 && !Xe) return SDPV_EARG;
    return tile_run(A, plane, ldb, ldr, L, nb, BT, Lout, X, Xe, hb, work, flag, as_stream(stream));
}

int sdpv_tile_trsv(const uint32_t* Lw, const uint32_t* RINV, uint32_t* V, int64_t nvec, int64_t BT, int64_t WL,
                   int64_t LF, void* stream) {
    if (nvec < 0 || BT < 1 || BT > 32 || LF < 1 || WL < LF + 2) return SDPV_EARG;
    if (nvec == 0) return SDPV_OK;
    if (!Lw || !RINV || !V) return SDPV_EARG;
    const size_t lds = (size_t)2 * WL * TT * 4;
    if (lds > 160 * 1024) return SDPV_ESIZE;
    const i64 grid = (nvec + TT / 32 - 1) / (TT / 32);
    if (grid > 0x7fffffffLL) return SDPV_ESIZE;
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)k_tile_trsv, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    hipLaunchKernelGGL(k_tile_trsv, dim3((unsigned)grid), dim3(TT), lds, as_stream(stream), Lw, RINV, V, nvec,
                       (int)BT, (int)WL, (int)LF);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

}  // extern "C"
