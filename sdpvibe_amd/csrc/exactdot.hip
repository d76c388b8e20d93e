// Exact products of a batch of matrices with one or two (a few) vectors, formed directly on the INT8 matrix
// cores without residues. The residue path pays for every entry of the matrix with a byte product
// against the tables of all primes, whatever the number of columns; with one column the byte-by-byte
// product itself is cheaper: with the bytes of row i at inner index (k, u), u < 4L, and a Toeplitz operand
// holding byte c - u of the vector's entry k in row (k, u) and column c, one integer product per row gives
// the column sums S_c = sum_k sum_u a_{i,k,u} b_{k,c-u}, and S = sum_c S_c 256^c is the exact dot product.
//
// Digits. The matrix enters with its own bytes less 128 (the top one signed as it is: a = a' + 128 R with
// R = sum_{u < 4L-1} 256^u), the vector with exact signed digits (4L + 1 of them, bytes of b + 128 ... less
// 128). sum_k a b = sum_k a' b + 128 R sum_k b, and the second term depends on the vector alone.
//
// One or two rows with many columns: k_narrow_few. Otherwise a
// workgroup takes 32 rows, one column and a slice of at most 128 k. It turns the vector's slice into
// reversed digit strings in LDS once; then, for 16 k (8 when the limb count is large) at a time, each
// thread rounds one or two entries of the matrix to their row's exponent (or copies their limbs) into LDS as
// bytes while the next ones load, and each wave multiplies a quarter of the k on v_mfma_i32_32x32x32_i8:
// KS = ceil(L / 8) byte chunks against KS + 1 shifts of the vector's string, which are unaligned 16-byte
// windows of it (the lanes of a Toeplitz fragment differ by one byte each). The four waves' column
// sums meet in LDS; a slice's sums leave as 64-bit words, or, when there is one slice, the waves propagate
// the carries themselves, a word per lane, and round.
//
// Bound: reading the matrix for large products, the latency of the passes over LDS for small ones. One MI355X,
// L = 24: 60 blocks of 162 x 3000 against one vector each (3.0 GB) 1.55 ms, 2.0 TB/s, against 5.83 ms through
// residues; a 32 x 32 tile against one vector, rounded to its column, 0.022 ms in one launch against
// 0.058 ms for the product with a wave per entry and column sums on the lanes, and eight more launches for
// the rounding. A solve with one vector against a 1000 x 1000 factor: 348 launches instead of 1838.
#include <type_traits>

#include "common.hpp"

namespace {

constexpr int SLICE = 128;       // k of a workgroup: 128 * 4L * 2^14 stays inside 32 bits
constexpr int ROWS = 32;

// LDS geometry of a workgroup for KS 32-byte chunks per entry
template <int KS>
struct Geo {
    static constexpr int KC = KS <= 4 ? 16 : 8;             // k per step
    // from four chunks on, two groups of four waves share the column tiles: one group's sums alone would take
    // more registers than a wave of two per SIMD has
    static constexpr int GRP = KS <= 3 ? 1 : 2, NT = 256 * GRP, NWV = NT / 64, TPG = 2 * KS / GRP;
    static constexpr int EPT = KC * ROWS > NT ? KC * ROWS / NT : 1;   // entries per thread and step
    static constexpr int XS = 32 * KS + 16;                 // bytes of an entry (odd multiple of 16: no conflicts
    static constexpr int KROW = ROWS * XS + 16;             //   along rows, nor along k)
    static constexpr int SB = 32 * KS + 80;                 // bytes of a reversed string
    static constexpr int OFF = 32 * KS + 35;                // place of digit 0 in it
    static constexpr int COLS = 64 * KS;                    // column sums of a row
    static constexpr int CST = COLS + 4;                    // their stride (16-byte reads without conflicts)
    static constexpr int NWP = COLS / 4;                    // words of a slice's sums
    static constexpr int H = 2 * (8 * KS) + 2 > 64 ? 2 : 1;  // words of a result per lane
    static constexpr int A_BYTES = KC * KROW, S_BYTES = SLICE * SB, D_BYTES = 4 * (32 * KS + 4) + 4 * COLS;
    static constexpr int RED_BYTES = ROWS * CST * 4;        // column sums, over the entries' area
    static constexpr int V_BYTES = ROWS * (NWP + 1) * 8;    // 64-bit words, over the strings
    static constexpr int W_BYTES = ROWS * 64 * H * 4;       // finished words, over the entries' area
    static constexpr int mx(int a, int b) { return a > b ? a : b; }
    static constexpr int S_OFF = mx(A_BYTES, mx(RED_BYTES, W_BYTES));
    static constexpr int D_OFF = S_OFF + mx(S_BYTES, V_BYTES);
    static constexpr int LDS = D_OFF + D_BYTES + 4 * ROWS + 16;
};

struct Operand {                 // entry (b, r, k): limb w at p[w * plane + b * ldb + r * ldr + k * ldk]
    const i32* p;
    const i64 *e, *E;            // exponents (same offsets) and row exponents E[b * rows + r], or null: limbs as they are
    i64 plane, ldb, ldr, ldk;
};

enum { OUT_WORDS = 0, OUT_NORMALIZE = SDPV_NARROW_NORMALIZE, OUT_FIXED = SDPV_NARROW_FIXED, OUT_COL = SDPV_NARROW_COL,
       OUT_ACC = SDPV_NARROW_ACC };

struct Result {
    int mode;
    i32* out;                    // limb w of entry (b, i, j) at out[w * plane + b * ob + i * oi + j * oj]
    i64 plane, ob, oi, oj;
    i64* oute;                   // NORMALIZE: exponents at the same offset; WORDS: bit lengths (e); COL: (nb, N)
    int NW;                      // words of the exact result (2L + 2, or the caller's)
    i64 e0;                      // exponent of the product: e0 + ea[b * lea] + eb[b * N + j]
    const i64 *ea, *eb;
    i64 lea, oexp;               // FIXED: output exponent
    const i32* X;                // COL: out = X + sgn * product, both rounded to one above the larger exponent
    i64 planeX, xb, xi, xj;
    const i64* eX;
    int sgn;
    i32* flag;
};

struct Dims {
    i64 nb, M, N, K;
    int L, ns, ksl;              // slices and k per slice
};

// ------------------------------------------------------------------ a word per lane
__device__ __forceinline__ u64 lane_read64(u64 v, int src) {
    return ((u64)lane_read((u32)(v >> 32), src) << 32) | lane_read((u32)v, src);
}

// words of sum_w (lo_w + hi_w 2^32) 2^(32 w), w = lane + 64 h: lo_w < 2^51, |hi_w| < 2^51 (up to 2^19
// slices), modulo 2^(32 NW). A bias of 2^52 per word keeps every sum positive; it is taken off the finished digits.
template <int H>
__device__ __forceinline__ void carry_words(const u64* lo, const i64* hi, int NW, u32* w) {
    const int l = lane_id();
    u64 inj = 0, top = 0, cin = 1;
#pragma unroll
    for (int h = 0; h < H; h++) {
        u64 hb = ((u64)lane_below((u32)((u64)hi[h] >> 32)) << 32) | lane_below((u32)hi[h]);
        if (h > 0 && l == 0) hb = top;
        if (H > 1) top = lane_read64((u64)hi[h], 63);
        const u64 t = lo[h] + hb + (1ull << 52);
        const u32 t1 = (u32)(t >> 32);
        const u64 d = (t & 0xffffffffull) + lane_below(t1) + (l == 0 ? inj : 0);
        const u32 d0 = (u32)d, c = (u32)(d >> 32), e = d0 + lane_below(c);
        const u64 G = ballot64(e < d0), P = ballot64(e == 0xffffffffu), X = G | P, s = X + G;
        const u32 dig = e + mask_bit(s ^ X ^ G);
        if (H > 1) inj = (u64)lane_read(t1, 63) + lane_read(c, 63) + (s < X ? 1u : 0u);
        // less the bias: 2^20 in every word but the first
        const u32 y = dig + ~((h == 0 && l == 0) ? 0u : 0x100000u);
        const u64 Gb = ballot64(y < dig), Pb = ballot64(y == 0xffffffffu), Xb = Gb | Pb;
        const u64 s1 = Xb + Gb, s2 = s1 + cin;
        w[h] = l + 64 * h < NW ? y + mask_bit(s2 ^ Xb ^ Gb) : 0u;
        cin = (s1 < Xb || s2 < s1) ? 1u : 0u;
    }
}

template <int H>
struct Value {                   // NW words, two's complement, word lane + 64 h in w[h]
    u32 w[H];
    int NW;
    u32 ext;
    __device__ __forceinline__ void sign() {
        const int t = NW - 1;
        ext = (lane_read(H > 1 && t >= 64 ? w[H - 1] : w[0], t & 63) >> 31) ? ~0u : 0u;
    }
    __device__ __forceinline__ u32 at(int t) const {          // word t of the infinite extension (any t per lane)
        u32 v = (u32)__shfl((int)w[0], t & 63, 64);
        if (H > 1) {
            const u32 v1 = (u32)__shfl((int)w[H - 1], t & 63, 64);
            if (t >= 64) v = v1;
        }
        return t < 0 ? 0u : (t >= NW ? ext : v);
    }
    // index of the top word where word ^ x is nonzero (x: ext or 0), -1 if none; the lowest one in z
    __device__ __forceinline__ int top(u32 x, int& z) const {
        int t = -1;
        z = -1;
#pragma unroll
        for (int h = 0; h < H; h++) {
            const u64 m = ballot64(lane_id() + 64 * h < NW && (w[h] ^ x) != 0u);
            if (m) {
                t = 64 * h + 63 - __builtin_clzll(m);
                if (z < 0) z = 64 * h + __builtin_ctzll(m);
            }
        }
        return t;
    }
    __device__ __forceinline__ u32 word(int t) const {        // word t (uniform), 0 <= t < NW
        return lane_read(H > 1 && t >= 64 ? w[H - 1] : w[0], t & 63);
    }
    // bit length of v, of ~v when v < 0
    __device__ __forceinline__ int bitlen() const {
        int z;
        const int t = top(ext, z);
        return t < 0 ? 0 : 32 * t + 32 - clz32(word(t) ^ ext);
    }
    // words 0..63 of floor(v / 2^s) + c (word t in lane t); s uniform
    __device__ __forceinline__ u32 shifted(i64 s, u32 c, int L) const {
        const i64 smax = 32 * (i64)NW + 32, smin = -32 * ((i64)L + 2);
        s = s > smax ? smax : (s < smin ? smin : s);
        const int q = (int)(s >> 5), r = (int)(s & 31), l = lane_id();
        const u32 x = (u32)((((u64)at(l + q + 1) << 32) | at(l + q)) >> r);
        const u64 P = ballot64(x == 0xffffffffu);
        return x + mask_bit((P + c) ^ P);
    }
    // round_half_up(v / 2^s) into L < 64 words (0 above); bad when it does not fit them
    __device__ __forceinline__ u32 rounded(i64 s, int L, bool& bad) const {
        u32 c = 0;
        if (s >= 1) {
            const i64 t = (s - 1) >> 5;
            c = (at(t < NW ? (int)t : NW) >> (int)((s - 1) & 31)) & 1u;
            c = lane_read(c, 0);
        }
        const u32 y = shifted(s, c, L);
        bad = lane_read(y, L) != ((lane_read(y, L - 1) >> 31) ? ~0u : 0u);
        return lane_id() < L ? y : 0u;
    }
};

__device__ __forceinline__ i64 product_exp(const Result& R, i64 N, i64 b, i64 j) {
    return R.e0 + (R.ea ? R.ea[b * R.lea] : 0) + (R.eb ? R.eb[b * N + j] : 0);
}

// a product rounded to words at its column's exponent ec (COL), added to X when there is one
__device__ __forceinline__ void emit_col(const Result& R, const Dims& D, i64 b, i64 i, i64 j, u32 cw, i64 ec) {
    const int l = lane_id(), L = D.L;
    if (R.X) {
        const i64 eX = R.eX[b * D.N + j], ex = (eX > ec ? eX : ec) + 1;
        Value<1> x, c;
        x.NW = c.NW = L;
        x.w[0] = l < L ? (u32)R.X[l * R.planeX + b * R.xb + i * R.xi + j * R.xj] : 0u;
        c.w[0] = cw;
        x.sign();
        c.sign();
        bool bad;
        const u32 xa = x.rounded(ex - eX, L, bad);
        u32 ca = c.rounded(ex - ec, L, bad);
        if (R.sgn < 0) ca = l < L ? ~ca : 0u;
        const u32 s = xa + ca;
        const u64 G = ballot64(s < xa), P = ballot64(s == 0xffffffffu), X = G | P;
        cw = s + mask_bit((X + G + (R.sgn < 0 ? 1u : 0u)) ^ X ^ G);
    }
    if (l < L) R.out[l * R.plane + b * R.ob + i * R.oi + j * R.oj] = (i32)cw;
}

// every mode but COL, from the exact words of entry (b, i, j)
template <int H>
__device__ __forceinline__ void emit(const Result& R, const Dims& D, const Operand& A, const Operand& B, i64 b, i64 i,
                                     i64 j, Value<H>& v) {
    const int l = lane_id(), L = D.L;
    const i64 e = (b * D.M + i) * D.N + j, o = b * R.ob + i * R.oi + j * R.oj;
    if (R.mode == OUT_WORDS) {
        v.sign();
#pragma unroll
        for (int h = 0; h < H; h++)
            if (l + 64 * h < v.NW) R.out[(i64)(l + 64 * h) * R.plane + e] = (i32)v.w[h];
        for (int t = v.NW + l; t < R.NW; t += 64) R.out[(i64)t * R.plane + e] = (i32)v.ext;
        const int bl = v.bitlen();
        if (l == 0) R.oute[e] = bl;
    } else if (R.mode == OUT_ACC) {                       // exact words added to those of the entry
        u64 cin = 0;
#pragma unroll
        for (int h = 0; h < H; h++) {
            const bool in = l + 64 * h < R.NW;
            i32* p = R.out + e * R.NW + l + 64 * h;
            const u32 a = in ? (u32)*p : 0u, s = a + v.w[h];
            const u64 G = ballot64(s < a), P = ballot64(s == 0xffffffffu), X = G | P, s1 = X + G, s2 = s1 + cin;
            if (in) *p = (i32)(s + mask_bit(s2 ^ X ^ G));
            cin = (s1 < X || s2 < s1) ? 1u : 0u;
        }
    } else if (R.mode == OUT_FIXED) {
        v.sign();
        bool bad;
        const u32 y = v.rounded(R.oexp - product_exp(R, D.N, b, j), L, bad);
        if (l < L) R.out[l * R.plane + o] = (i32)y;
        if (bad && R.flag && l == 0) atomicOr(R.flag, 1);
    } else {                                              // NORMALIZE: magnitude half up to 32 L - 2 bits
        v.sign();
        const bool neg = v.ext != 0u;
        int z, zz;
        const int T = v.top(v.ext, zz);
        (void)v.top(0u, z);                               // z: lowest nonzero word
        const u32 vz = z >= 0 ? v.word(z) : 0u;
        int bl;
        if (!neg) bl = T < 0 ? 0 : 32 * T + 32 - clz32(v.word(T));
        else bl = T > z ? 32 * T + 32 - clz32(~v.word(T)) : 32 * z + 32 - clz32(0u - vz);
        if (bl == 0) {
            if (l < L) R.out[l * R.plane + o] = 0;
            if (l == 0) R.oute[o] = EZV;
            return;
        }
        const int sv = bl - (32 * L - 2);
        u32 c = 0;
        if (sv > 0) {
            const u32 rb = (v.word((sv - 1) >> 5) >> ((sv - 1) & 31)) & 1u;
            c = (rb && (!neg || 32 * z + __builtin_ctz(vz) < sv - 1)) ? 1u : 0u;
        }
        const u32 y = v.shifted(sv, c, L);
        if (l < L) R.out[l * R.plane + o] = (i32)y;
        if (l == 0) R.oute[o] = (A.E ? A.E[b * D.M + i] : 0) + (B.E ? B.E[b * D.N + j] : 0) + sv;
    }
}

// ------------------------------------------------------------------ the product
struct PlaneWords {
    const i32* p;
    i64 plane;
    __device__ __forceinline__ u32 operator()(int k) const { return (u32)p[(i64)k * plane]; }
};
struct SlotWords {
    const u32* p;
    __device__ __forceinline__ u32 operator()(int k) const { return p[k]; }
};

__device__ __forceinline__ i64 round_shift(const Operand& X, i64 row, i64 off) {
    if (!X.e) return 0;
    const i64 e = X.e[off];
    return e == EZV ? (i64)1 << 30 : X.E[row] - e;
}

// KM: the entries' threads run along k (contiguous) instead of rows
template <int KS, bool KM>
__global__ void __launch_bounds__(Geo<KS>::NT, KS <= 3 ? 2 : 1) k_narrow(Operand A, Operand B, Dims D, Result R, i64* __restrict__ part,
                                                              u32* __restrict__ words, i32* __restrict__ bls) {
    using g = Geo<KS>;
    SDPV_DYNAMIC_LDS(unsigned char, lds);
    unsigned char* ent = lds;                             // [KC][ROWS] entries of XS bytes
    unsigned char* str = lds + g::S_OFF;                  // [SLICE] strings of SB bytes
    int* dsum = (int*)(lds + g::D_OFF);                   // digit sums of the slice's vector entries
    int* corr = dsum + 32 * KS + 4;                       // the columns' 128 R sum_k b
    int* blrow = corr + g::COLS;                          // bit lengths of the rows (COL)
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hsel = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = D.L, NB = 4 * L;
    const i64 nrt = (D.M + ROWS - 1) / ROWS;
    i64 id = blockIdx.x;
    const i64 rt = id % nrt;
    id /= nrt;
    const int sl = (int)(id % D.ns);
    id /= D.ns;
    const i64 j = id % D.N, b = id / D.N;
    const i64 k0 = (i64)sl * D.ksl, k1 = k0 + D.ksl < D.K ? k0 + D.ksl : D.K;
    const int nk = (int)(k1 - k0), steps = (nk + g::KC - 1) / g::KC;
    const i64 r0 = rt * ROWS;

    // this thread's entries of a step: rows er + q RQ (clamped to the matrix), k ek + q KQ
    constexpr int RQ = KM ? g::NT / g::KC : 0, KQ = KM ? 0 : g::NT / ROWS;
    const int er = KM ? tid / g::KC : tid % ROWS, ek = KM ? tid % g::KC : tid / ROWS;
    auto arow = [&](int q) { return r0 + er + q * RQ < D.M ? r0 + er + q * RQ : D.M - 1; };
    auto aoff = [&](int st, int q) {                      // k past the slice meets zero digits
        const i64 k = k0 + (i64)st * g::KC + ek + q * KQ;
        return b * A.ldb + arow(q) * A.ldr + (k < D.K ? k : 0) * A.ldk;
    };
    const bool act = g::KC * ROWS >= g::NT || tid < g::KC * ROWS;   // uniform per wave
    u32 pre[g::EPT][8 * KS];                              // limbs on their way
    i64 sh[g::EPT];
    auto fetch = [&](int st) {
#pragma unroll
        for (int q = 0; q < g::EPT; q++) {
            if (!act) break;
            const i64 off = aoff(st, q);
            sh[q] = round_shift(A, b * D.M + arow(q), off);
            const i32* p = A.p + off;
#pragma unroll
            for (int w = 0; w < 8 * KS; w++) {
                pre[q][w] = (u32)*p;                      // words past L - 1 re-read word L - 1
                if (w + 1 < L) p += A.plane;
            }
        }
    };
    constexpr bool AHEAD = KS <= 4;                       // the next step's limbs load beside the products (registers)
    if (AHEAD && steps > 0) fetch(0);

    // ---- the vector's slice as reversed signed digits, an entry per thread (its limbs requested at once)
    {
        const i64 kb = k0 + (tid < nk ? tid : 0);
        const i64 off = b * B.ldb + j * B.ldr + (kb < D.K ? kb : 0) * B.ldk;
        u32 y[8 * KS];
        i64 s = 0;
#pragma unroll
        for (int w = 0; w < 8 * KS; w++) y[w] = 0;
        if (tid < nk) {
            const i32* p = B.p + off;
#pragma unroll
            for (int w = 0; w < 8 * KS; w++) {
                y[w] = (u32)*p;
                if (w + 1 < L) p += B.plane;
            }
            s = round_shift(B, b * D.N + j, off);
        }
        for (int q = tid; q < SLICE * g::SB / 16; q += g::NT) ((v4i*)str)[q] = v4i{0, 0, 0, 0};
        for (int q = tid; q <= NB; q += g::NT) dsum[q] = 0;
        __syncthreads();
        u32 ext;
        if (tid < SLICE) round_words<8 * KS>(y, L, s < 0 ? 0 : s, ext, (v4i*)(ent + tid * g::XS));   // whole waves
        if (tid < nk) {
            u32* sw = (u32*)(str + tid * g::SB + g::OFF - 3);  // word w of the digits, reversed, at sw[-w]
            u32 c = 0, last = 0;
            auto put = [&](int w, u32 v) {
                const u64 t = (u64)v + 0x80808080u + c;
                c = (u32)(t >> 32);
                last = v;
                sw[-w] = __builtin_bswap32((u32)t ^ 0x80808080u);
            };
            if (s >= 0) {
#pragma unroll
                for (int w = 0; w < 8 * KS; w++)
                    if (w < L) put(w, y[w]);
            } else {                                      // an entry that is not normalised: a left shift
                (void)shr_round_batched(PlaneWords{B.p + off, B.plane}, L, s, L, put);
            }
            sw[-L] = ((c - (last >> 31)) & 0xffu) << 24;   // the digit above: -1, 0 or 1
        }
        __syncthreads();
    }
    // digit sums of the slice: a thread takes four places of every (NT / LD)-th entry
    {
        constexpr int LD = KS <= 1 ? 16 : KS <= 3 ? 32 : KS <= 7 ? 64 : 128;
        static_assert(LD >= 8 * KS + 1, "places");
        const int d = tid % LD;
        if (d <= L) {
            int s0 = 0, s1 = 0, s2 = 0, s3 = 0;
            for (int k = tid / LD; k < nk; k += g::NT / LD) {
                const u32 v = *((const u32*)(str + k * g::SB + g::OFF - 3) - d);
                s0 += (int)v >> 24;
                s1 += (int)(v << 8) >> 24;
                s2 += (int)(v << 16) >> 24;
                s3 += (int)(v << 24) >> 24;
            }
            atomicAdd(dsum + 4 * d, s0);
            if (d < L) {
                atomicAdd(dsum + 4 * d + 1, s1);
                atomicAdd(dsum + 4 * d + 2, s2);
                atomicAdd(dsum + 4 * d + 3, s3);
            }
        }
        __syncthreads();
        // prefix sums on wave 0 (four places a lane), then 128 R sum_k b per column: the digit sums of a window of
        // 4L - 1 places that ends at the column
        if (wave == 0) {
            int v[4], t = 0;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                t += 4 * lane + u <= NB ? dsum[4 * lane + u] : 0;
                v[u] = t;
            }
            int sc = t;
            for (int o = 1; o < 64; o <<= 1) {
                const int x = __shfl(sc, lane - o, 64);
                sc += lane >= o ? x : 0;
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (4 * lane + u <= NB) dsum[4 * lane + u] = v[u] + sc - t;
        }
        __syncthreads();
        for (int c = tid; c < g::COLS; c += g::NT)
            corr[c] = 128 * (dsum[c < NB ? c : NB] - (c - (NB - 1) >= 0 ? dsum[c - (NB - 1) < NB ? c - (NB - 1) : NB] : 0));
    }

    v16i acc[g::TPG];
#pragma unroll
    for (int t = 0; t < g::TPG; t++)
#pragma unroll
        for (int u = 0; u < 16; u++) acc[t][u] = 0;
    // column sums of this wave's k of a step, tiles [T0, T0 + TPG)
    auto products = [&](int st, auto t0) {
        constexpr int T0 = decltype(t0)::value;
        for (int kk = wave & 3; kk < g::KC; kk += 4) {
            const u32* sp = (const u32*)(str + (st * g::KC + kk) * g::SB);
            const int base = g::OFF + 16 * hsel - l32, sb = base & 3;
            v4i tf[KS + 1];
#pragma unroll
            for (int q = 0; q <= KS; q++) {               // digits c - u of the tiles q apart
                if (g::GRP == 2 && q == (T0 ? 0 : KS)) continue;   // meets no tile of this group
                const u32* p = sp + ((base - 32 * q) >> 2);
                u32 x[5];
#pragma unroll
                for (int u = 0; u < 5; u++) x[u] = p[u];
#pragma unroll
                for (int u = 0; u < 4; u++) tf[q][u] = (int)__builtin_amdgcn_alignbyte(x[u + 1], x[u], (u32)sb);
            }
            const unsigned char* ep = ent + kk * g::KROW + l32 * g::XS + 16 * hsel;
#pragma unroll
            for (int x = 0; x < KS; x++) {
                const v4i af = *(const v4i*)(ep + 32 * x);
#pragma unroll
                for (int q = 0; q <= KS; q++)
                    if (x + q >= T0 && x + q < T0 + g::TPG)
                        acc[x + q - T0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, tf[q], acc[x + q - T0], 0, 0, 0);
            }
        }
    };

    for (int st = 0; st < steps; st++) {
        if (!AHEAD) fetch(st);
        // ---- entries to bytes
#pragma unroll
        for (int q = 0; q < g::EPT; q++) {
            if (!act) break;
            unsigned char* slot = ent + (ek + q * KQ) * g::KROW + (er + q * RQ) * g::XS;
            if (A.e) {
                if (sh[q] < 0) {                          // an entry that is not normalised: a left shift
                    i32* sw = (i32*)slot;
                    (void)shr_round_batched(PlaneWords{A.p + aoff(st, q), A.plane}, L, sh[q], L,
                                            [&](int w, u32 v) { sw[w] = (i32)v; });
#pragma unroll
                    for (int w = 0; w < 8 * KS; w++) pre[q][w] = w < L ? (u32)sw[w] : 0u;
                }
                u32 ext;
                round_words<8 * KS>(pre[q], L, sh[q] < 0 ? 0 : sh[q], ext, (v4i*)slot);
            }
            // every byte less 128 but the signed top one, zeros above
#pragma unroll
            for (int w = 0; w < 2 * KS; w++) {
                u32 x[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int i = 4 * w + u;
                    x[u] = i < L ? pre[q][i] ^ (i == L - 1 ? 0x00808080u : 0x80808080u) : 0u;
                }
                ((v4i*)slot)[w] = v4i{(int)x[0], (int)x[1], (int)x[2], (int)x[3]};
            }
        }
        __syncthreads();
        if (AHEAD && st + 1 < steps) fetch(st + 1);
        if (g::GRP == 1 || wave < 4) products(st, std::integral_constant<int, 0>{});
        else products(st, std::integral_constant<int, (g::GRP == 1 ? 0 : KS)>{});
        __syncthreads();
    }

    // ---- the waves' sums together, as 64-bit words
    int* red = (int*)ent;
    for (int q = tid; q < ROWS * g::CST / 4; q += g::NT) ((v4i*)red)[q] = v4i{0, 0, 0, 0};
    __syncthreads();
#pragma unroll
    for (int t = 0; t < g::TPG; t++)
#pragma unroll
        for (int u = 0; u < 16; u++)
            atomicAdd(red + (8 * (u >> 2) + 4 * hsel + (u & 3)) * g::CST + 32 * (t + (wave >> 2) * g::TPG) + l32, acc[t][u]);
    __syncthreads();
    i64* vw = (i64*)str;
    for (int q = tid; q < ROWS * g::NWP; q += g::NT) {
        const int r = q / g::NWP, w = q % g::NWP;
        const v4i s = *(const v4i*)(red + r * g::CST + 4 * w);
        i64 v = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            v += ((i64)s[u] + corr[4 * w + u]) << (8 * u);
        }
        if (D.ns > 1) {
            if (r0 + r < D.M) part[(((i64)sl * D.nb + b) * D.M + r0 + r) * D.N * g::NWP + j * g::NWP + w] = v;
        } else {
            vw[r * (g::NWP + 1) + w] = v;
        }
    }
    if (D.ns > 1) return;
    __syncthreads();
    // ---- one slice: finished here
    u32* wl = (u32*)ent;                                  // COL: [ROWS][64 H] words
#pragma unroll 1
    for (int r4 = wave; r4 < ROWS; r4 += 4 * g::NWV) {    // four rows at a time: their carry chains interleave
        if (r0 + r4 >= D.M) break;                        // uniform
        Value<g::H> val[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            u64 lo[g::H];
            i64 hi[g::H];
#pragma unroll
            for (int h = 0; h < g::H; h++) {
                const int w = lane + 64 * h;
                const i64 v = w < g::NWP ? vw[(r4 + g::NWV * q) * (g::NWP + 1) + w] : 0;
                lo[h] = (u32)v;
                hi[h] = v >> 32;
            }
            val[q].NW = min(R.NW, 64 * g::H);
            carry_words<g::H>(lo, hi, val[q].NW, val[q].w);
            val[q].sign();
        }
        int bl[4];
        if (R.mode == OUT_COL) {
#pragma unroll
            for (int q = 0; q < 4; q++) bl[q] = val[q].bitlen();
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = r4 + g::NWV * q;
            if (r0 + r >= D.M) break;                     // uniform
            if (R.mode != OUT_COL) {
                emit<g::H>(R, D, A, B, b, r0 + r, j, val[q]);
            } else if (D.M <= ROWS) {
#pragma unroll
                for (int h = 0; h < g::H; h++) wl[(r * g::H + h) * 64 + lane] = val[q].w[h];
                if (lane == 0) blrow[r] = bl[q];
            } else {                                      // more rows elsewhere: k_narrow_round goes on
                const i64 e = (b * D.M + r0 + r) * D.N + j;
#pragma unroll
                for (int h = 0; h < g::H; h++) words[(e * g::H + h) * 64 + lane] = val[q].w[h];
                if (lane == 0) bls[e] = bl[q];
            }
        }
    }
    if (R.mode != OUT_COL || D.M > ROWS) return;
    __syncthreads();
    int mxb = lane < (int)D.M ? blrow[lane & 31] : 0;
    for (int o = 16; o >= 1; o >>= 1) mxb = max(mxb, __shfl_xor(mxb, o, 64));
    mxb = __builtin_amdgcn_readfirstlane(mxb);
    const i64 s = (i64)mxb - (32 * L - 32), ec = product_exp(R, D.N, b, j) + s;
    if (tid == 0) R.oute[b * D.N + j] = R.X ? max((long long)R.eX[b * D.N + j], (long long)ec) + 1 : ec;
#pragma unroll 1
    for (int r4 = wave; r4 < (int)D.M; r4 += 4 * g::NWV) {
        u32 cw[4];
        bool any = false;
#pragma unroll
        for (int q = 0; q < 4; q++) {                     // rows past M: words of an earlier use, not stored
            const int r = r4 + g::NWV * q;
            Value<g::H> val;
            val.NW = R.NW;
#pragma unroll
            for (int h = 0; h < g::H; h++) val.w[h] = r < (int)D.M ? wl[(r * g::H + h) * 64 + lane] : 0u;
            val.sign();
            bool bad;
            cw[q] = val.rounded(s, L, bad);
            any |= bad;
        }
        if (any && R.flag && lane == 0) atomicOr(R.flag, 1);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (r4 + g::NWV * q < (int)D.M) emit_col(R, D, b, r4 + g::NWV * q, j, cw[q], ec);
    }
}

// One or two rows: a workgroup of k_narrow has 32 of them and prepares its vector for all, so that most of its
// work would be done for nothing. Here a wave takes a column (or a slice of its k) and one row after the
// other: lane c sums column c (and c + 64) of the unsigned word products over k, 64 k at a time in LDS (odd
// stride: lanes at different words use different banks), with the corrections that make the top words
// signed (a = a_unsigned - s_a 2^(32 L)), then carries and rounds, or leaves the slice's word sums. Operands as
// they are (no exponents). Bound: LDS reads. 3000 columns of one row, K = 42, rounded to their column: 54 us
// at L = 24 (148 in k_narrow), 506 at L = 63 (2452).
constexpr int FEW_M = 2, FEW_KC = 64, FEW_KS = FEW_KC + 1;
template <int H>
__global__ void __launch_bounds__(256) k_narrow_few(Operand A, Operand B, Dims D, Result R, i64* __restrict__ part) {
    SDPV_DYNAMIC_LDS(unsigned char, lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), L = D.L;
    const i64 cols = D.nb * D.N, task = blockIdx.x * (i64)4 + wave;
    if (task >= cols * D.ns) return;                      // uniform per wave; no workgroup barrier below
    const i64 col = task % cols, sl = task / cols, b = col / D.N, j = col % D.N;
    const i64 k1 = (sl + 1) * D.ksl < D.K ? (sl + 1) * D.ksl : D.K;
    u32* As = (u32*)lds + wave * 2 * L * FEW_KS;
    u32* Bs = As + L * FEW_KS;
    Value<H> val[FEW_M];
    int mx = 0;
#pragma unroll
    for (int i = 0; i < FEW_M; i++) {
        if (i >= (int)D.M) break;                         // uniform
        const i32* ap = A.p + b * A.ldb + i * A.ldr;
        const i32* bp = B.p + b * B.ldb + j * B.ldr;
        i64 lo[H], hi[H];                                 // below 2^(12 + 6 + 32): within carry_words
#pragma unroll
        for (int h = 0; h < H; h++) lo[h] = hi[h] = 0;
        for (i64 k0 = sl * D.ksl; k0 < k1; k0 += FEW_KC) {
            const int kc = (int)(k1 - k0 < FEW_KC ? k1 - k0 : FEW_KC), kr = (kc + 3) & ~3;   // words past kc are zero
            wave_sync();                                  // the previous chunk has been read
            for (int u = 0; u < L; u++) {
                As[u * FEW_KS + lane] = lane < kc ? (u32)ap[u * A.plane + (k0 + lane) * A.ldk] : 0u;
                Bs[u * FEW_KS + lane] = lane < kc ? (u32)bp[u * B.plane + (k0 + lane) * B.ldk] : 0u;
            }
            wave_sync();
#pragma unroll
            for (int h = 0; h < H; h++) {
                const int c = lane + 64 * h;
                if (c > 2 * L) continue;
                const int u0 = c - (L - 1) > 0 ? c - (L - 1) : 0, u1 = c < L - 1 ? c : L - 1;
                for (int u = u0; u <= u1; u++) {
                    const u32 *x = As + u * FEW_KS, *y = Bs + (c - u) * FEW_KS;
                    for (int k = 0; k < kr; k += 4) {
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            const u64 q = (u64)x[k + t] * y[k + t];
                            lo[h] += (i64)(u32)q;
                            hi[h] += (i64)(q >> 32);
                        }
                    }
                }
                if (c >= L) {
                    const u32 *at = As + (L - 1) * FEW_KS, *bt = Bs + (L - 1) * FEW_KS;
                    const int q = c < 2 * L ? c - L : 0;
                    for (int k = 0; k < kc; k++) {
                        const u32 sa = at[k] >> 31, sb = bt[k] >> 31;
                        if (c < 2 * L) lo[h] -= (i64)(sa ? Bs[q * FEW_KS + k] : 0u) + (i64)(sb ? As[q * FEW_KS + k] : 0u);
                        else lo[h] += (i64)(sa & sb);
                    }
                }
            }
        }
        if (D.ns > 1) {                                   // word c gets the upper half of column c - 1
            i64* p = part + (sl * cols * D.M + (b * D.M + i) * D.N + j) * (2 * L + 2);
            u64 top = 0;
#pragma unroll
            for (int h = 0; h < H; h++) {
                u64 hb = ((u64)lane_below((u32)((u64)hi[h] >> 32)) << 32) | lane_below((u32)hi[h]);
                if (h > 0 && lane == 0) hb = top;
                if (H > 1) top = lane_read64((u64)hi[h], 63);
                if (lane + 64 * h < 2 * L + 2) p[lane + 64 * h] = lo[h] + (i64)hb;
            }
            continue;
        }
        val[i].NW = min(R.NW, 64 * H);
        carry_words<H>((const u64*)lo, hi, val[i].NW, val[i].w);
        if (R.mode != OUT_COL) {
            emit<H>(R, D, A, B, b, i, j, val[i]);
            continue;
        }
        val[i].sign();
        mx = max(mx, val[i].bitlen());
    }
    if (D.ns > 1 || R.mode != OUT_COL) return;
    const i64 s = (i64)mx - (32 * L - 32), ec = product_exp(R, D.N, b, j) + s;
    if (lane == 0) R.oute[b * D.N + j] = R.X ? max((long long)R.eX[b * D.N + j], (long long)ec) + 1 : ec;
#pragma unroll
    for (int i = 0; i < FEW_M; i++) {
        if (i >= (int)D.M) break;
        bool bad;
        const u32 cw = val[i].rounded(s, L, bad);
        if (bad && R.flag && lane == 0) atomicOr(R.flag, 1);
        emit_col(R, D, b, i, j, cw, ec);
    }
}

// the slices' words (nwp each) added and carried, a wave per entry; COL leaves words and bit lengths for
// k_narrow_round
template <int H>
__global__ void __launch_bounds__(256) k_narrow_finish(const i64* __restrict__ part, int nwp, Operand A, Operand B, Dims D,
                                                      Result R, u32* __restrict__ words, i32* __restrict__ bls) {
    const int lane = threadIdx.x & 63;
    const i64 E = D.nb * D.M * D.N, e = blockIdx.x * (i64)4 + (threadIdx.x >> 6);
    if (e >= E) return;                                   // uniform per wave; no workgroup barrier below
    u64 lo[H];
    i64 hi[H];
#pragma unroll
    for (int h = 0; h < H; h++) {
        lo[h] = 0;
        hi[h] = 0;
        const int w = lane + 64 * h;
        if (w < nwp) {
            const i64* p = part + e * nwp + w;
            const i64 step = E * nwp;
            int s = 0;
            for (; s + 8 <= D.ns; s += 8) {               // eight loads in flight
                i64 v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = p[(s + u) * step];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    lo[h] += (u32)v[u];
                    hi[h] += v[u] >> 32;
                }
            }
            for (; s < D.ns; s++) {
                const i64 v = p[s * step];
                lo[h] += (u32)v;
                hi[h] += v >> 32;
            }
        }
    }
    Value<H> val;
    val.NW = min(R.NW, 64 * H);
    carry_words<H>(lo, hi, val.NW, val.w);
    const i64 j = e % D.N, i = e / D.N % D.M, b = e / (D.N * D.M);
    if (R.mode != OUT_COL) {
        emit<H>(R, D, A, B, b, i, j, val);
        return;
    }
    val.sign();
    const int bl = val.bitlen();
#pragma unroll
    for (int h = 0; h < H; h++) words[(e * H + h) * 64 + lane] = val.w[h];
    if (lane == 0) bls[e] = bl;
}

// COL over more than 32 rows: the column's largest bit length (every workgroup reads the column's, 4 bytes a
// row), then a wave per entry rounds, adds and stores. rpw: rows of a workgroup
template <int H>
__global__ void __launch_bounds__(256) k_narrow_round(const u32* __restrict__ words, const i32* __restrict__ bls, Dims D,
                                                     Result R, i64 rpw) {
    __shared__ int part[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const i64 nrw = (D.M + rpw - 1) / rpw;
    i64 id = blockIdx.x;
    const i64 rw = id % nrw;
    id /= nrw;
    const i64 j = id % D.N, b = id / D.N;
    int mx = 0;
    for (i64 i = tid; i < D.M; i += 256) mx = max(mx, bls[(b * D.M + i) * D.N + j]);
    for (int o = 32; o >= 1; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) part[wave] = mx;
    __syncthreads();
    mx = max(max(part[0], part[1]), max(part[2], part[3]));
    const i64 s = (i64)__builtin_amdgcn_readfirstlane(mx) - (32 * D.L - 32), ec = product_exp(R, D.N, b, j) + s;
    if (rw == 0 && tid == 0) R.oute[b * D.N + j] = R.X ? max((long long)R.eX[b * D.N + j], (long long)ec) + 1 : ec;
    const i64 i1 = (rw + 1) * rpw < D.M ? (rw + 1) * rpw : D.M;
    for (i64 i = rw * rpw + wave; i < i1; i += 4) {
        const i64 e = (b * D.M + i) * D.N + j;
        Value<H> val;
        val.NW = R.NW;
#pragma unroll
        for (int h = 0; h < H; h++) val.w[h] = words[(e * H + h) * 64 + lane];
        val.sign();
        bool bad;
        const u32 cw = val.rounded(s, D.L, bad);
        if (bad && R.flag && lane == 0) atomicOr(R.flag, 1);
        emit_col(R, D, b, i, j, cw, ec);
    }
}

// accumulated words (OUT_ACC) -> normalised entries
template <int H>
__global__ void __launch_bounds__(256) k_narrow_result(const i32* __restrict__ acc, Operand A, Operand B, Dims D, Result R) {
    const int lane = threadIdx.x & 63;
    const i64 e = blockIdx.x * (i64)4 + (threadIdx.x >> 6);
    if (e >= D.nb * D.M * D.N) return;
    Value<H> val;
    val.NW = R.NW;
#pragma unroll
    for (int h = 0; h < H; h++) val.w[h] = lane + 64 * h < R.NW ? (u32)acc[e * R.NW + lane + 64 * h] : 0u;
    emit<H>(R, D, A, B, e / (D.N * D.M), e / D.N % D.M, e % D.N, val);
}

// slices of K: at most SLICE k, shorter ones (multiples of 16) while the launch has fewer than 512
// workgroups; the sums are exact, so the partition changes no result
inline void slices(i64 nb, i64 M, i64 N, i64 K, Dims& D) {
    const i64 wg = nb * N * ((M + ROWS - 1) / ROWS);
    i64 ns = (K + SLICE - 1) / SLICE;
    const i64 want = (512 + wg - 1) / (wg > 0 ? wg : 1), nmax = (K + 31) / 32;
    if (want > ns) ns = want < nmax ? want : nmax;
    if (ns < 1) ns = 1;
    i64 len = ((K + ns - 1) / ns + 15) / 16 * 16;
    if (len < 16) len = 16;
    D.ksl = (int)len;
    D.ns = (int)(K > 0 ? (K + len - 1) / len : 1);
}

// slices of k_narrow_few: multiples of 64 k, at most 4096, shorter ones while the launch has fewer than FEW_WAVES waves
constexpr i64 FEW_K = 4096, FEW_WAVES = 2048;
inline void few_slices(i64 nb, i64 N, i64 K, Dims& D) {
    const i64 cols = nb * N, nmax = (K + FEW_KC - 1) / FEW_KC;
    i64 ns = (K + FEW_K - 1) / FEW_K;
    const i64 want = (FEW_WAVES + cols - 1) / (cols > 0 ? cols : 1);
    if (want > ns) ns = want < nmax ? want : nmax;
    if (ns < 1) ns = 1;
    const i64 len = ((K + ns - 1) / ns + FEW_KC - 1) / FEW_KC * FEW_KC;
    D.ksl = (int)(len > 0 ? len : FEW_KC);
    D.ns = (int)(K > 0 ? (K + D.ksl - 1) / D.ksl : 1);
}
inline int chunks(i64 L) { return (int)((L + 7) / 8); }
inline int lane_words(i64 L) { return 16 * chunks(L) + 2 > 64 ? 2 : 1; }

// Whether one or two rows take k_narrow_few: its time grows with the rows and k, k_narrow's with the columns and the
// slices of 128 k that they start, the faster the more limbs. us for one row at 1024 columns of 42 k / 512 of 200 /
// 128 of 3000, few (k_narrow): L = 8 24 / 34 / 84 (22 / 27 / 74), L = 24 39 / 62 / 189 (52 / 82 / 257), L = 35
// 67 / 106 / 310 (133 / 220 / 727), L = 48 107 / 323 / 941 (322 / 642 / 2126); two rows and two columns a block, 512
// blocks of 42 k / 256 of 200 / 256 of 1000: L = 24 76 / 113 / 471 (53 / 84 / 334), L = 35 127 / 200 / 772
// (134 / 225 / 970), L = 48 206 / 605 / 2398 (325 / 649 / 2809)
inline bool takes_few(i64 L, i64 nb, i64 M, i64 N, i64 K) {
    if (M > FEW_M) return false;
    const int ks = chunks(L);
    const i64 w = nb * N * ((K + SLICE - 1) / SLICE);
    if (L == 40) return M == 1 && w >= 1024;              // its operands' LDS fits a CU once, to L = 39 twice
    if (ks <= 4) return (M == 1 || K <= SLICE / 2) && w >= (ks == 1 ? 2560 : 1024) * M;
    return w >= (ks == 5 ? 512 * M : ks == 6 ? 256 * M * M : 256 * M);
}

// 64-bit words of scratch: the slices' words; the words and bit lengths that k_narrow_round reads
inline i64 work_words(i64 L, i64 nb, i64 M, i64 N, i64 K) {
    Dims D;
    slices(nb, M, N, K, D);
    const i64 E = nb * M * N;
    i64 n = D.ns > 1 ? (i64)D.ns * E * 16 * chunks(L) : 0;
    if (D.ns > 1 || M > ROWS) n += E * 32 * lane_words(L) + (E + 1) / 2;
    if (takes_few(L, nb, M, N, K)) {
        few_slices(nb, N, K, D);
        const i64 f = D.ns > 1 ? (i64)D.ns * E * (2 * L + 2) + E * 32 * lane_words(L) + (E + 1) / 2 : 0;
        n = f > n ? f : n;
    }
    return n;
}

// after the products: the slices' sums, and COL's rounding over all rows
template <int H>
int launch_rest(const Operand& A, const Operand& B, const Dims& D, const Result& R, const i64* part, int nwp, u32* words,
                i32* bls, hipStream_t st) {
    const i64 E = D.nb * D.M * D.N;
    if (D.ns > 1) {
        hipLaunchKernelGGL(k_narrow_finish<H>, dim3((unsigned)((E + 3) / 4)), dim3(256), 0, st, part, nwp, A, B, D, R, words,
                           bls);
        SDPV_TRY_LAUNCH();
    }
    if (R.mode == OUT_COL && (D.ns > 1 || D.M > ROWS)) {
        const i64 rpw = D.M <= 4096 ? 4 : (D.M / 1024 + 3) / 4 * 4;
        hipLaunchKernelGGL(k_narrow_round<H>, dim3((unsigned)(D.nb * D.N * ((D.M + rpw - 1) / rpw))), dim3(256), 0, st,
                           words, bls, D, R, rpw);
        SDPV_TRY_LAUNCH();
    }
    return SDPV_OK;
}

template <int KS>
int launch_narrow(const Operand& A, const Operand& B, const Dims& D, const Result& R, i64* work, hipStream_t st) {
    using g = Geo<KS>;
    static_assert(g::LDS <= 160 * 1024, "LDS");
    const i64 E = D.nb * D.M * D.N, grid = D.nb * D.N * ((D.M + ROWS - 1) / ROWS) * D.ns;
    if (grid > 0x7fffffffLL) return SDPV_ESIZE;
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)k_narrow<KS, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void*)k_narrow<KS, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    i64* part = work;
    u32* words = (u32*)(work + (D.ns > 1 ? (i64)D.ns * E * g::NWP : 0));
    i32* bls = (i32*)(words + E * 64 * g::H);
    if (A.ldk == 1)
        hipLaunchKernelGGL((k_narrow<KS, true>), dim3((unsigned)grid), dim3(g::NT), (size_t)g::LDS, st, A, B, D, R, part, words, bls);
    else
        hipLaunchKernelGGL((k_narrow<KS, false>), dim3((unsigned)grid), dim3(g::NT), (size_t)g::LDS, st, A, B, D, R, part, words, bls);
    SDPV_TRY_LAUNCH();
    return launch_rest<g::H>(A, B, D, R, part, g::NWP, words, bls, st);
}

template <int H>
int launch_few(const Operand& A, const Operand& B, const Dims& D, const Result& R, i64* work, hipStream_t st) {
    const i64 E = D.nb * D.M * D.N, grid = (D.nb * D.N * D.ns + 3) / 4;
    if (grid > 0x7fffffffLL) return SDPV_ESIZE;
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)k_narrow_few<H>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    u32* words = (u32*)(work + (D.ns > 1 ? (i64)D.ns * E * (2 * D.L + 2) : 0));
    hipLaunchKernelGGL(k_narrow_few<H>, dim3((unsigned)grid), dim3(256), (size_t)32 * D.L * FEW_KS, st, A, B, D, R, work);
    SDPV_TRY_LAUNCH();
    if (D.ns == 1) return SDPV_OK;
    return launch_rest<H>(A, B, D, R, work, 2 * D.L + 2, words, (i32*)(words + E * 64 * H), st);
}

int narrow_run(const Operand& A, const Operand& B, i64 L, i64 nb, i64 M, i64 N, i64 K, const Result& R, i64* work,
               i64 nwork, hipStream_t st) {
    Dims D{nb, M, N, K, (int)L, 0, 0};
    slices(nb, M, N, K, D);
    const i64 need = work_words(L, nb, M, N, K);
    if (need > 0 && (!work || nwork < need)) return SDPV_EARG;
    if ((nb * M * N + 3) / 4 > 0x7fffffffLL) return SDPV_ESIZE;
    if (!A.e && !B.e && takes_few(L, nb, M, N, K)) {
        few_slices(nb, N, K, D);
        return lane_words(L) == 2 ? launch_few<2>(A, B, D, R, work, st) : launch_few<1>(A, B, D, R, work, st);
    }
    switch (chunks(L)) {
        case 1: return launch_narrow<1>(A, B, D, R, work, st);
        case 2: return launch_narrow<2>(A, B, D, R, work, st);
        case 3: return launch_narrow<3>(A, B, D, R, work, st);
        case 4: return launch_narrow<4>(A, B, D, R, work, st);
        case 5: return launch_narrow<5>(A, B, D, R, work, st);
        case 6: return launch_narrow<6>(A, B, D, R, work, st);
        case 7: return launch_narrow<7>(A, B, D, R, work, st);
        default: return launch_narrow<8>(A, B, D, R, work, st);
    }
}

}  // namespace

extern "C" {

int64_t sdpv_exact_dot_work(int64_t L, int64_t nb, int64_t M, int64_t N, int64_t K) {
    if (L < 1 || nb < 0 || M < 0 || N < 0 || K < 0) return SDPV_EARG;
    return nb * M * N == 0 ? 0 : work_words(L, nb, M, N, K);
}

int sdpv_exact_dot(const int32_t* A, int64_t planeA, int64_t ldAb, int64_t ldAr, int64_t ldAk, const int32_t* B,
                   int64_t planeB, int64_t ldBb, int64_t ldBr, int64_t ldBk, int64_t L, int64_t nb, int64_t M,
                   int64_t N, int64_t K, int32_t* W, int64_t NW, int64_t* bitlen, int64_t* work, int64_t nwork,
                   void* stream) {
    if (L < 1 || L > 63 || nb < 0 || M < 0 || N < 0 || K < 0) return SDPV_EARG;
    if (NW < 2 * L + 2 || NW > 128) return SDPV_EARG;
    if (nb * M * N == 0) return SDPV_OK;
    if (!W || !bitlen || (K > 0 && (!A || !B))) return SDPV_EARG;
    const Operand a{A, nullptr, nullptr, planeA, ldAb, ldAr, ldAk}, b{B, nullptr, nullptr, planeB, ldBb, ldBr, ldBk};
    Result R{};
    R.mode = OUT_WORDS;
    R.out = W;
    R.plane = nb * M * N;
    R.oute = bitlen;
    R.NW = (int)NW;
    return narrow_run(a, b, L, nb, M, N, K, R, work, nwork, as_stream(stream));
}

int sdpv_narrow(const int32_t* A, const int64_t* eA, const int64_t* EA, int64_t planeA, int64_t ldAb, int64_t ldAr,
                int64_t ldAk, const int32_t* B, const int64_t* eB, const int64_t* EB, int64_t planeB, int64_t ldBb,
                int64_t ldBr, int64_t ldBk, int64_t L, int64_t nb, int64_t M, int64_t N, int64_t K, int32_t mode,
                int32_t* out, int64_t plane, int64_t ob, int64_t oi, int64_t oj, int64_t* oute, int64_t e0,
                const int64_t* ea, int64_t lea, const int64_t* eb, int64_t oexp, const int32_t* X, int64_t planeX,
                int64_t xb, int64_t xi, int64_t xj, const int64_t* eX, int32_t sgn, int32_t* flag, int64_t* work,
                int64_t nwork, void* stream) {
    if (L < 1 || L > 63 || nb < 0 || M < 0 || N < 0 || K < 0 || K > (1 << 17)) return SDPV_EARG;
    if (mode < OUT_NORMALIZE || mode > OUT_ACC || (sgn != 1 && sgn != -1)) return SDPV_EARG;
    if (nb * M * N == 0) return SDPV_OK;
    if (!out || (K > 0 && (!A || !B)) || (eA && !EA) || (eB && !EB) || (X && !eX)) return SDPV_EARG;
    if ((mode == OUT_NORMALIZE || mode == OUT_COL) && !oute) return SDPV_EARG;
    const Operand a{A, eA, EA, planeA, ldAb, ldAr, ldAk}, b{B, eB, EB, planeB, ldBb, ldBr, ldBk};
    const Result R{mode, out, plane, ob, oi, oj, oute, (int)(2 * L + 2), e0, ea, eb, lea, oexp, X, planeX, xb, xi, xj,
                   eX, sgn, flag};
    return narrow_run(a, b, L, nb, M, N, K, R, work, nwork, as_stream(stream));
}

int sdpv_narrow_result(const int32_t* acc, int64_t L, int64_t nb, int64_t M, int64_t N, const int64_t* EA,
                       const int64_t* EB, int32_t* out, int64_t plane, int64_t ob, int64_t oi, int64_t oj, int64_t* oute,
                       void* stream) {
    if (L < 1 || L > 63 || nb < 0 || M < 0 || N < 0) return SDPV_EARG;
    const i64 E = nb * M * N;
    if (E == 0) return SDPV_OK;
    if (!acc || !EA || !EB || !out || !oute) return SDPV_EARG;
    if ((E + 3) / 4 > 0x7fffffffLL) return SDPV_ESIZE;
    const Operand a{nullptr, nullptr, EA, 0, 0, 0, 0}, b{nullptr, nullptr, EB, 0, 0, 0, 0};
    const Dims D{nb, M, N, 0, (int)L, 1, 0};
    Result R{};
    R.mode = OUT_NORMALIZE;
    R.out = out;
    R.plane = plane;
    R.ob = ob;
    R.oi = oi;
    R.oj = oj;
    R.oute = oute;
    R.NW = (int)(2 * L + 2);
    hipStream_t st = as_stream(stream);
    if (2 * L + 2 > 64)
        hipLaunchKernelGGL(k_narrow_result<2>, dim3((unsigned)((E + 3) / 4)), dim3(256), 0, st, acc, a, b, D, R);
    else
        hipLaunchKernelGGL(k_narrow_result<1>, dim3((unsigned)((E + 3) / 4)), dim3(256), 0, st, acc, a, b, D, R);
    SDPV_TRY_LAUNCH();
    return SDPV_OK;
}

}  // extern "C"
