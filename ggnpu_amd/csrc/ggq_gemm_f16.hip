// ggq_gemm_f16.hip -- dense GEMM on raw GGUF blocks for many activation rows
// (prompts and batches), C[m][n] = sum_k x[m][k] w[n][k], on the fp16 matrix
// cores of gfx950.
//
// Weights.  A block's integer scale is folded into its codes: Q4_K and Q5_K
// sub-blocks give sc*q <= 1953, exact in fp16, so one MFMA chain runs over a
// whole 256-value superblock and the fp32 scale is applied once per 256
// values instead of once per 32.  Q6_K (sc*q up to 4096), IQ4_XS
// ((ls-32)*kv), Q8_0 and IQ4_NL (q*d, d under a power of two common to the
// column's 256 values) are the sum of two fp16 values, hi = fp16(q*s) and the
// exact remainder lo = q*s - hi (a fused multiply-add), in two planes.  The
// K-quant mins are one more MFMA per superblock: the sums of x over the 32
// values of each sub-block against the 6-bit mins.
//
// Activations.  prep_* kernels write them once as fp16 planes in the order
// the MFMA reads: fp32 rows as hi + lo under a power of two per row (22
// bits), int8 codes as one exact plane.  For codes every product and, below
// 2^24, every partial sum of a superblock is an exact integer in fp32.
//
// Fragment order: the 16 values of MFMA step t = 2g + u (g: 32-value group)
// are k = 32 g + 16 h + 8 u + {0,2,1,3,4,6,5,7}, h = lane / 32.  The order
// inside 8 values is what masking the even and the odd bytes of two code
// dwords gives, so decoding needs no byte shuffles.
#include "ggq_device.h"

namespace ggq {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

// 16 bytes at a 2-byte aligned address (one global_load_dwordx4)
struct __attribute__((packed, aligned(2))) U4a2 { uint32_t x, y, z, w; };
__device__ __forceinline__ uint4 ld16_h(const uint8_t* p) {
    const U4a2 v = *(const U4a2*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h2 h2c(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h2 fma2(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
// Byte i of w twice, under the exponent byte of 1024: 1024 + byte in both halves.
__device__ __forceinline__ h2 dup_byte(uint32_t w, int i) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)i << 16 | (uint32_t)i));
}
constexpr uint32_t kExp = 0x64006400u;  // 1024.0 in both halves

struct Frag {  // one column tile's operand of one 32-value group: steps u = 0, 1
    h8 hi[2], lo[2];
};
__device__ __forceinline__ void put(h8& f, int i, h2 v) {
    f[2 * i] = v[0];
    f[2 * i + 1] = v[1];
}
// q * s as hi + lo (exact: q and s carry 8 and 11 significant bits at most)
__device__ __forceinline__ void put_split(Frag& f, int u, int i, h2 q, h2 s) {
    const h2 hi = q * s;
    put(f.hi[u], i, hi);
    put(f.lo[u], i, fma2(q, s, -hi));
}

// Per-format view of one column's 256 values.  A lane holds the column
// lane % 32 and, of every 32-value group, the values 16 h .. 16 h + 15.
//   load_head / load_part(c): raw bytes (c: 64-value part);
//   open(): scale bytes and the fp32 scale d (and dm of the mins) from the
//   head, after which the head can be reloaded;
//   group(g): the fragments of group g (part g / 2).
template <int T> struct Col;

// scale and min bytes of a K-quant head
struct KqHead {
    uint32_t sc[2], mn[2];
    float d, dm;
    __device__ __forceinline__ void open(uint4 hd) {
        d = h2f(hd.x & 0xFFFFu);
        dm = h2f(hd.x >> 16);
        sc[0] = hd.y & 0x3F3F3F3Fu;
        mn[0] = hd.z & 0x3F3F3F3Fu;
        sc[1] = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
        mn[1] = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
    }
    __device__ __forceinline__ h2 scale(int g) const { return dup_byte(sc[g >> 2], g & 3) - h2c(1024.0f); }
    // the 8 bytes of b as fp16
    static __device__ __forceinline__ h8 bytes(const uint32_t (&b)[2]) {
        h8 r;
#pragma unroll
        for (int i = 0; i < 4; i++)
            put(r, i, as_h2(__builtin_amdgcn_perm(0x64646464u, b[i >> 1], (i & 1) ? 0x04030402u : 0x04010400u)) - h2c(1024.0f));
        return r;
    }
    __device__ __forceinline__ h8 mins() const { return bytes(mn); }
    // the centre's share of a superblock against the sums of x / 32
    __device__ __forceinline__ h8 mids(float mid) const { return bytes(sc) * (_Float16)(32.0f * mid); }
};

template <> struct Col<T_Q4_K> {
    static constexpr bool kMin = true, kTwo = false;
    static constexpr float kMid = 8.0f;  // the centre of the codes
    uint4 hd, q[4];
    KqHead k;
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int, int) { hd = ld16_a(row + (size_t)sb * 144); }
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int h, int, int c) {
        q[c] = ld16_a(row + (size_t)sb * 144 + 16 + 32 * c + 16 * h);
    }
    __device__ __forceinline__ void open(int, int, int) { k.open(hd); }
    // (1024 + 16 q - 1024 - 16 c) sc / 16: every term exact in fp16, q nibbles in bits 4-7
    template <bool CENTER> __device__ __forceinline__ void group(int g, int, Frag& f) const {
        const uint4 v = q[g >> 1];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        const h2 sc = k.scale(g);
        // not centred, low nibbles stay in bits 0-3: (1024 + q - 1024) sc
        const bool low = !CENTER && !(g & 1);
        const uint32_t mask = low ? 0x000F000Fu : 0x00F000F0u;
        const h2 s = low ? sc : sc * h2c(0.0625f), o = sc * h2c(low ? -1024.0f : (CENTER ? -72.0f : -64.0f));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t even = CENTER && !(g & 1) ? w[j] << 4 : w[j], odd = CENTER && !(g & 1) ? w[j] >> 4 : w[j] >> 8;
            put(f.hi[j >> 1], 2 * (j & 1), fma2(as_h2((even & mask) | kExp), s, o));
            put(f.hi[j >> 1], 2 * (j & 1) + 1, fma2(as_h2((odd & mask) | kExp), s, o));
        }
    }
};

template <> struct Col<T_Q5_K> {
    static constexpr bool kMin = true, kTwo = false;
    static constexpr float kMid = 16.0f;
    uint4 hd, qh, q[4];
    KqHead k;
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int h, int) {
        hd = ld16_a(row + (size_t)sb * 176);
        qh_next = ld16_a(row + (size_t)sb * 176 + 16 + 16 * h);
    }
    uint4 qh_next;
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int h, int, int c) {
        q[c] = ld16_a(row + (size_t)sb * 176 + 48 + 32 * c + 16 * h);
    }
    __device__ __forceinline__ void open(int, int, int) {
        k.open(hd);
        qh = qh_next;
    }
    // as Q4_K with the fifth bit above the nibble
    template <bool CENTER> __device__ __forceinline__ void group(int g, int, Frag& f) const {
        const uint4 v = q[g >> 1];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w}, b[4] = {qh.x, qh.y, qh.z, qh.w};
        const bool low = !CENTER && !(g & 1);
        const int pos = low ? 4 : 8;
        const uint32_t mask = low ? 0x000F000Fu : 0x00F000F0u, bm = 0x00010001u << pos;
        const h2 sc = k.scale(g);
        const h2 s = low ? sc : sc * h2c(0.0625f), o = sc * h2c(low ? -1024.0f : (CENTER ? -80.0f : -64.0f));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t even = CENTER && !(g & 1) ? w[j] << 4 : w[j], odd = CENTER && !(g & 1) ? w[j] >> 4 : w[j] >> 8;
            const uint32_t be = pos >= g ? b[j] << (pos - g) : b[j] >> (g - pos);
            const uint32_t bo = pos >= g + 8 ? b[j] << (pos - g - 8) : b[j] >> (g + 8 - pos);
            put(f.hi[j >> 1], 2 * (j & 1), fma2(as_h2((even & mask) | kExp | (be & bm)), s, o));
            put(f.hi[j >> 1], 2 * (j & 1) + 1, fma2(as_h2((odd & mask) | kExp | (bo & bm)), s, o));
        }
    }
};

template <> struct Col<T_Q6_K> {
    static constexpr bool kMin = false, kTwo = true;
    uint4 hd, ql[4], qh[2];
    uint32_t dn, sc[2];
    struct { float d, dm; } k;
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int, int) {
        hd = ld16_h(row + (size_t)sb * 210 + 192);
        dn = *(const uint16_t*)(row + (size_t)sb * 210 + 208);
    }
    // the parts of a 128-value half share their bytes: loaded with the second
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int h, int, int c) {
        if (!(c & 1)) return;
        const uint8_t* b = row + (size_t)sb * 210;
        const int n = c >> 1;
        ql[2 * n] = ld16_h(b + 64 * n + 16 * h);
        ql[2 * n + 1] = ld16_h(b + 64 * n + 32 + 16 * h);
        qh[n] = ld16_h(b + 128 + 32 * n + 16 * h);
    }
    // byte qd of sc[n]: the scale of this lane half's 16 values of group 4 n + qd
    __device__ __forceinline__ void open(int, int h, int) {
        k.d = h2f(dn);
        const uint32_t sel = h ? 0x07050301u : 0x06040200u;
        sc[0] = __builtin_amdgcn_perm(hd.y, hd.x, sel) ^ 0x80808080u;
        sc[1] = __builtin_amdgcn_perm(hd.w, hd.z, sel) ^ 0x80808080u;
    }
    template <bool> __device__ __forceinline__ void group(int g, int, Frag& f) const {
        const int n = g >> 2, qd = g & 3;
        const uint4 v = ql[2 * n + (qd & 1)], y = qh[n];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w}, b[4] = {y.x, y.y, y.z, y.w};
        const h2 s = dup_byte(sc[n], qd) - h2c(1152.0f);
        const bool top = qd >= 2;  // high nibbles in place: 16 u
        const uint32_t mask = top ? 0x00F000F0u : 0x000F000Fu, bm = top ? 0x03000300u : 0x00300030u;
        const int pos = top ? 8 : 4, at = 2 * qd;
        const h2 one = h2c(top ? 0.0625f : 1.0f), o = h2c(top ? -96.0f : -1056.0f);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t be = pos >= at ? b[j] << (pos - at) : b[j] >> (at - pos);
            const uint32_t bo = pos >= at + 8 ? b[j] << (pos - at - 8) : b[j] >> (at + 8 - pos);
            put_split(f, j >> 1, 2 * (j & 1), fma2(as_h2((w[j] & mask) | kExp | (be & bm)), one, o), s);
            put_split(f, j >> 1, 2 * (j & 1) + 1, fma2(as_h2(((w[j] >> 8) & mask) | kExp | (bo & bm)), one, o), s);
        }
    }
};

// Scales of the column's 8 blocks of 32 under a common power of two 2^e:
// the largest in [2^8, 2^9), so that q*d' stays below 2^16 and lo exact for
// blocks down to 2^-22 of the largest; k.d = 2^-e.
struct BlockScales {
    uint32_t dn[8];
    h2 s[8];
    struct { float d, dm; } k;
    __device__ __forceinline__ void open(int nv) {  // blocks from nv on lie past the row: zero
        uint32_t mx = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            dn[i] = i < nv ? dn[i] : 0u;
            const uint32_t a = dn[i] & 0x7FFFu;
            mx = a > mx ? a : mx;
        }
        const int e = 9 - __builtin_amdgcn_frexp_expf(h2f(mx));
        k.d = ldexpf(1.0f, -e);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const _Float16 v = (_Float16)ldexpf(h2f(dn[i]), e);
            s[i] = h2{v, v};
        }
    }
};

template <> struct Col<T_Q8_0> : BlockScales {
    static constexpr bool kMin = false, kTwo = true;
    uint4 q[8];
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int, int nb) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            dn[i] = *(const uint16_t*)(row + (size_t)b * 34);
        }
    }
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int h, int nb, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            q[i] = ld16_h(row + (size_t)b * 34 + 2 + 16 * h);
        }
    }
    __device__ __forceinline__ void open(int sb, int, int nb) { BlockScales::open(nb - 8 * sb); }
    template <bool> __device__ __forceinline__ void group(int g, int, Frag& f) const {
        const uint4 v = q[g];
        const uint32_t w[4] = {v.x ^ 0x80808080u, v.y ^ 0x80808080u, v.z ^ 0x80808080u, v.w ^ 0x80808080u};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            put_split(f, j >> 1, 2 * (j & 1), as_h2((w[j] & 0x00FF00FFu) | kExp) - h2c(1152.0f), s[g]);
            put_split(f, j >> 1, 2 * (j & 1) + 1, as_h2(((w[j] >> 8) & 0x00FF00FFu) | kExp) - h2c(1152.0f), s[g]);
        }
    }
};

// codebook values of nibble h of 16 bytes, times s
__device__ __forceinline__ void iq4_group(uint4 v, int h, h2 s, Frag& f) {
    const uint32_t n[4] = {v.x >> (4 * h), v.y >> (4 * h), v.z >> (4 * h), v.w >> (4 * h)};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t w = lut16(n[j] & 0x0F0F0F0Fu, GGQ_IQ4U0, GGQ_IQ4U1, GGQ_IQ4U2, GGQ_IQ4U3);
        put_split(f, j >> 1, 2 * (j & 1), as_h2((w & 0x00FF00FFu) | kExp) - h2c(1152.0f), s);
        put_split(f, j >> 1, 2 * (j & 1) + 1, as_h2(((w >> 8) & 0x00FF00FFu) | kExp) - h2c(1152.0f), s);
    }
}

template <> struct Col<T_IQ4_NL> : BlockScales {
    static constexpr bool kMin = false, kTwo = true;
    uint4 q[8];
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int, int nb) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            dn[i] = *(const uint16_t*)(row + (size_t)b * 18);
        }
    }
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int, int nb, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            q[i] = ld16_h(row + (size_t)b * 18 + 2);
        }
    }
    __device__ __forceinline__ void open(int sb, int, int nb) { BlockScales::open(nb - 8 * sb); }
    template <bool> __device__ __forceinline__ void group(int g, int h, Frag& f) const { iq4_group(q[g], h, s[g], f); }
};

template <> struct Col<T_IQ4_XS> {
    static constexpr bool kMin = false, kTwo = true;
    uint2 hd;
    uint4 q[8];
    uint32_t ls[2];
    struct { float d, dm; } k;
    __device__ __forceinline__ void load_head(const uint8_t* row, int sb, int, int) {
        hd = *(const uint2*)(row + (size_t)sb * 136);
    }
    __device__ __forceinline__ void load_part(const uint8_t* row, int sb, int, int, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            const uint8_t* p = row + (size_t)sb * 136 + 8 + 16 * i;
            const uint2 lo = *(const uint2*)p, hi = *(const uint2*)(p + 8);
            q[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
    }
    __device__ __forceinline__ void open(int, int, int) {
        k.d = h2f(hd.x & 0xFFFFu);
        ls[0] = ls[1] = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t v = ((hd.y >> (4 * i)) & 15u) | (((hd.x >> (16 + 2 * i)) & 3u) << 4);
            ls[i >> 2] |= v << (8 * (i & 3));
        }
    }
    template <bool> __device__ __forceinline__ void group(int g, int h, Frag& f) const {
        iq4_group(q[g], h, dup_byte(ls[g >> 2], g & 3) - h2c(1056.0f), f);
    }
};

constexpr int kProb = 4;
struct Prob {
    const uint8_t* W;
    float* C;
    int64_t row_bytes;
    int N, ldc, nt0;  // nt0: first column tile
};
struct Args {
    Prob p[kProb];
    int np, nt, mt;  // problems, column tiles of all of them, row tiles
    int M, SB, nb;   // rows, 256-value superblocks, 32-value blocks
    const h8* XH;
    const h8* XL;
    const h8* XS;
    const float* rs;  // scale of each row
};

// One workgroup: 32 MF rows x 32 NF columns; its KW wavefronts take the
// superblocks w, w + KW, ... and add their sums through LDS in wavefront
// order.  Planes (AP = 2: hi, lo) are read straight from the caches, weights
// are decoded in registers.
template <int T, int AP, int MF, int NF, int KW>
__global__ __launch_bounds__(64 * KW, 2) void gemm_f16_ks_kernel(Args a) {
    constexpr int R = MF * NF * 16, RW = R / KW;
    __shared__ float red[KW][R][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    // workgroup -> (column tile, row tile): one column tile's row tiles run
    // on one XCD, whose L2 then holds its weights
    const int x = blockIdx.x & 7, r8 = blockIdx.x >> 3;
    const int mt = r8 % a.mt, nt = r8 / a.mt * 8 + x;
    if (nt >= a.nt) return;
    int pi = 0;
    while (pi + 1 < a.np && nt >= a.p[pi + 1].nt0) pi++;
    const Prob P_ = a.p[pi];
    const int n0 = (nt - P_.nt0) * 32 * NF, m0 = mt * 32 * MF;

    const uint8_t* row[NF];
#pragma unroll
    for (int j = 0; j < NF; j++) {
        int n = n0 + 32 * j + (lane & 31);
        n = n < P_.N ? n : P_.N - 1;
        row[j] = P_.W + (int64_t)n * P_.row_bytes;
    }
    const size_t tile = (size_t)a.SB * 16 * 64;  // h8 of one 32-row tile's plane
    const h8* xh = a.XH + (size_t)(m0 / 32) * tile + lane;
    const h8* xl = AP == 2 ? a.XL + (size_t)(m0 / 32) * tile + lane : nullptr;
    const h8* xs = a.XS + (size_t)(m0 / 32) * a.SB * 64 + lane;

    f16v acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++) acc[i][j] = f16v{};

    Col<T> col[NF];
    if (w < a.SB) {
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].load_head(row[j], w, h, a.nb);
#pragma unroll
            for (int c = 0; c < 4; c++) col[j].load_part(row[j], w, h, a.nb, c);
        }
    }
    constexpr int NB = AP == 2 ? 2 : 4;  // operand buffers: NB - 1 steps ahead
    h8 xa[NB][MF][AP];
    auto load_x = [&](int sb, int t, h8 (&d)[MF][AP]) {
        const size_t o = ((size_t)sb * 16 + t) * 64;
#pragma unroll
        for (int i = 0; i < MF; i++) {
            d[i][0] = xh[i * tile + o];
            if constexpr (AP == 2) d[i][1] = xl[i * tile + o];
        }
    };
    if (w < a.SB) {
#pragma unroll
        for (int t = 0; t < NB - 1; t++) load_x(w, t, xa[t]);
    }
    for (int sb = w; sb < a.SB; sb += KW) {
        const int nsb = sb + KW < a.SB ? sb + KW : sb;
        f16v P[MF][NF];
        h8 sm[MF];
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].open(sb, h, a.nb);
            col[j].load_head(row[j], nsb, h, a.nb);
        }
        if constexpr (Col<T>::kMin) {
#pragma unroll
            for (int i = 0; i < MF; i++) sm[i] = xs[((size_t)i * a.SB + sb) * 64];
        }
#pragma unroll
        for (int g = 0; g < 8; g++) {
            Frag f[NF];
#pragma unroll
            for (int j = 0; j < NF; j++) col[j].template group<AP == 2>(g, h, f[j]);
            if (g & 1) {
#pragma unroll
                for (int j = 0; j < NF; j++) col[j].load_part(row[j], nsb, h, a.nb, g >> 1);
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int t = 2 * g + u, ta = t + NB - 1;
                load_x(ta < 16 ? sb : nsb, ta & 15, xa[ta % NB]);
                const auto& x_ = xa[t % NB];
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++)
                        P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x_[i][0], f[j].hi[u], t ? P[i][j] : f16v{}, 0, 0, 0);
                if constexpr (AP == 2) {
#pragma unroll
                    for (int i = 0; i < MF; i++)
#pragma unroll
                        for (int j = 0; j < NF; j++)
                            P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x_[i][1], f[j].hi[u], P[i][j], 0, 0, 0);
                }
                if constexpr (Col<T>::kTwo) {
#pragma unroll
                    for (int i = 0; i < MF; i++)
#pragma unroll
                        for (int j = 0; j < NF; j++)
                            P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x_[i][0], f[j].lo[u], P[i][j], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NF; j++) {
            const float d = col[j].k.d, dm = -32.0f * col[j].k.dm;  // the sums carry 1 / 32
            h8 mn, mid;
            if constexpr (Col<T>::kMin) {
                mn = col[j].k.mins();
                if constexpr (AP == 2) mid = col[j].k.mids(Col<T>::kMid);
            }
#pragma unroll
            for (int i = 0; i < MF; i++) {
                if constexpr (Col<T>::kMin && AP == 2)
                    P[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm[i], mid, P[i][j], 0, 0, 0);
                if constexpr (Col<T>::kMin) {
                    const f16v S = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm[i], mn, f16v{}, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][j][e] = __builtin_fmaf(dm, S[e], acc[i][j][e]);
                }
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = __builtin_fmaf(d, P[i][j][e], acc[i][j][e]);
            }
        }
    }

#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) red[w][(i * NF + j) * 16 + e][lane] = acc[i][j][e];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RW; q++) {
        const int r = w * RW + q;
        float v = red[0][r][lane];
#pragma unroll
        for (int o = 1; o < KW; o++) v += red[o][r][lane];
        const int ij = r >> 4, e = r & 15;
        const int m = m0 + 32 * (ij / NF) + 8 * (e >> 2) + 4 * h + (e & 3);
        const int n = n0 + 32 * (ij % NF) + (lane & 31);
        if (m < a.M && n < P_.N) P_.C[(int64_t)m * P_.ldc + n] = v * a.rs[m];
    }
}

// ------------------------------------------------------ activation planes --
// One workgroup per row (rows from M on: zeros).  A thread takes pieces of 8
// consecutive values; piece p = 4 g + 2 h + u goes to lane slot 32 h + row %
// 32 of step 2 g + u.  S: the sums over 32 values, divided by 32, as fp16 hi
// + lo in one more fragment per superblock (hi in lane half 0, lo in 1; sub-
// block j in element j).
struct PrepArgs {
    const float* A;
    const int8_t* QA;
    const float* sa;
    int lda, M, K, SB, vec;
    h8* XH;
    h8* XL;
    _Float16* XS;
    float* rs;
};
constexpr int kPi[8] = {0, 2, 1, 3, 4, 6, 5, 7};

// MODE 0: fp32 rows as hi + lo; 1: fp32 rows quantized per row to int8 codes
// (the codes and scales of the row quantizer); 2: given int8 codes.
template <int MODE, int RP>
__global__ __launch_bounds__(256) void prep_kernel(PrepArgs a) {
    __shared__ float wmax[4];
    const int m = blockIdx.x, tid = threadIdx.x, np = a.SB * 32;
    const size_t tile = (size_t)(m >> 5) * a.SB;
    const int r = m & 31;
    float v[RP][8];
#pragma unroll
    for (int i = 0; i < RP; i++) {
        const int k = 8 * (tid + 256 * i);
#pragma unroll
        for (int e = 0; e < 8; e++) v[i][e] = 0.0f;
        if (m < a.M && k < a.K) {
            if constexpr (MODE == 2) {
                const uint2 c = *(const uint2*)(a.QA + (int64_t)m * a.K + k);
#pragma unroll
                for (int e = 0; e < 8; e++) v[i][e] = (float)(int8_t)((e < 4 ? c.x : c.y) >> (8 * (e & 3)));
            } else if (a.vec) {
                const float* p = a.A + (int64_t)m * a.lda + k;
                const float4 x = *(const float4*)p, y = *(const float4*)(p + 4);
                v[i][0] = x.x; v[i][1] = x.y; v[i][2] = x.z; v[i][3] = x.w;
                v[i][4] = y.x; v[i][5] = y.y; v[i][6] = y.z; v[i][7] = y.w;
            } else {
                const float* p = a.A + (int64_t)m * a.lda + k;
#pragma unroll
                for (int e = 0; e < 8; e++) v[i][e] = p[e];
            }
        }
    }
    int ex = 0;
    if constexpr (MODE != 2) {
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < RP; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[i][e]));
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        if ((tid & 63) == 0) wmax[tid >> 6] = amax;
        __syncthreads();
        amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
        if constexpr (MODE == 0) {
            if (amax > 0.0f) {  // the largest magnitude into [2^14, 2^15)
                int x2;
                (void)frexpf(amax, &x2);
                ex = 15 - x2 > 126 ? 126 : 15 - x2;
            }
            if (tid == 0 && m < a.M) a.rs[m] = ldexpf(1.0f, -ex);
        } else {
            const float sc = amax > 0.0f ? __fdiv_rn(amax, 127.0f) : 1.0f;
            const float inv = __fdiv_rn(1.0f, sc);
            if (tid == 0 && m < a.M) a.rs[m] = sc;
#pragma unroll
            for (int i = 0; i < RP; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) v[i][e] = (float)to_i8(__fmul_rn(v[i][e], inv));
        }
    }
#pragma unroll
    for (int i = 0; i < RP; i++) {
        const int p = tid + 256 * i;
        if (p >= np) break;
        h8 hi, lo;
        float gs = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float y = MODE == 0 ? ldexpf(v[i][kPi[e]], ex) : v[i][kPi[e]];
            hi[e] = (_Float16)y;
            lo[e] = (_Float16)(y - (float)hi[e]);
            gs += MODE == 0 ? (float)hi[e] + (float)lo[e] : y;
        }
        const int g = p >> 2, h = (p >> 1) & 1, u = p & 1;
        const size_t at = (tile * 16 + 2 * g + u) * 64 + 32 * h + r;
        a.XH[at] = hi;
        if constexpr (MODE == 0) a.XL[at] = lo;
        gs += __shfl_xor(gs, 1, 64);
        gs += __shfl_xor(gs, 2, 64);
        if ((p & 3) == 0) {
            const float y = gs * 0.03125f;
            const _Float16 sh = (_Float16)y;
            _Float16* s = a.XS + ((tile + (g >> 3)) * 64 + r) * 8 + (g & 7);
            s[0] = sh;
            s[32 * 8] = (_Float16)(y - (float)sh);
        }
    }
}

template <int MODE>
void launch_prep(const PrepArgs& a, hipStream_t s) {
    const int rows = (a.M + 63) & ~63, np = a.SB * 32;
    if (np <= 256) prep_kernel<MODE, 1><<<rows, 256, 0, s>>>(a);
    else if (np <= 1024) prep_kernel<MODE, 4><<<rows, 256, 0, s>>>(a);
    else prep_kernel<MODE, 16><<<rows, 256, 0, s>>>(a);
}

// Planes of one set of activation rows in a workspace.
struct Planes {
    size_t xh, xl, xs, rs, bytes;
};
Planes planes_of(int K, int M, bool two) {
    const size_t rows = ((size_t)M + 63) & ~size_t(63), sb = ((size_t)K + 255) / 256;
    Planes p;
    p.xh = 0;
    p.xl = p.xh + rows * sb * 512;
    p.xs = p.xl + (two ? rows * sb * 512 : 0);
    p.rs = p.xs + rows * sb * 32;
    p.bytes = p.rs + rows * 4;
    return p;
}

template <int T, int AP>
void launch_t(Args& a, int M, hipStream_t s) {
    auto tiles = [&](int nf, int mf) {
        a.nt = 0;
        for (int i = 0; i < a.np; i++) {
            a.p[i].nt0 = a.nt;
            a.nt += (a.p[i].N + 32 * nf - 1) / (32 * nf);
        }
        a.mt = (M + 32 * mf - 1) / (32 * mf);
        return dim3((unsigned)((a.nt + 7) / 8 * 8 * a.mt));
    };
    if (M <= 32) {
        const dim3 g = tiles(1, 1);
        gemm_f16_ks_kernel<T, AP, 1, 1, 4><<<g, 256, 0, s>>>(a);
    } else {
        const dim3 g = tiles(2, 2);
        gemm_f16_ks_kernel<T, AP, 2, 2, 4><<<g, 256, 0, s>>>(a);
    }
}

}  // namespace

size_t gemm_f16_ws_bytes(int K, int M, bool codes) { return planes_of(K, M, !codes).bytes; }

hipError_t launch_gemm_f16_prep(int mode, const float* A, int lda, const int8_t* qa, int K, int M, void* ws,
                                hipStream_t s) {
    const Planes pl = planes_of(K, M, mode == 0);
    char* b = (char*)ws;
    PrepArgs a{};
    a.A = A;
    a.QA = qa;
    a.lda = lda;
    a.M = M;
    a.K = K;
    a.SB = (K + 255) / 256;
    a.vec = A && ((uintptr_t)A & 15u) == 0 && lda % 4 == 0;
    a.XH = (h8*)(b + pl.xh);
    a.XL = (h8*)(b + pl.xl);
    a.XS = (_Float16*)(b + pl.xs);
    a.rs = (float*)(b + pl.rs);
    if (mode == 0) launch_prep<0>(a, s);
    else if (mode == 1) launch_prep<1>(a, s);
    else launch_prep<2>(a, s);
    return hipGetLastError();
}

hipError_t launch_gemm_f16(uint32_t type, const GemmDesc* d, int n, int K, int M, bool codes, const float* sa,
                           const void* ws, hipStream_t s) {
    if (n < 1 || n > kProb) return hipErrorInvalidValue;
    const Planes pl = planes_of(K, M, !codes);
    const char* b = (const char*)ws;
    Args a{};
    for (int i = 0; i < n; i++) a.p[i] = Prob{(const uint8_t*)d[i].W, d[i].C, row_bytes(type, K), d[i].N, d[i].ldc, 0};
    a.np = n;
    a.M = M;
    a.SB = (K + 255) / 256;
    a.nb = K / 32;
    a.XH = (const h8*)(b + pl.xh);
    a.XL = (const h8*)(b + pl.xl);
    a.XS = (const h8*)(b + pl.xs);
    a.rs = sa ? sa : (const float*)(b + pl.rs);
#define GO(TT)                                   \
    case TT:                                     \
        if (codes) launch_t<TT, 1>(a, M, s);     \
        else launch_t<TT, 2>(a, M, s);           \
        break
    switch (type) {
        GO(T_Q4_K);
        GO(T_Q5_K);
        GO(T_Q6_K);
        GO(T_Q8_0);
        GO(T_IQ4_NL);
        GO(T_IQ4_XS);
    default: return hipErrorInvalidValue;
    }
#undef GO
    return hipGetLastError();
}

}  // namespace ggq
