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
// Pieces: piece q (0..3) of a 32-value group g holds the values k = 32 g + 8 q
// + {0,2,1,3,4,6,5,7} of one row or column, one lane's operand of an MFMA.
// The order inside 8 values is what masking the even and the odd bytes of two
// code dwords gives, so decoding needs no byte shuffles.
// v_mfma_f32_32x32x16_f16 takes a group in two steps u (lane 32 h + i: row i,
// piece 2 h + u), v_mfma_f32_16x16x32_f16 in one (lane 16 q + i: row i, piece
// q).  The planes are stored in the order of the former, [32-row tile][step 2g
// + u][lane][8]; the latter's operand is four runs of 256 bytes of it.
#include "ggq_device.h"

namespace ggq {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f4v mfma(h8 a, h8 b, f4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f16v mfma(h8 a, h8 b, f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

// A weight row: the matrix's base and the row's 32-bit byte offset (a matrix
// stays below 4 GiB), so loads take the scalar-base form.
struct Row {
    const uint8_t* base;
    uint32_t off;
    __device__ __forceinline__ const uint8_t* at(uint32_t o) const { return base + (uint32_t)(off + o); }
};
// 8 and 16 bytes at a 2-byte aligned address (one load each)
struct __attribute__((packed, aligned(2))) U4a2 { uint32_t x, y, z, w; };
struct __attribute__((packed, aligned(2))) U2a2 { uint32_t x, y; };
__device__ __forceinline__ uint4 ld16_h(const uint8_t* p) {
    const U4a2 v = *(const U4a2*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 ld8_h(const uint8_t* p) {
    const U2a2 v = *(const U2a2*)p;
    return make_uint2(v.x, v.y);
}

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h2 h2c(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h2 fma2(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
// Byte i of w twice, under the exponent byte of 1024: 1024 + byte in both halves.
__device__ __forceinline__ h2 dup_byte(uint32_t w, int i) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)i << 16 | (uint32_t)i));
}
// Two codes (the bits of `mask`) as 1024 + code: 1024.0 in both halves is kept
// in a register, so that masking and setting it is one v_and_or_b32.
__device__ __forceinline__ h2 code2(uint32_t w, uint32_t mask, uint32_t k1024) { return as_h2((w & mask) | k1024); }

struct Frag {  // one column tile's operand of one MFMA
    h8 hi, lo;
};
__device__ __forceinline__ void put(h8& f, int i, h2 v) {
    f[2 * i] = v[0];
    f[2 * i + 1] = v[1];
}
// q * s as hi + lo (exact: q and s carry 8 and 11 significant bits at most)
__device__ __forceinline__ void put_split(Frag& f, int i, h2 q, h2 s) {
    const h2 hi = q * s;
    put(f.hi, i, hi);
    put(f.lo, i, fma2(q, s, -hi));
}

// Per-format view of one column's 256 values.  A lane holds, of every
// 32-value group of its column, NP pieces from piece q on (1, or 2 from an
// even one).
//   load_head / load_part(c): raw bytes (c: 64-value part; PB parts are kept,
//   part c replaces part c - PB);
//   open(): scale bytes and the fp32 scale d (and dm of the mins) from the
//   head, after which the head can be reloaded;
//   piece(g, u): the operand of piece q + u of group g (part g / 2).
template <int T, int PB, int NP> struct Col;
// 8 NP bytes
template <int NP> struct Bytes {
    uint2 v[NP];
    __device__ __forceinline__ void load_a(const uint8_t* p) {  // 8 NP-byte aligned
        if constexpr (NP == 1) v[0] = *(const uint2*)p;
        else {
            const uint4 x = *(const uint4*)p;
            v[0] = make_uint2(x.x, x.y);
            v[1] = make_uint2(x.z, x.w);
        }
    }
    __device__ __forceinline__ void load_h(const uint8_t* p) {  // 2-byte aligned
        if constexpr (NP == 1) v[0] = ld8_h(p);
        else {
            const uint4 x = ld16_h(p);
            v[0] = make_uint2(x.x, x.y);
            v[1] = make_uint2(x.z, x.w);
        }
    }
};

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

template <int PB, int NP> struct Col<T_Q4_K, PB, NP> {
    static constexpr bool kMin = true, kTwo = false;
    static constexpr float kMid = 8.0f;  // the centre of the codes
    uint4 hd;
    Bytes<NP> v[PB];
    KqHead k;
    __device__ __forceinline__ void load_head(Row row, int sb, int, int) { hd = ld16_a(row.at((uint32_t)sb * 144)); }
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int, int c) {
        v[c % PB].load_a(row.at((uint32_t)sb * 144 + 16 + 32 * c + 8 * q));
    }
    __device__ __forceinline__ void open(int, int, int) { k.open(hd); }
    // (1024 + 16 q - 1024 - 16 c) sc / 16: every term exact in fp16, q nibbles in bits 4-7
    template <bool CENTER> __device__ __forceinline__ void piece(int g, int u, int, uint32_t e, Frag& f) const {
        const uint2 l = v[(g >> 1) % PB].v[u];
        const uint32_t w[2] = {l.x, l.y};
        const h2 sc = k.scale(g);
        // not centred, low nibbles stay in bits 0-3: (1024 + q - 1024) sc
        const bool low = !CENTER && !(g & 1);
        const uint32_t mask = low ? 0x000F000Fu : 0x00F000F0u;
        const h2 s = low ? sc : sc * h2c(0.0625f), o = sc * h2c(low ? -1024.0f : (CENTER ? -72.0f : -64.0f));
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t even = CENTER && !(g & 1) ? w[j] << 4 : w[j], odd = CENTER && !(g & 1) ? w[j] >> 4 : w[j] >> 8;
            put(f.hi, 2 * j, fma2(code2(even, mask, e), s, o));
            put(f.hi, 2 * j + 1, fma2(code2(odd, mask, e), s, o));
        }
    }
};

template <int PB, int NP> struct Col<T_Q5_K, PB, NP> {
    static constexpr bool kMin = true, kTwo = false;
    static constexpr float kMid = 16.0f;
    uint4 hd;
    Bytes<NP> qh, qh_next, v[PB];
    KqHead k;
    __device__ __forceinline__ void load_head(Row row, int sb, int q, int) {
        hd = ld16_a(row.at((uint32_t)sb * 176));
        qh_next.load_a(row.at((uint32_t)sb * 176 + 16 + 8 * q));
    }
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int, int c) {
        v[c % PB].load_a(row.at((uint32_t)sb * 176 + 48 + 32 * c + 8 * q));
    }
    __device__ __forceinline__ void open(int, int, int) {
        k.open(hd);
        qh = qh_next;
    }
    // as Q4_K with the fifth bit above the nibble
    template <bool CENTER> __device__ __forceinline__ void piece(int g, int u, int, uint32_t e, Frag& f) const {
        const uint2 l = v[(g >> 1) % PB].v[u], y = qh.v[u];
        const uint32_t w[2] = {l.x, l.y}, b[2] = {y.x, y.y};
        const bool low = !CENTER && !(g & 1);
        const int pos = low ? 4 : 8;
        const uint32_t mask = low ? 0x000F000Fu : 0x00F000F0u, bm = 0x00010001u << pos;
        const h2 sc = k.scale(g);
        const h2 s = low ? sc : sc * h2c(0.0625f), o = sc * h2c(low ? -1024.0f : (CENTER ? -80.0f : -64.0f));
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t even = CENTER && !(g & 1) ? w[j] << 4 : w[j], odd = CENTER && !(g & 1) ? w[j] >> 4 : w[j] >> 8;
            const uint32_t be = pos >= g ? b[j] << (pos - g) : b[j] >> (g - pos);
            const uint32_t bo = pos >= g + 8 ? b[j] << (pos - g - 8) : b[j] >> (g + 8 - pos);
            put(f.hi, 2 * j, fma2(code2(even, mask, e | (be & bm)), s, o));
            put(f.hi, 2 * j + 1, fma2(code2(odd, mask, e | (bo & bm)), s, o));
        }
    }
};

template <int PB, int NP> struct Col<T_Q6_K, PB, NP> {
    static constexpr bool kMin = false, kTwo = true;
    uint4 hd;
    Bytes<NP> ql[4], qh[2];
    uint32_t dn, sc[2];
    struct { float d, dm; } k;
    __device__ __forceinline__ void load_head(Row row, int sb, int, int) {
        hd = ld16_h(row.at((uint32_t)sb * 210 + 192));
        dn = *(const uint16_t*)(row.at((uint32_t)sb * 210 + 208));
    }
    // the parts of a 128-value half share their bytes: loaded with the second
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int, int c) {
        if (!(c & 1)) return;
        const uint32_t b = (uint32_t)sb * 210;
        const int n = c >> 1;
        ql[2 * n].load_h(row.at(b + 64 * n + 8 * q));
        ql[2 * n + 1].load_h(row.at(b + 64 * n + 32 + 8 * q));
        qh[n].load_h(row.at(b + 128 + 32 * n + 8 * q));
    }
    // byte qd of sc[n]: the scale of the 16 values this lane's of group 4 n + qd belong to
    __device__ __forceinline__ void open(int, int q, int) {
        k.d = h2f(dn);
        const uint32_t sel = q >= 2 ? 0x07050301u : 0x06040200u;
        sc[0] = __builtin_amdgcn_perm(hd.y, hd.x, sel) ^ 0x80808080u;
        sc[1] = __builtin_amdgcn_perm(hd.w, hd.z, sel) ^ 0x80808080u;
    }
    template <bool> __device__ __forceinline__ void piece(int g, int u, int, uint32_t e, Frag& f) const {
        const int n = g >> 2, qd = g & 3;
        const uint2 l = ql[2 * n + (qd & 1)].v[u], y = qh[n].v[u];
        const uint32_t w[2] = {l.x, l.y}, b[2] = {y.x, y.y};
        const h2 s = dup_byte(sc[n], qd) - h2c(1152.0f);
        const bool top = qd >= 2;  // high nibbles in place: 16 u
        const uint32_t mask = top ? 0x00F000F0u : 0x000F000Fu, bm = top ? 0x03000300u : 0x00300030u;
        const int pos = top ? 8 : 4, at = 2 * qd;
        const h2 one = h2c(top ? 0.0625f : 1.0f), o = h2c(top ? -96.0f : -1056.0f);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t be = pos >= at ? b[j] << (pos - at) : b[j] >> (at - pos);
            const uint32_t bo = pos >= at + 8 ? b[j] << (pos - at - 8) : b[j] >> (at + 8 - pos);
            put_split(f, 2 * j, fma2(code2(w[j], mask, e | (be & bm)), one, o), s);
            put_split(f, 2 * j + 1, fma2(code2(w[j] >> 8, mask, e | (bo & bm)), one, o), s);
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

template <int PB, int NP> struct Col<T_Q8_0, PB, NP> : BlockScales {
    static constexpr bool kMin = false, kTwo = true;
    Bytes<NP> v[2 * PB];
    __device__ __forceinline__ void load_head(Row row, int sb, int, int nb) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            dn[i] = *(const uint16_t*)(row.at((uint32_t)b * 34));
        }
    }
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int nb, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            v[i % (2 * PB)].load_h(row.at((uint32_t)b * 34 + 2 + 8 * q));
        }
    }
    __device__ __forceinline__ void open(int sb, int, int nb) { BlockScales::open(nb - 8 * sb); }
    template <bool> __device__ __forceinline__ void piece(int g, int u, int, uint32_t e, Frag& f) const {
        const uint2 l = v[g % (2 * PB)].v[u];
        const uint32_t w[2] = {l.x ^ 0x80808080u, l.y ^ 0x80808080u};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            put_split(f, 2 * j, code2(w[j], 0x00FF00FFu, e) - h2c(1152.0f), s[g]);
            put_split(f, 2 * j + 1, code2(w[j] >> 8, 0x00FF00FFu, e) - h2c(1152.0f), s[g]);
        }
    }
};

// codebook values of 8 bytes' low (q < 2) or high nibbles, times s
__device__ __forceinline__ void iq4_piece(uint2 v, int q, h2 s, uint32_t e, Frag& f) {
    const uint32_t n[2] = {v.x >> (2 * (q & 2)), v.y >> (2 * (q & 2))};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t w = lut16(n[j] & 0x0F0F0F0Fu, GGQ_IQ4U0, GGQ_IQ4U1, GGQ_IQ4U2, GGQ_IQ4U3);
        put_split(f, 2 * j, code2(w, 0x00FF00FFu, e) - h2c(1152.0f), s);
        put_split(f, 2 * j + 1, code2(w >> 8, 0x00FF00FFu, e) - h2c(1152.0f), s);
    }
}

template <int PB, int NP> struct Col<T_IQ4_NL, PB, NP> : BlockScales {
    static constexpr bool kMin = false, kTwo = true;
    Bytes<NP> v[2 * PB];
    __device__ __forceinline__ void load_head(Row row, int sb, int, int nb) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            dn[i] = *(const uint16_t*)(row.at((uint32_t)b * 18));
        }
    }
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int nb, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            const int b = 8 * sb + i < nb ? 8 * sb + i : nb - 1;
            v[i % (2 * PB)].load_h(row.at((uint32_t)b * 18 + 2 + 8 * (q & 1)));
        }
    }
    __device__ __forceinline__ void open(int sb, int, int nb) { BlockScales::open(nb - 8 * sb); }
    template <bool> __device__ __forceinline__ void piece(int g, int u, int q, uint32_t e, Frag& f) const { iq4_piece(v[g % (2 * PB)].v[u], q, s[g], e, f); }
};

template <int PB, int NP> struct Col<T_IQ4_XS, PB, NP> {
    static constexpr bool kMin = false, kTwo = true;
    uint2 hd;
    Bytes<NP> v[2 * PB];
    uint32_t ls[2];
    struct { float d, dm; } k;
    __device__ __forceinline__ void load_head(Row row, int sb, int, int) {
        hd = *(const uint2*)(row.at((uint32_t)sb * 136));
    }
    __device__ __forceinline__ void load_part(Row row, int sb, int q, int, int c) {
#pragma unroll
        for (int i = 2 * c; i < 2 * c + 2; i++) {
            // 8-byte aligned: one 16-byte load all the same
            v[i % (2 * PB)].load_h(row.at((uint32_t)sb * 136 + 8 + 16 * i + 8 * (q & 1)));
        }
    }
    __device__ __forceinline__ void open(int, int, int) {
        k.d = h2f(hd.x & 0xFFFFu);
        ls[0] = ls[1] = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t x = ((hd.y >> (4 * i)) & 15u) | (((hd.x >> (16 + 2 * i)) & 3u) << 4);
            ls[i >> 2] |= x << (8 * (i & 3));
        }
    }
    template <bool> __device__ __forceinline__ void piece(int g, int u, int q, uint32_t e, Frag& f) const {
        iq4_piece(v[g % (2 * PB)].v[u], q, dup_byte(ls[g >> 2], g & 3) - h2c(1056.0f), e, f);
    }
};

constexpr int kProb = 4;
struct Prob {
    const uint8_t* W;
    float* C;
    uint32_t row_bytes;
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

// End of a superblock for one tile: its chain P under the column's scale and
// the mins onto the sums (sm: the sums of x).
template <int AP, class C, class V>
__device__ __forceinline__ void close(const C& col, h8 mn, h8 mid, h8 sm, V P, V& acc) {
    constexpr int E = sizeof(V) / 4;
    const float d = col.k.d, dm = -32.0f * col.k.dm;  // the sums carry 1 / 32
    if constexpr (C::kMin) {
        if constexpr (AP == 2) P = mfma(sm, mid, P);
        const V S = mfma(sm, mn, V{});
        // codes: both are exact integers; rows: P and S cancel in part, so they
        // meet before they round against the sum
#pragma unroll
        for (int e = 0; e < E; e++)
            acc[e] = AP == 2 ? acc[e] + __builtin_fmaf(d, P[e], dm * S[e]) : __builtin_fmaf(d, P[e], __builtin_fmaf(dm, S[e], acc[e]));
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = __builtin_fmaf(d, P[e], acc[e]);
    }
}
template <int AP, class C>
__device__ __forceinline__ void min_operands(const C& col, h8& mn, h8& mid) {
    if constexpr (C::kMin) {
        mn = col.k.mins();
        if constexpr (AP == 2) mid = col.k.mids(C::kMid);
    }
}
__device__ __forceinline__ void store(const Args& a, const Prob& p, int m, int n, float v) {
    if (m < a.M && n < p.N) p.C[(int64_t)m * p.ldc + n] = v * a.rs[m];
}
// Tile of a workgroup: one column tile's row tiles run on one XCD, whose L2
// then holds its weights.
__device__ __forceinline__ bool tile_of(const Args& a, int& mt, int& nt, int& pi) {
    const int x = blockIdx.x & 7, r8 = blockIdx.x >> 3;
    mt = r8 % a.mt;
    nt = r8 / a.mt * 8 + x;
    if (nt >= a.nt) return false;
    pi = 0;
    while (pi + 1 < a.np && nt >= a.p[pi + 1].nt0) pi++;
    return true;
}
// The lane's column of tile j (TW columns each); past the matrix its last one.
template <int TW, int NF>
__device__ __forceinline__ void rows_of(const Prob& p, int n0, int lane, Row (&row)[NF]) {
#pragma unroll
    for (int j = 0; j < NF; j++) {
        int n = n0 + TW * j + (lane & (TW - 1));
        n = n < p.N ? n : p.N - 1;
        row[j] = Row{p.W, (uint32_t)n * p.row_bytes};
    }
}

// Few rows or few tiles: a workgroup takes 16 MF rows x 16 NF columns; its KW
// wavefronts take the superblocks w, w + KW, ... and add their sums through
// LDS in wavefront order.  Latency bounds it, so each wavefront keeps the
// operands of the next NB groups and a superblock of weights in flight in
// registers (the scheduler otherwise sinks those loads to their use: 2048 x
// 2048 Q4_K, 64 rows with their planes 27 -> 16 us, 2048 x 8192, 32 rows 41 ->
// 23 us), and 16-column tiles put twice as many CUs to work as the 32-column
// MFMA shape would (2048 x 2048, 9 rows: 12.2 -> 9.2 us).
template <int T, int AP, int MF, int NF, int KW, int NB>
__global__ __launch_bounds__(64 * KW, 2) void gemm_f16_ks_kernel(Args a) {
    constexpr int R = MF * NF * 4, PB = 4;
    __shared__ float red[KW][R][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4;
    int mt, nt, pi;
    if (!tile_of(a, mt, nt, pi)) return;
    const Prob P_ = a.p[pi];
    const int n0 = (nt - P_.nt0) * 16 * NF, m0 = mt * 16 * MF;
    Row row[NF];
    rows_of<16, NF>(P_, n0, lane, row);
    // pieces of row tile i (half of a 32-row tile) and group g
    const size_t tile = (size_t)a.SB * 16 * 64;  // h8 of one 32-row tile's plane
    const int slot = 64 * (q & 1) + 32 * (q >> 1) + (lane & 15);
    auto at = [&](int i, int sb, int g) -> size_t {
        const int r = m0 / 16 + i;
        return (size_t)(r >> 1) * tile + ((size_t)sb * 8 + g) * 128 + 16 * (r & 1) + slot;
    };
    // sums: hi for piece 0, lo for piece 1, nothing above
    auto sums = [&](int i, int sb) -> h8 {
        const int r = m0 / 16 + i;
        const h8 v = a.XS[((size_t)(r >> 1) * a.SB + sb) * 64 + 32 * (q & 1) + 16 * (r & 1) + (lane & 15)];
        return q < 2 ? v : h8{};
    };

    f4v acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++) acc[i][j] = f4v{};
    typedef Col<T, PB, 1> C;
    C col[NF];
    const uint32_t k1024 = opaque(0x64006400u);
    h8 xa[NB][MF][AP];
    auto load_x = [&](int sb, int g, h8 (&d)[MF][AP]) {
#pragma unroll
        for (int i = 0; i < MF; i++) {
            d[i][0] = a.XH[at(i, sb, g)];
            if constexpr (AP == 2) d[i][1] = a.XL[at(i, sb, g)];
        }
    };
    if (w < a.SB) {
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].load_head(row[j], w, q, a.nb);
#pragma unroll
            for (int c = 0; c < 4; c++) col[j].load_part(row[j], w, q, a.nb, c);
        }
#pragma unroll
        for (int g = 0; g < NB; g++) load_x(w, g, xa[g]);
    }
    for (int sb = w; sb < a.SB; sb += KW) {
        const int nsb = sb + KW < a.SB ? sb + KW : sb;
        f4v P[MF][NF];
        h8 sm[MF];
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].open(sb, q, a.nb);
            col[j].load_head(row[j], nsb, q, a.nb);
        }
#pragma unroll
        for (int i = 0; i < MF; i++) sm[i] = C::kMin ? sums(i, sb) : h8{};
#pragma unroll
        for (int g = 0; g < 8; g++) {
            Frag f[NF];
#pragma unroll
            for (int j = 0; j < NF; j++) col[j].template piece<AP == 2>(g, 0, q, k1024, f[j]);
            const auto& x_ = xa[g % NB];
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int j = 0; j < NF; j++) P[i][j] = mfma(x_[i][0], f[j].hi, g ? P[i][j] : f4v{});
            if constexpr (AP == 2) {
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++) P[i][j] = mfma(x_[i][1], f[j].hi, P[i][j]);
            }
            if constexpr (C::kTwo) {
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++) P[i][j] = mfma(x_[i][0], f[j].lo, P[i][j]);
            }
            load_x(g + NB < 8 ? sb : nsb, (g + NB) & 7, xa[g % NB]);
            if (g & 1) {
#pragma unroll
                for (int j = 0; j < NF; j++) col[j].load_part(row[j], nsb, q, a.nb, g >> 1);
            }
            // the loads stay here, NB groups ahead of their use
            __builtin_amdgcn_sched_barrier(0x8F);
        }
#pragma unroll
        for (int j = 0; j < NF; j++) {
            h8 mn, mid;
            min_operands<AP>(col[j], mn, mid);
#pragma unroll
            for (int i = 0; i < MF; i++) close<AP>(col[j], mn, mid, sm[i], P[i][j], acc[i][j]);
        }
    }

#pragma unroll
    for (int r = 0; r < R; r++) red[w][r][lane] = acc[r / 4 / NF][r / 4 % NF][r & 3];
    __syncthreads();
    for (int r = w; r < R; r += KW) {
        float v = red[0][r][lane];
#pragma unroll
        for (int o = 1; o < KW; o++) v += red[o][r][lane];
        store(a, P_, m0 + 16 * (r / 4 / NF) + 4 * q + (r & 3), n0 + 16 * (r / 4 % NF) + (lane & 15), v);
    }
}

// 64 lanes' 16 bytes at src + 16 lane into LDS at lds + 16 lane (LDS offsets
// below 64 KB); the caller waits on the vector memory counter.
__device__ __forceinline__ void dma16(const h8* src, uint32_t lane16, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(lane16), "s"(src) : "memory");
}

// Many tiles: a workgroup of four wavefronts takes 64 rows; NWN of them sit
// side by side (64 columns each) and share the planes, which the memory
// system writes into a ring of four LDS slots three chunks (of CS steps)
// ahead; the 4 / NWN groups take the superblocks in turn and are added at
// the end through LDS.
// Bound: the matrix cores with two planes (1023 rows x 16384 x 2048 Q4_K 157
// us with the planes' 9: 0.93 PFLOP/s of fp16 products; 1.65 is what a loop
// of these MFMAs on random values reaches on this card, 1.1 its library's
// matmul), the decoding VALU with one (99 us).  128 x 32 values a wavefront
// decode a weight once per 128 rows: against 64 x 64, one plane 106 -> 99 us,
// Q6_K 394 -> 215 us (registers: that shape spilled).  Operands of a step are
// read during the step before it; weights straight from the caches, one part
// ahead.
template <int T, int AP, int MF, int NF, int NWN, int CS>
__global__ __launch_bounds__(256, 2) void gemm_f16_ring_kernel(Args a) {
    constexpr int PB = 2, KW = 4 / NWN, S = 4, R = MF * NF * 16;
    constexpr int CB = MF * AP * CS * 64;  // h8 of a chunk
    constexpr int PP = MF * AP * CS / NWN;  // loads of a wavefront per chunk
    constexpr int NC = 16 / CS;             // chunks of a superblock
    static_assert(NC % S == 0, "a superblock's chunks fill whole rounds of the ring");
    constexpr int kRed = KW > 1 ? 4 * R * 64 * 4 / 16 : 0;
    __shared__ h8 lds[KW * S * CB > kRed ? KW * S * CB : kRed];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int nw = w % NWN, kw = w / NWN;
    int mt, nt, pi;
    if (!tile_of(a, mt, nt, pi)) return;
    const Prob P_ = a.p[pi];
    const int n0 = ((nt - P_.nt0) * NWN + nw) * 32 * NF, m0 = mt * 32 * MF;

    Row row[NF];
    rows_of<32, NF>(P_, n0, lane, row);
    const size_t tile = (size_t)a.SB * 16 * 64;
    const h8* xh = a.XH + (size_t)(m0 / 32) * tile;
    const h8* xl = AP == 2 ? a.XL + (size_t)(m0 / 32) * tile : nullptr;
    const h8* xs = a.XS + (size_t)(m0 / 32) * a.SB * 64 + lane;
    h8* const ring = lds + kw * S * CB;
    const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) h8*)ring;
    const int iters = (a.SB + KW - 1) / KW;
    // chunk c of superblock kw + KW it of this wavefront's group (past the
    // end: the last superblock again, so that every chunk issues the same
    // number of loads)
    auto fetch = [&](int it, int c) {
        it += c / NC;
        c %= NC;
        int sb = kw + KW * it;
        sb = sb < a.SB ? sb : a.SB - 1;
#pragma unroll
        for (int i = 0; i < PP; i++) {
            const int p = nw + NWN * i, s = p % CS, pl = p / CS % AP, m = p / (CS * AP);
            const h8* src = (pl ? xl : xh) + m * tile + ((size_t)sb * 16 + c * CS + s) * 64;
            dma16(src, (uint32_t)lane * 16u, ring_at + (uint32_t)(c % S * CB + p * 64) * 16u);
        }
    };

    f16v acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++) acc[i][j] = f16v{};
    typedef Col<T, PB, 2> C;
    C col[NF];
    const uint32_t k1024 = opaque(0x64006400u);
    {
        const int sb = kw < a.SB ? kw : a.SB - 1;
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].load_head(row[j], sb, 2 * h, a.nb);
#pragma unroll
            for (int c = 0; c < (T == T_Q6_K ? 4 : PB); c++) col[j].load_part(row[j], sb, 2 * h, a.nb, c);
        }
    }
#pragma unroll
    for (int c = 0; c < S; c++) fetch(0, c);
    h8 xa[2][MF][AP];
    auto read = [&](int t) {  // step t of this superblock (16: step 0 of the next)
        const h8* src = ring + t / CS % S * CB + lane;
#pragma unroll
        for (int i = 0; i < MF; i++)
#pragma unroll
            for (int p = 0; p < AP; p++) xa[t & 1][i][p] = src[((i * AP + p) * CS + t % CS) * 64];
    };
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * PP) : "memory");
    read(0);
    for (int it = 0; it < iters; it++) {
        const int sb0 = kw + KW * it;
        const bool live = sb0 < a.SB;
        const int sb = live ? sb0 : a.SB - 1, nsb = sb + KW < a.SB ? sb + KW : sb;
        f16v P[MF][NF];
        h8 sm[MF];
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].open(sb, 2 * h, a.nb);
            col[j].load_head(row[j], nsb, 2 * h, a.nb);
        }
        if constexpr (C::kMin) {
#pragma unroll
            for (int i = 0; i < MF; i++) sm[i] = xs[((size_t)i * a.SB + sb) * 64];
        }
        Frag fr[2][NF];
#pragma unroll
        for (int j = 0; j < NF; j++) col[j].template piece<AP == 2>(0, 0, 2 * h, k1024, fr[0][j]);
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int c = t / CS;
            // operands of step t + 1 while step t multiplies
            if ((t + 1) % CS == 0) {
                // this wavefront's loads of chunk c + 1 have landed (at most
                // the last (S - 2) PP loads are outstanding, all issued after
                // them) and it has read chunk c; after the barrier both hold
                // for everyone: chunk c + 1 can be read, slot c is free
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * PP) : "memory");
                if ((t + 1) % 4 == 0) {  // the part just used makes room for the one PB ahead
                    const int p = t / 4 + (T == T_Q6_K ? 4 : PB);
#pragma unroll
                    for (int j = 0; j < NF; j++) col[j].load_part(row[j], p < 4 ? sb : nsb, 2 * h, a.nb, p & 3);
                }
                fetch(it, c + S);
            }
            read(t + 1);
            __builtin_amdgcn_sched_barrier(0x6);
            if (t < 15) {
#pragma unroll
                for (int j = 0; j < NF; j++) col[j].template piece<AP == 2>((t + 1) >> 1, (t + 1) & 1, 2 * h, k1024, fr[(t + 1) & 1][j]);
            }
            const auto& x_ = xa[t & 1];
            const auto& f = fr[t & 1];
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int j = 0; j < NF; j++)
                    P[i][j] = mfma(x_[i][0], f[j].hi, t ? P[i][j] : f16v{});
            if constexpr (AP == 2) {
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++)
                        P[i][j] = mfma(x_[i][1], f[j].hi, P[i][j]);
            }
            if constexpr (C::kTwo) {
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++)
                        P[i][j] = mfma(x_[i][0], f[j].lo, P[i][j]);
            }
            __builtin_amdgcn_sched_barrier(0x6);
        }
        if (!live) continue;
#pragma unroll
        for (int j = 0; j < NF; j++) {
            h8 mn, mid;
            min_operands<AP>(col[j], mn, mid);
#pragma unroll
            for (int i = 0; i < MF; i++) close<AP>(col[j], mn, mid, sm[i], P[i][j], acc[i][j]);
        }
    }
    // the last (repeated) loads land before the ring is reused or the workgroup ends
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    auto out = [&](int r, float v) {  // sum r of the lane: tile r / 16, register r % 16
        const int e = r & 15;
        store(a, P_, m0 + 32 * (r / 16 / NF) + 8 * (e >> 2) + 4 * h + (e & 3), n0 + 32 * (r / 16 % NF) + (lane & 31), v);
    };
    if constexpr (KW > 1) {
        float* red = (float*)lds;  // [KW][NWN][R][64]
#pragma unroll
        for (int r = 0; r < R; r++)
            red[((kw * NWN + nw) * R + r) * 64 + lane] = acc[r / 16 / NF][r / 16 % NF][r & 15];
        __syncthreads();
        constexpr int RW = R / KW;
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int r = kw * RW + i;
            float v = red[(nw * R + r) * 64 + lane];
#pragma unroll
            for (int o = 1; o < KW; o++) v += red[((o * NWN + nw) * R + r) * 64 + lane];
            out(r, v);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) out(r, acc[r / 16 / NF][r / 16 % NF][r & 15]);
    }
}

// ------------------------------------------------------ activation planes --
// A workgroup takes RW rows.  A thread takes pieces of 8 consecutive values of
// one row; piece p = 4 g + 2 h + u goes to lane slot 32 h + row % 32 of step
// 2 g + u.  S: the sums over 32 values, divided by 32, as fp16 hi + lo in one
// more operand per superblock (hi in lane half 0, lo in 1; sub-block j in
// element j).  Slots of rows from M on stay unwritten: each row is an output
// row of its own in the products, and those are not stored.
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
//
// Neighbouring lanes hold the same piece of RW neighbouring rows, which lie
// side by side in the planes (16 RW bytes a run; with a row per workgroup each
// lane's 16 bytes go to another line).  RP pieces a thread stay in registers
// between the row's maximum and the conversion; longer rows are read twice.
template <int MODE, int RW, int RP, bool VEC>
__global__ __launch_bounds__(1024) void prep_kernel(PrepArgs a) {
    __shared__ float wmax[16 * RW];
    const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
    // a row each: an XCD takes a contiguous range of them, so that their pieces
    // meet in one L2 (the grid is then a multiple of 8)
    const int wg = RW == 1 ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const int m = wg * RW + tid % RW, p0 = tid / RW, ps = blockDim.x / RW, np = a.SB * 32;
    const int64_t row = (int64_t)(m < a.M ? m : a.M - 1) * (MODE == 2 ? a.K : a.lda);
    const size_t tile = (size_t)(m >> 5) * a.SB;
    const int r = m & 31, chunk = ps * RP;
    float v[RP][8];
    auto load = [&](int c) {
#pragma unroll
        for (int i = 0; i < RP; i++) {
            const int k = 8 * (c + p0 + ps * i);
            const bool in = k < a.K;
            // no branch around the loads: places past the row read its start
            const int64_t at = row + (in ? k : 0);
            if constexpr (MODE == 2) {
                const uint2 q = *(const uint2*)(a.QA + at);
#pragma unroll
                for (int e = 0; e < 8; e++) v[i][e] = (float)(int8_t)((e < 4 ? q.x : q.y) >> (8 * (e & 3)));
            } else if (VEC) {
                const float4 x = *(const float4*)(a.A + at), y = *(const float4*)(a.A + at + 4);
                v[i][0] = x.x; v[i][1] = x.y; v[i][2] = x.z; v[i][3] = x.w;
                v[i][4] = y.x; v[i][5] = y.y; v[i][6] = y.z; v[i][7] = y.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[i][e] = a.A[at + e];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) v[i][e] = in ? v[i][e] : 0.0f;
        }
    };
    int ex = 0;
    float inv = 0.0f;
    if constexpr (MODE == 2) {
        load(0);
    } else {
        float amax = 0.0f;
        for (int c = 0; c < np; c += chunk) {
            load(c);
#pragma unroll
            for (int i = 0; i < RP; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[i][e]));
        }
#pragma unroll
        for (int off = 32; off >= RW; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        if (lane < RW) wmax[(tid >> 6) * RW + lane] = amax;
        __syncthreads();
        for (int o = 0; o < waves; o++) amax = fmaxf(amax, wmax[o * RW + tid % RW]);
        if constexpr (MODE == 0) {
            if (amax > 0.0f) {  // the largest magnitude into [2^14, 2^15)
                int x2;
                (void)frexpf(amax, &x2);
                ex = 15 - x2 > 126 ? 126 : 15 - x2;
            }
            if (tid < RW && m < a.M) a.rs[m] = ldexpf(1.0f, -ex);
        } else {
            const float sc = amax > 0.0f ? __fdiv_rn(amax, 127.0f) : 1.0f;
            inv = __fdiv_rn(1.0f, sc);
            if (tid < RW && m < a.M) a.rs[m] = sc;
        }
        if (np > chunk) load(0);
    }
    for (int c = 0;;) {
#pragma unroll
        for (int i = 0; i < RP; i++) {
            const int p = c + p0 + ps * i;
            if (p >= np || m >= a.M) break;
            h8 hi, lo;
            float gs = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = v[i][kPi[e]];
                const float y = MODE == 0 ? ldexpf(x, ex) : MODE == 1 ? (float)to_i8(__fmul_rn(x, inv)) : x;
                hi[e] = (_Float16)y;
                lo[e] = (_Float16)(y - (float)hi[e]);
                gs += MODE == 0 ? (float)hi[e] + (float)lo[e] : y;
            }
            const int g = p >> 2, h = (p >> 1) & 1, u = p & 1;
            const size_t at = (tile * 16 + 2 * g + u) * 64 + 32 * h + r;
            a.XH[at] = hi;
            if constexpr (MODE == 0) a.XL[at] = lo;
            gs += __shfl_xor(gs, RW, 64);  // the group's four pieces: all of them are in this loop
            gs += __shfl_xor(gs, 2 * RW, 64);
            const float y = gs * 0.03125f;
            const _Float16 sh = (_Float16)y, sl = (_Float16)(y - (float)sh);
            if (u == 0) a.XS[((tile + (g >> 3)) * 64 + 32 * h + r) * 8 + (g & 7)] = h ? sl : sh;
        }
        c += chunk;
        if (c >= np) break;
        load(c);
    }
}

// Four rows a workgroup from 512 rows on, where that still gives half of the
// CUs one; below that the time is the launch's and one row's latency, and a
// row per workgroup spreads it (fp32 rows, one against four: 100 x 2048 5.3,
// 6.8; 500 x 2048 6.8, 6.7; 1023 x 2048 7.4, 7.2; 1023 x 8192 18.6, 12.0 us).
template <int MODE, bool VEC>
void launch_prep_v(const PrepArgs& a, hipStream_t s) {
    const int np = a.SB * 32;  // pieces of a row
    if (a.M >= 512) {
        const int wgs = (a.M + 3) / 4;
        if (np <= 512) prep_kernel<MODE, 4, 2, VEC><<<wgs, np * 2, 0, s>>>(a);
        else prep_kernel<MODE, 4, 4, VEC><<<wgs, 1024, 0, s>>>(a);
    } else if (np <= 256) prep_kernel<MODE, 1, 1, VEC><<<(a.M + 7) & ~7, 256, 0, s>>>(a);
    else prep_kernel<MODE, 1, 4, VEC><<<(a.M + 7) & ~7, 256, 0, s>>>(a);
}
template <int MODE>
void launch_prep(const PrepArgs& a, hipStream_t s) {
    if (MODE == 2 || a.vec) launch_prep_v<MODE, true>(a, s);
    else launch_prep_v<MODE, false>(a, s);
}

// Planes of one set of activation rows in a workspace.
struct Planes {
    size_t xh, xl, xs, rs, bytes;
};
Planes planes_of(int K, int M, bool two) {
    const size_t rows = ((size_t)M + 127) & ~size_t(127), sb = ((size_t)K + 255) / 256;
    Planes p;
    p.xh = 0;
    p.xl = p.xh + rows * sb * 512;
    p.xs = p.xl + (two ? rows * sb * 512 : 0);
    p.rs = p.xs + rows * sb * 32;
    p.bytes = p.rs + rows * 4;
    return p;
}

// Kernel and tile of a launch, by how many workgroups each would give the 256
// CUs (times of 2048 x 2048 / 8192 x 2048 Q4_K, fp32 rows, in us):
//   K split over 8 wavefronts, 16 columns a workgroup, as long as every CU
//   gets at most one (64 rows: 16 / 29), then 32 columns (19 / 20);
//   128-row tiles from the ring otherwise: 128 columns a workgroup from two
//   workgroups a CU (1023 rows: 52 / 86), 64 columns and two K slices from one
//   (38 / 98), else four K slices: 32 columns.  With one weight plane 64 x 64
//   values a wavefront read half as much from LDS and fit the registers: with
//   two K slices 128 x 64 (8192 x 2048, 500 rows 56.1 -> 53.5; 2048 x 8192,
//   1023 rows 128 -> 118, codes 72 -> 68), with four 64 x 64 (29 -> 25).
// More K slices for longer rows keep the fp32 sums short: error against 64
// bits at K = 8192 2.4e-7, 2.25e-7, 2.15e-7 with one, two, four (the single-
// row kernels' 2.35e-7).
template <int T, int AP>
void launch_t(Args& a, int M, hipStream_t s) {
    constexpr int kCus = 256;
    // tiles of `cols` x `rows`; returns the grid
    auto tiles = [&](int cols, int rows) {
        a.nt = 0;
        for (int i = 0; i < a.np; i++) {
            a.p[i].nt0 = a.nt;
            a.nt += (a.p[i].N + cols - 1) / cols;
        }
        a.mt = (M + rows - 1) / rows;
        return dim3((unsigned)((a.nt + 7) / 8 * 8 * a.mt));
    };
    int cols16 = 0;  // 16-column tiles
    for (int i = 0; i < a.np; i++) cols16 += (a.p[i].N + 15) / 16;
    const int cols32 = (cols16 + 1) / 2, m64 = (M + 63) / 64, m128 = (M + 127) / 128;
    const bool narrow = m64 <= 8 && m64 * cols16 <= kCus;
    if (narrow || M <= 32 || (m64 <= 4 && m64 * cols32 <= kCus)) {
        const int rows = M <= 16 ? 16 : M <= 32 ? 32 : 64;
        const dim3 g = tiles(narrow ? 16 : 32, rows);
#define KS(MF, NB)                                                                       \
    (narrow ? gemm_f16_ks_kernel<T, AP, MF, 1, 8, NB><<<g, 512, 0, s>>>(a)               \
            : gemm_f16_ks_kernel<T, AP, MF, 2, 8, NB><<<g, 512, 0, s>>>(a))
        if (rows == 16) KS(1, 8);
        else if (rows == 32) KS(2, 8);
        else KS(4, 8 / AP);
#undef KS
    } else if (m128 * cols32 >= 8 * kCus && a.SB <= 16) {
        const dim3 g = tiles(128, 128);
        gemm_f16_ring_kernel<T, AP, 4, 1, 4, 4 / AP><<<g, 256, 0, s>>>(a);
    } else if (m128 * cols32 >= 2 * kCus && a.SB <= 32) {
        if constexpr (Col<T, 2, 2>::kTwo) {
            const dim3 g = tiles(64, 128);
            gemm_f16_ring_kernel<T, AP, 4, 1, 2, 2 / AP><<<g, 256, 0, s>>>(a);
        } else {
            const dim3 g = tiles(128, 64);
            gemm_f16_ring_kernel<T, AP, 2, 2, 2, 2 / AP><<<g, 256, 0, s>>>(a);
        }
    } else if constexpr (Col<T, 2, 2>::kTwo) {
        const dim3 g = tiles(32, 128);
        gemm_f16_ring_kernel<T, AP, 4, 1, 1, 1><<<g, 256, 0, s>>>(a);
    } else {
        const dim3 g = tiles(64, 64);
        gemm_f16_ring_kernel<T, AP, 2, 2, 1, 2 / AP><<<g, 256, 0, s>>>(a);
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
    for (int i = 0; i < n; i++) a.p[i] = Prob{(const uint8_t*)d[i].W, d[i].C, (uint32_t)row_bytes(type, K), d[i].N, d[i].ldc, 0};
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
