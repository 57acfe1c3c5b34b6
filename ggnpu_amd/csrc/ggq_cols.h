// ggq_cols.h -- weight columns of raw GGUF blocks as fp16 MFMA operands (gfx950).
//
// A block's integer scale is folded into its codes: Q4_K and Q5_K sub-blocks
// give sc*q <= 1953, exact in fp16, so one MFMA chain runs over a whole
// 256-value superblock and the fp32 scale is applied once per 256 values.
// Q6_K (sc*q up to 4096), IQ4_XS ((ls-32)*kv), Q8_0 and IQ4_NL (q*d, d under a
// power of two common to the column's 256 values) are the sum of two fp16
// values, hi = fp16(q*s) and the exact remainder lo = q*s - hi (a fused
// multiply-add), in two planes.  The K-quant mins are one more MFMA per
// superblock: the sums of x over the 32 values of each sub-block against the
// 6-bit mins.  fp32 rows are hi + lo as well; against two weight planes the
// product of the two low parts (2^-22 of a product) is left out.
//
// Pieces: piece q (0..3) of a 32-value group g holds the values k = 32 g + 8 q
// + {0,2,1,3,4,6,5,7} of one row or column, one lane's operand of an MFMA.
// The order inside 8 values is what masking the even and the odd bytes of two
// code dwords gives, so decoding needs no byte shuffles.
// v_mfma_f32_32x32x16_f16 takes a group in two steps u (lane 32 h + i: row i,
// piece 2 h + u), v_mfma_f32_16x16x32_f16 in one (lane 16 q + i: row i, piece
// q).
#pragma once
#include "ggq_device.h"

namespace ggq {


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

template <int CTRL> __device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// 2^(b - 127), b byte e of the words; 1 in kRowPower.
constexpr uint32_t kRowPower = 0x7F7F7F7Fu;
template <int W> __device__ __forceinline__ float power(const uint32_t (&w)[W], int e) {
    const uint32_t v = w[e >> 2];
    return __builtin_bit_cast(float, ((e & 3) == 3 ? v >> 1 : v << (23 - 8 * (e & 3))) & 0x7F800000u);
}
// End of a superblock for one tile.  with_mins: the chain P of fp32 rows under
// the column's scale with the mins (sm: the sums of x); they cancel in part, so
// they meet before they round against the sum.
template <class C, class V>
__device__ __forceinline__ void with_mins(const C& col, h8 mn, h8 mid, h8 sm, V& P) {
    const float d = col.k.d, dm = -32.0f * col.k.dm;  // the sums carry 1 / 32
    P = mfma(sm, mid, P);
    const V S = mfma(sm, mn, V{});
#pragma unroll
    for (int e = 0; e < (int)sizeof(V) / 4; e++) P[e] = __builtin_fmaf(d, P[e], dm * S[e]);
}
// close: the same and the chains without mins onto the sums; times(e, v): v
// under the power of two of element e's row.
struct NoPower {
    __device__ __forceinline__ float operator()(int, float v) const { return v; }
};
template <int AP, class C, class V, class F = NoPower>
__device__ __forceinline__ void close(const C& col, h8 mn, h8 mid, h8 sm, V P, V& acc, F times = NoPower{}) {
    constexpr int E = sizeof(V) / 4;
    const float d = col.k.d;
    if constexpr (C::kMin && AP == 2) {
        with_mins(col, mn, mid, sm, P);
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] += times(e, P[e]);
    } else if constexpr (C::kMin) {  // codes: both are exact integers
        const float dm = -32.0f * col.k.dm;
        const V S = mfma(sm, mn, V{});
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = __builtin_fmaf(d, P[e], __builtin_fmaf(dm, S[e], acc[e]));
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = __builtin_fmaf(d, times(e, P[e]), acc[e]);
    }
}
template <int AP, class C>
__device__ __forceinline__ void min_operands(const C& col, h8& mn, h8& mid) {
    if constexpr (C::kMin) {
        mn = col.k.mins();
        if constexpr (AP == 2) mid = col.k.mids(C::kMid);
    }
}
}  // namespace ggq
