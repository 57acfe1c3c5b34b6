// ggq_gemm_f16.hip -- dense GEMM on raw GGUF blocks for many activation rows
// (prompts and batches), C[m][n] = sum_k x[m][k] w[n][k], on the fp16 matrix
// cores of gfx950; the weights as ggq_cols.h decodes them.
//
// Activations.  prep_* kernels write them once as fp16 planes in the order
// the MFMA reads: fp32 rows as hi + lo (22 bits) under a power of two per row
// and superblock, int8 codes as one exact plane.  A power per row alone lost the
// values that lie far below a row's largest (rows with one value of 2^22 in a
// superblock of zero weights, K = 8192, 48 rows, Q5_K: relative error 8.3e-6;
// with a power per superblock 2.1e-7, fp32 FMA 2.3e-7).  For codes every product
// and, below 2^24, every partial sum of a superblock is an exact integer in
// fp32.
// The planes are stored in the piece order of the 32x32x16 MFMA, [32-row
// tile][step 2g + u][lane][8]; the 16x16x32 one's operand is four runs of 256
// bytes of it.
#include "ggq_cols.h"

namespace ggq {
namespace {

constexpr int kProb = 4;
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
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
    const uint32_t* XE;  // powers of two of each row and superblock (fp32 rows)
    const float* rs;     // scale of each row
};

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
    // powers of the lane's four rows
    auto powers = [&](int i, int sb, uint32_t (&e)[1]) {
        const int r = m0 / 16 + i;
        e[0] = a.XE[((size_t)(r >> 1) * a.SB + sb) * 8 + 4 * (q & 1) + 2 * (r & 1) + (q >> 1)];
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
        uint32_t pw[MF][1];
#pragma unroll
        for (int j = 0; j < NF; j++) {
            col[j].open(sb, q, a.nb);
            col[j].load_head(row[j], nsb, q, a.nb);
        }
#pragma unroll
        for (int i = 0; i < MF; i++) {
            sm[i] = C::kMin ? sums(i, sb) : h8{};
            if constexpr (AP == 2) powers(i, sb, pw[i]);
        }
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
            for (int i = 0; i < MF; i++) {
                if constexpr (AP == 2) close<AP>(col[j], mn, mid, sm[i], P[i][j], acc[i][j], [&](int e, float v) { return power(pw[i], e) * v; });
                else close<AP>(col[j], mn, mid, sm[i], P[i][j], acc[i][j]);
            }
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

// 64 lanes' 16 bytes at src + 16 lane into LDS at lds + 16 lane (offsets below
// 128 KB, the largest ring, which the tests run); the caller waits on the vector
// memory counter.  (m0 is reserved: the compiler keeps nothing in it, sets it
// right before its own uses, and takes it in no clobber list.  Its builtin for
// this load would wait for all of them before each read of LDS.)
__device__ __forceinline__ void dma16(const h8* src, uint32_t lane16, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(lane16), "s"(src) : "memory");
}

constexpr int kRing = 4;  // chunks
// Workgroups of a CU, by their LDS.
template <int AP, int MF, int NWN, int CS> constexpr int ring_wgs() {
    return 4 / NWN * kRing * MF * AP * CS * 1024 <= 64 * 1024 ? 2 : 1;
}
// Superblocks of the longest row of a ring kernel; more need more K slices.
constexpr int kMaxSB = 128;
template <int NWN> constexpr int ring_sb() { return NWN == 4 ? 16 : NWN == 2 ? 32 : kMaxSB; }

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
// Q6_K 394 -> 215 us (64 x 64 spilled most of its sums; here the fp32 rows of
// Q6_K still spill 26 registers and those of the other formats up to 7).
// Operands of a step are read during the step before it; weights straight from
// the caches, one part ahead.
template <int T, int AP, int MF, int NF, int NWN, int CS>
__global__ __launch_bounds__(256, (ring_wgs<AP, MF, NWN, CS>())) void gemm_f16_ring_kernel(Args a) {
    constexpr int PB = 2, KW = 4 / NWN, S = kRing, R = MF * NF * 16;
    constexpr int CB = MF * AP * CS * 64;  // h8 of a chunk
    constexpr int PP = MF * AP * CS / NWN;  // loads of a wavefront per chunk
    constexpr int NC = 16 / CS;             // chunks of a superblock
    static_assert(NC % S == 0, "a superblock's chunks fill whole rounds of the ring");
    static_assert(KW * S * CB * 16 <= 128 * 1024, "offsets of dma16");
    constexpr int kRed = KW > 1 ? 4 * R * 64 * 4 / 16 : 0;
    constexpr int kLds = KW * S * CB > kRed ? KW * S * CB : kRed;
    // behind the ring, the rows' powers for the whole K (a load near its use
    // would wait, in order, for the ring's: 2048 x 8192 Q6_K, 500 rows 81 -> 85
    // us).  Two workgroups stay below 160 KB: at 160 they took turns (18 -> 30).
    __shared__ h8 lds[kLds + (AP == 2 ? MF * ring_sb<NWN>() * 2 : 0)];
    u4v* const powers = (u4v*)(lds + kLds);
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
    const int tid = threadIdx.x, ne = a.SB * 2;  // 16 bytes of a row tile
    u4v pv[AP == 2 ? MF : 1];
    if constexpr (AP == 2) {
        static_assert(ring_sb<NWN>() * 2 <= 256, "a row tile's powers in one load");
        const u4v* src = (const u4v*)a.XE + (size_t)(m0 / 32) * ne + (tid < ne ? tid : 0);
#pragma unroll
        for (int k = 0; k < MF; k++) pv[k] = src[ne * k];
    }
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
    if constexpr (AP == 2) {  // (waits for its own loads, the first, and none of the ring's)
        if (tid < ne) {
#pragma unroll
            for (int k = 0; k < MF; k++) powers[tid + ne * k] = pv[k];
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
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 1) * PP) : "memory");
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
        // (K-quants of fp32 rows: products and mins are added first, then
        // scaled where a row's power differs: most superblocks have it)
        if constexpr (AP == 2) {
            if constexpr (C::kMin) {
#pragma unroll
                for (int j = 0; j < NF; j++) {
                    h8 mn, mid;
                    min_operands<AP>(col[j], mn, mid);
#pragma unroll
                    for (int i = 0; i < MF; i++) with_mins(col[j], mn, mid, sm[i], P[i][j]);
                }
            }
            uint32_t pw[MF][4], other = 0;
#pragma unroll
            for (int i = 0; i < MF; i++) {
                const u4v e = powers[(i * a.SB + sb) * 2 + h];
#pragma unroll
                for (int k = 0; k < 4; k++) pw[i][k] = e[k];
            }
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int k = 0; k < 4; k++) other |= pw[i][k] ^ kRowPower;
            if (__ballot(other != 0)) {
#pragma unroll
                for (int i = 0; i < MF; i++)
#pragma unroll
                    for (int j = 0; j < NF; j++)
#pragma unroll
                        for (int e = 0; e < 16; e++) P[i][j][e] *= power(pw[i], e);
            }
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int j = 0; j < NF; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        acc[i][j][e] = C::kMin ? acc[i][j][e] + P[i][j][e] : __builtin_fmaf(col[j].k.d, P[i][j][e], acc[i][j][e]);
        } else {
#pragma unroll
            for (int j = 0; j < NF; j++) {
                h8 mn, mid;
                min_operands<AP>(col[j], mn, mid);
#pragma unroll
                for (int i = 0; i < MF; i++) close<AP>(col[j], mn, mid, sm[i], P[i][j], acc[i][j]);
            }
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
// element j).  Rows from M to the end of their 128-row tile are zeros: the
// products of a tile with stale rows drew the power, and cost the clock, of a
// full one (128256 x 2048 Q4_K, 33 rows 125 -> 144 us).
struct PrepArgs {
    const float* A;
    const int8_t* QA;
    const float* bs;  // scales of 32 codes, [M][K / 32]
    int lda, M, K, SB, vec;
    h8* XH;
    h8* XL;
    _Float16* XS;
    uint8_t* XE;
    float* rs;
};
constexpr int kPi[8] = {0, 2, 1, 3, 4, 6, 5, 7};
// e of the power 2^e that brings the largest magnitude into [2^14, 2^15)
__device__ __forceinline__ int scale_exp(float amax) {
    const int ex = 15 - __builtin_amdgcn_frexp_expf(amax);
    return ex > 126 ? 126 : ex;
}

// MODE 0: fp32 rows as hi + lo; 1: fp32 rows quantized per row to int8 codes
// (the codes and scales of the row quantizer); 2: given int8 codes; 3: given
// int8 codes and block scales, whose products are fp32 rows as in 0.
//
// Neighbouring lanes hold the same piece of RW neighbouring rows, which lie
// side by side in the planes (16 RW bytes a run; with a row per workgroup each
// lane's 16 bytes go to another line).  RP pieces a thread stay in registers
// between the row's maximum and the conversion; longer rows are read twice.
// A superblock's pieces lie in one wavefront, PP neighbours in a lane.
template <int MODE, int RW, int RP, bool VEC>
__global__ __launch_bounds__(1024) void prep_kernel(PrepArgs a) {
    constexpr bool kCodes = MODE >= 2, kSplit = MODE == 0 || MODE == 3;
    __shared__ float wmax[16 * RW];
    const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
    // a row each: an XCD takes a contiguous range of them, so that their pieces
    // meet in one L2
    const int wg = RW == 1 ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const int m = wg * RW + tid % RW, p0 = tid / RW, ps = blockDim.x / RW, np = a.SB * 32;
    const int64_t row = (int64_t)(m < a.M ? m : a.M - 1) * (kCodes ? a.K : a.lda);
    const size_t tile = (size_t)(m >> 5) * a.SB;
    const int r = m & 31, chunk = ps * RP;
    constexpr int PP = RW == 1 ? 1 : 2;
    static_assert(RP % PP == 0, "");
    auto piece = [&](int i) { return PP * (p0 + ps * (i / PP)) + i % PP; };  // of a chunk, register i
    float v[RP][8];
    auto load = [&](int c) {
#pragma unroll
        for (int i = 0; i < RP; i++) {
            const int k = 8 * (c + piece(i));
            const bool in = m < a.M && k < a.K;
            // no branch around the loads: places past the row read its start
            const int64_t at = row + (in ? k : 0);
            if constexpr (kCodes) {
                const uint2 q = *(const uint2*)(a.QA + at);
                const float d = MODE == 3 ? a.bs[at >> 5] : 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float x = (float)(int8_t)((e < 4 ? q.x : q.y) >> (8 * (e & 3)));
                    v[i][e] = MODE == 3 ? __fmul_rn(x, d) : x;
                }
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
    // the largest magnitude of each superblock in hand
    float sx[RP / PP];
    auto largest = [&] {
#pragma unroll
        for (int i0 = 0; i0 < RP; i0 += PP) {
            float x = 0.0f;
#pragma unroll
            for (int j = 0; j < PP; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) x = fmaxf(x, fabsf(v[i0 + j][e]));
            // the other pieces: in the sixteen lanes, then in the others
            if constexpr (RW == 1) {
                x = fmaxf(x, dpp<0x121>(x));
                x = fmaxf(x, dpp<0x122>(x));
            }
            x = fmaxf(x, dpp<0x124>(x));
            x = fmaxf(x, dpp<0x128>(x));
            x = fmaxf(x, __shfl_xor(x, 16, 64));
            if constexpr (RW == 4) x = fmaxf(x, __shfl_xor(x, 32, 64));
            sx[i0 / PP] = x;
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
            largest();
#pragma unroll
            for (int i = 0; i < RP / PP; i++) amax = fmaxf(amax, sx[i]);
        }
        if constexpr (RW == 1) amax = fmaxf(amax, __shfl_xor(amax, 32, 64));  // a wavefront's other superblock
        if (lane < RW) wmax[(tid >> 6) * RW + lane] = amax;
        __syncthreads();
        for (int o = 0; o < waves; o++) amax = fmaxf(amax, wmax[o * RW + tid % RW]);
        if constexpr (kSplit) {
            if (amax > 0.0f) ex = scale_exp(amax);
            if (tid < RW && m < a.M) a.rs[m] = ldexpf(1.0f, -ex);
        } else {
            const float sc = amax > 0.0f ? __fdiv_rn(amax, 127.0f) : 1.0f;
            inv = __fdiv_rn(1.0f, sc);
            if (tid < RW && m < a.M) a.rs[m] = sc;
        }
        if (np > chunk) {
            load(0);
            if constexpr (kSplit) largest();
        }
    }
    for (int c = 0;;) {
#pragma unroll
        for (int i0 = 0; i0 < RP; i0 += PP) {
            const int q0 = c + piece(i0), g = q0 >> 2, h = (q0 >> 1) & 1;
            if (q0 >= np) break;
            int es = ex;
            if constexpr (kSplit) {
                const float smax = sx[i0 / PP];
                // its own from 2^4 below the row's on, at most 2^126 from it (a
                // byte, an fp32 exponent)
                if (smax > 0.0f && scale_exp(smax) - ex >= 4) es = min(scale_exp(smax), ex + 126);
                if ((q0 & 31) == 0) a.XE[(tile + (g >> 3)) * 32 + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3)] = (uint8_t)(127 - (es - ex));
            }
            float gs = 0.0f;
#pragma unroll
            for (int j = 0; j < PP; j++) {
                h8 hi, lo;
                float ps8 = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float x = v[i0 + j][kPi[e]];
                    const float y = kSplit ? ldexpf(x, es) : MODE == 1 ? (float)to_i8(__fmul_rn(x, inv)) : x;
                    hi[e] = (_Float16)y;
                    lo[e] = (_Float16)(y - (float)hi[e]);
                    ps8 += kSplit ? (float)hi[e] + (float)lo[e] : y;
                }
                const int u = (q0 + j) & 1;
                const size_t at = (tile * 16 + 2 * g + u) * 64 + 32 * h + r;
                a.XH[at] = hi;
                if constexpr (kSplit) a.XL[at] = lo;
                gs += ps8;
            }
            // the group's four pieces: all of them are in this loop
            if constexpr (PP == 1) gs += __shfl_xor(gs, RW, 64);
            gs += __shfl_xor(gs, 2 * RW / PP, 64);
            const float y = gs * 0.03125f;
            const _Float16 sh = (_Float16)y, sl = (_Float16)(y - (float)sh);
            if ((q0 & 1) == 0) a.XS[((tile + (g >> 3)) * 64 + 32 * h + r) * 8 + (g & 7)] = h ? sl : sh;
        }
        c += chunk;
        if (c >= np) break;
        load(c);
        if constexpr (kSplit) largest();
    }
}

// Four rows a workgroup from 512 rows on, where that still gives half of the
// CUs one; below that the time is the launch's and one row's latency, and a
// row per workgroup spreads it (fp32 rows, one against four: 100 x 2048 5.3,
// 6.8; 500 x 2048 6.8, 6.7; 1023 x 2048 7.4, 7.2; 1023 x 8192 18.6, 12.0 us).
template <int MODE, bool VEC>
void launch_prep_v(const PrepArgs& a, hipStream_t s) {
    const int np = a.SB * 32, rows = (a.M + 127) & ~127;  // pieces of a row
    if (a.M >= 512) {
        const int wgs = rows / 4;
        if (np <= 512) prep_kernel<MODE, 4, 2, VEC><<<wgs, np * 2, 0, s>>>(a);
        else prep_kernel<MODE, 4, 4, VEC><<<wgs, 1024, 0, s>>>(a);
    } else if (np <= 256) prep_kernel<MODE, 1, 1, VEC><<<rows, 256, 0, s>>>(a);
    else prep_kernel<MODE, 1, 4, VEC><<<rows, 256, 0, s>>>(a);
}
template <int MODE>
void launch_prep(const PrepArgs& a, hipStream_t s) {
    if constexpr (MODE >= 2) launch_prep_v<MODE, true>(a, s);
    else if (a.vec) launch_prep_v<MODE, true>(a, s);
    else launch_prep_v<MODE, false>(a, s);
}

// Planes of one set of activation rows in a workspace.
struct Planes {
    size_t xh, xl, xs, xe, rs, bytes;
};
Planes planes_of(int K, int M, bool two) {
    const size_t rows = ((size_t)M + 127) & ~size_t(127), sb = ((size_t)K + 255) / 256;
    Planes p;
    p.xh = 0;
    p.xl = p.xh + rows * sb * 512;
    p.xs = p.xl + (two ? rows * sb * 512 : 0);
    p.xe = p.xs + rows * sb * 32;
    p.rs = p.xe + (two ? rows * sb : 0);
    p.bytes = p.rs + rows * 4;
    return p;
}

// Kernel and tile of a launch, by how many workgroups each would give the CUs
// (of 256; times of 2048 x 2048 / 8192 x 2048 Q4_K, fp32 rows, in us):
//   K split over 8 wavefronts, 16 columns a workgroup, as long as every CU
//   gets at most one (64 rows: 16 / 29), then 32 columns (19 / 20);
//   128-row tiles from the ring otherwise: 128 columns a workgroup from two
//   workgroups a CU (1023 rows: 52 / 86), 64 columns and two K slices from one
//   (38 / 98), else four K slices: 32 columns.  With one weight plane 64 x 64
//   values a wavefront read half as much from LDS and fit the registers: with
//   two K slices 128 x 64 (8192 x 2048, 500 rows 56.1 -> 53.5; 2048 x 8192,
//   1023 rows 128 -> 118, codes 72 -> 68; 64 rows at any width, which fill
//   them: 128256 x 2048 140 -> 103), with four 64 x 64 (29 -> 25).
// More K slices for longer rows keep the fp32 sums short: error against 64
// bits at K = 8192 2.4e-7, 2.25e-7, 2.15e-7 with one, two, four (the single-
// row kernels' 2.35e-7).
template <int T, int AP>
void launch_t(Args& a, int M, hipStream_t s) {  // M: the rows of the whole call
    const int cus = cu_count();
    // tiles of `cols` x `rows`; returns the grid
    auto tiles = [&](int cols, int rows) {
        a.nt = 0;
        for (int i = 0; i < a.np; i++) {
            a.p[i].nt0 = a.nt;
            a.nt += (a.p[i].N + cols - 1) / cols;
        }
        a.mt = (a.M + rows - 1) / rows;
        return dim3((unsigned)((a.nt + 7) / 8 * 8 * a.mt));
    };
    int cols16 = 0;  // 16-column tiles
    for (int i = 0; i < a.np; i++) cols16 += (a.p[i].N + 15) / 16;
    const int cols32 = (cols16 + 1) / 2, m64 = (M + 63) / 64, m128 = (M + 127) / 128;
    const bool narrow = m64 <= 8 && m64 * cols16 <= cus;
    if (narrow || M <= 32 || (m64 <= 4 && m64 * cols32 <= cus)) {
        const int rows = M <= 16 ? 16 : M <= 32 ? 32 : 64;
        const dim3 g = tiles(narrow ? 16 : 32, rows);
#define KS(MF, NB)                                                                       \
    (narrow ? gemm_f16_ks_kernel<T, AP, MF, 1, 8, NB><<<g, 512, 0, s>>>(a)               \
            : gemm_f16_ks_kernel<T, AP, MF, 2, 8, NB><<<g, 512, 0, s>>>(a))
        if (rows == 16) KS(1, 8);
        else if (rows == 32) KS(2, 8);
        else KS(4, 8 / AP);
#undef KS
    } else if ((Col<T, 2, 2>::kTwo || M > 64) && m128 * cols32 >= 8 * cus && a.SB <= ring_sb<4>()) {
        const dim3 g = tiles(128, 128);
        gemm_f16_ring_kernel<T, AP, 4, 1, 4, 4 / AP><<<g, 256, 0, s>>>(a);
    } else if (m128 * cols32 >= 2 * cus && a.SB <= ring_sb<2>()) {
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

hipError_t launch_gemm_f16_prep(int mode, const float* A, int lda, const int8_t* qa, const float* bs, int K, int M,
                                void* ws, hipStream_t s) {
    const Planes pl = planes_of(K, M, mode == 0 || mode == 3);
    char* b = (char*)ws;
    PrepArgs a{};
    a.A = A;
    a.QA = qa;
    a.bs = bs;
    a.lda = lda;
    a.M = M;
    a.K = K;
    a.SB = (K + 255) / 256;
    a.vec = A && ((uintptr_t)A & 15u) == 0 && lda % 4 == 0;
    a.XH = (h8*)(b + pl.xh);
    a.XL = (h8*)(b + pl.xl);
    a.XS = (_Float16*)(b + pl.xs);
    a.XE = (uint8_t*)(b + pl.xe);
    a.rs = (float*)(b + pl.rs);
    if (mode == 0) launch_prep<0>(a, s);
    else if (mode == 1) launch_prep<1>(a, s);
    else if (mode == 2) launch_prep<2>(a, s);
    else launch_prep<3>(a, s);
    return hipGetLastError();
}

hipError_t launch_gemm_f16(uint32_t type, const GemmDesc* d, int n, int K, int M, int M_call, bool codes,
                           const float* sa, const void* ws, hipStream_t s) {
    if (n < 1 || n > kProb || K > 256 * kMaxSB) return hipErrorInvalidValue;
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
    a.XE = (const uint32_t*)(b + pl.xe);
    a.rs = sa ? sa : (const float*)(b + pl.rs);
#define GO(TT)                                    \
    case TT:                                      \
        if (codes) launch_t<TT, 1>(a, M_call, s); \
        else launch_t<TT, 2>(a, M_call, s);       \
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
