// ggq_gemm_rows.hip -- dense matmuls of 5..32 fp32 activation rows on the fp16
// matrix cores of gfx950, weights as ggq_cols.h decodes them.
//
// A batch this small is bound by what a CU reads beside its weights: with a
// workgroup per few columns the activations (4 bytes a value, against 0.56 of a
// Q4_K weight) come through L2 once per workgroup.  Here each wavefront keeps
// one superblock of all rows in registers, as fp16 hi + lo (22 bits) under a
// power of two per row and superblock, and the workgroup streams 16-column
// tiles past them: one workgroup a CU, its wavefronts side by side along K,
// their sums added through LDS in wavefront order.  K beyond the wavefronts of
// a workgroup is split over workgroups, whose partial sums a second launch adds
// in slice order.  The fp32 rows are split in registers, so no planes are
// written, and all weights of a level, of any types, share one launch.
//
// Measured (us, before -> here): 16384 x 2048 Q4_K, 8 / 16 / 32 rows 23 -> 12,
// 20 -> 12, 25 -> 17; 2048 x 8192 Q6_K 26 -> 13, 22 -> 14, 28 -> 17; 128256 x
// 2048 Q4_K, 8 / 32 rows 144 -> 54, 170 -> 67.  Bound: the start (launch, the
// rows' way into registers: about 6 us for 16 rows, 9 for 32) and past it the
// decoding VALU, 0.39 us per 1000 columns of K = 2048 (3.0 TB/s of Q4_K; 2.5
// with 32 rows).
// Error against 64 bits on N(0, 1) rows, in every format, over that of the fp32
// kernels (products of 24 bits): 0.8 in the middle and at most 1.0 up to K =
// 4096, 0.9 and 1.06 up to 16384 (fewer fp32 additions a sum).
#include "ggq_cols.h"

namespace ggq {
namespace {

typedef float f2v __attribute__((ext_vector_type(2)));
constexpr int kProb = 8, kWaves = 8;
struct Prob {
    const uint8_t* W;
    float* C;
    uint32_t row_bytes, type;
    int N, ldc;
    int col0;      // first of its columns in the partial sums
    int wg0, wgs;  // first workgroup (of a slice) and how many
};
struct Args {
    Prob p[kProb];
    int np, M, SB, nb, lda;
    int slices, per;  // K slices and their superblocks (= wavefronts)
    int cols;         // columns of a row of partial sums
    const float* A;
    float* part;  // [slice][row][cols], with more than one slice
};

// A wavefront's rows on their way to the operands' order: 64 values of 16 rows
// (an odd number of 16-byte places apart), the sums and the scales.
struct Stage {
    struct Row16 { union { uint2 u[18]; h8 p[9]; }; };
    struct Sum { union { _Float16 h[8]; h8 p; }; };
    Row16 hi[16], lo[16];
    Sum sum[2][16];
    float scale[16];
};
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int T, int MF>
__device__ __forceinline__ void rows_body(const Args& a, const Prob& p, int slice, int wg, char* lds) {
    Stage* const stage = (Stage*)lds;
    float* const red = (float*)lds;
    constexpr int PB = 4, R = 4 * MF;
    typedef Col<T, PB, 1> C;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4;
    const int left = a.SB - slice * a.per, live = left < a.per ? left : a.per;  // wavefronts with a superblock
    const bool on = w < live;
    const int sb = slice * a.per + (on ? w : 0);
    const int tiles = (p.N + 15) / 16;
    auto row_of = [&](int tile) {
        int n = tile * 16 + (lane & 15);
        n = n < p.N ? n : p.N - 1;
        return Row{p.W, (uint32_t)n * p.row_bytes};
    };
    int tile = wg;
    C col;
    {
        const Row r = row_of(tile);
        col.load_head(r, sb, q, a.nb);
#pragma unroll
        for (int c = 0; c < 4; c++) col.load_part(r, sb, q, a.nb, c);
    }

    // The superblock's rows: hi and lo of the pieces of each group, the scale
    // of the rows this lane's sums belong to, and the sums over 32 values,
    // divided by 32, as hi (piece 0) and lo (piece 1) of the mins' operand.
    // Sixteen lanes load 256 consecutive bytes of a row (in the operands' own
    // order, a row per lane, each load takes 64 lines: 32 rows cost 7 us of
    // them) and the halves change lanes through the wavefront's part of LDS,
    // 64 values at a time.
    h8 xh[MF][8], xl[MF][8], sm[MF];
    f4v sc[MF];
    Stage& st = stage[w];
    const int t = lane >> 4, c = lane & 15;
    const int Kv = (int)opaque((uint32_t)a.nb * 32);
    float4 v[MF][4][4];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = 16 * i + 4 * j + t;
            const float* const x = a.A + (int64_t)(m < a.M ? m : a.M - 1) * a.lda;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                // (only blocks of 32 values can end inside a superblock)
                const int k = 256 * sb + 64 * g + 4 * c;
                const bool in = (T != T_Q8_0 && T != T_IQ4_NL) || k < Kv;
                const float4 u = *(const float4*)(x + (in ? k : 0));
                v[i][j][g] = in ? u : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
#pragma unroll
    for (int i = 0; i < MF; i++) {
        float up[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float amax = 0.0f;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 u = v[i][j][g];
                amax = fmaxf(fmaxf(fmaxf(amax, fabsf(u.x)), fmaxf(fabsf(u.y), fabsf(u.z))), fabsf(u.w));
            }
            amax = fmaxf(amax, dpp<0xB1>(amax));   // neighbours
            amax = fmaxf(amax, dpp<0x4E>(amax));   // pairs of a quad
            amax = fmaxf(amax, dpp<0x141>(amax));  // quads of eight lanes
            amax = fmaxf(amax, dpp<0x140>(amax));  // halves of the sixteen
            int ex = 0;
            if (amax > 0.0f) {  // the largest magnitude into [2^14, 2^15)
                ex = 15 - __builtin_amdgcn_frexp_expf(amax);
                ex = ex > 126 ? 126 : ex;
            }
            up[j] = ldexpf(1.0f, ex);
            if (c == 0) st.scale[4 * j + t] = ldexpf(1.0f, -ex);
        }
#pragma unroll
        for (int g = 0; g < 4; g++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4 u = v[i][j][g];
                const f2v s0 = {u.x * up[j], u.z * up[j]}, s1 = {u.y * up[j], u.w * up[j]};
                const h2 h0 = __builtin_convertvector(s0, h2), h1 = __builtin_convertvector(s1, h2);
                const f2v d0 = {__builtin_fmaf((float)h0.x, -1.0f, s0.x), __builtin_fmaf((float)h0.y, -1.0f, s0.y)};
                const f2v d1 = {__builtin_fmaf((float)h1.x, -1.0f, s1.x), __builtin_fmaf((float)h1.y, -1.0f, s1.y)};
                st.hi[4 * j + t].u[c] = make_uint2(__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1));
                st.lo[4 * j + t].u[c] = make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(d0, h2)),
                                                   __builtin_bit_cast(uint32_t, __builtin_convertvector(d1, h2)));
                if constexpr (C::kMin) {
                    float gs = (s0.x + s0.y) + (s1.x + s1.y);
                    gs += dpp<0xB1>(gs);
                    gs += dpp<0x4E>(gs);
                    gs += dpp<0x141>(gs);
                    gs *= 0.03125f;
                    const _Float16 sh = (_Float16)gs;
                    if ((c & 7) == 0) {
                        st.sum[0][4 * j + t].h[2 * g + (c >> 3)] = sh;
                        st.sum[1][4 * j + t].h[2 * g + (c >> 3)] = (_Float16)(gs - (float)sh);
                    }
                }
            }
            // other lanes of the wavefront read these places: LDS serves a
            // wavefront in order, so only the compiler has to keep it
            wave_fence();
#pragma unroll
            for (int u = 0; u < 2; u++) {
                xh[i][2 * g + u] = st.hi[c].p[4 * u + q];
                xl[i][2 * g + u] = st.lo[c].p[4 * u + q];
            }
            wave_fence();
        }
        sm[i] = C::kMin && q < 2 ? st.sum[q & 1][c].p : h8{};
        sc[i] = *(const f4v*)&st.scale[4 * q];
        wave_fence();
    }
    __syncthreads();  // the places become the tiles' sums

    const uint32_t k1024 = opaque(0x64006400u);
    for (int par = 0; tile < tiles; tile += p.wgs, par ^= 1) {
        f4v acc[MF];
        if (on) {
            const Row next = row_of(tile + p.wgs < tiles ? tile + p.wgs : tile);
            f4v P[MF];
            col.open(sb, q, a.nb);
            col.load_head(next, sb, q, a.nb);
#pragma unroll
            for (int g = 0; g < 8; g++) {
                Frag f;
                col.template piece<true>(g, 0, q, k1024, f);
                if (g & 1) col.load_part(next, sb, q, a.nb, g >> 1);
#pragma unroll
                for (int i = 0; i < MF; i++) P[i] = mfma(xh[i][g], f.hi, g ? P[i] : f4v{});
#pragma unroll
                for (int i = 0; i < MF; i++) P[i] = mfma(xl[i][g], f.hi, P[i]);
                if constexpr (C::kTwo) {
#pragma unroll
                    for (int i = 0; i < MF; i++) P[i] = mfma(xh[i][g], f.lo, P[i]);
                }
                __builtin_amdgcn_sched_barrier(0x6);
            }
            h8 mn, mid;
            min_operands<2>(col, mn, mid);
#pragma unroll
            for (int i = 0; i < MF; i++) {
                acc[i] = f4v{};
                close<2>(col, mn, mid, sm[i], P[i], acc[i]);
            }
        }
        // two sets of places in turn: a tile's are read between its barrier
        // and the next one's, and written again after that
        float* const rp = red + par * kWaves * R * 64;
        if (on) {
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) rp[(w * R + 4 * i + e) * 64 + lane] = acc[i][e] * sc[i][e];
        }
        __syncthreads();
        for (int r = w; r < R; r += a.per) {
            float v = rp[r * 64 + lane];
            for (int o = 1; o < live; o++) v += rp[(o * R + r) * 64 + lane];
            const int m = 16 * (r >> 2) + 4 * q + (r & 3), n = tile * 16 + (lane & 15);
            if (m < a.M && n < p.N) {
                if (a.slices == 1) p.C[(int64_t)m * p.ldc + n] = v;
                else a.part[((int64_t)slice * a.M + m) * a.cols + p.col0 + n] = v;
            }
        }
    }
}

template <int MF>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_rows_kernel(Args a) {
    constexpr size_t kSums = 2 * kWaves * 4 * MF * 64 * sizeof(float), kStage = kWaves * sizeof(Stage);
    __shared__ __attribute__((aligned(16))) char red[kSums > kStage ? kSums : kStage];
    const int slice = blockIdx.x % a.slices, wg = blockIdx.x / a.slices;
    int i = 0;
    while (i + 1 < a.np && wg >= a.p[i + 1].wg0) i++;
    const Prob& p = a.p[i];
    switch (p.type) {
    case T_Q4_K: rows_body<T_Q4_K, MF>(a, p, slice, wg - p.wg0, red); break;
    case T_Q5_K: rows_body<T_Q5_K, MF>(a, p, slice, wg - p.wg0, red); break;
    case T_Q6_K: rows_body<T_Q6_K, MF>(a, p, slice, wg - p.wg0, red); break;
    case T_Q8_0: rows_body<T_Q8_0, MF>(a, p, slice, wg - p.wg0, red); break;
    case T_IQ4_NL: rows_body<T_IQ4_NL, MF>(a, p, slice, wg - p.wg0, red); break;
    default: rows_body<T_IQ4_XS, MF>(a, p, slice, wg - p.wg0, red); break;
    }
}

// C[m][n] = the slices' sums in slice order; workgroup (256 columns, row).
__global__ __launch_bounds__(256) void gemm_rows_reduce_kernel(Args a) {
    const int c = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (c >= a.cols) return;
    int i = 0;
    while (i + 1 < a.np && c >= a.p[i + 1].col0) i++;
    const float* src = a.part + (int64_t)m * a.cols + c;
    float v = src[0];
    for (int s = 1; s < a.slices; s++) v += src[(int64_t)s * a.M * a.cols];
    a.p[i].C[(int64_t)m * a.p[i].ldc + c - a.p[i].col0] = v;
}

int slices_of(int K) { return ((K + 255) / 256 + kWaves - 1) / kWaves; }

}  // namespace

size_t gemm_rows_ws_bytes(int K, int M, int64_t cols) {
    return slices_of(K) > 1 ? sizeof(float) * slices_of(K) * M * (size_t)cols : 0;
}

bool gemm_rows_eligible(int K, int M, const float* A, int lda) {
    return M >= 1 && M <= 32 && K % 32 == 0 && ((uintptr_t)A & 15u) == 0 && lda % 4 == 0;
}

hipError_t launch_gemm_rows(const GemmDesc* d, const uint32_t* types, int n, int K, const float* A, int lda, int M, void* ws,
                            hipStream_t s) {
    if (n < 1 || n > kProb || !gemm_rows_eligible(K, M, A, lda)) return hipErrorInvalidValue;
    const int cus = cu_count();
    Args a{};
    a.np = n;
    a.M = M;
    a.SB = (K + 255) / 256;
    a.nb = K / 32;
    a.lda = lda;
    a.A = A;
    a.part = (float*)ws;
    a.slices = slices_of(K);
    a.per = (a.SB + a.slices - 1) / a.slices;
    int64_t tiles = 0, cols = 0;
    for (int i = 0; i < n; i++) {
        tiles += (d[i].N + 15) / 16;
        cols += d[i].N;
    }
    a.cols = (int)cols;
    if (cols > INT32_MAX || (a.slices > 1 && !ws)) return hipErrorInvalidValue;
    // one workgroup of eight wavefronts fills a CU's registers; as many as
    // leave every workgroup the same number of tiles
    const int64_t cap = cus * (kWaves / a.per) / a.slices > 1 ? cus * (kWaves / a.per) / a.slices : 1;
    const int64_t rounds = (tiles + cap - 1) / cap;
    int wg = 0, col0 = 0;
    for (int i = 0; i < n; i++) {
        const int t = (d[i].N + 15) / 16, wgs = (int)((t + rounds - 1) / rounds);
        a.p[i] = Prob{(const uint8_t*)d[i].W, d[i].C, (uint32_t)row_bytes(types[i], K), types[i], d[i].N, d[i].ldc, col0, wg, wgs};
        wg += wgs;
        col0 += d[i].N;
    }
    if (M <= 16) gemm_rows_kernel<1><<<wg * a.slices, 64 * a.per, 0, s>>>(a);
    else gemm_rows_kernel<2><<<wg * a.slices, 64 * a.per, 0, s>>>(a);
    if (a.slices > 1) gemm_rows_reduce_kernel<<<dim3((a.cols + 255) / 256, M), 256, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace ggq
