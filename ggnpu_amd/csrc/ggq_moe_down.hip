// ggq_moe_down.hip -- one-launch tail of a MoE layer of few tokens (gfx950).
//
// A translation unit, and so a code object, of its own: among the other
// kernels its 24 variants shift where those lie in their code object, and the
// six launches of a fused decode layer (the same instructions; H = 2048, F =
// 8192, 6000 positions) took 41.9 us against 40.8.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ggq_device.h"
#include "ggq_launch.h"

namespace ggq {

// The rest of a layer behind gate and up for few tokens: SwiGLU, the routed
// and the shared expert's down projection and the weighted sum, in one launch.
// A workgroup takes kDownCols columns of a token, a wavefront an expert of its
// selection (then the shared expert): it makes the SwiGLU row from G and U in
// registers, a piece of 32 values a lane, and its column sums meet in LDS,
// where they are added in the order of moe_combine_kernel.  A token's layer is
// latency: four launches (SwiGLU 2.3, the grouped GEMV over a grid of every
// expert 11.4, the shared expert's 3.8, combine 3 us and the gaps) become one
// (256 experts, top 8, F = 512, Q4_K / Q6_K: the layer 38.4 -> 25.2 us).
// The SwiGLU row is the larger part of the arithmetic (an exponential and a
// division a value): where the 64 lanes hold several columns (S: F <= 1024) each
// makes its share of the row once and they exchange it through LDS (the layer
// 28.5 us with every lane making its own 32 values).
constexpr int kDownCols = 8;
__device__ __forceinline__ float4 swiglu4(float4 g, float4 u) {
    return make_float4((g.x / (1.0f + expf(-g.x))) * u.x, (g.y / (1.0f + expf(-g.y))) * u.y,
                       (g.z / (1.0f + expf(-g.z))) * u.z, (g.w / (1.0f + expf(-g.w))) * u.w);
}
template <int T, int U, bool S>
__global__ __launch_bounds__(1024) void moe_down_kernel(MoeDown a) {
    __shared__ float part[65][kDownCols];
    extern __shared__ float4 hrow[];  // [wavefronts][F], with S
    const int t = blockIdx.y, n0 = blockIdx.x * kDownCols;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int lg = a.lpr_log2, lp = lane & ((1 << lg) - 1), rsub = lane >> lg, rpi = 64 >> lg;
    const int P = a.F >> 5, pairs = a.topk + (a.Dsh ? 1 : 0);
    const bool ok = lp < P;
    const int p = ok ? lp : 0;
    pick_out(a.pick, a.wsel, t, a.topk);
    for (int j = wave; j < pairs; j += waves) {
        const uint8_t* W = a.Wsh;
        int64_t pair = (int64_t)a.T * a.topk + t;
        float* d = a.Dsh + (int64_t)t * a.H;
        if (j < a.topk) {
            W = a.W + expert_id(a.pick.sel[t * a.topk + j], a.E) * a.w_stride;
            pair = a.pos[t * a.topk + j];
            d = a.D + pair * a.H;
        }
        auto row = [&](int it) {
            const int n = n0 + it * rpi + rsub;
            return make_row(W, (uint32_t)(n < a.H ? n : a.H - 1) * a.row_bytes);
        };
        typename Piece<T>::Raw raw[U];
#pragma unroll
        for (int u = 0; u < U; u++) raw[u] = Piece<T>::fetch(row(u), p);
        float x[32], xs[2];
        float4* const hw = hrow + wave * (a.F >> 2);
        if constexpr (S) {
            float4 g[4], u[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int q = lane + 64 * c < a.F >> 2 ? lane + 64 * c : 0;
                g[c] = *((const float4*)(a.G + pair * a.F) + q);
                u[c] = *((const float4*)(a.U + pair * a.F) + q);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int q = lane + 64 * c;
                if (q >= a.F >> 2) break;
                const float4 h = swiglu4(g[c], u[c]);
                hw[q] = h;
                if (n0 == 0) *((float4*)(a.Hh + pair * a.F) + q) = h;
            }
            // the wavefront's own row: LDS serves it in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int k = Piece<T>::run_k(p, r);
            const int64_t at = pair * a.F + k;
            float4 h[4];
            if constexpr (S) {
#pragma unroll
                for (int c = 0; c < 4; c++) h[c] = hw[(k >> 2) + c];
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) h[c] = swiglu4(*(const float4*)(a.G + at + 4 * c), *(const float4*)(a.U + at + 4 * c));
            }
            xs[r] = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (!S && n0 == 0 && ok) *(float4*)(a.Hh + at + 4 * c) = h[c];
                x[16 * r + 4 * c] = ok ? h[c].x : 0.0f;
                x[16 * r + 4 * c + 1] = ok ? h[c].y : 0.0f;
                x[16 * r + 4 * c + 2] = ok ? h[c].z : 0.0f;
                x[16 * r + 4 * c + 3] = ok ? h[c].w : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 16; i++) xs[r] += x[16 * r + i];
        }
        if constexpr (S) {  // read before the next pair's row is written
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        for (int it = 0; it * rpi < kDownCols; it += U) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const PieceCodes pc = Piece<T>::decode(raw[u], row(it + u), p);
                float v = 0.0f;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    float f[16], s0 = 0.0f, s1 = 0.0f;
                    ubytes_to_f32(pc.u[r], f);
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        s0 = fmaf(x[16 * r + i], f[i], s0);
                        s1 = fmaf(x[16 * r + i + 1], f[i + 1], s1);
                    }
                    v = fmaf(pc.a[r], s0 + s1, fmaf(pc.b[r], xs[r], v));
                }
                v = group_sum(v, lg);
                const int c = (it + u) * rpi + rsub;
                if (lp == 0) {
                    part[j][c] = v;
                    if (n0 + c < a.H) d[n0 + c] = v;
                }
                if ((it + U) * rpi < kDownCols) raw[u] = Piece<T>::fetch(row(it + U + u), p);
            }
        }
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= kDownCols || n0 + c >= a.H) return;
    float acc = 0.0f;
    for (int j = 0; j < a.topk; j++) acc += a.wsel[t * a.topk + j] * part[j][c];
    if (a.Dsh) acc += (a.shared_w ? a.shared_w[t] : 1.0f) * part[a.topk][c];
    a.out[(int64_t)t * a.H + n0 + c] = acc;
}

bool moe_down_eligible(uint32_t type, int F, int topk) { return supported(type) && F % 32 == 0 && F <= 2048 && topk <= 64; }

hipError_t launch_moe_down(uint32_t type, MoeDown a, hipStream_t s) {
    if (!moe_down_eligible(type, a.F, a.topk) || a.T < 1) return hipErrorInvalidValue;
    a.row_bytes = (uint32_t)row_bytes(type, a.F);
    a.lpr_log2 = 3;
    while (1 << a.lpr_log2 < a.F / 32) a.lpr_log2++;
    const int pairs = a.topk + (a.Dsh ? 1 : 0), its = kDownCols >> (6 - a.lpr_log2);
    const int most = a.F <= 512 ? 16 : 12, waves = pairs < most ? pairs : most;  // rows in at most 48 KB of LDS
    const dim3 grid((a.H + kDownCols - 1) / kDownCols, a.T), block(64 * waves);
    const size_t lds = its <= 4 ? sizeof(float) * waves * a.F : 0;
#define GO(TT)                                                                    \
    case TT:                                                                      \
        if (its == 1) moe_down_kernel<TT, 1, true><<<grid, block, lds, s>>>(a);   \
        else if (its == 2) moe_down_kernel<TT, 2, true><<<grid, block, lds, s>>>(a); \
        else if (its == 4) moe_down_kernel<TT, 4, true><<<grid, block, lds, s>>>(a); \
        else moe_down_kernel<TT, 4, false><<<grid, block, 0, s>>>(a);             \
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
