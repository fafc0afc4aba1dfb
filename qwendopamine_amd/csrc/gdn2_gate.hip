// The decay gate activation and its VJP for the training path (gfx950).
//
// Forward (reference kda_gate_fwd, gdn2_ops/chunk_kda.py:3223-3251, kernel
// :3089-3148): per element of g [tokens, H, K]
//   x = g + dt_bias[h, c]
//   y = -exp(A_log[h]) * softplus(x)                     (default)
//   y = lower_bound * sigmoid(exp(A_log[h]) * x)         (GDN2_FLAG_LOWER_BOUND)
// in fp32, the same formula the chunk and token-serial kernels apply under
// GDN2_FLAG_GATE_IN_KERNEL (gate_activation in gdn2_common.h).  With
// GDN2_FLAG_LIBRARY_MATH the default form and its VJP take the library's expf and
// log1pf in the order of torch's float32 chain: y is that chain's bit for bit.
//
// Backward (reference kda_gate_bwd, chunk_kda.py:3254-3292, kernel
// :3151-3220): given dy = dL/dy,
//   dg       = dy * dy/dx       (-a sigmoid(x), or lower_bound a s (1 - s))
//   dA_log   = sum over tokens and channels of dy * dy/dA_log
//              (y itself, or dg * x for the bounded form)
//   ddt_bias = sum over tokens of dg
// One workgroup per (64-token block, head) writes its partial sums of dA_log
// and ddt_bias to a workspace; a second kernel adds the blocks in a fixed order,
// so the result does not depend on scheduling.
#include <hip/hip_runtime.h>

#include "gdn2_chunk.h"
#include "gdn2_internal.h"

namespace gdn2 {

namespace {

constexpr int kGateBT = 64;  // tokens per backward workgroup

struct GateParams {
    const void *g;
    const float *A_log, *dt_bias;
    float lower_bound;
    int use_lb;
    float *y;         // forward output (fp32)
    const float *dy;  // backward input (fp32)
    void *dg;         // backward output (g's dtype)
    float *part_a;    // [nblk, H] partial dA_log
    float *part_b;    // [nblk, H, K] partial ddt_bias (null without dt_bias)
    int64_t tokens;
    int H, K, vec_ok;
    int ql;           // backward: log2 of the lanes per row
};

// GDN2_FLAG_LIBRARY_MATH: softplus(x) and its VJP as torch forms them (threshold
// 20), from e = expf(x): log1p(e), and t e / (e + 1) for an upstream t.  For callers
// that held the decay in torch's float32 before; its rms error against float64 (4096
// tokens x 16 heads x 64 channels, raw gate N(0, 2) in bf16) is 1.2e-7 with these and
// 2.0e-7 with the hardware exp2 / log2 forms.  log1pf alone is about 130
// instructions, which then bound both passes: 28.3 us forward and 34.2 backward at
// 8192 tokens x 16 heads x 64 channels in bf16, 15.0 and 16.1 without.
__device__ __forceinline__ float softplus_of_exp(float x, float e) { return x > 20.0f ? x : log1pf(e); }

__device__ __forceinline__ float softplus_vjp(float x, float e, float t)
{
    return x > 20.0f ? t : t * e / (e + 1.0f);
}

// Channels 4q .. 4q+3 of row (token, h): one thread; K <= 256 (64 quads).
template <typename TG, bool LIB>
__global__ __launch_bounds__(256) void gate_fwd_kernel(GateParams p)
{
    const int64_t rows = p.tokens * p.H;
    const int quads = (p.K + 3) / 4;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t row = idx / quads;
    if (row >= rows) return;
    const int c0 = 4 * static_cast<int>(idx - row * quads);
    const int h = static_cast<int>(row % p.H);
    const int64_t off = row * p.K;
    float x[4], db[4] = {0.f, 0.f, 0.f, 0.f};
    load4(static_cast<const TG *>(p.g), off, c0, p.K, true, p.vec_ok, x);
    if (p.dt_bias) load4(p.dt_bias, static_cast<int64_t>(h) * p.K, c0, p.K, true, p.vec_ok, db);
    const float a_log = p.A_log[h];
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float xi = x[i] + db[i];
        y[i] = LIB ? -expf(a_log) * softplus_of_exp(xi, expf(xi))
                   : gate_activation(x[i], a_log, db[i], p.use_lb, p.lower_bound);
    }
    store4(p.y, off, c0, p.K, y);
}

// Workgroup (token block tb, head h): the QN = 2^ql lanes that cover a row's
// channel quads (K = 64: 16) times 256 / QN token lanes r; thread (r, q) takes
// channels 4q..4q+3 of tokens tb * 64 + r, r + 256 / QN, ..., kGateU of them
// requested at once.  Per-channel sums over its tokens, over the token lanes
// of a wave by shuffles, over the waves in LDS.  HBM-bound by its bytes (g, dy,
// dg: 8 a channel in bf16); with a fixed 64 lanes a row, three quarters of them idle at
// K = 64, and one row requested at a time it took 39.6 us at 8192 tokens x 16
// heads x 64 channels in bf16, now 16.1 (67 MB: 4.2 TB/s).
// VEC: K is a multiple of 4 and every row piece is aligned to its four values.
constexpr int kGateU = 4;
template <typename TG, bool VEC, bool LIB>
__global__ __launch_bounds__(256) void gate_bwd_kernel(GateParams p)
{
    __shared__ float s_b[4][256];
    __shared__ float s_a[4];
    const int tb = blockIdx.x / p.H, h = blockIdx.x % p.H;
    const int qn = 1 << p.ql, step = 256 >> p.ql;
    const int q = threadIdx.x & (qn - 1), r = threadIdx.x >> p.ql, wv = threadIdx.x >> 6;
    const bool live = 4 * q < p.K;
    const int c0 = live ? 4 * q : 0;
    const float a = expf(p.A_log[h]);
    float db[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.dt_bias) load4(p.dt_bias, static_cast<int64_t>(h) * p.K, c0, p.K, live, 0, db);
    float sb[4] = {0.f, 0.f, 0.f, 0.f}, sa = 0.f;
    const int64_t t_beg = static_cast<int64_t>(tb) * kGateBT;
    const int64_t t_end = p.tokens < t_beg + kGateBT ? p.tokens : t_beg + kGateBT;
    const TG *g = static_cast<const TG *>(p.g);
    using Raw = std::conditional_t<sizeof(TG) == 2, uint2, uint4>;
    for (int64_t t = t_beg + r; t < t_end; t += kGateU * step) {
        float x[kGateU][4], dy[kGateU][4];
        if constexpr (VEC) {
            // Rows past the block load its first row; their dy counts as zero.
            Raw xr[kGateU];
            float4 yr[kGateU];
#pragma unroll
            for (int u = 0; u < kGateU; ++u) {
                const int64_t tu = t + u * step < t_end ? t + u * step : t_beg;
                const int64_t off = (tu * p.H + h) * p.K + c0;
                xr[u] = *reinterpret_cast<const Raw *>(g + off);
                yr[u] = *reinterpret_cast<const float4 *>(p.dy + off);
            }
#pragma unroll
            for (int u = 0; u < kGateU; ++u) {
                const bool ok = live && t + u * step < t_end;
#pragma unroll
                for (int i = 0; i < 4; ++i) x[u][i] = io<TG>::ld(reinterpret_cast<const TG *>(&xr[u]), i);
                dy[u][0] = ok ? yr[u].x : 0.f;
                dy[u][1] = ok ? yr[u].y : 0.f;
                dy[u][2] = ok ? yr[u].z : 0.f;
                dy[u][3] = ok ? yr[u].w : 0.f;
            }
        } else {
#pragma unroll
            for (int u = 0; u < kGateU; ++u) {
                const bool ok = live && t + u * step < t_end;
                const int64_t off = ((ok ? t + u * step : t_beg) * p.H + h) * p.K;
                load4(g, off, c0, p.K, ok, 0, x[u]);
                load4(p.dy, off, c0, p.K, ok, 0, dy[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < kGateU; ++u) {
            if (!live || t + u * step >= t_end) continue;
            float dg[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float xi = x[u][i] + db[i];
                if constexpr (LIB) {
                    const float e = expf(xi);
                    dg[i] = softplus_vjp(xi, e, -a * dy[u][i]);
                    sa = fmaf(dy[u][i], -a * softplus_of_exp(xi, e), sa);
                } else if (p.use_lb) {
                    const float s = sigmoid_f(a * xi);
                    dg[i] = dy[u][i] * (p.lower_bound * s * (1.0f - s)) * a;
                    sa = fmaf(dg[i], xi, sa);
                } else {
                    dg[i] = -a * dy[u][i] * sigmoid_f(xi);
                    sa = fmaf(dy[u][i], -a * softplus_f(xi), sa);
                }
                sb[i] += dg[i];
            }
            // Rounded to g's dtype.
            store4(static_cast<TG *>(p.dg), ((t + u * step) * p.H + h) * p.K, c0, p.K, dg);
        }
    }
    // Channels beyond K were never loaded (zero sums).
    sa = wave_sum(sa);
    if ((threadIdx.x & 63) == 0) s_a[wv] = sa;
    for (int off = qn; off < kWave; off <<= 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sb[i] += __shfl_xor(sb[i], off, kWave);
    }
    if ((threadIdx.x & 63) < qn) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s_b[wv][4 * q + i] = sb[i];  // 4 q + 3 <= 255
    }
    __syncthreads();
    const int64_t blk = tb;
    if (threadIdx.x == 0) p.part_a[blk * p.H + h] = (s_a[0] + s_a[1]) + (s_a[2] + s_a[3]);
    if (p.part_b) {
        for (int c = threadIdx.x; c < p.K; c += 256)
            p.part_b[(blk * p.H + h) * p.K + c] = (s_b[0][c] + s_b[1][c]) + (s_b[2][c] + s_b[3][c]);
    }
}

// dA_log[h] and ddt_bias[h, c]: the blocks' partial sums in a fixed order, 64
// elements a workgroup (the first nba workgroups take dA_log).  One thread a sum
// over 128 blocks took 61.3 us at 16 heads x 64 channels, now 3.8.
__global__ __launch_bounds__(1024) void gate_bwd_sum_kernel(GateParams p, int nblk, int nba, float *dA_log,
                                                            float *ddt_bias)
{
    __shared__ float s_sum[16][64];
    const bool is_a = static_cast<int>(blockIdx.x) < nba;
    const int64_t E = is_a ? p.H : static_cast<int64_t>(p.H) * p.K;
    const int64_t e = static_cast<int64_t>(blockIdx.x - (is_a ? 0 : nba)) * 64 + (threadIdx.x & 63);
    const float s = sum_parts<16, 8>(is_a ? p.part_a : p.part_b, nblk, E, e < E ? e : E - 1, s_sum);
    if (threadIdx.x < 64 && e < E) (is_a ? dA_log : ddt_bias)[e] = s;
}

int64_t gate_blocks(int64_t tokens) { return (tokens + kGateBT - 1) / kGateBT; }

}  // namespace

size_t gate_bwd_workspace_bytes(int64_t tokens, int H, int K, bool has_bias)
{
    const int64_t nblk = gate_blocks(tokens);
    const int64_t a = round_up(nblk * H * 4, 256);
    return static_cast<size_t>(a + (has_bias ? round_up(nblk * H * static_cast<int64_t>(K) * 4, 256) : 0));
}

int launch_gate_fwd(const void *g, int g_dtype, const float *A_log, const float *dt_bias, float lower_bound,
                    unsigned flags, float *y, int64_t tokens, int H, int K, hipStream_t stream)
{
    GateParams p{};
    p.g = g;
    p.A_log = A_log;
    p.dt_bias = dt_bias;
    p.lower_bound = lower_bound;
    p.use_lb = (flags & GDN2_FLAG_LOWER_BOUND) != 0;
    p.y = y;
    p.tokens = tokens;
    p.H = H;
    p.K = K;
    p.vec_ok = (K % 4) == 0;
    const int64_t threads = tokens * H * ((K + 3) / 4);
    if (threads == 0) return GDN2_OK;
    const dim3 grid(static_cast<unsigned>((threads + 255) / 256));
    const auto go = [&](auto tag) {
        using TG = decltype(tag);
        if (flags & GDN2_FLAG_LIBRARY_MATH)
            hipLaunchKernelGGL((gate_fwd_kernel<TG, true>), grid, dim3(256), 0, stream, p);
        else
            hipLaunchKernelGGL((gate_fwd_kernel<TG, false>), grid, dim3(256), 0, stream, p);
    };
    switch (g_dtype) {
    case GDN2_DTYPE_F32: go(float{}); break;
    case GDN2_DTYPE_BF16: go(bf16_t{}); break;
    default: go(f16_t{}); break;
    }
    return hipGetLastError() == hipSuccess ? GDN2_OK : GDN2_ERR_LAUNCH;
}

int launch_gate_bwd(const void *g, int g_dtype, const float *A_log, const float *dt_bias, float lower_bound,
                    unsigned flags, const float *dy, void *dg, float *dA_log, float *ddt_bias, int64_t tokens,
                    int H, int K, void *workspace, hipStream_t stream)
{
    GateParams p{};
    p.g = g;
    p.A_log = A_log;
    p.dt_bias = dt_bias;
    p.lower_bound = lower_bound;
    p.use_lb = (flags & GDN2_FLAG_LOWER_BOUND) != 0;
    p.dy = dy;
    p.dg = dg;
    p.tokens = tokens;
    p.H = H;
    p.K = K;
    p.vec_ok = (K % 4) == 0;
    while ((4 << p.ql) < K) ++p.ql;  // K <= 256: at most 64 lanes
    const int64_t nblk = gate_blocks(tokens);
    p.part_a = static_cast<float *>(workspace);
    p.part_b = dt_bias ? reinterpret_cast<float *>(static_cast<unsigned char *>(workspace) +
                                                   round_up(nblk * H * 4, 256))
                       : nullptr;
    if (nblk > 0) {
        const dim3 grid(static_cast<unsigned>(nblk * H));
        const auto go = [&](auto tag) {
            using TG = decltype(tag);
            const uintptr_t odd = (reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(dg)) % (4 * sizeof(TG)) |
                                  reinterpret_cast<uintptr_t>(dy) % 16;
            const bool vec = p.vec_ok && odd == 0, lib = (flags & GDN2_FLAG_LIBRARY_MATH) != 0;
            if (vec && lib)
                hipLaunchKernelGGL((gate_bwd_kernel<TG, true, true>), grid, dim3(256), 0, stream, p);
            else if (vec)
                hipLaunchKernelGGL((gate_bwd_kernel<TG, true, false>), grid, dim3(256), 0, stream, p);
            else if (lib)
                hipLaunchKernelGGL((gate_bwd_kernel<TG, false, true>), grid, dim3(256), 0, stream, p);
            else
                hipLaunchKernelGGL((gate_bwd_kernel<TG, false, false>), grid, dim3(256), 0, stream, p);
        };
        switch (g_dtype) {
        case GDN2_DTYPE_F32: go(float{}); break;
        case GDN2_DTYPE_BF16: go(bf16_t{}); break;
        default: go(f16_t{}); break;
        }
        if (hipGetLastError() != hipSuccess) return GDN2_ERR_LAUNCH;
    }
    const int nba = (H + 63) / 64;
    const int64_t nbb = dt_bias ? (static_cast<int64_t>(H) * K + 63) / 64 : 0;
    hipLaunchKernelGGL(gate_bwd_sum_kernel, dim3(static_cast<unsigned>(nba + nbb)), dim3(1024), 0, stream, p,
                       static_cast<int>(nblk), nba, dA_log, ddt_bias);
    return hipGetLastError() == hipSuccess ? GDN2_OK : GDN2_ERR_LAUNCH;
}

}  // namespace gdn2
