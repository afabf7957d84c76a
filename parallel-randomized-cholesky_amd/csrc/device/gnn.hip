// gnn.hip -- forward and backward kernels of the ordering network.
//
// Network (no counterpart in the reference; the reference orders offline with
// Julia heuristics, write_graph.jl:46-78): node inputs x_v = (log degree,
// log weighted degree), centred per graph; three message-passing layers
//   M_l = Anorm H_{l-1}          (Anorm[v,u] = w_vu / wdeg_v)
//   Z_l = H_{l-1} Ws_l^T + M_l Wn_l^T + b_l,   H_l = relu(Z_l)
// with hidden width 64, and a linear score s_v = H_3 wo + bo.  Weights and
// layer inputs are rounded to bfloat16, products accumulate in FP32; the
// 128 -> 64 transforms of layers 2 and 3 run on MFMA (v_mfma_f32_16x16x16
// bf16), one wave per 16 rows.  The backward pass runs in FP32 on the
// bf16-rounded operands of the forward pass (straight-through for the
// rounding); weight gradients reduce over rows with fixed per-block partials,
// so gradients are deterministic.
#include <hip/hip_bf16.h>

#include <type_traits>

#include "common.cuh"
#include "kernels.h"

namespace rc {

namespace {

constexpr int kH = kGnnHidden;   // 64

__device__ __forceinline__ float bf16r(float x)
{   // round to nearest even bfloat16, returned as float
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7F800000u) == 0x7F800000u) return x;           // inf / nan unchanged
    uint32_t lsb = (u >> 16) & 1u;
    u += 0x7FFFu + lsb;
    return __uint_as_float(u & 0xFFFF0000u);
}

__device__ __forceinline__ unsigned short bf16bits(float x) { return (unsigned short)(__float_as_uint(bf16r(x)) >> 16); }

// ---------------------------------------------------------------- aggregation
// M[v, :] = sum_u a[v,u] H[u, :] (kAdd = false) or the transposed aggregation of
// the backward pass, M[u, :] += sum_{v in N(u)} a[v,u] H[v, :] with a[v,u] =
// w / wdeg_v stored at the (u -> v) entry.  Sixteen lanes per row, four features
// each; the row's entries eight at a time (indices, then the gathers, all in
// flight), summed in entry order.  Bound by the gathered rows; one wave per row
// with one entry in flight took 33 us at 64k rows, this 15 us.
template <bool kAdd>
__global__ void __launch_bounds__(256) k_agg64(int n, const int *ptr, const int *ind, const float *a, const float *H,
                                               float *M)
{
    constexpr int B = 8;
    const int c = (threadIdx.x & 15) * 4;
    for (int v = blockIdx.x * 16 + threadIdx.x / 16; v < n; v += gridDim.x * 16) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        if (kAdd) acc = *reinterpret_cast<const float4 *>(M + (size_t)v * kH + c);
        const int e1 = ptr[v + 1];
        for (int e = ptr[v]; e < e1; e += B) {
            int j[B];
            float w[B];
            float4 h[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int ee = e + u < e1 ? e + u : e1 - 1;
                j[u] = ind[ee];
                w[u] = a[ee];
            }
#pragma unroll
            for (int u = 0; u < B; ++u) h[u] = *reinterpret_cast<const float4 *>(H + (size_t)j[u] * kH + c);
#pragma unroll
            for (int u = 0; u < B; ++u)
                if (e + u < e1) {
                    acc.x = fmaf(w[u], h[u].x, acc.x);
                    acc.y = fmaf(w[u], h[u].y, acc.y);
                    acc.z = fmaf(w[u], h[u].z, acc.z);
                    acc.w = fmaf(w[u], h[u].w, acc.w);
                }
        }
        *reinterpret_cast<float4 *>(M + (size_t)v * kH + c) = acc;
    }
}

__global__ void k_agg2(int n, const int *ptr, const int *ind, const float *a, const float *H, float *M)
{
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        float a0 = 0.f, a1 = 0.f;
        for (int e = ptr[v]; e < ptr[v + 1]; ++e) {
            a0 = fmaf(a[e], H[(size_t)ind[e] * 2], a0);
            a1 = fmaf(a[e], H[(size_t)ind[e] * 2 + 1], a1);
        }
        M[(size_t)v * 2] = a0;
        M[(size_t)v * 2 + 1] = a1;
    }
}

// ---------------------------------------------------------------- layer 1 (2 -> 64)
__global__ void k_dense1(int n, const float *H0, const float *M1, const float *w, float *H)
{
    const float *Ws = w + kGnnWs1, *Wn = w + kGnnWn1, *b = w + kGnnB1;
    const int lane = lane_id();
    const float ws0 = bf16r(Ws[lane * 2]), ws1 = bf16r(Ws[lane * 2 + 1]);
    const float wn0 = bf16r(Wn[lane * 2]), wn1 = bf16r(Wn[lane * 2 + 1]);
    const float bb = b[lane];
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int nwaves = gridDim.x * blockDim.x / kWave;
    for (int v = wave; v < n; v += nwaves) {
        float h0 = bf16r(H0[(size_t)v * 2]), h1 = bf16r(H0[(size_t)v * 2 + 1]);
        float m0 = bf16r(M1[(size_t)v * 2]), m1 = bf16r(M1[(size_t)v * 2 + 1]);
        float z = bb;
        z = fmaf(ws0, h0, z);
        z = fmaf(ws1, h1, z);
        z = fmaf(wn0, m0, z);
        z = fmaf(wn1, m1, z);
        H[(size_t)v * kH + lane] = z > 0.f ? z : 0.f;
    }
}

// ---------------------------------------------------------------- layers 2, 3 (128 -> 64) on MFMA
// Z = [H | M] W^T + b with W = [Ws | Wn] (64 x 128) in bf16.  One wave per 16
// rows: 4 output tiles of 16 x 16, K = 128 in 8 steps of 16.
// v_mfma_f32_16x16x16_bf16 operand layout (per lane l): A holds row l % 16,
// k = 4 (l / 16) .. +3; B holds column l % 16, same k; D holds rows
// 4 (l / 16) .. +3 of column l % 16.
// All of W stays in the wave's registers (64 x 128 bf16 are 64 per lane); a lane
// loads its row 16 bytes at a time.  (Through LDS, 16 lanes met in one bank and
// every workgroup converted W for 64 rows: 50 us at 64k rows, now 16.)
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x4 to_bf16x4(float4 v)
{
    bf16x4 r;
    r[0] = (short)bf16bits(v.x);
    r[1] = (short)bf16bits(v.y);
    r[2] = (short)bf16bits(v.z);
    r[3] = (short)bf16bits(v.w);
    return r;
}

__global__ void __launch_bounds__(256) k_dense_mfma(int n, const float *Hin, const float *Min, const float *Ws,
                                                    const float *Wn, const float *b, float *Hout)
{
    const int lane = lane_id();
    const int r16 = lane % 16, kq = lane / 16;
    bf16x4 wv[8][4];
    float bias[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int col = c * 16 + r16;
        bias[c] = b[col];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const float *W = ks < 4 ? Ws : Wn;
            wv[ks][c] = to_bf16x4(*reinterpret_cast<const float4 *>(W + col * kH + (ks & 3) * 16 + kq * 4));
        }
    }
    const int ntiles = (n + 15) / 16;
    for (int tile = blockIdx.x * 4 + threadIdx.x / kWave; tile < ntiles; tile += gridDim.x * 4) {
        const int row = min(tile * 16 + r16, n - 1);          // rows past the end are not written
        float4 x[8];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
            x[ks] = *reinterpret_cast<const float4 *>((ks < 4 ? Hin : Min) + (size_t)row * kH + (ks & 3) * 16 + kq * 4);
        f32x4 acc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const bf16x4 av = to_bf16x4(x[ks]);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, wv[ks][c], acc[c], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int rr = tile * 16 + kq * 4 + t;
                const float z = acc[c][t] + bias[c];
                if (rr < n) Hout[(size_t)rr * kH + c * 16 + r16] = z > 0.f ? z : 0.f;
            }
    }
}

// ---------------------------------------------------------------- output
__global__ void k_score(int n, const float *H3, const float *w, float *s)
{
    const float *wo = w + kGnnWo;
    const float bo = w[kGnnBo];
    const int lane = lane_id();
    const float wl = bf16r(wo[lane]);
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int nwaves = gridDim.x * blockDim.x / kWave;
    for (int v = wave; v < n; v += nwaves) {
        float p = wl * bf16r(H3[(size_t)v * kH + lane]);
        for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off, kWave);
        if (lane == 0) s[v] = p + bo;
    }
}

// ---------------------------------------------------------------- backward
// dZ = dH where H > 0 (H = relu(Z)); at the output layer dH[v][o] = ds[v] wo[o]
// is formed on the fly.  Four consecutive features c..c+3 of row v.
template <bool kLast>
__device__ __forceinline__ void load_dz(int v, int c, const float *dH, const float *H, const float *ds,
                                        const float *wl, float *dz, float *h)
{
    const float4 hv = *reinterpret_cast<const float4 *>(H + (size_t)v * kH + c);
    h[0] = hv.x; h[1] = hv.y; h[2] = hv.z; h[3] = hv.w;
    if (kLast) {
        const float d = ds[v];
#pragma unroll
        for (int t = 0; t < 4; ++t) dz[t] = d * wl[t];
    } else {
        const float4 g = *reinterpret_cast<const float4 *>(dH + (size_t)v * kH + c);
        dz[0] = g.x; dz[1] = g.y; dz[2] = g.z; dz[3] = g.w;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) dz[t] = h[t] > 0.f ? dz[t] : 0.f;
}

// Weight-gradient partials of a 64-wide layer over this workgroup's rows:
// gWs[o][i] = sum_v dZ[v][o] bf16(X[v][i]), gWn likewise with M, gb[o] = sum_v
// dZ[v][o]; at the output layer also gwo[o] = sum_v ds[v] bf16(H[v][o]) and gbo =
// sum_v ds[v].  Products on v_mfma_f32_16x16x4_f32 (FP32 in and accumulated),
// four rows a step: lane l holds features 4 (l % 16) .. +3 of row l / 16, so
// tile t of an operand is made of the features 4 j + t.  A wave keeps all 64 x
// 128 sums; the workgroup's waves are added through LDS in order.  (One thread
// per output row and 250 rows one after the other took 567 us at 64k rows, this
// 25 us.)  The products add 0 times the input where dZ is zero, NaN where that
// input is not finite: k_sum_partials mends it.
// Layout of a partial: [Ws | Wn | b | wo | bo], as in the weights.
constexpr int kWgLen = 2 * kH * kH + kH + kH + 1;
template <bool kLast>
__global__ void __launch_bounds__(256) k_wgrad64(int n, int rows_per_wave, const float *dH, const float *H,
                                                 const float *ds, const float *wo, const float *X, const float *M,
                                                 float *part)
{
    __shared__ float red[2 * kH * kH];
    __shared__ float redb[4][2 * kH + 1];
    const int lane = lane_id(), w = threadIdx.x / kWave;
    const int c = (lane & 15) * 4, vq = lane >> 4;
    float wl[4] = {0.f, 0.f, 0.f, 0.f};
    if (kLast)
#pragma unroll
        for (int t = 0; t < 4; ++t) wl[t] = bf16r(wo[c + t]);
    f32x4 ax[4][4], am[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) ax[i][j] = am[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float gb[4] = {0.f, 0.f, 0.f, 0.f}, gwo[4] = {0.f, 0.f, 0.f, 0.f}, gbo = 0.f;
    const int v0 = min((blockIdx.x * 4 + w) * rows_per_wave, n);
    const int v1 = min(v0 + rows_per_wave, n);
    constexpr int U = 2;
    for (int vb = v0; vb < v1; vb += 4 * U) {
        float dz[U][4], h[U][4];
        float4 x[U], m[U];
        float d[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = min(vb + 4 * u + vq, v1 - 1);
            load_dz<kLast>(v, c, dH, H, ds, wl, dz[u], h[u]);
            x[u] = *reinterpret_cast<const float4 *>(X + (size_t)v * kH + c);
            m[u] = *reinterpret_cast<const float4 *>(M + (size_t)v * kH + c);
            d[u] = kLast ? ds[v] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = vb + 4 * u + vq < v1;
            const float xv[4] = {bf16r(x[u].x), bf16r(x[u].y), bf16r(x[u].z), bf16r(x[u].w)};
            const float mv[4] = {bf16r(m[u].x), bf16r(m[u].y), bf16r(m[u].z), bf16r(m[u].w)};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                dz[u][t] = in ? dz[u][t] : 0.f;
                gb[t] += dz[u][t];
                if (kLast && in) gwo[t] = fmaf(d[u], bf16r(h[u][t]), gwo[t]);
            }
            if (kLast && in) gbo += d[u];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ax[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(dz[u][i], xv[j], ax[i][j], 0, 0, 0);
                    am[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(dz[u][i], mv[j], am[i][j], 0, 0, 0);
                }
        }
    }
    // the four rows of a step sit in the lane groups of 16
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int off = 16; off < kWave; off <<= 1) {
            gb[t] += __shfl_xor(gb[t], off, kWave);
            gwo[t] += __shfl_xor(gwo[t], off, kWave);
        }
    gbo += __shfl_xor(gbo, 16, kWave);
    gbo += __shfl_xor(gbo, 32, kWave);
    if (lane < 16)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            redb[w][c + t] = gb[t];
            redb[w][kH + c + t] = gwo[t];
        }
    if (lane == 0) redb[w][2 * kH] = gbo;
    for (int s = 0; s < 4; ++s) {
        if (w == s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int o = 4 * (4 * vq + q) + i, col = c + j;     // row 4 (l / 16) + q of tile i
                        float &rx = red[o * kH + col], &rm = red[kH * kH + o * kH + col];
                        rx = s == 0 ? ax[i][j][q] : rx + ax[i][j][q];
                        rm = s == 0 ? am[i][j][q] : rm + am[i][j][q];
                    }
        __syncthreads();
    }
    float *p = part + (size_t)blockIdx.x * kWgLen;
    for (int i = threadIdx.x; i < 2 * kH * kH; i += 256) p[i] = red[i];
    if (threadIdx.x < 2 * kH + 1)
        p[2 * kH * kH + threadIdx.x] = ((redb[0][threadIdx.x] + redb[1][threadIdx.x]) + redb[2][threadIdx.x]) +
                                       redb[3][threadIdx.x];
}

// The same for the first layer (two inputs): lane = output, four rows in
// flight per wave.
constexpr int kWgLen2 = 2 * kH * 2 + kH;
__global__ void __launch_bounds__(256) k_wgrad2(int n, int rows_per_wave, const float *dH, const float *H,
                                                const float *X, const float *M, float *part)
{
    __shared__ float red[4][5][kWave];
    const int lane = lane_id(), w = threadIdx.x / kWave;
    float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    const int v0 = min((blockIdx.x * 4 + w) * rows_per_wave, n);
    const int v1 = min(v0 + rows_per_wave, n);
    constexpr int U = 8;
    for (int vb = v0; vb < v1; vb += U) {
        float d[U];
        float2 x[U], m[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = min(vb + u, v1 - 1);
            d[u] = H[(size_t)v * kH + lane] > 0.f ? dH[(size_t)v * kH + lane] : 0.f;
            x[u] = *reinterpret_cast<const float2 *>(X + (size_t)v * 2);
            m[u] = *reinterpret_cast<const float2 *>(M + (size_t)v * 2);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float dv = vb + u < v1 ? d[u] : 0.f;
            g[0] = fmaf(dv, bf16r(x[u].x), g[0]);
            g[1] = fmaf(dv, bf16r(x[u].y), g[1]);
            g[2] = fmaf(dv, bf16r(m[u].x), g[2]);
            g[3] = fmaf(dv, bf16r(m[u].y), g[3]);
            g[4] += dv;
        }
    }
    // 0 times an infinity is NaN: sums that are not finite are formed again, zeros
    // skipped (selecting in the loop took 6 us)
    if (!__builtin_isfinite(g[0]) || !__builtin_isfinite(g[1]) || !__builtin_isfinite(g[2]) || !__builtin_isfinite(g[3])) {
        g[0] = g[1] = g[2] = g[3] = 0.f;
        for (int v = v0; v < v1; ++v) {
            const float d = H[(size_t)v * kH + lane] > 0.f ? dH[(size_t)v * kH + lane] : 0.f;
            if (d == 0.f) continue;
            g[0] = fmaf(d, bf16r(X[(size_t)v * 2]), g[0]);
            g[1] = fmaf(d, bf16r(X[(size_t)v * 2 + 1]), g[1]);
            g[2] = fmaf(d, bf16r(M[(size_t)v * 2]), g[2]);
            g[3] = fmaf(d, bf16r(M[(size_t)v * 2 + 1]), g[3]);
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) red[w][i][lane] = g[i];
    __syncthreads();
    if (w != 0) return;
    float *p = part + (size_t)blockIdx.x * kWgLen2;
#pragma unroll
    for (int i = 0; i < 5; ++i) g[i] = ((red[0][i][lane] + red[1][i][lane]) + red[2][i][lane]) + red[3][i][lane];
    p[lane * 2] = g[0];
    p[lane * 2 + 1] = g[1];
    p[2 * kH + lane * 2] = g[2];
    p[2 * kH + lane * 2 + 1] = g[3];
    p[4 * kH + lane] = g[4];
}

// What the weight gradients of a 64-wide layer were formed from.
struct WgradRows {
    int n;
    const float *dH, *H, *ds, *wo, *X, *M;
};

// Sum of nblocks partials into out[0..len), eight threads per output, each over
// its share of the partials in order, then the eight in order.  A row whose dZ
// is zero contributes nothing, whatever its inputs hold: a weight's sum that is
// not finite is formed again from the rows, zeros skipped.  (Watching for such
// inputs in k_wgrad64 cost it its registers: 321 -> 331-350 us a gradient.)
template <bool kLast>
__global__ void __launch_bounds__(256) k_sum_partials(const float *part, int nblocks, int stride, int len, WgradRows w,
                                                      float *out)
{
    __shared__ float red[8][32];
    const int o = threadIdx.x & 31, s = threadIdx.x >> 5;
    const int i = blockIdx.x * 32 + o;
    const int per = (nblocks + 7) / 8;
    const int b0 = s * per, b1 = min(nblocks, b0 + per);
    float t = 0.f;
    if (i < len)
        for (int b = b0; b < b1; b += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = b + u < b1 ? part[(size_t)(b + u) * stride + i] : 0.f;
#pragma unroll
            for (int u = 0; u < 8; ++u) t += v[u];
        }
    red[s][o] = t;
    __syncthreads();
    if (threadIdx.x >= kWave) return;
    t = red[0][o];
    for (int q = 1; q < 8; ++q) t += red[q][o];
    const bool again = w.H && i < 2 * kH * kH && !__builtin_isfinite(t);
    if (ballot(again)) {                                 // the wave's halves take half of the rows each
        float r = 0.f;
        if (again) {
            const float *in = i < kH * kH ? w.X : w.M;
            const int row = (i / kH) % kH, col = i % kH;
            const float wl = kLast ? bf16r(w.wo[row]) : 0.f;
            const int half = w.n / 2, v1 = s == 0 ? half : w.n;
#pragma unroll 4
            for (int v = s == 0 ? 0 : half; v < v1; ++v) {
                const float g = kLast ? w.ds[v] * wl : w.dH[(size_t)v * kH + row];
                if (w.H[(size_t)v * kH + row] > 0.f && g != 0.f) r = fmaf(g, bf16r(in[(size_t)v * kH + col]), r);
            }
        }
        r += __shfl_xor(r, 32, kWave);
        if (again) t = r;
    }
    if (s == 0 && i < len) out[i] = t;
}

// dX[v][i] = sum_o dZ[v][o] bf16(Ws[o][i]);  G[v][i] = sum_o dZ[v][o] bf16(Wn[o][i]):
// 16 rows x 128 outputs per wave on v_mfma_f32_16x16x4_f32 with both weight
// matrices in registers (128 per lane): 20 us at 64k rows (one row per wave with
// 64 broadcasts, 98).
template <bool kLast>
__global__ void __launch_bounds__(256) k_back_dense(int n, const float *dH, const float *H, const float *ds,
                                                    const float *wo, const float *Ws, const float *Wn, float *dX,
                                                    float *G)
{
    const int lane = lane_id();
    const int r16 = lane % 16, kq = lane / 16;
    float wv[4][4][8];           // [k block][k in block][column tile]: W[16 b + 4 kq + j][16 c + r16]
    float wl[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int o = 16 * b + 4 * kq + j;
            wl[b][j] = kLast ? bf16r(wo[o]) : 0.f;
#pragma unroll
            for (int c = 0; c < 8; ++c) wv[b][j][c] = bf16r((c < 4 ? Ws : Wn)[o * kH + (c & 3) * 16 + r16]);
        }
    const int ntiles = (n + 15) / 16;
    for (int tile = blockIdx.x * 4 + threadIdx.x / kWave; tile < ntiles; tile += gridDim.x * 4) {
        const int row = min(tile * 16 + r16, n - 1);
        float dz[4][4], h[4][4];
#pragma unroll
        for (int b = 0; b < 4; ++b) load_dz<kLast>(row, 16 * b + 4 * kq, dH, H, ds, wl[b], dz[b], h[b]);
        f32x4 acc[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(dz[b][j], wv[b][j][c], acc[c], 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int rr = tile * 16 + kq * 4 + t;
                if (rr < n) (c < 4 ? dX : G)[(size_t)rr * kH + (c & 3) * 16 + r16] = acc[c][t];
            }
    }
}

int grid_for_waves(int n)
{
    int g = (n + 3) / 4;
    if (g > 8192) g = 8192;
    return g > 0 ? g : 1;
}

}  // namespace

// Workgroups of four waves over 16-row tiles, at most two per CU (the weights
// are loaded once per wave).
static int tile_grid(int n)
{
    const int t = (n + 63) / 64;
    return t < 512 ? t : 512;
}

void gnn_forward(const GnnArgs &g, const float *w, bool keep, float *scores, hipStream_t s)
{
    const int n = g.n;
    const int gw = grid_for_waves(n), ga = (n + 15) / 16 < 16384 ? (n + 15) / 16 : 16384;
    // layer 1
    hipLaunchKernelGGL(k_agg2, dim3(1024), dim3(256), 0, s, n, g.ptr, g.ind, g.a, g.H0, g.M1);
    hipLaunchKernelGGL(k_dense1, dim3(gw), dim3(256), 0, s, n, (const float *)g.H0, (const float *)g.M1, w, g.H[0]);
    // layers 2, 3
    for (int l = 1; l < 3; ++l) {
        const float *Hin = g.H[keep ? l - 1 : (l - 1) & 1];
        float *Mout = g.M[keep ? l : 0];
        float *Hout = g.H[keep ? l : (l & 1)];
        hipLaunchKernelGGL(k_agg64<false>, dim3(ga), dim3(256), 0, s, n, g.ptr, g.ind, g.a, Hin, Mout);
        const float *Ws = w + (l == 1 ? kGnnWs2 : kGnnWs3);
        const float *Wn = w + (l == 1 ? kGnnWn2 : kGnnWn3);
        const float *b = w + (l == 1 ? kGnnB2 : kGnnB3);
        hipLaunchKernelGGL(k_dense_mfma, dim3(tile_grid(n)), dim3(256), 0, s, n, Hin, (const float *)Mout, Ws, Wn, b,
                           Hout);
    }
    const float *H3 = g.H[keep ? 2 : 0];
    hipLaunchKernelGGL(k_score, dim3(gw), dim3(256), 0, s, n, H3, w, scores);
}

size_t gnn_partial_floats() { return (size_t)kGnnPartials * kWgLen; }

void gnn_backward(const GnnArgs &g, const float *w, const float *ds, float *dw, hipStream_t s)
{
    const int n = g.n;
    const int ga = (n + 15) / 16 < 16384 ? (n + 15) / 16 : 16384;
    // rows per wave of the weight gradients: four waves a workgroup, at most
    // kGnnPartials workgroups, at least one 8-row step a wave
    int rows = (n + 4 * kGnnPartials - 1) / (4 * kGnnPartials);
    rows = (rows + 7) / 8 * 8;
    const int nb = (n + 4 * rows - 1) / (4 * rows);
    auto sum = [&](auto last, int stride, int len, const WgradRows &r, float *out) {
        hipLaunchKernelGGL((k_sum_partials<decltype(last)::value>), dim3((len + 31) / 32), dim3(256), 0, s,
                           (const float *)g.part, nb, stride, len, r, out);
    };
    float *dH = g.dA, *dX = g.dB, *G = g.dC;
    // layer 3 with the output layer (its gradients follow the layer's in dw)
    hipLaunchKernelGGL(k_wgrad64<true>, dim3(nb), dim3(256), 0, s, n, rows, (const float *)nullptr,
                       (const float *)g.H[2], ds, w + kGnnWo, (const float *)g.H[1], (const float *)g.M[2], g.part);
    sum(std::true_type(), kWgLen, kWgLen, WgradRows{n, nullptr, g.H[2], ds, w + kGnnWo, g.H[1], g.M[2]}, dw + kGnnWs3);
    hipLaunchKernelGGL(k_back_dense<true>, dim3(tile_grid(n)), dim3(256), 0, s, n, (const float *)nullptr,
                       (const float *)g.H[2], ds, w + kGnnWo, w + kGnnWs3, w + kGnnWn3, dH, G);
    hipLaunchKernelGGL(k_agg64<true>, dim3(ga), dim3(256), 0, s, n, g.ptr, g.ind, g.at, (const float *)G, dH);
    // layer 2
    hipLaunchKernelGGL(k_wgrad64<false>, dim3(nb), dim3(256), 0, s, n, rows, (const float *)dH, (const float *)g.H[1],
                       (const float *)nullptr, (const float *)nullptr, (const float *)g.H[0], (const float *)g.M[1],
                       g.part);
    sum(std::false_type(), kWgLen, 2 * kH * kH + kH, WgradRows{n, dH, g.H[1], nullptr, nullptr, g.H[0], g.M[1]},
        dw + kGnnWs2);
    hipLaunchKernelGGL(k_back_dense<false>, dim3(tile_grid(n)), dim3(256), 0, s, n, (const float *)dH,
                       (const float *)g.H[1], (const float *)nullptr, (const float *)nullptr, w + kGnnWs2, w + kGnnWn2,
                       dX, G);
    hipLaunchKernelGGL(k_agg64<true>, dim3(ga), dim3(256), 0, s, n, g.ptr, g.ind, g.at, (const float *)G, dX);
    // layer 1
    hipLaunchKernelGGL(k_wgrad2, dim3(nb), dim3(256), 0, s, n, rows, (const float *)dX, (const float *)g.H[0],
                       (const float *)g.H0, (const float *)g.M1, g.part);
    sum(std::false_type(), kWgLen2, kWgLen2, WgradRows{}, dw + kGnnWs1);
}

}  // namespace rc
