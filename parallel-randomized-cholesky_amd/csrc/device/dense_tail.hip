// dense_tail.hip -- the narrow trailing levels of the triangular sweeps.
//
// The level order ends in hundreds of levels of a few rows each (solver.hpp:
// 149-233 leaves them to cuSPARSE's level scheduler).  Walking them one after
// the other costs a dependency round trip per level: about 1 us (FP32) to
// 1.3 us (FP64) from LDS in one workgroup, 2.2 us through device-scope memory.
// Here the tail rows are cut into blocks of at most kTailBlock consecutive
// positions and every block's unit lower triangle is inverted at assembly, so
// a sweep spends two short launches per block (about 5 us each, a launch
// inside a graph costs 1.8 us) whatever the block's number of levels.
//
// Accuracy: the off-diagonal entries of a factor column are -w/S, so N = I - L
// is non-negative with column sums <= 1 and L^-1 = sum N^k holds visiting
// probabilities: every entry lies in [0, 1] and is a sum of non-negative
// products, with no cancellation.  The inversion runs in FP64 on the matrix
// cores and is rounded once to the factor's precision, so applying it is as
// accurate as the substitution it replaces (a longer chain of roundings).
#include "common.cuh"
#include "kernels.h"

namespace rc {

namespace {

constexpr int kTB = 256;

__device__ __forceinline__ int entry_pos(const EllSrc &src, int e)
{
    const int col = src.rowk ? src.rowk[e] : src.ind[e];
    return src.colmap ? src.colmap[col] : col;
}

// ---------------------------------------------------------------- assembly
// One wave per tail row.
template <typename T>
__global__ void k_tail_count(TailBuild tb, int fwd, EllSrc src, int *cnt, int *flag)
{
    const int lane = lane_id();
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int nwaves = gridDim.x * blockDim.x / kWave;
    const T *sval = (const T *)src.val;
    for (int q = wave; q < tb.ntail; q += nwaves) {
        const int row = tb.order[tb.tp0 + q];
        const int b = src.ptr[row], len = src.ptr[row + 1] - b;
        const int lo = tb.tp0 + q / tb.m * tb.m, hi = lo + tb.m;
        int no = 0;
        double sum = 0.0;
        for (int t = lane; t < len; t += kWave) {
            const int e = src.eidx ? src.eidx[b + t] : b + t;
            const int pos = entry_pos(src, e);
            no += (fwd ? pos < lo : pos >= hi) ? 1 : 0;
            if (!fwd) sum += fabs((double)sval[e]);
        }
        no = wave_sum_int(no);
        if (!fwd) sum = wave_sum(sum);
        if (lane == 0) {
            cnt[q] = no;
            if (!fwd && !(sum <= 1.001)) atomicOr(flag, 1);
        }
    }
}

// One wave per tail row: stable compaction of the outer entries; forward, the
// block's own entries are written to its dense matrix.  A loaded factor may hold
// an entry in several parts; they lie side by side (rows are sorted by column),
// and the first one's lane adds them in order.
template <typename T>
__global__ void k_tail_split(TailBuild tb, int fwd, EllSrc src, const int *ptr, int *ind, T *val, double *D)
{
    const int lane = lane_id();
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int nwaves = gridDim.x * blockDim.x / kWave;
    const T *sval = (const T *)src.val;
    for (int q = wave; q < tb.ntail; q += nwaves) {
        const int row = tb.order[tb.tp0 + q];
        const int b = src.ptr[row], len = src.ptr[row + 1] - b;
        const int blk = q / tb.m, lo = tb.tp0 + blk * tb.m, hi = lo + tb.m;
        double *drow = D + ((size_t)blk * tb.m + (size_t)(q - blk * tb.m)) * tb.m;
        int o = ptr[q];
        for (int base = 0; base < len; base += kWave) {
            const int t = base + lane;
            int pos = 0, e = 0;
            bool outer = false;
            if (t < len) {
                e = src.eidx ? src.eidx[b + t] : b + t;
                pos = entry_pos(src, e);
                outer = fwd ? pos < lo : pos >= hi;
                if (fwd && !outer) {
                    auto part = [&](int u) { return src.eidx ? src.eidx[b + u] : b + u; };
                    if (t == 0 || entry_pos(src, part(t - 1)) != pos) {
                        double v = (double)sval[e];
                        for (int u = t + 1; u < len && entry_pos(src, part(u)) == pos; ++u) v += (double)sval[part(u)];
                        drow[pos - lo] = v;
                    }
                }
            }
            const uint64_t mo = ballot(outer);
            if (outer) {
                const int at = o + lanes_below(mo);
                ind[at] = pos;
                val[at] = sval[e];
            }
            o += __popcll(mo);
        }
    }
}

// Inverse of every 64 x 64 diagonal tile (unit lower triangular), in place:
// lane j holds column j, row i is X_ij = d_ij - sum_{k<i} L_ik X_kj.
__global__ void __launch_bounds__(kWave) k_tail_base(int m, double *D)
{
    __shared__ double L[kTailTile][kTailTile], X[kTailTile][kTailTile];
    const int lane = lane_id();
    double *d = D + (size_t)blockIdx.y * m * m + (size_t)blockIdx.x * kTailTile * (m + 1);
    for (int i = 0; i < kTailTile; ++i) L[i][lane] = d[(size_t)i * m + lane];
    __syncthreads();
    for (int i = 0; i < kTailTile; ++i) {
        double a0 = i == lane ? 1.0 : 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
        int k = 0;
        for (; k + 4 <= i; k += 4) {
            a0 = __builtin_fma(-L[i][k], X[k][lane], a0);
            a1 = __builtin_fma(-L[i][k + 1], X[k + 1][lane], a1);
            a2 = __builtin_fma(-L[i][k + 2], X[k + 2][lane], a2);
            a3 = __builtin_fma(-L[i][k + 3], X[k + 3][lane], a3);
        }
        for (; k < i; ++k) a0 = __builtin_fma(-L[i][k], X[k][lane], a0);
        X[i][lane] = (a0 + a1) + (a2 + a3);          // column `lane` is read by this lane only
    }
    for (int i = 0; i < kTailTile; ++i) d[(size_t)i * m + lane] = X[i][lane];
}

// One doubling step of the inversion: with A and B the inverted diagonal parts
// of s rows and C the part of L below A and left of B,
//   kSecond = false: E = C A^-1;   kSecond = true: C <- -B^-1 E.
// One 64 x 64 tile per workgroup, 32 x 32 per wave, v_mfma_f64_16x16x4_f64
// (operands: lane l holds A row l % 16 / B column l % 16 at k = l / 16; result
// register i of lane l is row 4 i + l / 16 of column l % 16).  Tiles above the
// triangles are skipped, which halves the products.
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kGK = 16;                              // k per LDS stage

template <bool kSecond>
__global__ void __launch_bounds__(kTB) k_tail_gemm(int m, int s, double *Dall, double *Eall)
{
    __shared__ double As[64][kGK + 2], Bs[kGK][64 + 4];
    const int nt = s / kTailTile;                    // tiles per side of A
    const int ti = blockIdx.x / nt, tj = blockIdx.x % nt;
    const int r0 = (2 * blockIdx.y + 1) * s, c0 = 2 * blockIdx.y * s;
    if (r0 + ti * 64 >= m) return;                   // the last part may be shorter than s
    double *D = Dall + (size_t)blockIdx.z * m * m, *E = Eall + (size_t)blockIdx.z * m * m;
    const double *A, *B;
    double *out;
    int k0, k1;
    if (!kSecond) {
        A = D + (size_t)(r0 + ti * 64) * m + c0;     // C, rows of this tile
        B = D + (size_t)c0 * m + c0 + tj * 64;       // A^-1, columns of this tile: rows k >= column
        out = E + (size_t)(r0 + ti * 64) * m + c0 + tj * 64;
        k0 = tj * 64;
        k1 = s;
    } else {
        A = D + (size_t)(r0 + ti * 64) * m + r0;     // B^-1: columns k <= row
        B = E + (size_t)r0 * m + c0 + tj * 64;
        out = D + (size_t)(r0 + ti * 64) * m + c0 + tj * 64;
        k0 = 0;
        k1 = (ti + 1) * 64;
    }
    const int t = threadIdx.x, lane = lane_id(), w = t / kWave;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
    const int lr = lane % 16, lk = lane / 16;
    f64x4 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    // stage loads: A 64 x 16 (thread: row t / 4, 4 values), B 16 x 64 (row t / 16, 4 values)
    const int ar = t / 4, ac = (t % 4) * 4, br = t / 16, bc = (t % 16) * 4;
    double2 a0, a1, b0, b1;
    auto load = [&](int k) {
        const double2 *pa = reinterpret_cast<const double2 *>(A + (size_t)ar * m + k + ac);
        const double2 *pb = reinterpret_cast<const double2 *>(B + (size_t)(k + br) * m + bc);
        a0 = pa[0]; a1 = pa[1];
        b0 = pb[0]; b1 = pb[1];
    };
    load(k0);
    for (int k = k0; k < k1; k += kGK) {
        As[ar][ac] = a0.x; As[ar][ac + 1] = a0.y; As[ar][ac + 2] = a1.x; As[ar][ac + 3] = a1.y;
        Bs[br][bc] = b0.x; Bs[br][bc + 1] = b0.y; Bs[br][bc + 2] = b1.x; Bs[br][bc + 3] = b1.y;
        __syncthreads();
        if (k + kGK < k1) load(k + kGK);             // the next stage's loads run under the products
#pragma unroll
        for (int kk = 0; kk < kGK; kk += 4) {
            double av[2], bv[2];
            for (int i = 0; i < 2; ++i) av[i] = As[wr + i * 16 + lr][kk + lk];
            for (int j = 0; j < 2; ++j) bv[j] = Bs[kk + lk][wc + j * 16 + lr];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int q = 0; q < 4; ++q) {
                const double v = acc[i][j][q];
                out[(size_t)(wr + i * 16 + 4 * q + lk) * m + wc + j * 16 + lr] = kSecond ? -v : v;
            }
}

// Wf = D and Wb = D^T in precision T, one 64 x 64 tile per workgroup.  (FP64:
// Wf is D itself.)  Only tiles on and below the diagonal of D hold entries;
// the mirrored tiles of Wb are the ones that are read.
template <typename T>
__global__ void __launch_bounds__(kTB) k_tail_store(int m, const double *Dall, T *Wf, T *Wb)
{
    __shared__ double tile[64][64 + 1];
    const int nt = m / 64;
    const int ti = blockIdx.x / nt, tj = blockIdx.x % nt;
    if (ti < tj) return;
    const size_t base = (size_t)blockIdx.y * m * m;
    const double *D = Dall + base;
    for (int i = threadIdx.x; i < 64 * 64; i += kTB) {
        const int r = i / 64, c = i % 64;
        const double v = D[(size_t)(ti * 64 + r) * m + tj * 64 + c];
        tile[r][c] = v;
        if constexpr (sizeof(T) == 4) Wf[base + (size_t)(ti * 64 + r) * m + tj * 64 + c] = (T)v;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += kTB) {
        const int r = i / 64, c = i % 64;
        Wb[base + (size_t)(tj * 64 + r) * m + ti * 64 + c] = (T)tile[c][r];
    }
}

// ---------------------------------------------------------------- sweeps
// Right-hand side of block blk, one wave per row (a row has up to a few
// hundred outer entries: four loads per lane in flight).  Forward: r (updated
// to r - alpha Ap, with x += alpha p) minus the entries in earlier positions;
// backward: D+ y (solver.hpp:64-84) minus the entries in later blocks.
template <typename T, bool kFwd>
__global__ void __launch_bounds__(kTB) k_tail_rhs(SolveArgs a, int blk, const double *p_cur, int update_rx)
{
    PcgScalars *sc = a.sc;
    if (sc->done) return;
    const double alpha0 = (kFwd && update_rx) ? sc->alpha : 0.0;
    const int *ptr = kFwd ? a.tf_ptr : a.tb_ptr, *ind = kFwd ? a.tf_ind : a.tb_ind;
    const T *val = (const T *)(kFwd ? a.tf_val : a.tb_val);
    const T *y = (const T *)a.y;
    const T *vec = kFwd ? y : (const T *)a.z;
    const int lane = lane_id();
    const int i = (blockIdx.x * kTB + threadIdx.x) / kWave;
    const int q = blk * a.tail_m + i;
    if (i >= a.tail_m || q >= a.ntail) return;
    const int k = a.tail_pos0 + q;
    const bool lead = lane == kWave - 1;             // receives the group sum
    double rk = 0.0, apk = 0.0, xk = 0.0, pk = 0.0;
    T own = (T)0, dk = (T)0;
    if (lead) {
        if (kFwd) {
            rk = a.r[k];
            if (update_rx) {
                apk = a.ap[k];
                xk = a.x[k];
                pk = p_cur[k];
            }
        } else {
            own = y[k];
            dk = ((const T *)a.diag)[k];
        }
    }
    const int e0 = ptr[q], e1 = ptr[q + 1];
    T acc = (T)0;
    for (int e = e0 + lane; e < e1; e += 4 * kWave) {
        int j[4];
        T l[4], v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool in = e + u * kWave < e1;
            j[u] = in ? ind[e + u * kWave] : a.n;    // the dummy slot holds 0
            l[u] = in ? val[e + u * kWave] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = vec[j[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = fma_t(-l[u], v[u], acc);
    }
    acc = group_sum(acc, kWave);
    if (lead) {
        if (kFwd) {
            if (update_rx) {
                const double al = a.alpha_sys ? a.alpha_sys[a.sys_of[k]] : alpha0;
                rk = fma_t(-al, apk, rk);
                a.r[k] = rk;
                a.x[k] = fma_t(al, pk, xk);
            }
            own = (T)rk;
        } else if (dk != (T)0) {
            own = own / dk;
        }
        ((T *)a.tacc)[i] = own + acc;
    }
}

// Applies block blk's inverse: one wave per row of Wf (columns 0..i) or Wb
// (columns i..m-1), 16-byte loads, up to eight in flight per lane.  Bound by
// the bytes of the triangle and one memory round trip.  Short and long rows
// alternate between the waves of a workgroup.  An entry that is exactly zero
// contributes nothing whatever the right-hand side holds, as in the
// substitution: systems of a batch stay independent of each other's values.
template <typename T, bool kFwd>
__global__ void __launch_bounds__(kTB) k_tail_apply(SolveArgs a, int blk)
{
    constexpr int V = 16 / (int)sizeof(T);
    constexpr int U = 8;
    if (a.sc->done) return;
    const int m = a.tail_m, rows = min(m, a.ntail - blk * m);
    const int lane = lane_id();
    const int w = (blockIdx.x * kTB + threadIdx.x) / kWave;
    if (w >= rows) return;
    const int i = (w & 1) ? rows - 1 - (w >> 1) : (w >> 1);
    const T *W = (const T *)(kFwd ? a.tail_wf : a.tail_wb) + ((size_t)blk * m + i) * m;
    const T *tv = (const T *)a.tacc;
    const int c0 = kFwd ? 0 : i / V * V, c1 = kFwd ? i + 1 : rows;
    T acc = (T)0;
    for (int c = c0 + lane * V; c < c1; c += U * kWave * V) {
        T wv[U][V], xv[U][V];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int cc = c + u * kWave * V;
            if (cc < c1) {                            // rows of W and tacc are padded to the tile size
                if constexpr (sizeof(T) == 4) {
                    const float4 p = *reinterpret_cast<const float4 *>(W + cc);
                    const float4 x = *reinterpret_cast<const float4 *>(tv + cc);
                    wv[u][0] = p.x; wv[u][1] = p.y; wv[u][2] = p.z; wv[u][3] = p.w;
                    xv[u][0] = x.x; xv[u][1] = x.y; xv[u][2] = x.z; xv[u][3] = x.w;
                } else {
                    const double2 p = *reinterpret_cast<const double2 *>(W + cc);
                    const double2 x = *reinterpret_cast<const double2 *>(tv + cc);
                    wv[u][0] = p.x; wv[u][1] = p.y;
                    xv[u][0] = x.x; xv[u][1] = x.y;
                }
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v) { wv[u][v] = (T)0; xv[u][v] = (T)0; }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) acc = fma_t(wv[u][v], wv[u][v] != (T)0 ? xv[u][v] : (T)0, acc);
    }
    acc = group_sum(acc, kWave);
    if (lane == kWave - 1) ((T *)(kFwd ? a.y : a.z))[a.tail_pos0 + blk * m + i] = unsent(acc);
}

int waves_grid(int items)
{
    int g = (items + 3) / 4;
    if (g > 16384) g = 16384;
    return g < 1 ? 1 : g;
}

}  // namespace

template <typename T>
void launch_tail_count(const TailBuild &t, bool fwd, EllSrc src, int *cnt, int *flag, hipStream_t s)
{
    hipLaunchKernelGGL(k_tail_count<T>, dim3(waves_grid(t.ntail)), dim3(kTB), 0, s, t, fwd ? 1 : 0, src, cnt, flag);
}

template <typename T>
void launch_tail_split(const TailBuild &t, bool fwd, EllSrc src, const int *ptr, int *ind, T *val, double *D,
                       hipStream_t s)
{
    hipLaunchKernelGGL(k_tail_split<T>, dim3(waves_grid(t.ntail)), dim3(kTB), 0, s, t, fwd ? 1 : 0, src, ptr, ind, val,
                       D);
}

void launch_tail_invert(const TailBuild &t, double *D, double *E, hipStream_t s)
{
    hipLaunchKernelGGL(k_tail_base, dim3(t.m / kTailTile, t.nb), dim3(kWave), 0, s, t.m, D);
    for (int sz = kTailTile; sz < t.m; sz *= 2) {
        const int pairs = (t.m + sz - 1) / (2 * sz);        // pairs whose second part is not empty
        const int nt = sz / kTailTile;
        const dim3 g(nt * nt, pairs, t.nb);
        hipLaunchKernelGGL(k_tail_gemm<false>, g, dim3(kTB), 0, s, t.m, sz, D, E);
        hipLaunchKernelGGL(k_tail_gemm<true>, g, dim3(kTB), 0, s, t.m, sz, D, E);
    }
}

template <typename T>
void launch_tail_store(const TailBuild &t, const double *D, T *Wf, T *Wb, hipStream_t s)
{
    const int nt = t.m / 64;
    hipLaunchKernelGGL(k_tail_store<T>, dim3(nt * nt, t.nb), dim3(kTB), 0, s, t.m, D, Wf, Wb);
}

template <typename T>
void launch_tail_fwd(const SolveArgs &a, const double *p_cur, int update_rx, hipStream_t s)
{
    for (int b = 0; b < a.tail_nb; ++b) {
        const int g = waves_grid(a.ntail - b * a.tail_m < a.tail_m ? a.ntail - b * a.tail_m : a.tail_m);
        hipLaunchKernelGGL((k_tail_rhs<T, true>), dim3(g), dim3(kTB), 0, s, a, b, p_cur, update_rx);
        hipLaunchKernelGGL((k_tail_apply<T, true>), dim3(g), dim3(kTB), 0, s, a, b);
    }
}

template <typename T>
void launch_tail_bwd(const SolveArgs &a, hipStream_t s)
{
    for (int b = a.tail_nb - 1; b >= 0; --b) {
        const int g = waves_grid(a.ntail - b * a.tail_m < a.tail_m ? a.ntail - b * a.tail_m : a.tail_m);
        hipLaunchKernelGGL((k_tail_rhs<T, false>), dim3(g), dim3(kTB), 0, s, a, b, (const double *)nullptr, 0);
        hipLaunchKernelGGL((k_tail_apply<T, false>), dim3(g), dim3(kTB), 0, s, a, b);
    }
}

#define RC_TAIL_INST(T)                                                                                         \
    template void launch_tail_count<T>(const TailBuild &, bool, EllSrc, int *, int *, hipStream_t);             \
    template void launch_tail_split<T>(const TailBuild &, bool, EllSrc, const int *, int *, T *, double *,      \
                                       hipStream_t);                                                            \
    template void launch_tail_store<T>(const TailBuild &, const double *, T *, T *, hipStream_t);               \
    template void launch_tail_fwd<T>(const SolveArgs &, const double *, int, hipStream_t);                      \
    template void launch_tail_bwd<T>(const SolveArgs &, hipStream_t);
RC_TAIL_INST(float)
RC_TAIL_INST(double)
#undef RC_TAIL_INST

}  // namespace rc
