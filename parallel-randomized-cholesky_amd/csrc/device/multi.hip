// multi.hip -- PCG for k <= 64 right-hand sides sharing one factor.
//
// Same recurrence as pcg.hip (solver.hpp:457-569) run independently for every
// right-hand side q: its own alpha, beta, r'z, stop test and iteration count;
// a converged right-hand side is frozen (its x and r no longer change) while
// the others continue.  Vectors are row-major n x K (K = next power of two
// >= k) in the level-order position numbering, so the K values of a row are
// contiguous: a wave handles 64/K rows with K lanes each, the index and value
// of every matrix entry are one broadcast load, and the gather of row j's K
// values is one coalesced access.  Matrices are CSR in position numbering.
// The sweeps keep the sentinel protocol of the single-RHS sweeps (per value);
// the tail rows are solved by the blocks' dense inverses on the matrix cores.
#include "common.cuh"
#include "kernels.h"

namespace rc {

namespace {

// Reduction kernels: few large workgroups, so that the last one adds 256
// partials per right-hand side (1024 workgroups of 256 threads left it with
// 1024 dependent device-scope loads per right-hand side: 300 us of the 350 us
// of k_mspmv at 148k rows x 64).
constexpr int kMB = 1024;
constexpr int kMBlocks = 256;
int mblocks(const MultiArgs &a)
{
    const long long need = ((long long)a.n * a.K + kMB - 1) / kMB;
    return need >= kMBlocks ? kMBlocks : (need < 8 ? 8 : (int)(need / 8 * 8));   // a multiple of the XCDs
}

// The partials are written by the first wave (K <= 64 threads) with agent-scope
// stores and read the same way, so that wave's drain_stores orders them before
// the arrival.

// Sum over the workgroup of every right-hand side's v (thread t holds one of
// right-hand side t % K), valid in threads t < K.
__device__ __forceinline__ double msum(double v, int K, double *red)
{
    red[threadIdx.x] = v;
    __syncthreads();
    for (int h = (int)blockDim.x / 2; h >= K; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    const double s = red[threadIdx.x & (K - 1)];
    __syncthreads();
    return s;
}

// The workgroups' partials (nb x K) summed by one workgroup, valid in threads t < K.
__device__ __forceinline__ double mfinal(const double *partials, int nb, int K, double *red)
{
    double s = 0.0;
    const int total = nb * K;
    for (int i = threadIdx.x; i < total; i += 4 * (int)blockDim.x) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int e = i + u * (int)blockDim.x;
            v[u] = e < total ? ld_relaxed_val(partials + e) : 0.0;
        }
        s += (v[0] + v[1]) + (v[2] + v[3]);
    }
    return msum(s, K, red);
}

// Replaces the sentinels among w[u][v] = vec[j[u] * K + q0 + v] by their values,
// awaiting them: a lane's pending values are polled together (as await_values
// of the single sweeps), and a wave in which a lane awaits several entries, so
// some levels ahead of the sweep, polls less often.  Polled one after the other
// with a status load each, a solve with 5 right-hand sides x 101520 rows took
// 25.0 ms, together 19.6 (64 x 147840 rows: 38.2 and 37.1).
template <typename T, int B, int V>
__device__ __forceinline__ void mawait_values(T (&w)[B][V], const int (&j)[B], T *vec, int K, int q0,
                                              long long spin_ticks, MultiScalars *sc)
{
    const auto pending = [&](int u) {
        bool p = false;
#pragma unroll
        for (int v = 0; v < V; ++v) p |= is_sent(w[u][v]);
        return p;
    };
    int np = 0;
#pragma unroll
    for (int u = 0; u < B; ++u) np += pending(u);
    if (np == 0) return;
    long long t0 = 0;
    int tries = 0;
    while (true) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
            T *p = vec + (size_t)j[u] * K + q0;
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (is_sent(w[u][v])) w[u][v] = ld_relaxed_val(p + v);
        }
        np = 0;
#pragma unroll
        for (int u = 0; u < B; ++u) np += pending(u);
        if (np == 0) return;
        if ((++tries & 63) == 0) {               // bounded: see kPcgTimeout
            const long long now = wall_clock64();
            if (t0 == 0) t0 = now;
            bool stop = (ld_relaxed(&sc->status) & kPcgTimeout) != 0;
            if (now - t0 > spin_ticks) {
                atomicOr(&sc->status, kPcgTimeout);
                stop = true;
            }
            if (stop) {
#pragma unroll
                for (int u = 0; u < B; ++u)
#pragma unroll
                    for (int v = 0; v < V; ++v) w[u][v] = is_sent(w[u][v]) ? (T)0 : w[u][v];
                return;
            }
        }
        if (ballot(np >= 2)) __builtin_amdgcn_s_sleep(8);
    }
}

// ---------------------------------------------------------------- SpMM
// p_new = z + beta_q p_old (streaming); then Ap = A p_new and per-q partials
// of p'Ap.
template <typename T>
__global__ void __launch_bounds__(256) k_mpupdate(MultiArgs a, const double *p_old, double *p_new)
{
    MultiScalars *sc = a.sc;
    if (sc->all_done) return;
    const int K = a.K;
    const T *z = (const T *)a.z;
    const size_t total = (size_t)a.n * K;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int q = (int)(i & (size_t)(K - 1));
        const double beta = q < a.k ? sc->beta[q] : 0.0;
        p_new[i] = fma_t(beta, p_old[i], (double)z[i]);
    }
}

template <typename T>
__global__ void __launch_bounds__(kMB) k_mspmv(MultiArgs a, const double *p)
{
    __shared__ double red[kMB];
    __shared__ int flag;
    MultiScalars *sc = a.sc;
    if (sc->all_done) return;
    if (blockIdx.x == 0) reset_claims(a.ctr_fwd, a.ctr_bwd, threadIdx.x);
    const int K = a.K;
    const int q = threadIdx.x % K;
    const int rows_per_block = kMB / K;
    double acc_dot = 0.0;
    // rows visited in the input numbering (a row's neighbours are near it
    // there, not in positions), the workgroups of each XCD (workgroup b runs
    // on XCD b % 8) walking one contiguous eighth of it
    int r0 = blockIdx.x * rows_per_block + threadIdx.x / K, r1 = a.n, rstep = gridDim.x * rows_per_block;
    if (gridDim.x % 8 == 0) {
        const int x = blockIdx.x % 8, per = (a.n + 7) / 8;
        const int lo = min(a.n, x * per);
        r1 = min(a.n, lo + per);
        r0 = lo + (blockIdx.x / 8) * rows_per_block + threadIdx.x / K;
        rstep = (gridDim.x / 8) * rows_per_block;
    }
    // two rows per pass, the first kE entries of both loaded together, so the
    // dependent loads of one row (row index, row bounds, entries, gathers)
    // overlap with the other's; each row still sums its entries in order
    constexpr int kE = 8;
    for (int ru = r0; ru < r1; ru += 2 * rstep) {
        const bool two = ru + rstep < r1;
        int row[2], eb[2], ee[2];
        row[0] = a.row_ord[ru];
        row[1] = two ? a.row_ord[ru + rstep] : row[0];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            eb[h] = a.a_ptr[row[h]];
            ee[h] = a.a_ptr[row[h] + 1];
        }
        if (!two) ee[1] = eb[1];
        int j[2][kE];
        double v[2][kE], pj[2][kE];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < kE; ++u) {
                const bool has = eb[h] + u < ee[h];
                j[h][u] = has ? a.a_ind[eb[h] + u] : 0;
                v[h][u] = has ? a.a_val[eb[h] + u] : 0.0;
            }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < kE; ++u) pj[h][u] = p[(size_t)j[h][u] * K + q];
        double acc[2] = {0.0, 0.0};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int u = 0; u < kE; ++u)
                if (eb[h] + u < ee[h]) acc[h] = fma_t(v[h][u], pj[h][u], acc[h]);
            for (int e = eb[h] + kE; e < ee[h]; ++e) acc[h] = fma_t(a.a_val[e], p[(size_t)a.a_ind[e] * K + q], acc[h]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 1 && !two) break;
            const size_t o = (size_t)row[h] * K + q;
            a.ap[o] = acc[h];
            acc_dot += p[o] * acc[h];
        }
    }
    // per-q block partial: threads t, t+K, t+2K, ... share q
    const double bs = msum(acc_dot, K, red);
    if ((int)threadIdx.x < K) st_relaxed_val(a.partials + (size_t)blockIdx.x * K + threadIdx.x, bs);
    __syncthreads();
    if (threadIdx.x == 0) {
        drain_stores();
        unsigned int old = atomicAdd(&sc->arrive_spmv, 1u);
        flag = old == gridDim.x - 1;
    }
    __syncthreads();
    if (!flag) return;
    const double pap = mfinal(a.partials, gridDim.x, K, red);
    if ((int)threadIdx.x < K) {
        const int qq = threadIdx.x;
        if (qq < a.k && !sc->done[qq]) {
            if (!(pap > 0.0) || !isfinite(pap)) {
                sc->alpha[qq] = 0.0;
                sc->done[qq] = 1;
                sc->breakdown[qq] = 1;
            } else {
                sc->alpha[qq] = sc->rz[qq] / pap;
            }
        } else if (qq < a.k) {
            sc->alpha[qq] = 0.0;
        }
        if (qq == 0) sc->arrive_spmv = 0u;
    }
}

// ---------------------------------------------------------------- sweeps
// A row takes L x S lanes of one wave: L = K / V lanes hold V right-hand sides
// each (V = 4 in FP32, 2 in FP64, so a gather of row j's values is one 16-byte
// access per lane), S entry slots share the row's entries (slot s holds
// entries s, s + S, ..., at most eight of them in flight) and are summed by
// shuffles.  S grows with the row length, so a long row costs one memory round
// trip per eight entries of a slot, not per eight entries.
template <typename T, int V>
__device__ __forceinline__ void vload(const T *p, T *v)
{
    if constexpr (V == 4 && sizeof(T) == 4) {
        const float4 q = *reinterpret_cast<const float4 *>(p);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else if constexpr (V >= 2 && sizeof(T) == 8) {
#pragma unroll
        for (int h = 0; h < V; h += 2) {
            const double2 q = *reinterpret_cast<const double2 *>(p + h);
            v[h] = q.x; v[h + 1] = q.y;
        }
    } else if constexpr (V == 2) {
        const float2 q = *reinterpret_cast<const float2 *>(p);
        v[0] = q.x; v[1] = q.y;
    } else {
        v[0] = *p;
    }
}
template <typename T, int V>
__device__ __forceinline__ void vstore(T *p, const T *v)
{
    if constexpr (V == 4) {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    } else if constexpr (V == 2 && sizeof(T) == 4) {
        *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
    } else if constexpr (V == 2) {
        *reinterpret_cast<double2 *>(p) = make_double2(v[0], v[1]);
    } else {
        *p = v[0];
    }
}
template <int V>
__device__ __forceinline__ void dload(const double *p, double *v)
{
    if constexpr (V == 1) v[0] = *p;
    else
#pragma unroll
        for (int h = 0; h < V; h += 2) {
            const double2 q = *reinterpret_cast<const double2 *>(p + h);
            v[h] = q.x; v[h + 1] = q.y;
        }
}
template <int V>
__device__ __forceinline__ void dstore(double *p, const double *v)
{
    if constexpr (V == 1) *p = v[0];
    else
#pragma unroll
        for (int h = 0; h < V; h += 2) *reinterpret_cast<double2 *>(p + h) = make_double2(v[h], v[h + 1]);
}
// Published values: agent-scope stores of at most 8 bytes (two FP32 values
// share one; a reader checks every value for the sentinel by itself).
template <typename T, int V>
__device__ __forceinline__ void vpublish(T *p, const T *v)
{
    if constexpr (sizeof(T) == 4 && V >= 2) {
#pragma unroll
        for (int h = 0; h < V; h += 2)
            st_relaxed(reinterpret_cast<unsigned long long *>(p + h),
                       ((unsigned long long)__float_as_uint(unsent(v[h + 1])) << 32) | __float_as_uint(unsent(v[h])));
    } else {
#pragma unroll
        for (int h = 0; h < V; ++h) st_relaxed_val(p + h, unsent(v[h]));
    }
}

// Sum over the S entry slots (lane bits above the L right-hand-side lanes).
template <typename T, int V>
__device__ __forceinline__ void slot_sum(T *acc, int L, int LS)
{
    for (int o = L; o < LS; o <<= 1)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += __shfl_xor(acc[v], o, kWave);
}

// The row update of the forward sweep: r <- r - alpha Ap, x <- x + alpha p per
// right-hand side (a frozen one has alpha 0 and keeps its values).
template <int V>
__device__ __forceinline__ void row_update(const MultiArgs &a, size_t o, const double *alpha, double *rk,
                                           const double *ap, const double *pk, const double *xk)
{
    bool any = false;
    double xn[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        any = any || alpha[v] != 0.0;
        xn[v] = xk[v];
        if (alpha[v] != 0.0) {
            rk[v] = fma_t(-alpha[v], ap[v], rk[v]);
            xn[v] = fma_t(alpha[v], pk[v], xk[v]);
        }
    }
    if (any) {
        dstore<V>(a.r + o, rk);
        dstore<V>(a.x + o, xn);
    }
}

// Persistent sweep over the levels before the tail: workgroups claim chunks in
// level order, three ahead (the same protocol and the same argument against
// deadlock as k_sweep_bulk); while chunk i is solved, chunk i + 1's descriptor,
// row bounds and entries are loaded into registers, so a chunk costs one
// gather round trip and, as there, thread 0's claim.  Entries go through LDS: all
// lanes of a row read them.
template <typename T, bool kFwd, int V>
__global__ void __launch_bounds__(kMSweepThreads) k_msweep(MultiArgs a, const double *p_cur, int update_rx)
{
    constexpr int PE = kMChunkEntries / kMSweepThreads;
    __shared__ int s_ind[kMChunkEntries];
    __shared__ T s_val[kMChunkEntries];
    __shared__ int s_init[3], s_claim[2], s_stop;
    MultiScalars *sc = a.sc;
    if (sc->all_done) return;
    const int K = a.K;
    const int L = K / V, lb = __builtin_ctz(L);
    const int t = threadIdx.x;
    const int q0 = (t & (L - 1)) * V;
    double alpha[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int q = q0 + v;
        alpha[v] = (kFwd && update_rx && q < a.k && !sc->done[q]) ? sc->alpha[q] : 0.0;
    }
    T *y = (T *)a.y;
    T *z = (T *)a.z;
    T *vec = kFwd ? y : z;
    const T *val = (const T *)(kFwd ? a.l_val : a.lt_val);
    const int *ptr = kFwd ? a.l_ptr : a.lt_ptr;
    const int *ind = kFwd ? a.l_ind : a.lt_ind;
    const T *diag = (const T *)a.diag;
    const int nb = a.nchunks;
    const int4 *meta = kFwd ? a.cm_f : a.cm_b;
    // claim queue of this workgroup: its j-th claim is chunk j * nq + cq
    const int nq = (int)gridDim.x < kClaimQueues ? (int)gridDim.x : kClaimQueues;
    const int cq = (int)(blockIdx.x % (unsigned int)nq);
    unsigned int *ctr = (kFwd ? a.ctr_fwd : a.ctr_bwd) + cq * kClaimStride;
    auto desc = [&](int c) {              // a claim past the end is never processed
        const int cc = c < nb ? c : nb - 1;
        return meta[kFwd ? cc : nb - 1 - cc];
    };
    // log2 of the lanes per row: as many entry slots as the chunk's rows leave
    auto row_bits = [&](const int4 &m) {
        const int p2 = m.y <= 1 ? 0 : 32 - __builtin_clz((unsigned)(m.y - 1));
        const int b = kMSweepBits - p2;
        return b > 6 ? 6 : b;
    };
    int c_pend = 0;
    unsigned int st_pend = 0;
    if (t == 0) {
        s_init[0] = (int)atomicAdd(ctr, 1u) * nq + cq;
        s_init[1] = (int)atomicAdd(ctr, 1u) * nq + cq;
        s_init[2] = (int)atomicAdd(ctr, 1u) * nq + cq;
        c_pend = (int)atomicAdd(ctr, 1u) * nq + cq;
        st_pend = ld_relaxed(&sc->status);
    }
    __syncthreads();
    int c_cur = s_init[0], c_nxt = s_init[1], c_nxt2 = s_init[2];
    int4 m_cur = desc(c_cur), m_nxt = desc(c_nxt);
    int j_nxt[PE], r0_nxt, r1_nxt;
    T l_nxt[PE];
    // chunk m's entries and this lane's row bounds
    auto fetch = [&](const int4 &m) {
#pragma unroll
        for (int u = 0; u < PE; ++u) {
            const int e = u * kMSweepThreads + t;
            const int ee = m.z + (e < m.w ? e : 0);
            j_nxt[u] = ind[ee];
            l_nxt[u] = val[ee];
        }
        const int i = t >> row_bits(m);
        const int k = m.x + (i < m.y ? i : 0);
        r0_nxt = ptr[k];
        r1_nxt = ptr[k + 1];
    };
    fetch(m_cur);
    int par = 0;
    while (c_cur < nb) {
#pragma unroll
        for (int u = 0; u < PE; ++u) {
            s_ind[u * kMSweepThreads + t] = j_nxt[u];
            s_val[u * kMSweepThreads + t] = l_nxt[u];
        }
        const int r0 = r0_nxt - m_cur.z, r1 = r1_nxt - m_cur.z;
        __syncthreads();
        fetch(m_nxt);
        const int4 m_nxt2 = desc(c_nxt2);
        // ---- solve the chunk
        const int bits = row_bits(m_cur);
        const int S = 1 << (bits - lb);
        const int i = t >> bits, s = (t >> lb) & (S - 1);
        const bool active = i < m_cur.y;
        const bool lead = active && s == 0;
        const int k = m_cur.x + (active ? i : 0);
        const size_t o = (size_t)k * K + q0;
        T acc[V];
        double rk[V], ap[V], xk[V], pk[V];
        T own[V];
        T dk = (T)0;
#pragma unroll
        for (int v = 0; v < V; ++v) { acc[v] = (T)0; own[v] = (T)0; rk[v] = ap[v] = xk[v] = pk[v] = 0.0; }
        if (lead) {
            if (kFwd) {
                dload<V>(a.r + o, rk);
                if (update_rx) {
                    dload<V>(a.ap + o, ap);
                    dload<V>(a.x + o, xk);
                    dload<V>(p_cur + o, pk);
                }
            } else {
                vload<T, V>(y + o, own);
                dk = diag[k];
            }
        }
        if (active) {
            constexpr int B = 8;
            const bool in_lds = m_cur.w <= kMChunkEntries;
            for (int e = r0 + s; e < r1; e += B * S) {
                int j[B];
                T l[B];
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    const int ee = e + u * S;
                    const bool in = ee < r1;
                    const int at = in ? ee : r0;
                    if (in_lds) {
                        j[u] = in ? s_ind[at] : a.n;      // dummy slot n holds zeros
                        l[u] = in ? s_val[at] : (T)0;
                    } else {
                        j[u] = in ? ind[m_cur.z + at] : a.n;
                        l[u] = in ? val[m_cur.z + at] : (T)0;
                    }
                }
                T w[B][V];
#pragma unroll
                for (int u = 0; u < B; ++u) vload<T, V>(vec + (size_t)j[u] * K + q0, w[u]);
                mawait_values<T, B, V>(w, j, vec, K, q0, a.spin_ticks, sc);
#pragma unroll
                for (int u = 0; u < B; ++u)
#pragma unroll
                    for (int v = 0; v < V; ++v) acc[v] = fma_t(-l[u], w[u][v], acc[v]);
            }
        }
        slot_sum<T, V>(acc, L, 1 << bits);
        if (lead) {
            T sent[V];
#pragma unroll
            for (int v = 0; v < V; ++v) sent[v] = sent_value(T());
            if (kFwd) {
                if (update_rx) row_update<V>(a, o, alpha, rk, ap, pk, xk);
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] += (T)rk[v];
                vpublish<T, V>(y + o, acc);
                vstore<T, V>(z + o, sent);
            } else {
                vstore<T, V>(y + o, sent);
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] += dk != (T)0 ? own[v] / dk : own[v];   // solver.hpp:64-84
                vpublish<T, V>(z + o, acc);
            }
        }
        if (t == 0) {
            s_claim[par] = c_pend;
            s_stop = (int)st_pend;
            c_pend = (int)atomicAdd(ctr, 1u) * nq + cq;
            st_pend = ld_relaxed(&sc->status);
        }
        __syncthreads();
        if (s_stop & kPcgTimeout) break;
        c_cur = c_nxt;
        c_nxt = c_nxt2;
        c_nxt2 = s_claim[par];
        m_cur = m_nxt;
        m_nxt = m_nxt2;
        par ^= 1;
    }
}

// ---------------------------------------------------------------- tail
// Right-hand sides of block blk of the tail (rows of tacc, K values each), one
// wave per row, as k_tail_rhs; rows past the last are zero (the products read
// them).
template <typename T, bool kFwd, int V>
__global__ void __launch_bounds__(256) k_mtail_rhs(MultiArgs a, int blk, const double *p_cur, int update_rx)
{
    MultiScalars *sc = a.sc;
    if (sc->all_done) return;
    const int K = a.K, L = K / V, S = kWave / L;
    const int lane = lane_id();
    const int q0 = (lane & (L - 1)) * V, s = lane / L;
    const int i = (blockIdx.x * 256 + threadIdx.x) / kWave;
    if (i >= a.tail_m) return;
    const int q = blk * a.tail_m + i;
    T *out = (T *)a.tacc + (size_t)i * K + q0;
    T acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = (T)0;
    if (q >= a.ntail) {
        if (s == 0) vstore<T, V>(out, acc);
        return;
    }
    const int k = a.tail_pos0 + q;
    const size_t o = (size_t)k * K + q0;
    const int *ptr = kFwd ? a.tf_ptr : a.tb_ptr, *ind = kFwd ? a.tf_ind : a.tb_ind;
    const T *val = (const T *)(kFwd ? a.tf_val : a.tb_val);
    const T *vec = (const T *)(kFwd ? a.y : a.z);
    double rk[V], ap[V], xk[V], pk[V];
    T own[V];
    T dk = (T)0;
    if (s == 0) {
        if (kFwd) {
            dload<V>(a.r + o, rk);
            if (update_rx) {
                dload<V>(a.ap + o, ap);
                dload<V>(a.x + o, xk);
                dload<V>(p_cur + o, pk);
            }
        } else {
            vload<T, V>((const T *)a.y + o, own);
            dk = ((const T *)a.diag)[k];
        }
    }
    constexpr int B = 8;
    const int e1 = ptr[q + 1];
    for (int e = ptr[q] + s; e < e1; e += B * S) {
        int j[B];
        T l[B], w[B][V];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const bool in = e + u * S < e1;
            j[u] = in ? ind[e + u * S] : a.n;
            l[u] = in ? val[e + u * S] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < B; ++u) vload<T, V>(vec + (size_t)j[u] * K + q0, w[u]);
#pragma unroll
        for (int u = 0; u < B; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v] = fma_t(-l[u], w[u][v], acc[v]);
    }
    slot_sum<T, V>(acc, L, kWave);
    if (s != 0) return;
    if (kFwd) {
        if (update_rx) {
            double alpha[V];
#pragma unroll
            for (int v = 0; v < V; ++v) alpha[v] = (q0 + v < a.k && !sc->done[q0 + v]) ? sc->alpha[q0 + v] : 0.0;
            row_update<V>(a, o, alpha, rk, ap, pk, xk);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += (T)rk[v];
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += dk != (T)0 ? own[v] / dk : own[v];
    }
    vstore<T, V>(out, acc);
}

// Block blk's inverse times its right-hand sides.  A workgroup takes 16 rows x K
// columns of the result and kMTailCols columns of the triangle, dealt to eight
// waves; the last workgroup of a row tile to finish adds the tile's parts in
// order.  (Without the split over workgroups a 2048-row block of 64 right-hand
// sides took 23 us, bound by the product and load rate of the few CUs that hold
// the long rows.)
// FP32 in, FP32 accumulated (v_mfma_f32_16x16x4_f32), or FP64.  A lane loads 16
// bytes of its row of W, i.e. VK consecutive k; product j takes element j of
// every lane group, so its k are VK (l / 16) + j for both operands.
typedef float mf32x4 __attribute__((ext_vector_type(4)));
typedef double mf64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mf32x4 mtail_mfma(float x, float y, mf32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}
__device__ __forceinline__ mf64x4 mtail_mfma(double x, double y, mf64x4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0);
}
template <typename T> struct MAcc { typedef mf32x4 type; };
template <> struct MAcc<double> { typedef mf64x4 type; };

template <typename T, bool kFwd, int NT>
__global__ void __launch_bounds__(512) k_mtail_apply(MultiArgs a, int blk)
{
    constexpr int VK = 16 / (int)sizeof(T), KS = 4 * VK;      // k per lane, per wave step
    constexpr int NW = 8, kU = 4;
    static_assert(kMTailCols % (NW * KS * kU) == 0, "whole batches of loads");
    typedef typename MAcc<T>::type acc_t;
    __shared__ T part[NW][16][NT * 16];
    __shared__ int last;
    if (a.sc->all_done) return;
    const int m = a.tail_m, K = a.K;
    const int rows = min(m, a.ntail - blk * m);
    const int tile = blockIdx.x, i0 = tile * 16;
    const int c0 = kFwd ? 0 : i0, c1 = kFwd ? i0 + 16 : m;
    const int k0 = c0 + blockIdx.y * kMTailCols, k1 = min(c1, k0 + kMTailCols);
    if (k0 >= c1) return;
    const int parts = (c1 - c0 + kMTailCols - 1) / kMTailCols;
    const int t = threadIdx.x, lane = lane_id(), w = t / kWave;
    const int lr = lane % 16, lg = lane / 16;
    const T *W = (const T *)(kFwd ? a.tail_wf : a.tail_wb) + (size_t)blk * m * m + (size_t)(i0 + lr) * m;
    const T *B = (const T *)a.tacc;
    acc_t acc[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[c] = acc_t{(T)0, (T)0, (T)0, (T)0};
    for (int kb = k0 + w * KS; kb < k1; kb += kU * NW * KS) {
        T wv[kU][VK], bv[kU][VK][NT];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int k = kb + u * NW * KS;
            const bool in = k < k1;                   // steps past the end multiply zeros
            const int kk = in ? k : kb;
            vload<T, VK>(W + kk + lg * VK, wv[u]);
#pragma unroll
            for (int j = 0; j < VK; ++j) {
                wv[u][j] = in ? wv[u][j] : (T)0;
#pragma unroll
                for (int c = 0; c < NT; ++c) {
                    const int col = c * 16 + lr;
                    bv[u][j][c] = (in && col < K) ? B[(size_t)(kk + lg * VK + j) * K + col] : (T)0;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < VK; ++j)
#pragma unroll
                for (int c = 0; c < NT; ++c) acc[c] = mtail_mfma(wv[u][j], bv[u][j][c], acc[c]);
    }
    // result register q of lane l: FP32 row 4 (l / 16) + q, FP64 row 4 q + l / 16
#pragma unroll
    for (int c = 0; c < NT; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) part[w][sizeof(T) == 4 ? 4 * lg + q : 4 * q + lg][c * 16 + lr] = acc[c][q];
    __syncthreads();
    T *out = (T *)(kFwd ? a.y : a.z) + ((size_t)a.tail_pos0 + (size_t)blk * m + i0) * K;
    T *mine = (T *)a.tail_part + ((size_t)blockIdx.y * m + i0) * K;
    for (int e = t; e < 16 * K; e += 512) {
        const int i = e / K, c = e - i * K;
        T s = part[0][i][c];
#pragma unroll
        for (int p = 1; p < NW; ++p) s += part[p][i][c];
        if (parts > 1) st_relaxed_val(mine + e, s);
        else if (i0 + i < rows) out[e] = unsent(s);
    }
    if (parts == 1) return;
    drain_stores();                                   // every thread's part is visible before the arrival
    __syncthreads();
    if (t == 0) last = atomicAdd(a.tail_arrive + tile, 1u) == (unsigned int)(parts - 1);
    __syncthreads();
    if (!last) return;
    if (t == 0) a.tail_arrive[tile] = 0u;             // for the next launch
    const T *all = (const T *)a.tail_part + (size_t)i0 * K;
    for (int e = t; e < 16 * K; e += 512) {
        if (i0 + e / K >= rows) break;
        T s = ld_relaxed_val(all + e);
        for (int p = 1; p < parts; ++p) s += ld_relaxed_val(all + (size_t)p * m * K + e);
        out[e] = unsent(s);
    }
}

// Chunks of the sweeps: the rows of a level segment cut into runs of
// mchunk_rows(widest row) rows.
__device__ __forceinline__ int mchunk_rows(int width, int L)
{
    int S = 1;
    while (S * L < kWave && S * 8 < width) S <<= 1;
    const int by_threads = kMSweepThreads / (L * S), by_entries = kMChunkEntries / (8 * S);
    return by_threads < by_entries ? by_threads : by_entries;
}
__global__ void k_mchunk_count(int nseg, const int *seg_ptr, const int *width, int L, int *cnt)
{
    for (int g = blockIdx.x * blockDim.x + threadIdx.x; g < nseg; g += gridDim.x * blockDim.x) {
        const int r = mchunk_rows(width[g], L);
        cnt[g] = (seg_ptr[g + 1] - seg_ptr[g] + r - 1) / r;
    }
}
// cm[c] = {first row, rows, first entry, entries} of both sweeps
__global__ void k_mchunk_fill(int nchunks, int nseg, const int *seg_ptr, const int *chunk_ptr, const int *width, int L,
                              const int *l_ptr, const int *lt_ptr, int4 *cm_f, int4 *cm_b)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < nchunks; c += gridDim.x * blockDim.x) {
        int lo = 0, hi = nseg - 1;          // last segment with chunk_ptr <= c
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (chunk_ptr[mid] <= c) lo = mid; else hi = mid - 1;
        }
        const int r = mchunk_rows(width[lo], L);
        const int start = seg_ptr[lo] + (c - chunk_ptr[lo]) * r;
        const int cnt = min(r, seg_ptr[lo + 1] - start);
        cm_f[c] = make_int4(start, cnt, l_ptr[start], l_ptr[start + cnt] - l_ptr[start]);
        cm_b[c] = make_int4(start, cnt, lt_ptr[start], lt_ptr[start + cnt] - lt_ptr[start]);
    }
}

// ---------------------------------------------------------------- dots
template <typename T>
__global__ void __launch_bounds__(kMB) k_mdot(MultiArgs a, int init)
{
    __shared__ double red[kMB];
    __shared__ int flag;
    MultiScalars *sc = a.sc;
    if (sc->all_done) return;
    const int K = a.K;
    const int q = threadIdx.x % K;
    const int rows_per_block = kMB / K;
    const T *z = (const T *)a.z;
    const bool need_rr = sc->stop_rule == 1;
    double acc = 0.0, acc_rr = 0.0;
    for (int row = blockIdx.x * rows_per_block + threadIdx.x / K; row < a.n; row += gridDim.x * rows_per_block) {
        const size_t o = (size_t)row * K + q;
        const double ri = a.r[o];
        acc += ri * (double)z[o];
        if (need_rr) acc_rr += ri * ri;
    }
    const double s1 = msum(acc, K, red), s2 = need_rr ? msum(acc_rr, K, red) : 0.0;
    if ((int)threadIdx.x < K) {
        st_relaxed_val(a.partials + (size_t)blockIdx.x * K + threadIdx.x, s1);
        st_relaxed_val(a.partials + (size_t)(gridDim.x + blockIdx.x) * K + threadIdx.x, s2);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        drain_stores();
        unsigned int old = atomicAdd(&sc->arrive_dot, 1u);
        flag = old == gridDim.x - 1;
    }
    __syncthreads();
    if (!flag) return;
    const double rz = mfinal(a.partials, gridDim.x, K, red);
    const double rr = need_rr ? mfinal(a.partials + (size_t)gridDim.x * K, gridDim.x, K, red) : 0.0;
    if ((int)threadIdx.x < K) {
        const int qq = threadIdx.x;
        if (qq < a.k) {
            if (need_rr && !(!init && sc->done[qq])) sc->rr[qq] = rr;
            if (init) {
                sc->rz0[qq] = rz;
                sc->rz[qq] = rz;
                sc->beta[qq] = 0.0;
                sc->iter[qq] = 0;
                bool go = need_rr ? (sc->bb[qq] > 0.0 && sqrt(rr) / sqrt(sc->bb[qq]) > sc->tol) : (rz > sc->tol);
                sc->done[qq] = go ? 0 : 1;
            } else if (!sc->done[qq]) {
                sc->beta[qq] = rz / sc->rz[qq];
                sc->rz[qq] = rz;
                sc->iter[qq] += 1;
                bool go = need_rr ? (sqrt(rr) / sqrt(sc->bb[qq]) > sc->tol) : (sqrt(rz) / sqrt(sc->rz0[qq]) > sc->tol);
                if (!go || sc->iter[qq] >= sc->maxit) sc->done[qq] = 1;
            } else {
                sc->beta[qq] = 0.0;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 1;
        for (int qq = 0; qq < a.k; ++qq) all &= sc->done[qq] ? 1 : 0;
        if (sc->status != 0) all = 1;
        sc->all_done = all;
        sc->arrive_dot = 0u;
    }
}

// ||A x_q - b_q||^2 and ||b_q||^2 per q (solver.hpp:549-569)
__global__ void __launch_bounds__(kMB) k_mresidual(MultiArgs a, int bnorm_only)
{
    __shared__ double red[kMB];
    __shared__ int flag;
    MultiScalars *sc = a.sc;
    const int K = a.K;
    const int q = threadIdx.x % K;
    const int rows_per_block = kMB / K;
    double acc = 0.0, accb = 0.0;
    for (int row = blockIdx.x * rows_per_block + threadIdx.x / K; row < a.n; row += gridDim.x * rows_per_block) {
        const size_t o = (size_t)row * K + q;
        if (!bnorm_only) {
            double s = 0.0;
            for (int e = a.a_ptr[row]; e < a.a_ptr[row + 1]; ++e)
                s = fma_t(a.a_val[e], a.x[(size_t)a.a_ind[e] * K + q], s);
            double d = s - a.b[o];
            acc += d * d;
        }
        accb += a.b[o] * a.b[o];
    }
    const double s1 = msum(acc, K, red), s2 = msum(accb, K, red);
    if ((int)threadIdx.x < K) {
        st_relaxed_val(a.partials + (size_t)blockIdx.x * K + threadIdx.x, s1);
        st_relaxed_val(a.partials + (size_t)(gridDim.x + blockIdx.x) * K + threadIdx.x, s2);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        drain_stores();
        unsigned int old = atomicAdd(&sc->arrive_res, 1u);
        flag = old == gridDim.x - 1;
    }
    __syncthreads();
    if (!flag) return;
    const double r2 = mfinal(a.partials, gridDim.x, K, red);
    const double b2 = mfinal(a.partials + (size_t)gridDim.x * K, gridDim.x, K, red);
    if ((int)threadIdx.x < K) {
        const int qq = threadIdx.x;
        if (!bnorm_only) sc->res2[qq] = r2;
        sc->bb[qq] = b2;
        if (qq == 0) sc->arrive_res = 0u;
    }
}

template <typename T>
__global__ void k_mprepare(MultiArgs a)
{
    const size_t total = (size_t)(a.n + 1) * a.K;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const bool dummy = i >= (size_t)a.n * a.K;
        a.r[i] = dummy ? 0.0 : a.b[i];
        a.x[i] = 0.0;
        a.p0[i] = 0.0;
        a.p1[i] = 0.0;
        a.ap[i] = 0.0;
        ((T *)a.y)[i] = dummy ? (T)0 : sent_value(T());
        ((T *)a.z)[i] = dummy ? (T)0 : sent_value(T());
    }
    if (blockIdx.x == 0) reset_claims(a.ctr_fwd, a.ctr_bwd, threadIdx.x);
}

// b (positions, K-strided) from the user's column-major B (n x k):
// b[p*K + q] = B[q*n_user + idx_user[p]]
__global__ void k_mgather(const double *B, const int *idx_user, int n, int k, int K, double *b)
{
    const size_t total = (size_t)n * K;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int p = (int)(i / K), q = (int)(i % K);
        b[i] = q < k ? B[(size_t)q * n + idx_user[p]] : 0.0;
    }
}
__global__ void k_mscatter(const double *x, const int *idx_user, int n, int k, int K, double *X)
{
    const size_t total = (size_t)n * K;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int p = (int)(i / K), q = (int)(i % K);
        if (q < k) X[(size_t)q * n + idx_user[p]] = x[i];
    }
}

template <typename T, bool kFwd, int V>
void launch_msweep_v(const MultiArgs &a, const double *p_cur, int update_rx, hipStream_t s)
{
    auto bulk = [&]() {
        const int g = a.nchunks < a.sweep_blocks ? a.nchunks : a.sweep_blocks;
        if (g > 0)
            hipLaunchKernelGGL((k_msweep<T, kFwd, V>), dim3(g), dim3(kMSweepThreads), 0, s, a, p_cur, update_rx);
    };
    auto tail = [&](int b) {
        const int rows = a.ntail - b * a.tail_m < a.tail_m ? a.ntail - b * a.tail_m : a.tail_m;
        const dim3 gb((rows + 15) / 16, (a.tail_m + kMTailCols - 1) / kMTailCols);
        hipLaunchKernelGGL((k_mtail_rhs<T, kFwd, V>), dim3(a.tail_m / 4), dim3(256), 0, s, a, b, p_cur, update_rx);
        if (a.K <= 16) hipLaunchKernelGGL((k_mtail_apply<T, kFwd, 1>), gb, dim3(512), 0, s, a, b);
        else if (a.K == 32) hipLaunchKernelGGL((k_mtail_apply<T, kFwd, 2>), gb, dim3(512), 0, s, a, b);
        else hipLaunchKernelGGL((k_mtail_apply<T, kFwd, 4>), gb, dim3(512), 0, s, a, b);
    };
    if (kFwd) {
        bulk();
        for (int b = 0; b < a.tail_nb; ++b) tail(b);
    } else {
        for (int b = a.tail_nb - 1; b >= 0; --b) tail(b);
        bulk();
    }
}

// One sweep, V right-hand sides per lane.
template <typename T, bool kFwd>
void launch_msweep(const MultiArgs &a, const double *p_cur, int update_rx, hipStream_t s)
{
    const int V = multi_lane_rhs(a.K, (int)sizeof(T));
    if constexpr (sizeof(T) == 4) {
        if (V == 4) {
            launch_msweep_v<T, kFwd, 4>(a, p_cur, update_rx, s);
            return;
        }
    }
    if (V == 2) launch_msweep_v<T, kFwd, 2>(a, p_cur, update_rx, s);
    else launch_msweep_v<T, kFwd, 1>(a, p_cur, update_rx, s);
}

}  // namespace

void launch_mchunk_count(int nseg, const int *seg_ptr, const int *width, int L, int *cnt, hipStream_t s)
{
    hipLaunchKernelGGL(k_mchunk_count, dim3(256), dim3(256), 0, s, nseg, seg_ptr, width, L, cnt);
}
void launch_mchunk_fill(int nchunks, int nseg, const int *seg_ptr, const int *chunk_ptr, const int *width, int L,
                        const int *l_ptr, const int *lt_ptr, int4 *cm_f, int4 *cm_b, hipStream_t s)
{
    hipLaunchKernelGGL(k_mchunk_fill, dim3(1024), dim3(256), 0, s, nchunks, nseg, seg_ptr, chunk_ptr, width, L, l_ptr,
                       lt_ptr, cm_f, cm_b);
}

template <typename T>
void launch_multi_init(const MultiArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_mprepare<T>, dim3(2048), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_mresidual, dim3(mblocks(a)), dim3(kMB), 0, s, a, 1);
    launch_msweep<T, true>(a, (const double *)a.p0, 0, s);
    launch_msweep<T, false>(a, (const double *)nullptr, 0, s);
    hipLaunchKernelGGL(k_mdot<T>, dim3(mblocks(a)), dim3(kMB), 0, s, a, 1);
}

template <typename T>
void launch_multi_iteration(const MultiArgs &a, int parity, hipStream_t s)
{
    double *p_old = parity ? a.p1 : a.p0;
    double *p_new = parity ? a.p0 : a.p1;
    hipLaunchKernelGGL(k_mpupdate<T>, dim3(4096), dim3(256), 0, s, a, (const double *)p_old, p_new);
    hipLaunchKernelGGL(k_mspmv<T>, dim3(mblocks(a)), dim3(kMB), 0, s, a, (const double *)p_new);
    launch_msweep<T, true>(a, (const double *)p_new, 1, s);
    launch_msweep<T, false>(a, (const double *)nullptr, 0, s);
    hipLaunchKernelGGL(k_mdot<T>, dim3(mblocks(a)), dim3(kMB), 0, s, a, 0);
}

template <typename T>
__global__ void k_msentinel(T *v, size_t total)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x)
        v[i] = sent_value(T());
}

template <typename T>
void launch_multi_spmm_only(const MultiArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_mspmv<T>, dim3(mblocks(a)), dim3(kMB), 0, s, a, (const double *)a.p0);
}

template <typename T>
void launch_multi_fwd_only(const MultiArgs &a, hipStream_t s)
{
    launch_msweep<T, true>(a, (const double *)a.p0, 0, s);
}

template <typename T>
void launch_multi_bwd_only(const MultiArgs &a, hipStream_t s)
{
    launch_msweep<T, false>(a, (const double *)nullptr, 0, s);
}

template <typename T>
void launch_multi_sentinels(const MultiArgs &a, bool y, bool z, hipStream_t s)
{
    const size_t total = (size_t)a.n * a.K;         // the dummy row n keeps its zeros
    if (y) hipLaunchKernelGGL(k_msentinel<T>, dim3(2048), dim3(256), 0, s, (T *)a.y, total);
    if (z) hipLaunchKernelGGL(k_msentinel<T>, dim3(2048), dim3(256), 0, s, (T *)a.z, total);
}

void launch_multi_residual(const MultiArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_mresidual, dim3(mblocks(a)), dim3(kMB), 0, s, a, 0);
}

void launch_multi_gather(const double *B, const int *idx_user, int n, int k, int K, double *b, hipStream_t s)
{
    hipLaunchKernelGGL(k_mgather, dim3(2048), dim3(256), 0, s, B, idx_user, n, k, K, b);
}
void launch_multi_scatter(const double *x, const int *idx_user, int n, int k, int K, double *X, hipStream_t s)
{
    hipLaunchKernelGGL(k_mscatter, dim3(2048), dim3(256), 0, s, x, idx_user, n, k, K, X);
}

template void launch_multi_init<float>(const MultiArgs &, hipStream_t);
template void launch_multi_init<double>(const MultiArgs &, hipStream_t);
template void launch_multi_iteration<float>(const MultiArgs &, int, hipStream_t);
template void launch_multi_iteration<double>(const MultiArgs &, int, hipStream_t);
template void launch_multi_spmm_only<float>(const MultiArgs &, hipStream_t);
template void launch_multi_spmm_only<double>(const MultiArgs &, hipStream_t);
template void launch_multi_fwd_only<float>(const MultiArgs &, hipStream_t);
template void launch_multi_fwd_only<double>(const MultiArgs &, hipStream_t);
template void launch_multi_bwd_only<float>(const MultiArgs &, hipStream_t);
template void launch_multi_bwd_only<double>(const MultiArgs &, hipStream_t);
template void launch_multi_sentinels<float>(const MultiArgs &, bool, bool, hipStream_t);
template void launch_multi_sentinels<double>(const MultiArgs &, bool, bool, hipStream_t);

}  // namespace rc
