// factor.hip -- randomized elimination on gfx950, one round per DAG level.
//
// Semantics follow cpu_implementation/driver_local.cpp:302-707 and
// gpu_implementation/driver.cu:43-1302 (the reference's per-column step):
// gather the column's strict-lower entries and pending fill edges, merge
// duplicate rows (summing weight and multiplicity), sort by weight, take the
// forward cumulative sums C and S = C[d-1], and for every entry i < d-1 draw
// u in (0,1], pick the first j > i with C[j] - C[i] >= u (S - C[i]) and emit
// the fill edge (max, min, w_i (S - C[i]) / S) into column min; the factor
// column holds -w/S and the pivot is S.  The last column is never eliminated
// (driver.cu:184-197): it keeps count 0 and pivot 0.
//
// MI355X design:
//   * rounds: one launch eliminates every column made ready by the previous
//     launch (a wave64 per column, or per four where many are ready,
//     grid-stride over the round's list), so the kernel boundary orders all
//     communication -- no fences, no waits;
//   * gather, duplicate merge, sorts and the prefix sum run in LDS (global
//     per-workgroup scratch for columns above the LDS capacity); columns of more
//     than 128 entries, and of more than 64 where few are ready, are eliminated
//     by eight waves;
//   * the sampling draw is Philox4x32-10 keyed by (seed, i, column): with the
//     canonical (row, weight) merge order and (weight, row) sampling order the
//     factor is a pure function of (matrix, seed), independent of schedule;
//   * each neighbour's dependency counter gets ONE atomic add of
//     (new fills with it as the larger end) - (retired multiplicity); the
//     column whose add reaches zero appends the neighbour to the next round's
//     list with one wave-aggregated atomic;
//   * a column's pending fill records hang off kFillLists linked lists
//     (record index mod kFillLists), so its gather walks them in lockstep,
//     one lane per list, instead of chasing one long chain;
//   * fill records and factor entries are carved from per-wave chunks of two
//     global pools, so pool counters see one atomic per few thousand entries;
//   * pool or scratch exhaustion raises a status bit, later rounds drain, and
//     the host regrows and reruns (same result).
#include "common.cuh"
#include "kernels.h"

namespace rc {

namespace {

constexpr int kLdsCap = 128;                                   // entries per wave in LDS (round kernel)
static_assert(kLdsCap <= 2 * 64, "the round kernel sorts two entries per lane");
constexpr int kBytesPerEntry = 16 + 8 + 8 + 4 + 4 + 4 + 4;  // s mw C mrow mmult minc jt
// global scratch of a column above kBigCap entries: the column buffer, the
// sorts' second entry array, and eight bytes per 64 entries (one an entry is
// more than that) for the scan's block sums
constexpr int kScratchBytesPerEntry = kBytesPerEntry + 16 + 1;
constexpr long long kFillChunk = 2048;
constexpr long long kOutChunk = 2048;

// An entry being sorted: row, payload (multiplicity, later the merged index)
// and weight in one 16-byte record, so a comparator moves two records with
// one LDS instruction each instead of six.
struct __attribute__((aligned(16))) SEnt {
    int row;
    int pay;
    double w;
};

// A pointer of the argument block, known to be device memory: the block itself
// is read from memory, and without this its pointers would be dereferenced with
// flat accesses, which occupy the LDS queue as well.
template <typename T>
using Global = __attribute__((address_space(1))) T;
template <typename T>
__device__ __forceinline__ Global<T> *gp(T *p)
{
    return (Global<T> *)p;
}
// ... and as an operand of an atomic (global still, as the compiler sees where
// it comes from)
template <typename T>
__device__ __forceinline__ T *at(Global<T> *p)
{
    return (T *)p;
}

struct ColBuf {
    SEnt *s;
    double *mw, *C;
    int *mrow, *mmult, *minc, *jt;   // jt: sampled partner of every fill
};

__device__ __forceinline__ ColBuf carve(char *base, int cap)
{
    ColBuf b;
    b.s = reinterpret_cast<SEnt *>(base);
    b.mw = reinterpret_cast<double *>(b.s + cap);
    b.C = b.mw + cap;
    b.mrow = reinterpret_cast<int *>(b.C + cap);
    b.mmult = b.mrow + cap;
    b.minc = b.mmult + cap;
    b.jt = b.minc + cap;
    return b;
}

__device__ __forceinline__ int next_pow2(int v)
{
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

// Orders the accesses of one wave's lanes among each other (they are executed in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int kWaves>
__device__ __forceinline__ void sync_waves()
{
    if constexpr (kWaves == 1) wave_fence();
    else __syncthreads();
}

// The sorts place an entry by counting those before it, in the order (row, w) or
// (w, row): entries are compared against one broadcast entry at a time, with
// independent reads, where a network is a chain of shuffles (64 entries: 5.0 us
// for the network's 21 stages).  Equal entries (unit weights) go by their
// index.  A weight that is not a number counts as infinity, so that every place
// is taken once whatever the weights.
__device__ __forceinline__ double sort_key(double w) { return w != w ? __builtin_inf() : w; }
template <bool kByRow>
__device__ __forceinline__ bool ent_before(int xr, double xw, int vr, double vw, bool tie)
{
    const bool lr = xr < vr, er = xr == vr, lw = xw < vw, ew = xw == vw;    // no branches
    return kByRow ? lr | (er & (lw | (ew & tie))) : lw | (ew & (lr | (er & tie)));
}

constexpr int kCountBatch = 8;
// For entry index i (key vr, vw): entries among e[j0..j1) that come before it.
// Weights in e are sort keys.
template <bool kByRow, int R>
__device__ __forceinline__ void count_before(const SEnt *e, int j0, int j1, const int (&i)[R], const int (&vr)[R],
                                             const double (&vw)[R], int (&c)[R])
{
    for (; j0 < j1; j0 += kCountBatch) {
        SEnt x[kCountBatch];
#pragma unroll
        for (int u = 0; u < kCountBatch; ++u) x[u] = e[min(j0 + u, j1 - 1)];
#pragma unroll
        for (int u = 0; u < kCountBatch; ++u)
#pragma unroll
            for (int s = 0; s < R; ++s)
                c[s] += (j0 + u < j1) & ent_before<kByRow>(x[u].row, x[u].w, vr[s], vw[s], j0 + u < i[s]);
    }
}

// Sorts e[0..len) by one wave, len <= 64 R, the payload travelling along.
template <bool kByRow, int R>
__device__ __forceinline__ void wave_sort(SEnt *e, int len)
{
    const int lane = lane_id();
    SEnt v[R];
    int i[R], row[R], c[R];
    double key[R];
#pragma unroll
    for (int s = 0; s < R; ++s) {
        i[s] = s * kWave + lane;
        v[s] = e[min(i[s], len - 1)];
        row[s] = v[s].row;
        key[s] = sort_key(v[s].w);
        c[s] = 0;
        if (v[s].w != v[s].w && i[s] < len) e[i[s]].w = key[s];
    }
    wave_fence();
    count_before<kByRow, R>(e, 0, len, i, row, key, c);
    wave_fence();
#pragma unroll
    for (int s = 0; s < R; ++s)
        if (i[s] < len) e[c[s]] = v[s];
    wave_fence();
}

__device__ __forceinline__ void raise_status(unsigned long long *ctr, unsigned long long bits)
{
    atomicOr(&ctr[kCtrStatus], bits);
}

struct Cursor {
    long long cur, end;
};

// Wave-uniform carve of `count` entries from a per-wave chunk of a pool.
__device__ __forceinline__ bool carve_pool(Cursor &c, long long count, long long chunk, unsigned long long *top,
                                           long long cap, long long &base)
{
    if (c.cur + count > c.end) {
        long long size = count > chunk ? count : chunk;
        long long b = 0;
        if (lane_id() == 0) b = (long long)atomicAdd(top, (unsigned long long)size);
        b = bcast(b, 0);
        if (b + size > cap) return false;
        c.cur = b;
        c.end = b + size;
    }
    base = c.cur;
    c.cur += count;
    return true;
}

// ---- segmented ready lists ------------------------------------------------
__device__ __forceinline__ unsigned int *list_set(const FactorArgs &a, int round)
{
    return a.seg_count + (size_t)(round % 3) * kListSlots;
}

// Lane q: effective entry count c of slot q of a list and the inclusive
// prefix over slots; the list's length is the prefix at lane 63.
__device__ __forceinline__ void list_counts(const FactorArgs &a, const unsigned int *set, unsigned int &c,
                                            unsigned int &incl)
{
    const int lane = lane_id();
    const unsigned int v = set[lane];
    c = lane < kListSegs ? min(v, (unsigned int)a.seg_cap) : v;
    incl = c;
    for (int off = 1; off < kWave; off <<= 1) {
        const unsigned int o = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += o;
    }
}

// Storage index of entry i (wave-uniform, below the length) of a list.
__device__ __forceinline__ size_t list_index(const FactorArgs &a, unsigned int c, unsigned int incl, unsigned int i)
{
    const int s = __popcll(ballot(incl <= i));          // slots wholly before entry i
    const unsigned int excl = __shfl(incl - c, s, kWave);
    return (size_t)s * (size_t)a.seg_cap + (i - excl);
}

// Appends `value` of every lane with `ready` to the list of counter set `set`:
// one atomic on this workgroup's segment counter, and one on the overflow
// counter for entries past the segment's capacity.
__device__ __forceinline__ void list_append(const FactorArgs &a, unsigned int *set, int *list, bool ready, int value)
{
    const uint64_t mask = ballot(ready);
    if (!mask) return;
    const unsigned int cnt = (unsigned int)__popcll(mask);
    const unsigned int cap = (unsigned int)a.seg_cap;
    const int seg = (int)(blockIdx.x % kListSegs);
    unsigned int base = 0;
    if (lane_id() == 0) base = atomicAdd(at(gp(set) + seg), cnt);
    base = bcast(base, 0);
    const unsigned int pos = base + (unsigned int)lanes_below(mask);
    if (base + cnt > cap) {
        const unsigned int lo = base > cap ? base : cap;
        unsigned int ob = 0;
        if (lane_id() == 0) ob = atomicAdd(&set[kListSegs], base + cnt - lo);
        ob = bcast(ob, 0);
        if (ready && pos >= cap) gp(list)[(size_t)kListSegs * cap + ob + (pos - lo)] = value;
    }
    if (ready && pos < cap) gp(list)[(size_t)seg * cap + pos] = value;
}

// A fill record through agent-scope accesses (two words of 8 bytes).
__device__ __forceinline__ FillRec load_record(const FillRec *p)
{
    const unsigned long long *q = reinterpret_cast<const unsigned long long *>(p);
    const unsigned long long rn = ld_relaxed(q), w = ld_relaxed(q + 1);
    FillRec r;
    r.row = (int)(unsigned int)rn;
    r.next = (int)(unsigned int)(rn >> 32);
    r.w = __longlong_as_double((long long)w);
    return r;
}
__device__ __forceinline__ void store_record(FillRec *p, const FillRec &r)
{
    unsigned long long *q = reinterpret_cast<unsigned long long *>(p);
    st_relaxed(q, ((unsigned long long)(unsigned int)r.next << 32) | (unsigned int)r.row);
    st_relaxed(q + 1, (unsigned long long)__double_as_longlong(r.w));
}

// Gathers column k: its strict-lower entries ...
__device__ __forceinline__ void gather_original(const FactorArgs &a, int lo0, int norig, const ColBuf &b, int cap, int t,
                                                int nt)
{
    for (; t < norig && t < cap; t += nt) {
        SEnt v;
        v.row = gp(a.lo_row)[lo0 + t];
        v.pay = 1;
        v.w = gp(a.lo_w)[lo0 + t];
        b.s[t] = v;
    }
}
// ... and its pending fills (kFillLists linked lists, walked in lockstep by one
// wave, one lane per list; f = this lane's list head), writing the first `cap`
// entries; returns the total count, or with kStopOverCap any count above `cap`
// as soon as one is reached (the column is then handed on without walking the
// rest of its lists).  kCoherent (queue-driven kernel): records written by
// running waves of the same launch are read with agent-scope loads.  The order
// of the gathered entries does not matter: the (row, weight) sort makes it canonical.
template <bool kStopOverCap, bool kCoherent>
__device__ __forceinline__ int gather_fills(const FactorArgs &a, int norig, int f, const ColBuf &b, int cap)
{
    int t = norig;
    while (true) {
        if (kStopOverCap && t > cap) break;
        const bool act = f >= 0;
        const uint64_t mask = ballot(act);
        if (!mask) break;
        if (act) {
            const FillRec rec = kCoherent ? load_record(at(gp(a.pool) + f)) : *at(gp(a.pool) + f);
            const int pos = t + lanes_below(mask);
            if (pos < cap) {
                SEnt v;
                v.row = rec.row;
                v.pay = 1;
                v.w = rec.w;
                b.s[pos] = v;
            }
            f = rec.next;
        }
        t += __popcll(mask);
    }
    return t;
}

// A run of one row in the (row, weight) order starting at entry i: summed left
// to right (ascending weight), kRun records per LDS round trip.
constexpr int kRun = 8;
struct RowRun {
    bool head;
    int row, mult;
    double w;
};
__device__ __forceinline__ RowRun row_run(const SEnt *s, int i, int m)
{
    RowRun r;
    const SEnt first = s[i];
    r.row = first.row;
    r.head = i == 0 || s[i - 1].row != first.row;
    r.mult = first.pay;
    r.w = first.w;
    if (r.head) {
        bool more = true;
        for (int t0 = i + 1; more; t0 += kRun) {
            SEnt x[kRun];
#pragma unroll
            for (int u = 0; u < kRun; ++u) x[u] = s[t0 + u < m ? t0 + u : m - 1];
#pragma unroll
            for (int u = 0; u < kRun; ++u) {
                more = more && t0 + u < m && x[u].row == r.row;
                if (more) {
                    r.w += x[u].w;
                    r.mult += x[u].pay;
                }
            }
        }
    }
    return r;
}
__device__ __forceinline__ void put_merged(const ColBuf &b, int pos, const RowRun &r)
{
    b.mrow[pos] = r.row;
    b.mw[pos] = r.w;
    b.mmult[pos] = r.mult;
    b.minc[pos] = 0;
}
__device__ __forceinline__ SEnt merged_entry(const ColBuf &b, int i)
{
    SEnt v;
    v.row = b.mrow[i];
    v.pay = i;
    v.w = b.mw[i];
    return v;
}

// Doubling scan of 64 values, one per lane (each step from the previous step's
// values).
__device__ __forceinline__ double block_scan64(double x)
{
    const int lane = lane_id();
    for (int off = 1; off < kWave; off <<= 1) {
        const double o = __shfl_up(x, off, kWave);
        if (lane >= off) x = x + o;
    }
    return x;
}

// Partner j of fill i and the new dependency of the larger row (:598-631; gpu
// auxilliary.hpp:543-592).
__device__ __forceinline__ void sample_partner(const FactorArgs &a, int k, const ColBuf &b, int i, int d, double S)
{
    const double u = sample_uniform(a.seed, (uint32_t)i, (uint32_t)k);
    const double Ci = b.C[i];
    const double rest = S - Ci;
    const double tgt = u * rest;
    int lo = i + 1, hi = d - 1;
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (b.C[mid] - Ci < tgt) lo = mid + 1; else hi = mid;
    }
    b.jt[i] = lo;
    const SEnt ei = b.s[i], el = b.s[lo];
    atomicAdd(&b.minc[ei.row > el.row ? ei.pay : el.pay], 1);   // the larger row gains a dependency
}

// Pushes fill e as record rec onto its column's lists; returns the old head.
__device__ __forceinline__ int push_head(const FactorArgs &a, const ColBuf &b, int e, int rec)
{
    const int ri = b.s[e].row, rj = b.s[b.jt[e]].row;
    const int c = ri > rj ? rj : ri;
    return atomicExch(at(&gp(a.head)[(size_t)c * kFillLists + (rec & (kFillLists - 1))]), rec);
}
__device__ __forceinline__ FillRec fill_record(const ColBuf &b, int e, double S, int next)
{
    const SEnt se = b.s[e];
    const int ri = se.row, rj = b.s[b.jt[e]].row;
    FillRec fr;
    fr.row = ri > rj ? ri : rj;
    fr.next = next;
    fr.w = (se.w * (S - b.C[e])) / S;
    return fr;
}

// ---- columns by a whole workgroup -------------------------------------------
// The large-LDS kernels (deferred columns, narrow rounds, the queue-driven
// rest) run one workgroup per CU, and their time is the latency of one column
// after the other.  The first wave takes the columns and eliminates those of at
// most kWave entries by itself, without a barrier; for a larger one all kWgWaves
// waves work together.  One wave with sorting networks took 14 us for up to 64
// entries, 30 us for 129-256 and 45 us for 257-512, two thirds of it sorting;
// the queue-driven rest of a 192^3 grid (learned order) took 26 ms that way and
// takes 15.7 ms, its whole factorization 58.5 and 47.4 ms (101 x 83 x 89: 18.9
// and 14.2 ms; 64^2: 0.76 and 0.70 ms).
constexpr int kWgWaves = 8;
constexpr int kWgThreads = kWgWaves * kWave;

struct WgShared {
    int k;                             // the large column (< 0: the end)
    int m;                             // its gathered entries
    int round;                         // its level
    int ok;                            // pools not exhausted
    int cnt[kWgWaves];                 // merged rows per wave
    long long fbase, obase;            // its pool entries
    double tot[kBigCap / kWave];       // block sums of the scan
};

// Sorts e[0..m) by the workgroup with tmp[0..m) as the second array; returns
// the array that holds the result.  Up to kCountMax entries, every wave counts
// over its share of them and the shares are added.  Above, a wave sorts
// 64-entry runs; within groups of kGroup runs an entry's place is then its place
// in its run plus the number of smaller entries in every other run (bisections,
// kPar at a time: one pass where pairwise merges take three), and groups are
// merged in pairs.  The second weight sort has distinct rows and the runs are
// compared in index order, so equal entries keep their order throughout.
constexpr int kCountMax = 2 * kWave;
template <bool kByRow>
__device__ __forceinline__ SEnt *wg_sort(SEnt *e, SEnt *tmp, int m)
{
    constexpr int kPar = 4, kGroup = 8;
    const int lane = lane_id(), w = threadIdx.x / kWave;
    if (m <= kCountMax) {
        const int parts = m <= kWave ? kWgWaves : kWgWaves / 2;
        const int share = (m + parts - 1) / parts;
        const int part = w % parts;
        const int i[1] = {w / parts * kWave + lane};
        const SEnt v = e[min(i[0], m - 1)];
        const int row[1] = {v.row};
        const double key[1] = {sort_key(v.w)};
        int c[1] = {0};
        int *cnt = reinterpret_cast<int *>(tmp);          // per wave and lane
        __syncthreads();
        if (v.w != v.w && part == 0 && i[0] < m) e[i[0]].w = key[0];
        __syncthreads();
        count_before<kByRow, 1>(e, part * share, min(part * share + share, m), i, row, key, c);
        cnt[w * kWave + lane] = c[0];
        __syncthreads();
        if (part == 0 && i[0] < m) {
            int rank = 0;
            for (int p = 0; p < parts; ++p) rank += cnt[(w + p) * kWave + lane];
            e[rank] = v;
        }
        __syncthreads();
        return e;
    }
    const int nr = (m + kWave - 1) / kWave;
    for (int r = w; r < nr; r += kWgWaves) wave_sort<kByRow, 1>(e + r * kWave, min(m - r * kWave, kWave));
    __syncthreads();
    for (int r = w; r < nr; r += kWgWaves) {
        const int i = r * kWave + lane;
        if (i < m) {
            const SEnt v = e[i];
            const double key = sort_key(v.w);
            const int g0 = r / kGroup * kGroup, g1 = min(g0 + kGroup, nr);
            int rank = g0 * kWave + lane;
            for (int q0 = g0; q0 < g1; q0 += kPar) {
                int lo[kPar], hi[kPar];
#pragma unroll
                for (int u = 0; u < kPar; ++u) {
                    const int q = q0 + u;
                    lo[u] = 0;
                    hi[u] = q < g1 && q != r ? min(m - q * kWave, kWave) : 0;
                }
                for (int step = 0; step < 7; ++step) {    // 65 possible counts
                    SEnt x[kPar];
                    int mid[kPar];
#pragma unroll
                    for (int u = 0; u < kPar; ++u) {
                        mid[u] = (lo[u] + hi[u]) >> 1;
                        const int at = (q0 + u) * kWave + mid[u];
                        x[u] = e[at < m ? at : 0];
                    }
#pragma unroll
                    for (int u = 0; u < kPar; ++u)
                        if (lo[u] < hi[u]) {
                            const bool before = ent_before<kByRow>(x[u].row, sort_key(x[u].w), v.row, key, q0 + u < r);
                            lo[u] = before ? mid[u] + 1 : lo[u];
                            hi[u] = before ? hi[u] : mid[u];
                        }
                }
#pragma unroll
                for (int u = 0; u < kPar; ++u) rank += lo[u];
            }
            tmp[rank] = v;
        }
    }
    __syncthreads();
    SEnt *src = tmp, *dst = e;
    for (int len = kGroup * kWave; len < m; len *= 2) {
        for (int base = 0; base < m; base += kWgThreads) {
            const int i = base + (int)threadIdx.x;
            if (i >= m) continue;
            const SEnt v = src[i];
            const double key = sort_key(v.w);
            const int block = i / len * len;
            const bool second = (i / len) & 1;
            const int p0 = second ? block - len : block + len;   // the partner's first entry
            int lo = 0, hi = max(0, min(m - p0, len));
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                const SEnt x = src[p0 + mid];
                if (ent_before<kByRow>(x.row, sort_key(x.w), v.row, key, second)) lo = mid + 1;
                else hi = mid;
            }
            dst[i - block + (second ? p0 : block) + lo] = v;
        }
        __syncthreads();
        SEnt *s = src;
        src = dst;
        dst = s;
    }
    return src;
}

// Steps 2-5 of a column whose m >= 1 entries are gathered in b, by kWaves waves;
// one wave: m <= 64 R.  tmp (m entries) and tot (a double per 64 entries): only
// for more than one wave.  The cursors are the first wave's.  Returns false if
// the pools are exhausted (status set).
template <bool kAsync, int kWaves, int R>
__device__ __forceinline__ bool process_column(const FactorArgs &a, WgShared *sh, int k, int round, const ColBuf &b,
                                               SEnt *tmp, double *tot, int m, Cursor &fcur, Cursor &ocur, int *next,
                                               unsigned int *next_set)
{
    constexpr int kT = kWaves * kWave;
    const int lane = lane_id(), w = kWaves == 1 ? 0 : threadIdx.x / kWave;
    const int t = w * kWave + lane;
    const int last = a.n - 1;
    // ---- 2. sort by (row, w); merge duplicates left to right (:520-560)
    const SEnt *rs = b.s;
    if constexpr (kWaves > 1) {
        rs = wg_sort<true>(b.s, tmp, m);
    } else {
        if (R == 1 || m <= kWave) wave_sort<true, 1>(b.s, m);
        else wave_sort<true, R>(b.s, m);
    }
    int d = 0;
    for (int base = 0; base < m; base += kT) {
        const int i = base + t;
        RowRun run;
        run.head = false;
        if (i < m) run = row_run(rs, i, m);
        const uint64_t mask = ballot(run.head);
        int off = d, all = __popcll(mask);
        if constexpr (kWaves > 1) {
            if (lane == 0) sh->cnt[w] = all;
            __syncthreads();
            all = 0;
            for (int q = 0; q < kWaves; ++q) {
                const int c = sh->cnt[q];
                off += q < w ? c : 0;
                all += c;
            }
        }
        if (run.head) put_merged(b, off + lanes_below(mask), run);
        d += all;
        sync_waves<kWaves>();
    }

    // ---- 3. sort merged entries by (w, row), carrying the merged index;
    //         forward cumulative sums (:573-593)
    for (int i = t; i < d; i += kT) b.s[i] = merged_entry(b, i);
    sync_waves<kWaves>();
    if constexpr (kWaves > 1) {
        const SEnt *vs = wg_sort<false>(b.s, tmp, d);
        if (vs != b.s) {
            for (int i = t; i < d; i += kT) b.s[i] = vs[i];
            __syncthreads();
        }
    } else {
        if (R == 1 || d <= kWave) wave_sort<false, 1>(b.s, d);
        else wave_sort<false, R>(b.s, d);
    }
    // canonical blocked scan (shared with the oracle): per 64-entry block the
    // doubling scan x_i += x_{i-off}, off = 1..32, then the previous block's
    // last sum is added
    if constexpr (kWaves > 1) {
        // the blocks by all waves, the sums before each by one thread
        for (int q = w; q * kWave < d; q += kWaves) {
            const int i = q * kWave + lane;
            const double x = block_scan64(i < d ? b.s[i].w : 0.0);
            if (i < d) b.C[i] = x;
            if (lane == kWave - 1) tot[q] = x;
        }
        __syncthreads();
        if (d > kWave) {
            if (t == 0) {
                double carry = tot[0];
                for (int q = 1; q * kWave < d; ++q) {
                    const double x = tot[q];
                    tot[q] = carry;
                    carry = carry + x;
                }
            }
            __syncthreads();
            for (int i = kWave + t; i < d; i += kT) b.C[i] = tot[i / kWave] + b.C[i];
            __syncthreads();
        }
    } else {
        double carry = 0.0;
        for (int base = 0; base < d; base += kWave) {
            const int i = base + lane;
            const double x = block_scan64(i < d ? b.s[i].w : 0.0);
            const double c = base == 0 ? x : carry + x;
            if (i < d) b.C[i] = c;
            carry = __shfl(c, kWave - 1, kWave);
        }
        wave_fence();
    }
    const double S = b.C[d - 1];

    // ---- 4. sampled partners
    const int nfill_out = d - 1;
    for (int i = t; i < nfill_out; i += kT) sample_partner(a, k, b, i, d, S);
    long long fbase = 0, obase = 0;
    bool ok = true;
    if (w == 0) {
        if (nfill_out > 0 && !carve_pool(fcur, nfill_out, kFillChunk, &a.ctr[kCtrFillTop], a.pool_cap, fbase)) {
            if (lane == 0) raise_status(a.ctr, kStatusFillPool);
            ok = false;
        }
        if (ok && !carve_pool(ocur, d, kOutChunk, &a.ctr[kCtrOutTop], a.out_cap, obase)) {
            if (lane == 0) raise_status(a.ctr, kStatusOutPool);
            ok = false;
        }
        if (ok && lane == 0) {
            // a column is eliminated in the round after its last dependency, so
            // its level in the triangular-solve DAG is its round (:638-645); the
            // queue-driven levels come from atomicMax
            if (!kAsync) gp(a.level)[k] = round;
            gp(a.out_start)[k] = obase;
            gp(a.out_cnt)[k] = d;
            gp(a.diag)[k] = S;
        }
        if (kWaves > 1 && lane == 0) {
            sh->fbase = fbase;
            sh->obase = obase;
            sh->ok = ok;
        }
    }
    sync_waves<kWaves>();   // minc and jt complete
    if constexpr (kWaves > 1) {
        fbase = sh->fbase;
        obase = sh->obase;
        ok = sh->ok != 0;
    }
    if (!ok) return false;

    // ---- 5. per entry: the neighbour's net dependency update (:653-687), the
    //         fill edge (max, min, w_i (S - C_i) / S) pushed onto column min's
    //         lists, and the factor entry -w/S in row order.  In a round the
    //         column's returning atomics (list-head exchanges, dependency adds)
    //         are all in flight at once: nothing orders them but the kernel
    //         boundary.  Queue-driven: every push and raised level is complete
    //         before any dependency add (a neighbour may be taken by another
    //         workgroup as soon as its count reaches zero); they are agent-scope
    //         accesses, so the wait alone makes them visible, and factor
    //         entries are read by later launches only.
    constexpr int kB = kWaves == 1 ? R : 4;
    for (int sb = 0; sb < d; sb += kB * kT) {
        int old[kB], r[kB], nd[kB];
        bool upd[kB];
#pragma unroll
        for (int u = 0; u < kB; ++u) {
            const int e = sb + u * kT + t;
            old[u] = -1;
            r[u] = -1;
            upd[u] = false;
            nd[u] = 1;
            if (e < nfill_out) old[u] = push_head(a, b, e, (int)(fbase + e));
            if (!kAsync && e < d) {
                r[u] = b.mrow[e];
                const int delta = b.minc[e] - b.mmult[e];
                upd[u] = r[u] != last && delta != 0;
                if (upd[u]) nd[u] = atomicAdd(at(&gp(a.dep)[r[u]]), delta) + delta;
            }
        }
#pragma unroll
        for (int u = 0; u < kB; ++u) {
            const int e = sb + u * kT + t;
            if (e < d) {
                const int rr = b.mrow[e];
                gp(a.out_row)[obase + e] = rr;
                gp(a.out_val)[obase + e] = -(b.mw[e] / S);
                if (kAsync && rr != last) atomicMax(at(&gp(a.level)[rr]), round + 1);
            }
            if (e < nfill_out) {
                const FillRec fr = fill_record(b, e, S, old[u]);
                if (kAsync) store_record(at(gp(a.pool) + (int)(fbase + e)), fr);
                else *at(gp(a.pool) + (int)(fbase + e)) = fr;
            }
        }
        if constexpr (!kAsync) {
#pragma unroll
            for (int u = 0; u < kB; ++u) list_append(a, next_set, next, upd[u] && nd[u] == 0, r[u]);
        }
    }
    if constexpr (kAsync) {
        drain_stores();
        sync_waves<kWaves>();
        for (int sb = 0; sb < d; sb += kB * kT) {
            int r[kB], nd[kB];
            bool upd[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                const int e = sb + u * kT + t;
                r[u] = -1;
                upd[u] = false;
                nd[u] = 1;
                if (e < d) {
                    r[u] = b.mrow[e];
                    const int delta = b.minc[e] - b.mmult[e];
                    upd[u] = r[u] != last && delta != 0;
                    if (upd[u]) nd[u] = atomicAdd(at(&gp(a.dep)[r[u]]), delta) + delta;
                }
            }
            // the ready neighbours of this wave, one queue atomic for all
            unsigned int cnt = 0;
            uint64_t mk[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                mk[u] = ballot(upd[u] && nd[u] == 0);
                cnt += (unsigned int)__popcll(mk[u]);
            }
            if (cnt) {
                unsigned int qb = 0;
                if (lane == 0) qb = atomicAdd(at(gp(a.aq_ctr) + kAqTail), cnt);
                qb = bcast(qb, 0);
#pragma unroll
                for (int u = 0; u < kB; ++u) {
                    // every remaining column is queued once: a slot past the
                    // queue's end means inconsistent dependency counts
                    const bool ready = (mk[u] >> lane) & 1ull;
                    const unsigned int slot = qb + (unsigned int)lanes_below(mk[u]);
                    if (ready && slot < a.aq_total) st_relaxed(at(gp(next) + slot), r[u]);
                    if (ready && slot >= a.aq_total) raise_status(a.ctr, kStatusInconsistent);
                    qb += (unsigned int)__popcll(mk[u]);
                }
            }
        }
    }
    sync_waves<kWaves>();
    return true;
}

// A column without entries: zero pivot (driver_local.cpp:491-498).  One lane.
template <bool kAsync>
__device__ __forceinline__ void empty_column(const FactorArgs &a, int k, int round)
{
    if (!kAsync) gp(a.level)[k] = round;
    gp(a.out_start)[k] = 0;
    gp(a.out_cnt)[k] = 0;
    gp(a.diag)[k] = 0.0;
}

// Eliminates column k in the round kernel; newly ready neighbours are appended
// to `next`.  A column larger than the LDS buffer is appended to the round's
// deferred list.  Returns false if the pools are exhausted (status set).
__device__ __forceinline__ bool eliminate_column(const FactorArgs &a, int k, int round, char *lds, Cursor &fcur,
                                                 Cursor &ocur, int *next, unsigned int *next_set,
                                                 unsigned int *defer_count)
{
    const int lane = lane_id();
    // the list heads do not depend on the column's slice: one memory trip for both
    const int f0 = gp(a.head)[(size_t)k * kFillLists + lane];
    const int lo0 = gp(a.lo_ptr)[k];
    const int norig = gp(a.lo_ptr)[k + 1] - lo0;
    // ---- 1. gather (driver_local.cpp:459-487; cpu auxilliary.hpp:89-173);
    // the entries are counted as they come (no fill counter is kept)
    const ColBuf b = carve(lds, kLdsCap);
    gather_original(a, lo0, norig, b, kLdsCap, lane, kWave);
    const int m = gather_fills<true, false>(a, norig, f0, b, kLdsCap);
    wave_fence();
    if (m == 0) {
        if (lane == 0) empty_column<false>(a, k, round);
        return true;
    }
    if (m > kLdsCap) {                 // the round's large-LDS kernel takes it
        if (lane == 0) gp(a.big_list)[atomicAdd(defer_count, 1u)] = k;
        return true;
    }
    return process_column<false, 1, kLdsCap / kWave>(a, nullptr, k, round, b, nullptr, nullptr, m, fcur,
                                                     ocur, next, next_set);
}

// ---- several small columns per wave -------------------------------------------
// The first rounds of a large matrix hold hundreds of thousands of columns of a
// few entries each; one wave per column leaves most lanes idle and is bound by
// the column's chain of memory trips times the waves in flight.  Here a wave
// eliminates kPack columns at a time, kPackLanes lanes (and entries) each:
// the first round of a 192^3 grid (learned order) 2.9 -> 1.4 ms, its first
// twenty 18.6 -> 10.3 ms.  Four waves per SIMD (125 registers) issue most of the
// time: reading the next columns' lists ahead gained nothing, a fifth wave by
// spilling lost 3 %.
constexpr int kPackLanes = 16;
constexpr int kPack = kWave / kPackLanes;

// Sorts a group's b.s[0..len) (wave_sort, by kPackLanes lanes).
template <bool kByRow>
__device__ __forceinline__ void pack_sort(const ColBuf &b, int gl, int len)
{
    SEnt v;
    v.row = 0;
    v.pay = 0;
    v.w = 0.0;
    if (gl < len) v = b.s[gl];
    const double key = sort_key(v.w);
    if (v.w != v.w && gl < len) b.s[gl].w = key;
    wave_fence();
    int c = 0;
#pragma unroll
    for (int j0 = 0; j0 < kPackLanes; j0 += kCountBatch) {
        if (ballot(j0 < len) == 0ull) break;
        SEnt x[kCountBatch];
#pragma unroll
        for (int u = 0; u < kCountBatch; ++u) x[u] = b.s[j0 + u];
#pragma unroll
        for (int u = 0; u < kCountBatch; ++u)
            c += (j0 + u < len) & ent_before<kByRow>(x[u].row, x[u].w, v.row, key, j0 + u < gl);
    }
    wave_fence();
    if (gl < len) b.s[c] = v;
    wave_fence();
}

// Eliminates the groups' columns (k: this lane's group's, < 0: none) with
// entries in b.  over: a lane of every group whose column has more than
// kPackLanes entries (left as it was).  Returns false if the pools are exhausted.
__device__ __forceinline__ bool eliminate_packed(const FactorArgs &a, int k, int round, char *lds, Cursor &fcur,
                                                 Cursor &ocur, int *next, unsigned int *next_set, uint64_t &over)
{
    constexpr int G = kPackLanes, kHeads = kFillLists / G;
    static_assert(kWave * kBytesPerEntry <= kLdsCap * kBytesPerEntry, "the groups share one column buffer");
    const int lane = lane_id(), gl = lane % G, gb = lane - gl;
    const int last = a.n - 1;
    const uint64_t below = (1ull << lane) - 1ull, group = ((1ull << G) - 1ull) << gb;
    ColBuf b = carve(lds, kLdsCap);
    b.s += gb; b.mw += gb; b.C += gb; b.mrow += gb; b.mmult += gb; b.minc += gb; b.jt += gb;

    // ---- 1. gather: originals one per lane, kHeads lists per lane
    const bool act = k >= 0;
    int m = 0, f[kHeads];
#pragma unroll
    for (int u = 0; u < kHeads; ++u) f[u] = -1;
    if (act) {
#pragma unroll
        for (int u = 0; u < kHeads; ++u) f[u] = gp(a.head)[(size_t)k * kFillLists + gl * kHeads + u];
        const int lo0 = gp(a.lo_ptr)[k];
        m = gp(a.lo_ptr)[k + 1] - lo0;
        if (gl < m && m <= G) {
            SEnt v;
            v.row = gp(a.lo_row)[lo0 + gl];
            v.pay = 1;
            v.w = gp(a.lo_w)[lo0 + gl];
            b.s[gl] = v;
        }
    }
    while (true) {
        uint64_t mask[kHeads], any = 0;
        FillRec rec[kHeads];
#pragma unroll
        for (int u = 0; u < kHeads; ++u) {
            const bool more = f[u] >= 0 && m <= G;
            mask[u] = ballot(more);
            any |= mask[u];
            if (more) rec[u] = *at(gp(a.pool) + f[u]);
        }
        if (!any) break;
#pragma unroll
        for (int u = 0; u < kHeads; ++u) {
            if ((mask[u] >> lane) & 1ull) {
                const int pos = m + __popcll(mask[u] & group & below);
                if (pos < G) {
                    SEnt v;
                    v.row = rec[u].row;
                    v.pay = 1;
                    v.w = rec[u].w;
                    b.s[pos] = v;
                }
                f[u] = rec[u].next;
            }
            m += __popcll(mask[u] & group);
        }
    }
    over = ballot(m > G && gl == 0);
    const bool live = m > 0 && m <= G;
    if (act && m == 0 && gl == 0) empty_column<false>(a, k, round);
    if (!live) m = 0;
    if (ballot(live) == 0ull) return true;
    wave_fence();

    // ---- 2. sort by (row, w), merge (as process_column, a group's lanes)
    pack_sort<true>(b, gl, m);
    RowRun run;
    run.head = false;
    if (gl < m) run = row_run(b.s, gl, m);
    const uint64_t heads = ballot(run.head) & group;
    if (run.head) put_merged(b, __popcll(heads & below), run);
    const int d = __popcll(heads);
    wave_fence();

    // ---- 3. sort by (w, row); sums (one block of the canonical scan)
    if (gl < d) b.s[gl] = merged_entry(b, gl);
    wave_fence();
    pack_sort<false>(b, gl, d);
    double x = gl < d ? b.s[gl].w : 0.0;
    for (int off = 1; off < G; off <<= 1) {
        const double o = __shfl_up(x, off, G);
        if (gl >= off) x = x + o;
    }
    if (gl < d) b.C[gl] = x;
    wave_fence();
    const double S = d > 0 ? b.C[d - 1] : 0.0;

    // ---- 4. sampled partners; the groups' pool entries in one piece
    const bool fill = gl < d - 1, ent = gl < d;
    if (fill) sample_partner(a, k, b, gl, d, S);
    const uint64_t fmask = ballot(fill), emask = ballot(ent);
    long long fbase = 0, obase = 0;
    if (fmask && !carve_pool(fcur, __popcll(fmask), kFillChunk, &a.ctr[kCtrFillTop], a.pool_cap, fbase)) {
        if (lane == 0) raise_status(a.ctr, kStatusFillPool);
        return false;
    }
    if (!carve_pool(ocur, __popcll(emask), kOutChunk, &a.ctr[kCtrOutTop], a.out_cap, obase)) {
        if (lane == 0) raise_status(a.ctr, kStatusOutPool);
        return false;
    }
    const int rec = (int)(fbase + __popcll(fmask & below));
    const long long oe = obase + __popcll(emask & below);
    if (live && gl == 0) {
        gp(a.level)[k] = round;
        gp(a.out_start)[k] = oe;
        gp(a.out_cnt)[k] = d;
        gp(a.diag)[k] = S;
    }
    wave_fence();   // minc and jt complete

    // ---- 5. fills, dependency updates, factor entries
    int old = -1, r = -1, nd = 1;
    bool upd = false;
    if (fill) old = push_head(a, b, gl, rec);
    if (ent) {
        r = b.mrow[gl];
        const int delta = b.minc[gl] - b.mmult[gl];
        upd = r != last && delta != 0;
        if (upd) nd = atomicAdd(at(&gp(a.dep)[r]), delta) + delta;
        gp(a.out_row)[oe] = r;
        gp(a.out_val)[oe] = -(b.mw[gl] / S);
    }
    if (fill) *at(gp(a.pool) + rec) = fill_record(b, gl, S, old);
    list_append(a, next_set, next, upd && nd == 0, r);
    wave_fence();
    return true;
}

// LDS of the large-LDS kernels: the column buffer, the sorts' second entry
// array and the workgroup's words.
constexpr size_t kWgColBytes = (size_t)kBigCap * kBytesPerEntry;
constexpr size_t kWgTmpBytes = (size_t)kBigCap * sizeof(SEnt);
constexpr size_t kWgLds = kWgColBytes + kWgTmpBytes + sizeof(WgShared);
static_assert(kWgLds <= 160 * 1024, "one workgroup's LDS");

// A column of more than kBigCap entries, in this workgroup's global scratch
// (column buffer, entry array, block sums).  Not inlined: it is rare, and the
// kernels' code stays half as long without it.
template <bool kAsync>
__device__ __attribute__((noinline)) bool eliminate_in_scratch(const FactorArgs *pa, WgShared *psh, int k, int round,
                                                               int m, Cursor *fcur, Cursor *ocur, int *next,
                                                               unsigned int *next_set)
{
    const FactorArgs &a = *pa;
    WgShared &sh = *psh;
    const int t = threadIdx.x;
    const int P = next_pow2(m);
    if (P > a.scratch_cap) {
        if (t == 0) {
            atomicMax(&a.ctr[kCtrScratchNeed], (unsigned long long)P);
            raise_status(a.ctr, kStatusScratch);
        }
        return false;
    }
    const int lo0 = gp(a.lo_ptr)[k];
    const int norig = gp(a.lo_ptr)[k + 1] - lo0;
    char *mine = at(gp(a.scratch) + (size_t)blockIdx.x * (size_t)a.scratch_cap * kScratchBytesPerEntry);
    const ColBuf g = carve(mine, a.scratch_cap);
    SEnt *tmp = reinterpret_cast<SEnt *>(mine + (size_t)a.scratch_cap * kBytesPerEntry);
    double *tot = reinterpret_cast<double *>(tmp + a.scratch_cap);
    gather_original(a, lo0, norig, g, a.scratch_cap, t, kWgThreads);
    if (t < kWave) {
        const int *hd = at(gp(a.head) + (size_t)k * kFillLists + t);
        const int c = gather_fills<false, kAsync>(a, norig, kAsync ? ld_relaxed(hd) : *hd, g, a.scratch_cap);
        if (t == 0) sh.ok = c == m;
    }
    __syncthreads();
    if (!sh.ok) {
        if (t == 0) raise_status(a.ctr, kStatusInconsistent);
        return false;
    }
    return process_column<kAsync, kWgWaves, 0>(a, &sh, k, round, g, tmp, tot, m, *fcur, *ocur, next, next_set);
}

// The columns that pop() hands to this workgroup's first wave (column < 0: no
// more; round: its level), until there are none or the pools are exhausted.
template <bool kAsync, typename Pop>
__device__ __forceinline__ void wg_columns(const FactorArgs &a, char *lds, Pop pop, int *next, unsigned int *next_set)
{
    static_assert(kFillLists == kWave, "one list per lane");
    WgShared &sh = *reinterpret_cast<WgShared *>(lds + kWgColBytes + kWgTmpBytes);
    SEnt *tmp = reinterpret_cast<SEnt *>(lds + kWgColBytes);
    const ColBuf b = carve(lds, kBigCap);
    const int t = threadIdx.x, lane = lane_id();
    long long *ws = a.wave_state + 4 * ((size_t)a.big_ws + blockIdx.x);
    Cursor fcur, ocur;
    fcur.cur = ws[0]; fcur.end = ws[1];
    ocur.cur = ws[2]; ocur.end = ws[3];
    while (true) {
        if (t < kWave) {
            int k, m = 0, round = 0;
            while (true) {
                k = pop(round);
                if (k < 0) break;
                // ---- 1. gather (as the round kernel, up to kBigCap entries)
                const int *hd = at(gp(a.head) + (size_t)k * kFillLists + lane);
                const int f0 = kAsync ? ld_relaxed(hd) : *hd;
                const int lo0 = gp(a.lo_ptr)[k];
                const int norig = gp(a.lo_ptr)[k + 1] - lo0;
                gather_original(a, lo0, norig, b, kWave, lane, kWave);
                m = gather_fills<false, kAsync>(a, norig, f0, b, kBigCap);
                wave_fence();
                if (m > kWave) break;
                if (m == 0) {
                    if (lane == 0) empty_column<kAsync>(a, k, round);
                    continue;
                }
                if (!process_column<kAsync, 1, 1>(a, &sh, k, round, b, nullptr, nullptr, m, fcur, ocur, next, next_set)) {
                    k = -1;
                    break;
                }
            }
            if (lane == 0) {
                sh.k = k;
                sh.m = m;
                sh.round = round;
            }
        }
        __syncthreads();
        const int k = sh.k, m = sh.m, round = sh.round;
        if (k < 0) break;
        bool ok;
        if (m <= kBigCap) {
            // original entries past the first kWave (few columns have them)
            const int lo0 = gp(a.lo_ptr)[k];
            const int norig = gp(a.lo_ptr)[k + 1] - lo0;
            if (norig > kWave) {
                gather_original(a, lo0, norig, b, kBigCap, kWave + t, kWgThreads);
                __syncthreads();
            }
            ok = process_column<kAsync, kWgWaves, 0>(a, &sh, k, round, b, tmp, sh.tot, m, fcur, ocur, next, next_set);
        } else {
            Cursor fc = fcur, oc = ocur;       // copies: the call takes addresses
            ok = eliminate_in_scratch<kAsync>(&a, &sh, k, round, m, &fc, &oc, next, next_set);
            fcur = fc;
            ocur = oc;
        }
        if (!ok) break;
    }
    if (t == 0) {
        ws[0] = fcur.cur; ws[1] = fcur.end;
        ws[2] = ocur.cur; ws[3] = ocur.end;
    }
}

}  // namespace

// One elimination round: every column of `cur` (count counts[round]).
__global__ void __launch_bounds__(kWave) k_factor_round(const FactorArgs *__restrict__ pa, int round, const int *cur,
                                                        int *next)
{
    const FactorArgs &a = *pa;
    __shared__ __attribute__((aligned(16))) char lds[kLdsCap * kBytesPerEntry];
    // this round's list counters (one per lane) with the status in one trip;
    // workgroup 0 clears the counter set of round + 2 (last used by round - 1)
    // and records the round's length for the host
    unsigned int c, incl;
    list_counts(a, list_set(a, round), c, incl);
    const unsigned long long status = a.ctr[kCtrStatus];
    const unsigned int ncur = __shfl(incl, kWave - 1, kWave);
    if (blockIdx.x == 0) {
        list_set(a, round + 2)[lane_id()] = 0u;
        if (lane_id() == 0) gp(a.round_count)[round] = ncur;
    }
    if (ncur <= (unsigned int)kBigGrid) return;     // a narrow round: the large-LDS kernel takes all of it
    if (status != 0ull) return;
    Cursor fcur, ocur;
    long long *ws = a.wave_state + 4 * (size_t)blockIdx.x;
    fcur.cur = ws[0]; fcur.end = ws[1];
    ocur.cur = ws[2]; ocur.end = ws[3];
    unsigned int *next_set = list_set(a, round + 1);
    // several columns per wave where every group has one to do: below, the
    // second pass over columns too large for a group costs more than it saves
    // (12000 columns: 53 us, one per wave 45 us; 20000: 104 and 143 us)
    const bool packed = ncur > (unsigned int)kPack * gridDim.x;
    const unsigned int per = packed ? kPack : 1;
    bool ok = true;
    for (unsigned int i = blockIdx.x * per; ok && i < ncur; i += gridDim.x * per) {
        int col = -1;
        for (unsigned int q = 0; q < per; ++q) {
            const unsigned int j = min(i + q, ncur - 1);
            const int kq = cur[list_index(a, c, incl, j)];
            if (!packed || (unsigned int)(lane_id() / kPackLanes) == q) col = i + q < ncur ? kq : -1;
        }
        uint64_t left = 1ull;
        if (packed) ok = eliminate_packed(a, col, round, lds, fcur, ocur, next, next_set, left);
        for (; ok && left; left &= left - 1ull)
            ok = eliminate_column(a, bcast(col, __ffsll((unsigned long long)left) - 1), round, lds, fcur, ocur, next, next_set,
                                  &a.big_count[round]);
    }
    if (lane_id() == 0) {
        ws[0] = fcur.cur; ws[1] = fcur.end;
        ws[2] = ocur.cur; ws[3] = ocur.end;
    }
}

// The round's columns deferred by k_factor_round (more than kLdsCap entries):
// one workgroup per column with kBigCap entries of LDS (columns above that use the
// per-workgroup global scratch).  Runs after k_factor_round of the same round.
__global__ void __launch_bounds__(kWgThreads) k_factor_round_big(const FactorArgs *__restrict__ pa, int round,
                                                                 const int *cur, int *next)
{
    const FactorArgs &a = *pa;
    extern __shared__ __attribute__((aligned(16))) char lds_big[];
    // a round of at most kBigGrid columns is eliminated here entirely (one
    // column per workgroup); otherwise the columns k_factor_round deferred
    unsigned int c, incl;
    list_counts(a, list_set(a, round), c, incl);
    const unsigned int ndef = gp(a.big_count)[round];
    const unsigned long long status = a.ctr[kCtrStatus];
    const unsigned int ncur = __shfl(incl, kWave - 1, kWave);
    const bool narrow = ncur <= (unsigned int)kBigGrid;
    const unsigned int nbig = narrow ? ncur : ndef;
    if (nbig == 0) return;
    unsigned int i = blockIdx.x;
    wg_columns<false>(a, lds_big, [&](int &level) {
        if (i >= nbig || status != 0ull) return -1;
        const int k = narrow ? cur[list_index(a, c, incl, i)] : gp(a.big_list)[i];
        level = round;
        i += gridDim.x;
        return k;
    }, next, list_set(a, round + 1));
}

// ---- queue-driven tail -----------------------------------------------------
// Once a round holds at most kBigGrid columns, the rest of the elimination runs
// in this one persistent launch: every workgroup takes the next queue index,
// waits until that slot holds a column (slots start at -1), eliminates it and
// appends the neighbours it made ready.  A column's level
// is 1 + the largest level of its lower neighbours (atomicMax by each of them
// before its dependency update), the same value the rounds assign.  Slot h is
// written by the workgroup that made its column ready, which is running, so every
// wait ends; the waits are bounded all the same (status bit on expiry).
__device__ __forceinline__ bool factor_should_stop(const FactorArgs &a)
{
    return ld_relaxed(&a.ctr[kCtrStatus]) != 0ull;
}

__global__ void __launch_bounds__(kWgThreads) k_factor_async(const FactorArgs *__restrict__ pa, unsigned int total)
{
    const FactorArgs &a = *pa;
    extern __shared__ __attribute__((aligned(16))) char lds_big[];
    wg_columns<true>(a, lds_big, [&](int &level) {
        unsigned int h = 0;
        int k = -1;
        if (lane_id() == 0) {
            h = atomicAdd(at(gp(a.aq_ctr) + kAqHead), 1u);
            if (h < total) k = ld_relaxed(at(&gp(a.aq)[h]));
            if (h < total && k < 0) {
                const long long t0 = wall_clock64();
                int nap = 1;
                while ((k = ld_relaxed(at(&gp(a.aq)[h]))) < 0) {
                    if (factor_should_stop(a)) break;
                    if (wall_clock64() - t0 > a.spin_ticks) {
                        raise_status(a.ctr, kStatusTimeout);
                        break;
                    }
                    for (int t = 0; t < nap; ++t) __builtin_amdgcn_s_sleep(2);
                    nap = nap < 8 ? nap * 2 : 8;
                }
            }
        }
        k = bcast(k, 0);
        asm volatile("" ::: "memory");             // the column's loads follow the slot's
        if (k >= 0) level = ld_relaxed(at(&gp(a.level)[k]));
        return k;                                  // < 0: all columns taken, or stopped (status raised)
    }, a.aq, nullptr);
}

// The queue starts with round `round`'s list (its columns' level is the round).
// One workgroup.  Entry i of the list is found per thread from the slot
// counts kept in LDS (list_index needs a wave-uniform entry).
__global__ void k_factor_async_init(FactorArgs a, int round, const int *cur, unsigned int total)
{
    __shared__ unsigned int s_c[kWave], s_incl[kWave];
    if (threadIdx.x < kWave) {
        unsigned int c, incl;
        list_counts(a, list_set(a, round), c, incl);
        s_c[threadIdx.x] = c;
        s_incl[threadIdx.x] = incl;
    }
    for (unsigned int i = threadIdx.x; i < total; i += blockDim.x) gp(a.aq)[i] = -1;
    __syncthreads();
    const unsigned int ncur = min(s_incl[kWave - 1], total);
    for (unsigned int i = threadIdx.x; i < ncur; i += blockDim.x) {
        int s = 0;                                   // slot of entry i: the first with incl > i
        while (s < kWave - 1 && s_incl[s] <= i) ++s;
        const size_t idx = (size_t)s * (size_t)a.seg_cap + (i - (s_incl[s] - s_c[s]));
        const int col = cur[idx];
        gp(a.aq)[i] = col;
        gp(a.level)[col] = round;
    }
    if (threadIdx.x == 0) {
        gp(a.aq_ctr)[kAqHead] = 0u;
        gp(a.aq_ctr)[kAqTail] = ncur;
    }
}

// ---- set-up kernels ------------------------------------------------------

__global__ void k_factor_init(int n, const int *dep_init, int *dep, int *head, int *level, int *out_cnt,
                              long long *out_start, double *diag)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)n * kFillLists;
         i += (size_t)gridDim.x * blockDim.x)
        head[i] = -1;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        dep[i] = dep_init[i];
        level[i] = 0;
        out_cnt[i] = 0;
        out_start[i] = 0;
        diag[i] = 0.0;
    }
}

// Round 0: every column without lower-index neighbours, except the last.
__global__ void k_factor_seed(FactorArgs a, const int *dep)
{
    for (int base = blockIdx.x * blockDim.x; base < a.n; base += gridDim.x * blockDim.x) {
        const int i = base + threadIdx.x;
        list_append(a, list_set(a, 0), a.list0, i < a.n - 1 && dep[i] == 0, i);
    }
}

void launch_factor_setup(const FactorArgs &a, const int *dep_init, hipStream_t s)
{
    hipLaunchKernelGGL(k_factor_init, dim3(1024), dim3(256), 0, s, a.n, dep_init, a.dep, a.head, a.level,
                       a.out_cnt, a.out_start, a.diag);
    hipLaunchKernelGGL(k_factor_seed, dim3(1024), dim3(256), 0, s, a, (const int *)a.dep);
}

void launch_factor_rounds(const FactorArgs &a, const FactorArgs *da, int num_blocks, int first_round, int nrounds,
                          hipStream_t s)
{
    for (int r = first_round; r < first_round + nrounds; ++r) {
        const int *cur = (r & 1) ? a.list1 : a.list0;
        int *next = (r & 1) ? a.list0 : a.list1;
        hipLaunchKernelGGL(k_factor_round, dim3(num_blocks), dim3(kWave), 0, s, da, r, cur, next);
        hipLaunchKernelGGL(k_factor_round_big, dim3(kBigGrid), dim3(kWgThreads), kWgLds, s, da, r,
                           cur, next);
    }
}

void factor_kernel_setup()
{
    (void)hipFuncSetAttribute((const void *)k_factor_round_big, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kWgLds);
    (void)hipFuncSetAttribute((const void *)k_factor_async, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kWgLds);
}

void launch_factor_async(const FactorArgs &a0, const FactorArgs *da, int round, unsigned int total, hipStream_t s)
{
    FactorArgs a = a0;
    a.aq_total = total;            // total <= n - 1 slots of the n-entry queue
    const int *cur = (round & 1) ? a.list1 : a.list0;
    // one block: the init kernel's slot clearing must finish before it seeds the queue
    hipLaunchKernelGGL(k_factor_async_init, dim3(1), dim3(1024), 0, s, a, round, cur, total);
    hipLaunchKernelGGL(k_factor_async, dim3(kBigGrid), dim3(kWgThreads), kWgLds, s, da, total);
}

int factor_lds_capacity() { return kLdsCap; }
int factor_scratch_bytes_per_entry() { return kScratchBytesPerEntry; }
long long factor_pool_slack(int num_blocks) { return (long long)(num_blocks + kBigGrid) * (kFillChunk + kOutChunk); }

int factor_occupancy_blocks(int device)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_factor_round, kWave, 0) != hipSuccess) per_cu = 8;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) cus = 256;
    if (per_cu < 1) per_cu = 1;
    return per_cu * cus;
}

// Statistics after the factor: nnz_off, fills, max degree, zero pivots
// (over the first n-1 columns; the last column is a zero pivot by definition),
// and the level of the last column (never eliminated): 1 + max level of the
// columns whose factor column holds it (rows are sorted, so it is their last
// entry).  One atomic per workgroup and word: with one per wave (4,096 of
// them on each word) the two passes took 150 us whatever the size.
constexpr int kStatBlock = 1024;
__global__ void __launch_bounds__(kStatBlock) k_factor_stats(int n, const long long *out_start, const int *out_cnt,
                                                             const int *out_row, int *level, unsigned long long *ctr)
{
    __shared__ unsigned long long red[5][kStatBlock / kWave];
    unsigned long long v[5] = {0, 0, 0, 0, 0};       // nnz, fills, zero pivots, max degree, level + 1
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned long long d = (unsigned long long)out_cnt[i];
        v[0] += d;
        v[1] += d > 0 ? d - 1 : 0;
        v[2] += d == 0 ? 1 : 0;
        v[3] = d > v[3] ? d : v[3];
        if (d > 0 && i < n - 1 && out_row[out_start[i] + (long long)d - 1] == n - 1) {
            const unsigned long long l = (unsigned long long)level[i] + 1;
            v[4] = l > v[4] ? l : v[4];
        }
    }
    for (int q = 0; q < 5; ++q) {
        v[q] = q < 3 ? (unsigned long long)wave_sum_u64(v[q]) : (unsigned long long)wave_max((int64_t)v[q]);
        if (lane_id() == 0) red[q][threadIdx.x / kWave] = v[q];
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return;
    for (int q = 0; q < 5; ++q) {
        const unsigned long long t = threadIdx.x < kStatBlock / kWave ? red[q][threadIdx.x] : 0;
        v[q] = q < 3 ? wave_sum_u64(t) : (unsigned long long)wave_max((int64_t)t);
    }
    if (threadIdx.x == 0) {
        atomicAdd(&ctr[kCtrNnzOff], v[0]);
        atomicAdd(&ctr[kCtrFills], v[1]);
        atomicAdd(&ctr[kCtrZeroPivots], v[2]);
        atomicMax(&ctr[kCtrMaxDeg], v[3]);
        if (v[4] > 0) atomicMax(&level[n - 1], (int)v[4]);
    }
}

void launch_factor_finish(const FactorArgs &a, hipStream_t s)
{
    const int g = a.n < 128 * kStatBlock ? (a.n + kStatBlock - 1) / kStatBlock : 128;
    hipLaunchKernelGGL(k_factor_stats, dim3(g), dim3(kStatBlock), 0, s, a.n, (const long long *)a.out_start,
                       (const int *)a.out_cnt, (const int *)a.out_row, a.level, a.ctr);
}

}  // namespace rc
