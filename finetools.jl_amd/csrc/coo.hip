// Device sparse(I, J, V, m, n): the COO -> CSC stage of makematrix!
// (src/AssemblyModule.jl:304-329), i.e. Julia's SparseArrays.sparse with its
// documented semantics: duplicates combined with + as a left fold in input
// order, explicit zeros kept, rows sorted within every column.
//
//   1. key = col * m + row (64 bit), payload = input position; the same pass
//      flags any index outside [0, m) x [0, n) (the stdlib raises an error);
//   2. stable LSD radix sort over the key bits actually used -- stability
//      keeps equal keys in input order;
//   3. segment heads where the key changes, scanned to segment numbers;
//   4. one thread per segment folds its values left to right in that order
//      (the same additions, in the same order, as the stdlib), and writes
//      rowval / nzval; column pointers come from the sorted segment columns.
//
// Steps 1-3 (phase A) end with one read-back of the entry count and the range
// flag; step 4 (phase B) then writes the outputs.
//
// Triples that come in runs of one column -- assemble! buffers element matrices
// column by column, 24 triples at a time for an H8 elasticity element -- take a
// shorter way (sparse_by_columns): the runs are listed by column, then one
// wavefront per column sorts the column's rows in registers and folds the
// duplicates, reading every triple once and in place.  A look at a few of the
// triples decides; columns too long for a wavefront's registers are taken out
// and sorted by steps 1-4 alone.
#include "common.hpp"
#include "wavesort.hpp"

#include <limits>

#include <rocprim/rocprim.hpp>

namespace feasm {

namespace {

__global__ void k_zero_flag(unsigned int *__restrict__ flag) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0u;
}

__global__ void k_keys(const int32_t *__restrict__ I, const int32_t *__restrict__ J, int64_t nt, int64_t m, int64_t n,
                       uint64_t *__restrict__ keys, uint32_t *__restrict__ idx, unsigned int *__restrict__ bad) {
    bool out = false;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nt; t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t i = I[t], j = J[t];
        out |= (i < 0) | ((int64_t)i >= m) | (j < 0) | ((int64_t)j >= n);
        keys[t] = (uint64_t)(uint32_t)j * (uint64_t)m + (uint64_t)(uint32_t)i;
        idx[t] = (uint32_t)t;
    }
    if (out) atomicOr(bad, 1u);
}

__global__ void k_heads(const uint64_t *__restrict__ keys, int64_t nt, int32_t *__restrict__ head) {
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nt; t += (int64_t)gridDim.x * blockDim.x)
        head[t] = (t == 0 || keys[t] != keys[t - 1]) ? 1 : 0;
}

// nnz = last segment number + last head; copied back with the range flag
__global__ void k_count(const int32_t *__restrict__ head, const int64_t *__restrict__ seg, int64_t nt,
                        const unsigned int *__restrict__ bad, int64_t *__restrict__ out) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        out[0] = seg[nt - 1] + head[nt - 1];
        out[1] = (int64_t)*bad;
    }
}

__global__ void k_seg_start(const int32_t *__restrict__ head, const int64_t *__restrict__ seg, int64_t nt,
                            int64_t *__restrict__ start) {
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nt; t += (int64_t)gridDim.x * blockDim.x)
        if (head[t]) start[seg[t]] = t;
}

__global__ void k_seg_sum(const uint64_t *__restrict__ keys, const uint32_t *__restrict__ idx,
                          const double *__restrict__ V, const int64_t *__restrict__ start, int64_t nnz, int64_t nt,
                          int64_t m, int32_t *__restrict__ rowval, double *__restrict__ nzval) {
    for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < nnz; s += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = start[s], e = (s + 1 < nnz) ? start[s + 1] : nt;
        double v = V[idx[b]];
        for (int64_t t = b + 1; t < e; t++) v = v + V[idx[t]];
        nzval[s] = v;
        rowval[s] = (int32_t)(keys[b] % (uint64_t)m);
    }
}

// One thread per segment fills the column pointers since the last column; a gap
// of many empty columns is the whole wavefront's (25 ns a column for one thread).
__global__ void k_colptr(const uint64_t *__restrict__ keys, const int64_t *__restrict__ start, int64_t nnz,
                         int64_t m, int64_t n, int64_t *__restrict__ colptr) {
    const int lane = threadIdx.x & 63;
    for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s - lane <= nnz;
         s += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = -1, prev = -1;
        if (s <= nnz) {
            c = (s < nnz) ? (int64_t)(keys[start[s]] / (uint64_t)m) : n;
            prev = (s == 0) ? -1 : (int64_t)(keys[start[s - 1]] / (uint64_t)m);
        }
        const bool gap = c - prev > 16;
        if (!gap)
            for (int64_t j = prev + 1; j <= c; j++) colptr[j] = s;
        for (uint64_t todo = __ballot(gap); todo; todo &= todo - 1) {
            const int l = __ffsll((unsigned long long)todo) - 1;
            const int64_t b = __shfl(prev, l, 64), e = __shfl(c, l, 64), v = __shfl(s, l, 64);
            for (int64_t j = b + 1 + lane; j <= e; j += 64) colptr[j] = v;
        }
    }
}

// colptr of a matrix with no entries (a fill kernel rather than a memset)
__global__ void k_fill_i64(int64_t *__restrict__ p, int64_t n, int64_t v) {
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        p[t] = v;
}

// ---- sparse_by_columns
// What bounds it: one read of I, J and V and one write of the result (240 MB for
// the 11.3 M triples of H8 29x27x25 elasticity), against a radix sort of 64-bit
// keys that moves them through memory four times (886 us in all; this way
// 302 us).
//
// A run is a stretch of triples of one column within 64 consecutive triples
// (one wavefront's load).  The runs are put into lists by column with counting
// atomics, in any order; a column's wavefront orders its few runs by their
// first triple.

constexpr int kSmallColumn = 256, kMaxColumn = 1024;  // triples of one column the wavefront sorts hold
// (longer ones -- a constraint, a vertex of 35 T10 elasticity elements -- are
// taken out and sorted by themselves: H8 11.3 M triples with one of 5000 670 us,
// 1060 when it sent all to the sort, after most of this way's work)
// mean run length from which this way pays: the lists take 8 bytes a run
constexpr int64_t kMinRun = 4;
// state bits: a row or column out of range; a column of more than kSmallColumn
// triples; rows of a column too far apart for 31-bit keys; runs too short
constexpr unsigned kBadRow = 1, kBadColumn = 2, kBigColumn = 4, kWideRows = 8, kShortRuns = 16;
// states in which this way is given up: the kernels that follow return at once
constexpr unsigned kGiveUp = kBadColumn | kShortRuns;
// (also when more than half of the nt triples are in columns too long: their
// number is the 8-byte word after the state's)
__device__ __forceinline__ bool given_up(const unsigned int *state, int64_t nt) {
    return (*state & kGiveUp) || 2 * reinterpret_cast<const unsigned long long *>(state)[1] > (unsigned long long)nt;
}
constexpr int kWide = -1;  // sort_column: the rows are too far apart for its keys
constexpr int kSampleWindows = 256, kFarTriples = kMaxColumn;
constexpr int64_t kMinTriples = 1 << 16;

// What the triples look like, from up to kSampleWindows stretches of 64 spread
// over them: out[0] the runs, out[1] the triples that have the column of the one
// kFarTriples further on (columns too long for the wavefront sorts).
__global__ __launch_bounds__(1024) void k_run_sample(const int32_t *__restrict__ J, int64_t nt,
                                                     unsigned int *__restrict__ out) {
    __shared__ unsigned int sum[2];
    if (threadIdx.x < 2) sum[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t all = (nt + 63) / 64, windows = min(all, (int64_t)kSampleWindows);
    // all of a wavefront's stretches are loaded before any is looked at (one after
    // the other they took 13 us, so 10)
    constexpr int W = kSampleWindows / 16;
    int32_t j[W], f[W];
    bool in[W];
#pragma unroll
    for (int i = 0; i < W; i++) {
        const int64_t k = wave + 16 * i, t = all * k / windows * 64 + lane;
        in[i] = k < windows && t < nt;
        j[i] = in[i] ? J[t] : 0;
        f[i] = in[i] && t + kFarTriples < nt ? J[t + kFarTriples] : -1;
    }
    unsigned int runs = 0, far = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const int32_t prev = __shfl_up(j[i], 1, 64);
        runs += (unsigned)__popcll(__ballot(in[i] && (lane == 0 || prev != j[i])));
        far += (unsigned)__popcll(__ballot(in[i] && f[i] == j[i] && j[i] >= 0));
    }
    if (lane == 0) {
        atomicAdd(&sum[0], runs);
        atomicAdd(&sum[1], far);
    }
    __syncthreads();
    if (threadIdx.x < 2) out[threadIdx.x] = sum[threadIdx.x];
}

// the run that starts at this lane's triple: its length, 0 when none does
__device__ __forceinline__ int run_at(int32_t j, bool in, int lane) {
    const int32_t prev = __shfl_up(j, 1, 64);
    const uint64_t heads = __ballot(in && (lane == 0 || prev != j)), all = __ballot(in);
    if (!((heads >> lane) & 1)) return 0;
    const uint64_t above = lane < 63 ? heads >> (lane + 1) : 0;
    return above ? __ffsll((unsigned long long)above) : __popcll(all >> lane);
}

// per column: its runs (high word) and triples (low word); kBadColumn for a
// column index outside [0, n)
__global__ __launch_bounds__(256) void k_run_count(const int32_t *__restrict__ J, int64_t nt, int64_t n,
                                                   unsigned long long *__restrict__ cnt,
                                                   unsigned int *__restrict__ state) {
    const int lane = threadIdx.x & 63;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t - lane < nt; t += step) {
        const int32_t j = t < nt ? J[t] : 0;
        const bool ok = j >= 0 && (int64_t)j < n;
        const int len = run_at(j, t < nt, lane);
        if (len > 0) {
            if (ok)
                atomicAdd(&cnt[j], (1ull << 32) | (unsigned)len);
            else
                atomicOr(state, kBadColumn);
        }
    }
}

// the runs into their columns' lists: (first triple, length), counting the
// column's runs down.  place[c]: the column's first run (high word) and first
// place in column order (low word).
__global__ __launch_bounds__(256) void k_run_fill(const int32_t *__restrict__ J, int64_t nt,
                                                  const uint64_t *__restrict__ place,
                                                  unsigned long long *__restrict__ cnt, uint2 *__restrict__ runs,
                                                  const unsigned int *__restrict__ state) {
    if (given_up(state, nt)) return;
    const int lane = threadIdx.x & 63;
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t - lane < nt; t += step) {
        const int32_t j = t < nt ? J[t] : 0;
        const int len = run_at(j, t < nt, lane);
        if (len > 0) {
            const unsigned left = (unsigned)(atomicAdd(&cnt[j], ~0ull << 32) >> 32);  // one run fewer
            runs[(place[j] >> 32) + left - 1] = make_uint2((uint32_t)t, (uint32_t)len);
        }
    }
}

// (cnt: the end of the columns' entry counts, which the scan of them reads;
// longs: the triples of the columns of more than kMaxColumn)
__global__ __launch_bounds__(256) void k_col_check(const uint64_t *__restrict__ place, int64_t n, int64_t nt,
                                                   int32_t *__restrict__ cnt, unsigned int *__restrict__ state,
                                                   unsigned long long *__restrict__ longs) {
    unsigned st = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        cnt[n] = 0;
        if ((int64_t)(place[n] >> 32) > nt / kMinRun) st = kShortRuns;
    }
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t L = (uint32_t)place[c + 1] - (uint32_t)place[c];
        st |= L > kSmallColumn ? kBigColumn : 0u;
        if (L > kMaxColumn) atomicAdd(longs, (unsigned long long)L);  // few: each is more than 1024 triples
    }
    if (st) atomicOr(state, st);
}

// One column of L <= 64 E triples in nr runs: its runs ordered, its rows sorted
// (ties by input order: the key's low B bits are the place in the column),
// duplicates folded left to right.  The distinct rows and their sums go to
// trow / tval; returns their number.  Keys of 31 bits (T int32_t) hold rows up to
// 2^(31-B) apart, else kWide is returned; keys of 63 any row.  lds: 4 * 64 E words
// of the wavefront's own.
template <int E, int B, typename T>
__device__ __forceinline__ int sort_column(const int32_t *__restrict__ I, const double *__restrict__ V, int64_t m,
                                           const uint2 *__restrict__ runs, int nr, int L, int lane, int32_t *lds,
                                           int32_t *__restrict__ trow, double *__restrict__ tval, unsigned int &state) {
    constexpr T kPad = std::numeric_limits<T>::max();
    // the places of the runs, in order of their first triple (by counting the
    // triples of earlier runs), and what takes a place to its triple
    uint32_t *const sS = reinterpret_cast<uint32_t *>(lds), *const sN = sS + 64 * E, *const sAt = sN + 64 * E,
                    *const sSh = sAt + 64 * E;
    for (int j = lane; j < nr; j += 64) {
        const uint2 r = runs[j];
        sS[j] = r.x;
        sN[j] = r.y;
    }
    wave_fence();
    for (int j = lane; j < nr; j += 64) {
        const uint32_t s = sS[j];
        uint32_t at = 0, rank = 0;
        for (int k = 0; k < nr; k++) {
            const bool before = sS[k] < s;
            at += before ? sN[k] : 0u;
            rank += before ? 1u : 0u;
        }
        sAt[rank] = at;
        sSh[rank] = s - at;
    }
    wave_fence();
    uint32_t t[E];
    const int top = nr > 1 ? 1 << (31 - __clz(nr - 1)) : 0;  // the largest power of two below nr
#pragma unroll
    for (int e = 0; e < E; e++) {
        const uint32_t p = lane + 64 * e;
        int r = 0;  // the last run at or before place p
        for (int w = top; w > 0; w >>= 1)
            if (r + w < nr && sAt[r + w] <= p) r += w;
        t[e] = p + sSh[r];
    }
    wave_fence();
    double *const sV = reinterpret_cast<double *>(lds);
    T *const sK = reinterpret_cast<T *>(lds + 2 * 64 * E);
    int32_t row[E], lo = 0x7fffffff, hi = -1;
    T x[E];
    double v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int p = lane + 64 * e;
        row[e] = p < L ? I[t[e]] : 0;
        v[e] = p < L ? V[t[e]] : 0.0;
    }
    bool out = false;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const bool in = lane + 64 * e < L;
        out |= in && (row[e] < 0 || (int64_t)row[e] >= m);
        lo = in ? min(lo, row[e]) : lo;
        hi = in ? max(hi, row[e]) : hi;
        sV[lane + 64 * e] = v[e];
    }
#pragma unroll
    for (int j = 1; j < 64; j <<= 1) {
        lo = min(lo, lane_xor(lo, j, lane));
        hi = max(hi, lane_xor(hi, j, lane));
    }
    if (__any(out)) {
        state |= kBadRow;
        wave_fence();  // the words are reused for the next column
        return 0;
    }
    if constexpr (sizeof(T) == 4) {
        if (hi - lo >= (1 << (31 - B)) - 1) {
            wave_fence();
            return kWide;
        }
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int p = lane + 64 * e;
        x[e] = p < L ? ((T)(row[e] - lo) << B) | p : kPad;
    }
    wave_sort(x, lane);
#pragma unroll
    for (int e = 0; e < E; e++) sK[lane + 64 * e] = x[e];
    wave_fence();
    int base = 0;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int i = lane + 64 * e;
        const bool head = i < L && (i == 0 || (sK[i > 0 ? i - 1 : 0] >> B) != (x[e] >> B));
        const uint64_t hm = __ballot(head);
        if (head) {
            const T r = x[e] >> B;
            double a = sV[(int)x[e] & ((1 << B) - 1)];
            for (int q = i + 1; q < L; q++) {
                const T y = sK[q];
                if ((y >> B) != r) break;
                a = a + sV[(int)y & ((1 << B) - 1)];
            }
            const int at = base + __popcll(hm & ((1ull << lane) - 1ull));
            trow[at] = (int32_t)r + lo;
            tval[at] = a;
        }
        base += __popcll(hm);
    }
    wave_fence();
    return base;
}

// One wavefront per column: kSmall the columns of up to kSmallColumn triples,
// kBig the longer ones; kWideKeys those that either found wide (cnt kWide), with
// 63-bit keys: quadratic elements whose edge nodes are numbered after 700k
// corners have such columns.  (A kernel of their own: in kBig's they would take
// its registers from 121 to 194.)  A column's distinct rows and sums go to trow /
// tval from its first place on, their number to cnt.
enum { kSmall, kBig, kWideKeys };
template <int WHICH>
__global__ __launch_bounds__(64) void k_columns(const int32_t *__restrict__ I, const double *__restrict__ V, int64_t nt,
                                                int64_t m, int64_t n, const uint64_t *__restrict__ place,
                                                const uint2 *__restrict__ runs, int32_t *__restrict__ cnt,
                                                int32_t *__restrict__ trow, double *__restrict__ tval,
                                                unsigned int *__restrict__ state) {
    __shared__ __align__(16) int32_t lds[4 * (WHICH == kSmall ? kSmallColumn : kMaxColumn)];
    const unsigned before = *state;
    if (given_up(state, nt) || (WHICH == kBig && !(before & kBigColumn))) return;
    const int lane = threadIdx.x;
    unsigned int st = 0;
    for (int64_t c = blockIdx.x; c < n; c += gridDim.x) {
        const uint64_t a = place[c], b = place[c + 1];
        const int L = (int)((uint32_t)b - (uint32_t)a), nr = (int)((b >> 32) - (a >> 32));
        if (WHICH == kWideKeys ? cnt[c] != kWide : (WHICH == kBig) != ((uint32_t)L > kSmallColumn)) continue;
        if (WHICH == kBig && (uint32_t)L > kMaxColumn) {  // sorted with the other long columns' triples
            if (lane == 0) cnt[c] = 0;
            continue;
        }
        const uint2 *ru = runs + (a >> 32);
        int32_t *tr = trow + (uint32_t)a;
        double *tv = tval + (uint32_t)a;
        int k = 0;
        if constexpr (WHICH == kWideKeys)
            k = L <= 256   ? sort_column<4, 10, int64_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st)
                : L <= 512 ? sort_column<8, 10, int64_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st)
                           : sort_column<16, 10, int64_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st);
        else if constexpr (WHICH == kBig)
            k = L <= 512 ? sort_column<8, 10, int32_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st)
                         : sort_column<16, 10, int32_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st);
        else if (L > 0)
            k = L <= 64    ? sort_column<1, 8, int32_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st)
                : L <= 128 ? sort_column<2, 8, int32_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st)
                           : sort_column<4, 8, int32_t>(I, V, m, ru, nr, L, lane, lds, tr, tv, st);
        if (k == kWide) st |= kWideRows;
        if (lane == 0) cnt[c] = k;
    }
    if (st && lane == 0) atomicOr(state, st);
}

// what the host decides by, into pinned memory: one launch for two copies
struct ColumnsEnd {
    int64_t nnz;
    uint64_t nlong;
    unsigned int state;
};
__global__ void k_columns_end(const int64_t *__restrict__ colptr_end, const unsigned int *__restrict__ state,
                              ColumnsEnd *__restrict__ out) {
    if (threadIdx.x == 0)
        *out = ColumnsEnd{*colptr_end, reinterpret_cast<const unsigned long long *>(state)[1], *state};
}

// the triples of the columns of more than kMaxColumn
struct InLongColumn {
    const int32_t *J;
    const uint64_t *place;
    __device__ bool operator()(uint32_t t) const {
        const int32_t j = J[t];
        return (uint32_t)place[j + 1] - (uint32_t)place[j] > (uint32_t)kMaxColumn;
    }
};

__global__ __launch_bounds__(256) void k_take(const uint32_t *__restrict__ at, int64_t n, const int32_t *__restrict__ I,
                                              const int32_t *__restrict__ J, const double *__restrict__ V,
                                              int32_t *__restrict__ i, int32_t *__restrict__ j,
                                              double *__restrict__ v) {
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t t = at[k];
        i[k] = I[t];
        j[k] = J[t];
        v[k] = V[t];
    }
}

// the long columns' entry counts, from the matrix of their triples
__global__ __launch_bounds__(256) void k_long_counts(const int64_t *__restrict__ colptr, int64_t n,
                                                     int32_t *__restrict__ cnt) {
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
        if (colptr[c + 1] != colptr[c]) cnt[c] = (int32_t)(colptr[c + 1] - colptr[c]);
}

// the columns' entries, packed; LONG: the long columns' alone, from the matrix of
// their triples (place: its column pointers)
template <bool LONG>
__global__ __launch_bounds__(256) void k_columns_pack(const uint64_t *__restrict__ place, int64_t n, const int64_t *__restrict__ colptr,
                                                      const int32_t *__restrict__ trow, const double *__restrict__ tval,
                                                      int32_t *__restrict__ rowval, double *__restrict__ nzval) {
    const int lane = threadIdx.x & 63;
    for (int64_t c = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6; c < n;
         c += ((int64_t)gridDim.x * blockDim.x) >> 6) {
        const int64_t src = LONG ? (int64_t)place[c] : (int64_t)(uint32_t)place[c], dst = colptr[c];
        const int64_t k = LONG ? (int64_t)(place[c + 1] - place[c]) : colptr[c + 1] - dst;
        for (int64_t i = lane; i < k; i += 64) {
            rowval[dst + i] = trow[src + i];
            nzval[dst + i] = tval[src + i];
        }
    }
}

}  // namespace

void fill_i64(hipStream_t s, int64_t *p, int64_t n, int64_t v) {
    hipLaunchKernelGGL(k_fill_i64, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    FEASM_HIP(hipGetLastError());
}

static feasm_matrix *sparse_by_sort(feasm_ctx *ctx, int64_t nt, const int32_t *I, const int32_t *J, const double *V,
                                    int64_t m, int64_t n);

// The shorter way; null when the triples are few or not in runs, or most are in
// columns too long for the wavefront sort.  Throws FEASM_EDOF for an index out
// of range, as the general way does.
static feasm_matrix *sparse_by_columns(feasm_ctx *ctx, int64_t nt, const int32_t *I, const int32_t *J, const double *V,
                                       int64_t m, int64_t n) {
    // few triples: both ways are launches and waits, and the sort has fewer of
    // them (H8 elasticity in runs: 37k triples 135 us by the sort, 146 this way; 72k
    // 169, 127); but the sort fills a wide matrix's column pointers gap by gap, a
    // wavefront each (37k triples of 20 M columns 7.9 ms, this way 2.5)
    if (nt < kMinTriples && n <= nt) return nullptr;
    hipStream_t s = ctx->stream;
    // A look at a few of the triples first: what this way does before it knows
    // all the runs (an atomic a run, two passes over the columns) would cost
    // triples in no order half of their sort again (11.3 M: 1030 us, 560 more).
    void *const pinned = pinned_buffer(sizeof(ColumnsEnd));
    unsigned int *sample = static_cast<unsigned int *>(pinned);
    hipLaunchKernelGGL(k_run_sample, dim3(1), dim3(1024), 0, s, J, nt, sample);
    FEASM_HIP(hipGetLastError());
    FEASM_HIP(hipStreamSynchronize(s));
    const int64_t seen = std::min<int64_t>(nt, 64 * kSampleWindows);
    if (seen < kMinRun * (int64_t)sample[0] || 2 * (int64_t)sample[1] > seen) return nullptr;
    DevPtr ccnt = dev_alloc((n + 3) * 8), place = dev_alloc((n + 1) * 8);
    unsigned int *state = reinterpret_cast<unsigned int *>(dp<int64_t>(ccnt) + n + 1);
    unsigned long long *longs = dp<unsigned long long>(ccnt) + n + 2;  // where given_up() looks
    fill_i64(s, dp<int64_t>(ccnt), n + 3, 0);
    const unsigned gt = grid_for(nt, 256, 1u << 14);
    hipLaunchKernelGGL(k_run_count, dim3(gt), dim3(256), 0, s, J, nt, n, dp<unsigned long long>(ccnt), state);
    FEASM_HIP(hipGetLastError());
    // both words of an entry stay below 2^32 (at most a run a triple), so they
    // are scanned as one number and read back unsigned
    exclusive_scan_i64(ctx, dp<int64_t>(ccnt), dp<int64_t>(place), n + 1);
    DevPtr cnt = dev_alloc((n + 1) * 4), trow = dev_alloc(nt * 4), tval = dev_alloc(nt * 8);
    hipLaunchKernelGGL(k_col_check, dim3(grid_for(n, 256)), dim3(256), 0, s, dp<uint64_t>(place), n, nt,
                       dp<int32_t>(cnt), state, longs);
    DevPtr runs = dev_alloc(std::max<int64_t>(nt / kMinRun, 1) * sizeof(uint2));  // k_col_check: no more of them
    hipLaunchKernelGGL(k_run_fill, dim3(gt), dim3(256), 0, s, J, nt, dp<uint64_t>(place),
                       dp<unsigned long long>(ccnt), dp<uint2>(runs), state);
    FEASM_HIP(hipGetLastError());
    const auto columns = [&](auto kern, unsigned most) {
        hipLaunchKernelGGL(kern, dim3(grid_for(n, 1, most)), dim3(64), 0, s, I, V, nt, m, n, dp<uint64_t>(place),
                           dp<uint2>(runs), dp<int32_t>(cnt), dp<int32_t>(trow), dp<double>(tval), state);
        FEASM_HIP(hipGetLastError());
    };
    columns(k_columns<kSmall>, 1u << 17);
    columns(k_columns<kBig>, 1u << 11);  // what the LDS of 256 CUs holds; most matrices have no such column
    std::unique_ptr<feasm_matrix> M(new feasm_matrix);
    M->ctx = ctx;
    M->m = m;
    M->n = n;
    M->colptr = dev_alloc((n + 1) * sizeof(int64_t));
    exclusive_scan_i32_to_i64(ctx, dp<int32_t>(cnt), dp<int64_t>(M->colptr), n + 1);
    hipLaunchKernelGGL(k_columns_end, dim3(1), dim3(64), 0, s, dp<int64_t>(M->colptr) + n, state,
                       static_cast<ColumnsEnd *>(pinned));
    FEASM_HIP(hipGetLastError());
    FEASM_HIP(hipStreamSynchronize(s));
    const ColumnsEnd end = *static_cast<const ColumnsEnd *>(pinned);
    M->nnz = end.nnz;
    const uint64_t nlong = end.nlong;
    const unsigned int st = end.state;
    FEASM_REQUIRE(!(st & (kBadRow | kBadColumn)), FEASM_EDOF, "sparse: row or column index out of range");
    if ((st & kGiveUp) || 2 * (int64_t)nlong > nt) return nullptr;
    // the long columns' triples by the sort of theirs alone, in input order
    std::unique_ptr<feasm_matrix> far;
    if (nlong > 0) {
        DevPtr at = dev_alloc(nlong * 4), count = dev_alloc(8);
        DevPtr li = dev_alloc(nlong * 4), lj = dev_alloc(nlong * 4), lv = dev_alloc(nlong * 8);
        const InLongColumn pick{J, dp<uint64_t>(place)};
        const auto select = [&](void *tmp, size_t &bytes) {
            FEASM_HIP(rocprim::select(tmp, bytes, rocprim::counting_iterator<uint32_t>(0), dp<uint32_t>(at),
                                      dp<unsigned long long>(count), (size_t)nt, pick, s));
        };
        size_t bytes = 0;
        select(nullptr, bytes);
        void *tmp = ctx->scratch_get(bytes);
        select(tmp, bytes);
        hipLaunchKernelGGL(k_take, dim3(grid_for(nlong, 256)), dim3(256), 0, s, dp<uint32_t>(at), (int64_t)nlong, I, J, V,
                           dp<int32_t>(li), dp<int32_t>(lj), dp<double>(lv));
        FEASM_HIP(hipGetLastError());
        far.reset(sparse_by_sort(ctx, nlong, dp<int32_t>(li), dp<int32_t>(lj), dp<double>(lv), m, n));
        hipLaunchKernelGGL(k_long_counts, dim3(grid_for(n, 256)), dim3(256), 0, s, dp<int64_t>(far->colptr), n,
                           dp<int32_t>(cnt));
        FEASM_HIP(hipGetLastError());
    }
    if (nlong > 0 || (st & kWideRows)) {  // the entry counts are complete now
        if (st & kWideRows) columns(k_columns<kWideKeys>, 1u << 11);
        exclusive_scan_i32_to_i64(ctx, dp<int32_t>(cnt), dp<int64_t>(M->colptr), n + 1);
        read_back(s, &M->nnz, dp<int64_t>(M->colptr) + n, sizeof(int64_t));
    }
    M->rowval = dev_alloc(std::max<int64_t>(M->nnz, 1) * sizeof(int32_t));
    M->nzval = dev_alloc(std::max<int64_t>(M->nnz, 1) * sizeof(double));
    const auto pack = [&](auto kern, const void *from, const DevPtr &row, const DevPtr &val) {
        hipLaunchKernelGGL(kern, dim3(grid_for(n, 4)), dim3(256), 0, s, static_cast<const uint64_t *>(from), n,
                           dp<int64_t>(M->colptr), dp<int32_t>(row), dp<double>(val), dp<int32_t>(M->rowval),
                           dp<double>(M->nzval));
        FEASM_HIP(hipGetLastError());
    };
    pack(k_columns_pack<false>, place->p, trow, tval);
    if (far) pack(k_columns_pack<true>, far->colptr->p, far->rowval, far->nzval);
    FEASM_HIP(hipStreamSynchronize(s));
    return M.release();
}

int bits_for(uint64_t v) {
    int b = 0;
    while (b < 64 && (v >> b) != 0) b++;
    return b < 1 ? 1 : b;
}

size_t sort_tmp_bytes(int64_t nt, unsigned end_bit, hipStream_t s) {
    size_t a = 0, b = 0;
    rocprim::double_buffer<uint64_t> kb(nullptr, nullptr);
    rocprim::double_buffer<uint32_t> vb(nullptr, nullptr);
    FEASM_HIP(rocprim::radix_sort_pairs(nullptr, a, kb, vb, (size_t)nt, 0u, end_bit, s));
    FEASM_HIP(rocprim::exclusive_scan(nullptr, b, (const int32_t *)nullptr, (int64_t *)nullptr, (int64_t)0,
                                      (size_t)nt, rocprim::plus<int64_t>(), s));
    return std::max(a, b);
}

// Phase A: keys + range check, stable sort, segment heads and numbers; one
// read-back.  Returns nnz; FEASM_EDOF when an index is out of range.
int64_t sparse_phase_a(hipStream_t s, int64_t nt, const int32_t *I, const int32_t *J, int64_t m, int64_t n,
                       unsigned end_bit, SparseWork &w, bool pinned) {
    hipLaunchKernelGGL(k_zero_flag, dim3(1), dim3(64), 0, s, w.flag);
    hipLaunchKernelGGL(k_keys, dim3(grid_for(nt, 256)), dim3(256), 0, s, I, J, nt, m, n, w.keys, w.idx, w.flag);
    FEASM_HIP(hipGetLastError());
    rocprim::double_buffer<uint64_t> kb(w.keys, w.keys_alt);
    rocprim::double_buffer<uint32_t> vb(w.idx, w.idx_alt);
    size_t bytes = w.tmp_bytes;
    FEASM_HIP(rocprim::radix_sort_pairs(w.tmp, bytes, kb, vb, (size_t)nt, 0u, end_bit, s));
    w.skeys = kb.current();
    w.sidx = vb.current();
    w.head = reinterpret_cast<int32_t *>(vb.alternate());
    w.seg = reinterpret_cast<int64_t *>(kb.alternate());
    hipLaunchKernelGGL(k_heads, dim3(grid_for(nt, 256)), dim3(256), 0, s, w.skeys, nt, w.head);
    bytes = w.tmp_bytes;
    FEASM_HIP(rocprim::exclusive_scan(w.tmp, bytes, (const int32_t *)w.head, w.seg, (int64_t)0, (size_t)nt,
                                      rocprim::plus<int64_t>(), s));
    hipLaunchKernelGGL(k_count, dim3(1), dim3(64), 0, s, (const int32_t *)w.head, (const int64_t *)w.seg, nt,
                       (const unsigned int *)w.flag, w.count);
    FEASM_HIP(hipGetLastError());
    int64_t hc[2] = {0, 0};
    if (pinned) {
        read_back(s, hc, w.count, sizeof(hc));
    } else {
        FEASM_HIP(hipMemcpyAsync(hc, w.count, sizeof(hc), hipMemcpyDeviceToHost, s));
        FEASM_HIP(hipStreamSynchronize(s));
    }
    FEASM_REQUIRE(hc[1] == 0, FEASM_EDOF, "sparse: row or column index out of range");
    return hc[0];
}

// Phase B: segment starts, ordered sums, column pointers.
void sparse_phase_b(hipStream_t s, int64_t nt, const double *V, int64_t m, int64_t n, int64_t nnz,
                    const SparseWork &w, int64_t *colptr, int32_t *rowval, double *nzval) {
    hipLaunchKernelGGL(k_seg_start, dim3(grid_for(nt, 256)), dim3(256), 0, s, (const int32_t *)w.head,
                       (const int64_t *)w.seg, nt, w.start);
    hipLaunchKernelGGL(k_seg_sum, dim3(grid_for(nnz, 256)), dim3(256), 0, s, w.skeys, w.sidx, V,
                       (const int64_t *)w.start, nnz, nt, m, rowval, nzval);
    hipLaunchKernelGGL(k_colptr, dim3(grid_for(nnz + 1, 256)), dim3(256), 0, s, w.skeys, (const int64_t *)w.start,
                       nnz, m, n, colptr);
    FEASM_HIP(hipGetLastError());
}

void check_sparse_args(int64_t nt, int64_t m, int64_t n) {
    FEASM_REQUIRE(nt >= 0 && m >= 0 && n >= 0, FEASM_EINVAL, "negative size");
    FEASM_REQUIRE(nt < (1ll << 32), FEASM_EUNSUPPORTED, "more than 2^32 triples");
    FEASM_REQUIRE(m < (1ll << 31) && n < (1ll << 31), FEASM_EUNSUPPORTED, "more than 2^31 rows or columns");
    FEASM_REQUIRE(nt == 0 || (m >= 1 && n >= 1), FEASM_EDOF, "sparse: row or column index out of range");
}

// The radix sort of all triples (nt > 0).
static feasm_matrix *sparse_by_sort(feasm_ctx *ctx, int64_t nt, const int32_t *I, const int32_t *J, const double *V,
                                    int64_t m, int64_t n) {
    hipStream_t s = ctx->stream;
    std::unique_ptr<feasm_matrix> M(new feasm_matrix);
    M->ctx = ctx;
    M->m = m;
    M->n = n;
    M->colptr = dev_alloc((n + 1) * sizeof(int64_t));
    const unsigned end_bit = (unsigned)bits_for((uint64_t)m * (uint64_t)n);
    SparseWork w;
    DevPtr keys = dev_alloc(nt * sizeof(uint64_t)), keys2 = dev_alloc(nt * sizeof(uint64_t));
    DevPtr idx = dev_alloc(nt * sizeof(uint32_t)), idx2 = dev_alloc(nt * sizeof(uint32_t));
    DevPtr small = dev_alloc(256);
    w.keys = dp<uint64_t>(keys);
    w.keys_alt = dp<uint64_t>(keys2);
    w.idx = dp<uint32_t>(idx);
    w.idx_alt = dp<uint32_t>(idx2);
    w.count = dp<int64_t>(small);
    w.flag = reinterpret_cast<unsigned int *>(dp<int64_t>(small) + 2);
    w.tmp_bytes = sort_tmp_bytes(nt, end_bit, s);
    w.tmp = ctx->scratch_get(w.tmp_bytes);
    const int64_t nnz = sparse_phase_a(s, nt, I, J, m, n, end_bit, w, true);
    DevPtr start = dev_alloc(nnz * sizeof(int64_t));
    w.start = dp<int64_t>(start);
    M->nnz = nnz;
    M->rowval = dev_alloc(nnz * sizeof(int32_t));
    M->nzval = dev_alloc(nnz * sizeof(double));
    sparse_phase_b(s, nt, V, m, n, nnz, w, dp<int64_t>(M->colptr), dp<int32_t>(M->rowval), dp<double>(M->nzval));
    FEASM_HIP(hipStreamSynchronize(s));
    return M.release();
}

feasm_matrix *sparse_device(feasm_ctx *ctx, int64_t nt, const int32_t *I, const int32_t *J, const double *V,
                            int64_t m, int64_t n) {
    check_sparse_args(nt, m, n);
    if (nt > 0) {
        try {
            if (feasm_matrix *M = sparse_by_columns(ctx, nt, I, J, V, m, n)) return M;
        } catch (const Error &e) {
            if (e.code != FEASM_ENOMEM) throw;  // it takes more than the sort in a matrix of many columns
        }
        return sparse_by_sort(ctx, nt, I, J, V, m, n);
    }
    std::unique_ptr<feasm_matrix> M(new feasm_matrix);
    M->ctx = ctx;
    M->m = m;
    M->n = n;
    M->nnz = 0;
    M->colptr = dev_alloc((n + 1) * sizeof(int64_t));
    fill_i64(ctx->stream, dp<int64_t>(M->colptr), n + 1, 0);
    FEASM_HIP(hipStreamSynchronize(ctx->stream));
    return M.release();
}

}  // namespace feasm
