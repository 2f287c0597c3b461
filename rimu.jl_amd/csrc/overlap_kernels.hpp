// overlap_kernels.hpp -- overlaps of two device vectors: dot(t, u) and the three-way
// dot(t, op, u) = dot_from_right(t, op, u) (DictVectors/abstractdvec.jl:313-324), a sum over
// the entries (k, v) of u of  t[k] * diagonal_element(op, k) * v  plus, for an operator with
// off-diagonals,  t[k'] * h' * v  over every off-diagonal (k', h') of k.  These are the
// reductions behind AllOverlaps (replicastrategy.jl:112-183).
//
// Two kernels share the work.  overlap_kernel takes the dot and the diagonal operators: one
// thread per entry, a tile of consecutive entries of u per workgroup, t[k] found in the range
// of t that the tile's first and last key bound (staged in LDS when it holds at most ov_lds
// keys).  overlap_ham_kernel takes a Hamiltonian: OV_LANES lanes per entry share its
// off-diagonals, each a search of its own in t -- through an index of t by the top P key bits
// when the keys are stored mixed (spread evenly over their B bits: ranges of one or two
// keys), else with the first levels taken from OV_SPLIT evenly spaced keys of t staged in LDS.
// Per-workgroup partial sums are reduced in a fixed order (deterministic).
#pragma once

#include "step_kernels.hpp"

namespace rimu {

// Entries per thread of overlap_kernel: eight for long vectors, two while that leaves fewer
// than OV_MIN_TILES workgroups (a call with H and G2 on 20,000 entries takes 90 us with eight
// and 58 us with two, on 360,000 entries 359 and 328 us).
constexpr int OV_IPT = 8, OV_IPT_SHORT = 2;
constexpr int64_t OV_MIN_TILES = 1024;
constexpr int OV_LANES = 8;    // lanes per entry of overlap_ham_kernel
constexpr int OV_HAM_GRID = 4096;  // workgroups of overlap_ham_kernel at most
constexpr int OV_SPLIT = 1024;
constexpr int OV_MAX_OPS = 8;
constexpr int OV_LDS = 3072;   // t's keys of a tile's range staged in LDS when they fit
constexpr int OV_INDEX_MAX_BITS = 24;   // top-bit index of t for mixed keys: at most 2^24 + 1 entries
constexpr int64_t OV_INDEX_MIN = 1 << 12;  // smaller t: the LDS splitters suffice
template <class K> struct ov_lds { static constexpr int value = sizeof(K) == 8 ? OV_LDS : 2048; };

enum { OP_HAMILTONIAN = 1, OP_G2_REAL = 2, OP_DENSITY = 3 };

// The diagonal operators of a call, in the order of their output columns.
struct DiagOps {
    int n;
    int kind[OV_MAX_OPS];
    int param[OV_MAX_OPS];  // G2RealCorrelator: d; DensityMatrixDiagonal: mode (1-based)
};

// Where the partial sums of each output column lie.
struct OvColumns {
    int64_t first[1 + OV_MAX_OPS], count[1 + OV_MAX_OPS];
};

// G2RealCorrelator(d): (1/M) sum_i n_i (n_{i+d} - delta_{0d}), periodic
// (correlation_functions.jl:82-92); the integer sum is exact, then one division.
template <class A>
__device__ inline double g2_real(A bits, int M, int d) {
    const int dd = ((d % M) + M) % M;
    int64_t acc = 0;
    A x = bits;
    int mode = 1;
    while (x) {
        const int z = ctzA(x);
        mode += z;
        x = shrA(x, z);
        const int n = ctzA((A)~x);
        if (dd == 0) {
            acc += (int64_t)n * (n - 1);
        } else {
            int j = mode + dd;
            if (j > M) j -= M;
            acc += (int64_t)n * occupation(bits, j);
        }
        x = shrA(x, n);
    }
    return (double)acc / (double)M;
}

// Position of key in keys[a, b), or -1.
template <class K>
__device__ inline int64_t find_in(const K* __restrict__ keys, int64_t a, int64_t b, K key) {
    const int64_t end = b;
    while (a < b) {
        const int64_t mid = (a + b) >> 1;
        if (keys[mid] < key) a = mid + 1; else b = mid;
    }
    return (a < end && keys[a] == key) ? a : -1;
}

// Position of key in keys[0, L), or -1; s_split[j] = keys[j * L / OV_SPLIT].
template <class K>
__device__ inline int64_t find_split(const K* __restrict__ keys, int64_t L, const K* s_split, K key) {
    int lo = 0, hi = OV_SPLIT;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s_split[mid] <= key) lo = mid + 1; else hi = mid;
    }
    if (lo == 0) return -1;
    const int64_t a = (int64_t)(lo - 1) * L / OV_SPLIT;
    const int64_t b = lo < OV_SPLIT ? (int64_t)lo * L / OV_SPLIT : L;
    return find_in(keys, a, b, key);
}

// idx[b] = the first position in keys[0, L) whose top P of the B key bits are at least b,
// b = 0 .. 2^P (idx[2^P] = L < 2^32).  Position i writes idx[b] for b in (top(i - 1), top(i)]
// (i = 0 from b = 0; i = L up to 2^P), one coalesced pass over the keys.
template <class K>
__global__ __launch_bounds__(NT) void overlap_index_kernel(const K* __restrict__ keys, int64_t L, int B, int P,
                                                           uint32_t* __restrict__ idx) {
    const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (i > L) return;
    const int sh = B - P;
    const int64_t nb = (int64_t)1 << P;
    const int64_t lo = i == 0 ? 0 : (int64_t)(keys[i - 1] >> sh) + 1;
    const int64_t hi = i == L ? nb : (int64_t)(keys[i] >> sh);
    for (int64_t b = lo; b <= hi; ++b) idx[b] = (uint32_t)i;
}

// Position of key in its index range [idx[b], idx[b + 1]), b its top bits, or -1.  keys holds
// L >= 4 keys; four consecutive keys are read at once (two 16-byte loads for one-word keys,
// which need no more than the keys' own alignment), the window moved down where it would pass
// the end: a match anywhere in it is the key, since t's keys are unique.  So a lookup is
// mostly two dependent loads on two or three cache lines.  (Halving a range of 16 keys reads
// one key after another; with hundreds of thousands of lookups in flight their lines left the
// caches in between: 8.5e6 entries of a 20-site chain took 10.9 ms so with few workgroups in
// flight and 16.8 ms with many; with the index 9.2 ms.)
template <class K>
__device__ inline int64_t find_index(const K* __restrict__ keys, int64_t L, const uint32_t* __restrict__ idx, int tsh,
                                     K key) {
    uint32_t r[2];
    __builtin_memcpy(r, idx + (int64_t)(key >> tsh), sizeof(r));
    for (uint32_t a = r[0]; a < r[1]; a += 4) {
        const int64_t w = min((int64_t)a, L - 4);
        K k[4];
        __builtin_memcpy(k, keys + w, sizeof(k));
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (k[j] == key) return w + j;
    }
    return -1;
}

// ranges[t] = lower bound in t of u's key at t * tile (t < ntiles), ranges[ntiles] = Lt.
// u's keys are unique, so tile t's keys lie in t[ranges[t], ranges[t + 1]).
template <class K>
__global__ __launch_bounds__(NT) void overlap_ranges_kernel(const K* __restrict__ tk, int64_t Lt,
                                                            const K* __restrict__ uk, int64_t tile,
                                                            int64_t ntiles, int64_t* __restrict__ ranges) {
    const int64_t t = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (t > ntiles) return;
    if (t == ntiles) { ranges[t] = Lt; return; }
    const K key = uk[t * tile];
    int64_t a = 0, b = Lt;
    while (a < b) {
        const int64_t mid = (a + b) >> 1;
        if (tk[mid] < key) a = mid + 1; else b = mid;
    }
    ranges[t] = a;
}

// partials[o * gridDim.x + block], o = 0 (dot) .. ops.n (operators).  Lt >= 1, Lu >= 1.
template <class K, class VT, class VU, int IPT>
__global__ __launch_bounds__(NT) void overlap_kernel(const K* __restrict__ tk,
                                                     const VT* __restrict__ tv, int64_t Lt,
                                                     const K* __restrict__ uk,
                                                     const VU* __restrict__ uv, int64_t Lu,
                                                     DiagOps ops, KeyMix mix, int M,
                                                     const int64_t* __restrict__ ranges,
                                                     double* __restrict__ partials) {
    constexpr int LDSN = ov_lds<K>::value;
    __shared__ K s_lk[LDSN];
    __shared__ double s_sum[1 + OV_MAX_OPS][NT / WAVE];
    const int64_t t0 = (int64_t)blockIdx.x * (NT * IPT);
    const int64_t lo = ranges[blockIdx.x], hi = ranges[blockIdx.x + 1];
    const bool staged = hi - lo <= LDSN;
    if (staged) {
        const int n = (int)(hi - lo);
        for (int j = threadIdx.x; j < n; j += NT) s_lk[j] = tk[lo + j];
    }
    __syncthreads();

    K k[IPT];
    double v[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const int64_t i = t0 + (int64_t)j * NT + threadIdx.x;
        const int64_t ic = min(i, Lu - 1);
        k[j] = uk[ic];
        v[j] = i < Lu ? (double)uv[ic] : 0.0;
    }
    double acc[1 + OV_MAX_OPS];
#pragma unroll
    for (int o = 0; o <= OV_MAX_OPS; ++o) acc[o] = 0.0;
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const int64_t i = t0 + (int64_t)j * NT + threadIdx.x;
        if (i >= Lu) continue;
        int64_t p;
        if (staged) {
            int a = 0, b = (int)(hi - lo);
            const int n = b;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (s_lk[mid] < k[j]) a = mid + 1; else b = mid;
            }
            p = (a < n && s_lk[a] == k[j]) ? lo + a : -1;
        } else {
            p = find_in(tk, lo, hi, k[j]);
        }
        const double tval = p >= 0 ? (double)tv[p] : 0.0;
        acc[0] += tval * v[j];
        const K key = unmix_key(mix, k[j]);  // the address
#pragma unroll
        for (int o = 0; o < OV_MAX_OPS; ++o) {
            if (o < ops.n)
                acc[1 + o] += tval * (ops.kind[o] == OP_G2_REAL ? g2_real(key, M, ops.param[o])
                                                                : (double)occupation(key, ops.param[o])) * v[j];
        }
    }
    block_sums<NT, 1 + OV_MAX_OPS>(acc, s_sum);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int o = 0; o <= OV_MAX_OPS; ++o)
            if (o <= ops.n) partials[(int64_t)o * gridDim.x + blockIdx.x] = acc[o];
    }
}

// partials[block] = sum over u's entries (k, v) of t[k] diag(k) v + sum t[k'] h' v over the
// off-diagonals (k', h') of k.  Bound by the dependent loads of a search (an index
// range, its keys, the value): OV_LANES lanes take every OV_LANES-th off-diagonal
// of an entry, lane 0 its diagonal too, so a short vector still fills the chip (20,000 entries
// of a 20-site chain took 754 us a call with one thread per entry and its 26 searches in a
// row, now 55 us; 360,000 entries 668 and 226 us).
// tidx null: no index, the LDS splitters are used.
template <bool RS, class K, class VT, class VU>
__global__ __launch_bounds__(NT) void overlap_ham_kernel(ModelDev h, KeyMix mix, const K* __restrict__ tk,
                                                         const VT* __restrict__ tv, int64_t Lt,
                                                         const K* __restrict__ uk, const VU* __restrict__ uv,
                                                         int64_t Lu, const uint32_t* __restrict__ tidx, int tsh,
                                                         double* __restrict__ partials) {
    __shared__ K s_split[OV_SPLIT];
    __shared__ double s_sum[1][NT / WAVE];
    if (!tidx)
        for (int j = threadIdx.x; j < OV_SPLIT; j += NT) s_split[j] = tk[(int64_t)j * Lt / OV_SPLIT];
    __syncthreads();
    auto position = [&](K key) -> int64_t {  // of key in t, or -1
        return tidx ? find_index(tk, Lt, tidx, tsh, key) : find_split(tk, Lt, s_split, key);
    };
    constexpr int EPB = NT / OV_LANES;  // entries per workgroup and round
    const int sub = threadIdx.x % OV_LANES;
    double acc[1] = {0.0};
    for (int64_t e = (int64_t)blockIdx.x * EPB + threadIdx.x / OV_LANES; e < Lu; e += (int64_t)gridDim.x * EPB) {
        const K skey = uk[e];
        const double v = (double)uv[e];
        const K key = unmix_key(mix, skey);
        if (sub == 0) {
            const int64_t q = position(skey);
            acc[0] += (q >= 0 ? (double)tv[q] : 0.0) * model_diagonal_element<RS>(h, key) * v;
        }
        const int64_t n = model_num_offdiagonals<RS>(h, key);
        for (int64_t c = 1 + sub; c <= n; c += OV_LANES) {
            double hv;
            const K nb = mix_key(mix, model_offdiagonal<RS>(h, key, c, &hv));
            if (hv == 0.0) continue;
            const int64_t q = position(nb);
            if (q >= 0) acc[0] += (double)tv[q] * hv * v;
        }
    }
    block_sums<NT, 1>(acc, s_sum);
    if (threadIdx.x == 0) partials[blockIdx.x] = acc[0];
}

// out[o] = sum of column o's partials in a fixed order; one workgroup per column.  out is
// pinned host memory.
__global__ __launch_bounds__(NT) void overlap_final_kernel(const double* __restrict__ partials, OvColumns c,
                                                           double* __restrict__ out) {
    __shared__ double s_sum[1][NT / WAVE];
    const int o = blockIdx.x;
    const double* p = partials + c.first[o];
    const int64_t n = c.count[o];
    double acc[1] = {0.0};
    for (int64_t b0 = 0; b0 < n; b0 += 8 * NT) {
        double x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t b = b0 + j * NT + threadIdx.x;
            x[j] = b < n ? p[b] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[0] += x[j];
    }
    block_sums<NT, 1>(acc, s_sum);
    if (threadIdx.x == 0) out[o] = acc[0];
}

}  // namespace rimu
