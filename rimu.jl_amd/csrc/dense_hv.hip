// dense_hv.hip -- deterministic H.v on the ranked basis of HubbardReal1D, its adjoint, and
// the checkpointed adjoint of a K-step projection (the C ABI rimu_dense_* of rimu_hip.h).
//
// Row r of a vector is the address of colex rank r: the N one-bits of the address at
// positions p_0 < p_1 < ... give rank = sum_j C(p_j, j+1), and colex order equals
// ascending numeric order of the bit strings.  A hop moves one boson by one bit, so the
// rank of a neighbour follows from the row's own rank with one binomial, which depends only on
// the bond and on the bosons below it (a small table in LDS).  Hops across the periodic
// boundary rotate the string; their ranks are laid out with the basis.
//
// Vectors are row-major [dim][R] (R right-hand sides, one per Hamiltonian): a neighbour's
// R amplitudes are one contiguous 8R-byte load.  Every reduction is a fixed-order tree,
// so results are deterministic.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "bosefs_device.hpp"
#include "capi_util.hpp"
#include "device_common.hpp"

using namespace rimu;

namespace {

constexpr int DT = 256;          // workgroup size
constexpr int MAXR = 8;          // right-hand sides per launch
constexpr int BINOM_N = 65;      // C(n, k) for 0 <= n, k <= 64

struct DenseParams {
    double a[MAXR], b[MAXR], u[MAXR], t[MAXR];
    int M, N;
};

// Colex rank from scratch.
__device__ inline int64_t colex_rank(uint64_t bits, const int64_t* __restrict__ binom) {
    int64_t r = 0;
    int j = 1;
    while (bits) {
        const int p = __builtin_ctzll(bits);
        r += binom[p * BINOM_N + j];
        ++j;
        bits &= bits - 1;
    }
    return r;
}

// Tables of one (M, N), built on the host and copied to LDS by every workgroup of a product:
//   delta[i * (N + 2) + s] = C(s + i - 2, s - 1): the rank change of a hop from mode i to mode
//     i + 1 (1 <= i < M) when modes 1 .. i hold s bosons before it (0 for s = 0); the hop back
//     from mode i + 1 when they hold s - 1 changes the rank by the same amount down;
//   root[x] = sqrt(x), x <= (N + 1)^2 / 4 >= n (n' + 1), the hop amplitudes.
struct HopTables {
    const uint32_t* delta;
    const double* root;
    int n_delta, n_root;
};

__device__ inline void stage_hop_tables(const HopTables& t, double* s_root, uint32_t* s_delta) {
    for (int j = threadIdx.x; j < t.n_root; j += DT) s_root[j] = t.root[j];
    for (int j = threadIdx.x; j < t.n_delta; j += DT) s_delta[j] = t.delta[j];
    __syncthreads();
}

// Rank of the neighbour across the periodic boundary: rot[r].x after a hop from mode M to
// mode 1 (the string rotates up), rot[r].y after one from mode 1 to mode M; r where that mode
// is empty.  Every bit moves, so these are ranked once, when the basis is laid out.
__global__ __launch_bounds__(DT) void dense_rotations_kernel(const uint64_t* __restrict__ basis, int64_t D, int B,
                                                             const int64_t* __restrict__ binom,
                                                             uint2* __restrict__ rot) {
    const int64_t r = (int64_t)blockIdx.x * DT + threadIdx.x;
    if (r >= D) return;
    const uint64_t bits = basis[r];
    const uint64_t top = 1ull << (B - 1);
    uint2 o = {(uint32_t)r, (uint32_t)r};
    if (bits & top) o.x = (uint32_t)colex_rank(((bits << 1) | 1ull) & low_mask(B), binom);
    if (bits & 1ull) o.y = (uint32_t)colex_rank((bits >> 1) | top, binom);
    rot[r] = o;
}

// Workgroup -> tile of rows.  Workgroups go to the eight XCDs in turn; giving each XCD a
// contiguous eighth of the rows keeps the near neighbours of its rows in its own L2.
__device__ inline int64_t dense_tile(int64_t b, int64_t n) {
    const int64_t per = n >> 3;
    return b < per * 8 ? (b & 7) * per + (b >> 3) : b;
}

// acc[i] += -s_root[x] * v[k][i], or zero where the row r has no such hop (it loads itself).
template <int R>
__device__ inline void add_hop(bool has, int64_t r, int64_t k, int x, const double* s_root,
                               const double* __restrict__ v, double (&acc)[R]) {
    const double* vk = v + (has ? k : r) * R;
    const double amp = -s_root[has ? x : 0];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const double y = vk[i];
        acc[i] = fma(amp, has ? y : 0.0, acc[i]);
    }
}

// K v at row r (K: the hopping with unit amplitude, elements -sqrt(n (n' + 1))): acc[i] =
// sum over hops of -sqrt * v[neighbour][i]; returns sum n(n - 1) / 2 of the address.
// One pass over the M - 1 bonds and the boundary, both directions of a bond from the same
// occupations, the same instructions in every lane: a hop that the address does not have loads
// the row itself and adds zero.  Per bond two table reads, two gathers of 8R bytes and 2R fused
// multiply-adds.  Bound by the gathers that miss the L2: at dimension 1,352,078, R = 4 they
// bring in 265 MB a product (v alone is 43 MB) at 4.8 TB/s.  (Walking each lane's own occupied
// modes with popcounts, clz and an f64 sqrt per hop took 106 us a product there.)
template <int R>
__device__ inline int hop_sum_bonds(uint64_t bits, int64_t r, int M, int row_len, uint2 rot,
                                    const double* s_root, const uint32_t* s_delta,
                                    const double* __restrict__ v, double (&acc)[R]) {
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = 0.0;
    uint64_t x = bits;
    const int n1 = __builtin_ctzll(~x);  // M >= 2: an address has a zero bit
    x = shr(x, n1 + 1);
    int nc = n1, s = n1;
    int pairs = n1 * (n1 - 1) / 2;
    const uint32_t* dl = s_delta + row_len;  // mode 1
#pragma unroll 2
    for (int m = 1; m < M; ++m, dl += row_len) {
        const int nn = ctz64(~x);
        x = shr(x, nn + 1);
        add_hop<R>(nc > 0, r, r + dl[s], nc * (nn + 1), s_root, v, acc);
        add_hop<R>(nn > 0, r, r - (int64_t)dl[s + 1], nn * (nc + 1), s_root, v, acc);
        s += nn;
        nc = nn;
        pairs += nn * (nn - 1) / 2;
    }
    add_hop<R>(nc > 0, r, rot.x, nc * (n1 + 1), s_root, v, acc);
    add_hop<R>(n1 > 0, r, rot.y, n1 * (nc + 1), s_root, v, acc);
    return pairs;
}

// The same sum over the occupied modes only, left hop then right hop, modes ascending: the
// hops in the order of their bonds, so the same additions and the same bits as hop_sum_bonds.
template <int R>
__device__ inline int hop_sum_occupied(uint64_t bits, int64_t r, int M, int row_len, uint2 rot,
                                       const double* s_root, const uint32_t* s_delta,
                                       const double* __restrict__ v, double (&acc)[R]) {
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = 0.0;
    const int n1 = __builtin_ctzll(~bits);
    uint64_t x = bits;
    int m = 1, n = 0, s = 0, pairs = 0;  // the last run's mode and bosons, the bosons so far
    while (x) {
        const int z = __builtin_ctzll(x);  // modes further on
        const int before = z == 1 ? n : 0;
        m += z;
        x >>= z;
        n = ctz64(~x);
        x = shr(x, n);
        const int after = __builtin_ctzll(~(x >> 1));
        add_hop<R>(m > 1, r, r - (int64_t)s_delta[(m - 1) * row_len + s + 1], n * (before + 1), s_root, v, acc);
        s += n;
        add_hop<R>(m < M, r, r + s_delta[(m < M ? m : 0) * row_len + s], n * (after + 1), s_root, v, acc);
        pairs += n * (n - 1) / 2;
    }
    const int nM = m == M ? n : 0;
    add_hop<R>(nM > 0, r, rot.x, nM * (n1 + 1), s_root, v, acc);
    add_hop<R>(n1 > 0, r, rot.y, n1 * (nM + 1), s_root, v, acc);
    return pairs;
}

template <int R, bool OCC>
__device__ inline int hop_sum(uint64_t bits, int64_t r, int M, int row_len, uint2 rot, const double* s_root,
                              const uint32_t* s_delta, const double* __restrict__ v, double (&acc)[R]) {
    return OCC ? hop_sum_occupied<R>(bits, r, M, row_len, rot, s_root, s_delta, v, acc)
               : hop_sum_bonds<R>(bits, r, M, row_len, rot, s_root, s_delta, v, acc);
}

// Whether a product walks the occupied modes instead of all bonds.  A wavefront takes as many turns
// as its fullest row has occupied modes, up to N, against M: but a turn that finds a run costs more
// than a bond, and a bond that holds no boson only loads its own row (8R bytes, from the caches).
// Where the line lies, in ms for 200 projector steps with their adjoint, walk against bonds:
//   R = 4: N/M = 0.07 (60 modes) 14.5 : 48.2, 0.25 (24) 14.6 : 22.0, 0.42 (12) 4.1 : 4.2,
//          0.50 (12) 4.4 : 4.2, 0.64 (14) 17.5 : 17.5, 1 (12) 43.4 : 38.8
//   R = 1: 0.42 3.35 : 3.35, 0.50 3.6 : 3.4, 0.64 8.0 : 7.9, 1 17.2 : 15.0
//   R = 8: 0.50 (16) 40.0 : 47.9, 0.67 (12) 10.3 : 12.0, 0.83 (12) 32.6 : 31.2 (5 and 6 alike)
bool walk_occupied(int M, int N, int R) { return R > 4 ? 3 * N <= 2 * M : 2 * N < M; }

// w = (a + b H) v, one thread per row.  DOT: also per-block partials[i][block] of <v|w>.
template <int R, bool DOT, bool OCC>
__global__ __launch_bounds__(DT) void dense_apply_kernel(const uint64_t* __restrict__ basis,
                                                         const uint2* __restrict__ rot, int64_t D,
                                                         DenseParams p, HopTables t,
                                                         const double* __restrict__ v,
                                                         double* __restrict__ w, double* __restrict__ partials) {
    extern __shared__ double s_tab[];
    uint32_t* s_delta = (uint32_t*)(s_tab + t.n_root);
    stage_hop_tables(t, s_tab, s_delta);
    const int64_t tile = dense_tile(blockIdx.x, gridDim.x);
    const int64_t r = tile * DT + threadIdx.x;
    double dt[R];
#pragma unroll
    for (int i = 0; i < R; ++i) dt[i] = 0.0;
    if (r < D) {
        double acc[R];
        const double dr = (double)hop_sum<R, OCC>(basis[r], r, p.M, p.N + 2, rot[r], s_tab, s_delta, v, acc);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const double vr = v[r * R + i];
            const double x = (p.a[i] + p.b[i] * (p.u[i] * dr)) * vr + p.b[i] * (p.t[i] * acc[i]);
            w[r * R + i] = x;
            dt[i] = vr * x;
        }
    }
    if constexpr (DOT) {
        __shared__ double s_sum[R][DT / WAVE];
        block_sums<DT, R>(dt, s_sum);
        if (threadIdx.x == 0)
#pragma unroll
            for (int i = 0; i < R; ++i) partials[(int64_t)i * gridDim.x + tile] = dt[i];
    }
}

// Pullback: vbar = (a + b H) ybar; per-block partial sums of b <ybar|D|v> and b <ybar|K|v>
// written to partials[2R][blocks].  K is real symmetric, so <ybar|K|v> = sum_r v_r (K ybar)_r
// and only ybar is gathered at the neighbours.
template <int R, bool OCC>
__global__ __launch_bounds__(DT) void dense_pullback_kernel(const uint64_t* __restrict__ basis,
                                                            const uint2* __restrict__ rot, int64_t D,
                                                            DenseParams p, HopTables t,
                                                            const double* __restrict__ v,
                                                            const double* __restrict__ ybar,
                                                            double* __restrict__ vbar,
                                                            double* __restrict__ partials) {
    extern __shared__ double s_tab[];
    __shared__ double s_sum[2 * R][DT / WAVE];
    uint32_t* s_delta = (uint32_t*)(s_tab + t.n_root);
    stage_hop_tables(t, s_tab, s_delta);
    const int64_t tile = dense_tile(blockIdx.x, gridDim.x);
    const int64_t r = tile * DT + threadIdx.x;
    double ps[2 * R];
#pragma unroll
    for (int i = 0; i < 2 * R; ++i) ps[i] = 0.0;
    if (r < D) {
        double ky[R];
        const double dr = (double)hop_sum<R, OCC>(basis[r], r, p.M, p.N + 2, rot[r], s_tab, s_delta, ybar, ky);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const double yr = ybar[r * R + i];
            const double vr = v[r * R + i];
            vbar[r * R + i] = (p.a[i] + p.b[i] * (p.u[i] * dr)) * yr + p.b[i] * (p.t[i] * ky[i]);
            ps[i] = p.b[i] * (yr * (dr * vr));
            ps[R + i] = p.b[i] * (vr * ky[i]);
        }
    }
    block_sums<DT, 2 * R>(ps, s_sum);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < 2 * R; ++i) partials[(int64_t)i * gridDim.x + tile] = ps[i];
}

// out[i] = sum_r x[r][i] * y[r][i] as per-block partials[R][blocks].
template <int R>
__global__ __launch_bounds__(DT) void dense_dot_kernel(const double* __restrict__ x, const double* __restrict__ y,
                                                       int64_t D, double* __restrict__ partials) {
    __shared__ double s_sum[R][DT / WAVE];
    const int64_t r = (int64_t)blockIdx.x * DT + threadIdx.x;
    double ps[R];
#pragma unroll
    for (int i = 0; i < R; ++i) ps[i] = r < D ? x[r * R + i] * y[r * R + i] : 0.0;
    block_sums<DT, R>(ps, s_sum);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < R; ++i) partials[(int64_t)i * gridDim.x + blockIdx.x] = ps[i];
}

// out[c] (+)= sum over blocks of partials[c][block], one workgroup per c; every thread's loads
// are in flight together (with one load at a time 9.1 us at 5282 blocks).
constexpr int RED_NT = 1024;
__global__ __launch_bounds__(RED_NT) void reduce_rows_kernel(const double* __restrict__ partials, int64_t blocks,
                                                             double* __restrict__ out, int accumulate) {
    __shared__ double s[RED_NT / WAVE];
    const double* p = partials + (int64_t)blockIdx.x * blocks;
    double acc = 0;
    for (int64_t b0 = 0; b0 < blocks; b0 += 8 * RED_NT) {
        double x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t b = b0 + j * RED_NT + threadIdx.x;
            x[j] = b < blocks ? p[b] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += x[j];
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) s[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = s[0];
        for (int w = 1; w < RED_NT / WAVE; ++w) t += s[w];
        out[blockIdx.x] = accumulate ? out[blockIdx.x] + t : t;
    }
}

// lambda = 2 (Hv - E v) / <v|v>, per right-hand side (gradient of the Rayleigh quotient).
template <int R>
__global__ __launch_bounds__(DT) void rq_gradient_kernel(const double* __restrict__ v, const double* __restrict__ hv,
                                                         const double* __restrict__ dots /* [vv R][vHv R] */,
                                                         int64_t D, double* __restrict__ lam) {
    const int64_t r = (int64_t)blockIdx.x * DT + threadIdx.x;
    if (r >= D) return;
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const double vv = dots[i], e = dots[R + i] / vv;
        lam[r * R + i] = 2.0 * (hv[r * R + i] - e * v[r * R + i]) / vv;
    }
}

// 1 / sqrt(n2), or zero where the norm has fallen to `floor2` or below: a right-hand side whose
// Krylov space is exhausted goes on with zero vectors.
__device__ inline double lanczos_scale(double n2, double floor2) { return n2 > floor2 ? 1.0 / sqrt(n2) : 0.0; }

// The start vector over its norm, n2 = |x|^2, and one for the squared norm that the first update
// takes: <x|Hx> of a vector as it was given may overflow or underflow where |x|^2 does not.
__global__ __launch_bounds__(DT) void lanczos_start_kernel(double* __restrict__ x, int64_t D, int R,
                                                           const double* __restrict__ n2, double* __restrict__ x2) {
    const int64_t r = (int64_t)blockIdx.x * DT + threadIdx.x;
    for (int i = 0; i < R; ++i) {
        if (r < D) x[r * R + i] = n2[i] > 0.0 ? x[r * R + i] / sqrt(n2[i]) : 0.0;
        if (r == 0) x2[i] = 1.0;
    }
}

// One three-term Lanczos update per right-hand side.  The vectors are kept unnormalised with
// their squared norms in device memory: v_j = x / sqrt(x2), v_{j-1} = y / sqrt(y2), and w = H x,
// so H v_j = w / sqrt(x2) and alpha_j = <v_j|H v_j> = xw / x2.  Writes
// w <- H v_j - alpha_j v_j - beta_j v_{j-1} (beta_j = sqrt(x2), the norm x had as w) with the
// partial sums of |w|^2 of each block in partials[R][blocks], and alpha_j.  (Writing v_{j+1} out
// was a pass of its own: 7.7 of 46 us an iteration at dimension 352,716, R = 4.)
template <int R>
__global__ __launch_bounds__(DT) void lanczos_orth_kernel(double* __restrict__ w, const double* __restrict__ x,
                                                          const double* __restrict__ y,
                                                          const double* __restrict__ xw, const double* __restrict__ x2,
                                                          const double* __restrict__ y2, double floor_x, double floor_y, int first,
                                                          int64_t D, double* __restrict__ alpha,
                                                          double* __restrict__ partials) {
    __shared__ double s_sum[R][DT / WAVE];
    __shared__ double s_c[4][R];
    // the row's loads travel while one thread per right-hand side prepares the scalars (square
    // roots and divisions in every thread, or before the loads, cost 15 to 19 us a call)
    const int64_t r = (int64_t)blockIdx.x * DT + threadIdx.x;
    const int64_t rc = min(r, D - 1);
    double wr[R], xr[R], yr[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        wr[i] = w[rc * R + i];
        xr[i] = x[rc * R + i];
        yr[i] = first ? 0.0 : y[rc * R + i];
    }
    if (threadIdx.x < R) {
        const int i = threadIdx.x;
        const double s = lanczos_scale(x2[i], floor_x);
        s_c[0][i] = s;
        s_c[1][i] = first ? 0.0 : lanczos_scale(y2[i], floor_y);
        s_c[2][i] = (xw[i] * s) * s;
        s_c[3][i] = first ? 0.0 : sqrt(x2[i]);
        if (blockIdx.x == 0) alpha[i] = s_c[2][i];
    }
    __syncthreads();
    double ps[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const double sx = s_c[0][i], vp = yr[i] * s_c[1][i];
        const double z = wr[i] * sx - s_c[2][i] * (xr[i] * sx) - s_c[3][i] * vp;
        if (r < D) w[r * R + i] = z;
        ps[i] = r < D ? z * z : 0.0;
    }
    block_sums<DT, R>(ps, s_sum);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < R; ++i) partials[(int64_t)i * gridDim.x + blockIdx.x] = ps[i];
}

}  // namespace

struct rimu_dense {
    int R = 0;
    int M = 0, N = 0, B = 0;
    int64_t D = 0;
    rimu_model models[MAXR];
    hipStream_t stream = nullptr;
    DevBuf<uint64_t> basis;
    DevBuf<uint2> rot;
    DevBuf<double> tab;  // root table, then the hop table (uint32), then the binomials (int64)
    DevBuf<double> x, y, z, hist, partials, scal;
    double* h_scal = nullptr;  // pinned, 8 * MAXR
};

namespace {

DenseParams params(const rimu_dense* d, const double* a, const double* b) {
    DenseParams p{};
    for (int i = 0; i < d->R; ++i) {
        p.a[i] = a[i];
        p.b[i] = b[i];
        p.u[i] = d->models[i].u;
        p.t[i] = d->models[i].t;
    }
    p.M = d->M;
    p.N = d->N;
    return p;
}

HopTables tables(const rimu_dense* d) {
    const int n_root = (d->N + 1) * (d->N + 1) / 4 + 1;
    return HopTables{(const uint32_t*)(d->tab.p + n_root), d->tab.p, d->M * (d->N + 2), n_root};
}
size_t table_bytes(const HopTables& t) { return sizeof(double) * t.n_root + sizeof(uint32_t) * t.n_delta; }

// w = (a + b H) v; with out also out[i] = <v_i|w_i>
template <int R>
int launch_apply(rimu_dense* d, const DenseParams& p, const double* v, double* w, double* out) {
    const HopTables t = tables(d);
    const int64_t blocks = ceil_div(d->D, DT);
    const bool occ = walk_occupied(d->M, d->N, R);
    if (out) {
        HIP_TRY(d->partials.alloc((size_t)blocks * R));
        const auto product = occ ? dense_apply_kernel<R, true, true> : dense_apply_kernel<R, true, false>;
        product<<<blocks, DT, table_bytes(t), d->stream>>>(d->basis.p, d->rot.p, d->D, p, t, v, w, d->partials.p);
        reduce_rows_kernel<<<R, RED_NT, 0, d->stream>>>(d->partials.p, blocks, out, 0);
    } else {
        const auto product = occ ? dense_apply_kernel<R, false, true> : dense_apply_kernel<R, false, false>;
        product<<<blocks, DT, table_bytes(t), d->stream>>>(d->basis.p, d->rot.p, d->D, p, t, v, w, nullptr);
    }
    HIP_TRY(hipGetLastError());
    return RIMU_OK;
}

int apply(rimu_dense* d, const DenseParams& p, const double* v, double* w, double* out = nullptr) {
    switch (d->R) {
        case 1: return launch_apply<1>(d, p, v, w, out);
        case 2: return launch_apply<2>(d, p, v, w, out);
        case 3: return launch_apply<3>(d, p, v, w, out);
        case 4: return launch_apply<4>(d, p, v, w, out);
        case 5: return launch_apply<5>(d, p, v, w, out);
        case 6: return launch_apply<6>(d, p, v, w, out);
        case 7: return launch_apply<7>(d, p, v, w, out);
        default: return launch_apply<8>(d, p, v, w, out);
    }
}

// vbar and the (u, t) cotangents; cot receives [ubar R][tbar R] (added to it if accumulate)
template <int R>
int launch_pullback(rimu_dense* d, const DenseParams& p, const double* v, const double* ybar,
                    double* vbar, double* cot, int accumulate) {
    const HopTables t = tables(d);
    const int64_t blocks = ceil_div(d->D, DT);
    HIP_TRY(d->partials.alloc((size_t)blocks * 2 * R));
    const auto product = walk_occupied(d->M, d->N, R) ? dense_pullback_kernel<R, true> : dense_pullback_kernel<R, false>;
    product<<<blocks, DT, table_bytes(t), d->stream>>>(d->basis.p, d->rot.p, d->D, p, t, v, ybar, vbar, d->partials.p);
    reduce_rows_kernel<<<2 * R, RED_NT, 0, d->stream>>>(d->partials.p, blocks, cot, accumulate);
    HIP_TRY(hipGetLastError());
    return RIMU_OK;
}

int pullback(rimu_dense* d, const DenseParams& p, const double* v, const double* ybar, double* vbar,
             double* cot, int accumulate) {
    switch (d->R) {
        case 1: return launch_pullback<1>(d, p, v, ybar, vbar, cot, accumulate);
        case 2: return launch_pullback<2>(d, p, v, ybar, vbar, cot, accumulate);
        case 3: return launch_pullback<3>(d, p, v, ybar, vbar, cot, accumulate);
        case 4: return launch_pullback<4>(d, p, v, ybar, vbar, cot, accumulate);
        case 5: return launch_pullback<5>(d, p, v, ybar, vbar, cot, accumulate);
        case 6: return launch_pullback<6>(d, p, v, ybar, vbar, cot, accumulate);
        case 7: return launch_pullback<7>(d, p, v, ybar, vbar, cot, accumulate);
        default: return launch_pullback<8>(d, p, v, ybar, vbar, cot, accumulate);
    }
}

template <int R>
int launch_dot(rimu_dense* d, const double* x, const double* y, double* out) {
    const int64_t blocks = ceil_div(d->D, DT);
    HIP_TRY(d->partials.alloc((size_t)blocks * R));
    dense_dot_kernel<R><<<blocks, DT, 0, d->stream>>>(x, y, d->D, d->partials.p);
    reduce_rows_kernel<<<R, RED_NT, 0, d->stream>>>(d->partials.p, blocks, out, 0);
    HIP_TRY(hipGetLastError());
    return RIMU_OK;
}

int dot(rimu_dense* d, const double* x, const double* y, double* out) {
    switch (d->R) {
        case 1: return launch_dot<1>(d, x, y, out);
        case 2: return launch_dot<2>(d, x, y, out);
        case 3: return launch_dot<3>(d, x, y, out);
        case 4: return launch_dot<4>(d, x, y, out);
        case 5: return launch_dot<5>(d, x, y, out);
        case 6: return launch_dot<6>(d, x, y, out);
        case 7: return launch_dot<7>(d, x, y, out);
        default: return launch_dot<8>(d, x, y, out);
    }
}

int rq_gradient(rimu_dense* d, const double* v, const double* hv, const double* dots, double* lam) {
    const int64_t blocks = ceil_div(d->D, DT);
    switch (d->R) {
        case 1: rq_gradient_kernel<1><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 2: rq_gradient_kernel<2><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 3: rq_gradient_kernel<3><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 4: rq_gradient_kernel<4><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 5: rq_gradient_kernel<5><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 6: rq_gradient_kernel<6><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        case 7: rq_gradient_kernel<7><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
        default: rq_gradient_kernel<8><<<blocks, DT, 0, d->stream>>>(v, hv, dots, d->D, lam); break;
    }
    HIP_TRY(hipGetLastError());
    return RIMU_OK;
}

template <int R>
int launch_lanczos(rimu_dense* d, double* w, const double* x, const double* y, const double* xw, const double* x2,
                   const double* y2, double floor_x, double floor_y, int first, double* alpha,
                   double* norm2_out) {
    const int64_t blocks = ceil_div(d->D, DT);
    HIP_TRY(d->partials.alloc((size_t)blocks * R));
    lanczos_orth_kernel<R><<<blocks, DT, 0, d->stream>>>(w, x, y, xw, x2, y2, floor_x, floor_y, first, d->D, alpha,
                                                         d->partials.p);
    reduce_rows_kernel<<<R, RED_NT, 0, d->stream>>>(d->partials.p, blocks, norm2_out, 0);
    HIP_TRY(hipGetLastError());
    return RIMU_OK;
}

int lanczos_update(rimu_dense* d, double* w, const double* x, const double* y, const double* xw, const double* x2,
                   const double* y2, double floor_x, double floor_y, int first, double* alpha,
                   double* norm2_out) {
    switch (d->R) {
        case 1: return launch_lanczos<1>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 2: return launch_lanczos<2>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 3: return launch_lanczos<3>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 4: return launch_lanczos<4>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 5: return launch_lanczos<5>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 6: return launch_lanczos<6>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        case 7: return launch_lanczos<7>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
        default: return launch_lanczos<8>(d, w, x, y, xw, x2, y2, floor_x, floor_y, first, alpha, norm2_out);
    }
}

// Lowest eigenvalue of the symmetric tridiagonal matrix with diagonal a[0..m) and squared
// off-diagonal b2[1..m) (b2[k] couples k-1 and k), by bisection on the Sturm count: the
// number of negative pivots of T - x I is the number of eigenvalues below x.
double tridiag_lowest(const double* a, const double* b2, int64_t m) {
    double lo = INFINITY, hi = -INFINITY;
    for (int64_t k = 0; k < m; ++k) {
        const double off = (k > 0 ? sqrt(b2[k]) : 0.0) + (k + 1 < m ? sqrt(b2[k + 1]) : 0.0);
        lo = std::min(lo, a[k] - off);
        hi = std::max(hi, a[k] + off);
    }
    auto below = [&](double x) {
        int64_t c = 0;
        double piv = 1.0;
        for (int64_t k = 0; k < m; ++k) {
            piv = a[k] - x - (k > 0 ? b2[k] / piv : 0.0);
            if (piv == 0.0) piv = -1e-300;
            if (piv < 0) ++c;
        }
        return c;
    };
    for (int it = 0; it < 200 && hi - lo > 1e-15 * std::max(1.0, std::fabs(lo)); ++it) {
        const double mid = 0.5 * (lo + hi);
        if (below(mid) >= 1) hi = mid; else lo = mid;
    }
    return 0.5 * (lo + hi);
}

bool binomial64(int n, int k, int64_t* out) {
    if (k < 0 || k > n) { *out = 0; return true; }
    unsigned __int128 c = 1;
    for (int i = 1; i <= k; ++i) {
        c = c * (unsigned)(n - k + i) / (unsigned)i;
        if (c > (unsigned __int128)INT64_MAX) return false;
    }
    *out = (int64_t)c;
    return true;
}

}  // namespace

extern "C" {

int rimu_basis_size(int32_t M, int32_t N, int64_t* dim) {
    if (!dim) return fail(RIMU_ERR_ARG, "dim is null");
    if (M < 1 || N < 0 || M + N - 1 > 64) return fail(RIMU_ERR_ARG, "need N + M - 1 <= 64");
    if (!binomial64(N + M - 1, N, dim)) return fail(RIMU_ERR_ARG, "dimension overflows int64");
    return RIMU_OK;
}

int rimu_dense_create(const rimu_model* models, int32_t nrhs, rimu_dense** out) {
    if (!out || !models) return fail(RIMU_ERR_ARG, "null argument");
    *out = nullptr;
    if (nrhs < 1 || nrhs > MAXR) return fail(RIMU_ERR_ARG, "nrhs must be in 1..8");
    const rimu_model& m0 = models[0];
    for (int i = 0; i < nrhs; ++i) {
        if (models[i].kind != RIMU_MODEL_HUBBARD_REAL_1D)
            return fail(RIMU_ERR_ARG, "ranked-basis products support HubbardReal1D");
        if (models[i].M != m0.M || models[i].N != m0.N)
            return fail(RIMU_ERR_ARG, "all right-hand sides must share M and N");
    }
    if (m0.M < 2 || m0.N < 1 || m0.M + m0.N - 1 > 64) return fail(RIMU_ERR_ARG, "need M >= 2, N >= 1, N + M - 1 <= 64");
    int64_t D;
    if (int rc = rimu_basis_size(m0.M, m0.N, &D)) return rc;
    if (D > (int64_t)1 << 31) return fail(RIMU_ERR_ARG, "basis larger than 2^31 addresses");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(RIMU_ERR_NODEVICE, "no HIP device");
    rimu_dense* d = new rimu_dense();
    d->R = nrhs;
    d->M = m0.M;
    d->N = m0.N;
    d->B = m0.M + m0.N - 1;
    d->D = D;
    for (int i = 0; i < nrhs; ++i) d->models[i] = models[i];
    auto bad = [&](const char* what, hipError_t e) {
        std::string msg = std::string(what) + ": " + hipGetErrorString(e);
        rimu_dense_destroy(d);
        return fail(RIMU_ERR_HIP, msg);
    };
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking)) != hipSuccess) return bad("stream", e);
    // binomial and hop tables, and the sorted basis (next bit pattern with the same popcount)
    std::vector<int64_t> binom(BINOM_N * BINOM_N, 0);
    for (int n = 0; n < BINOM_N; ++n)
        for (int k = 0; k < BINOM_N; ++k) {
            int64_t c;
            binom[n * BINOM_N + k] = binomial64(n, k, &c) ? c : INT64_MAX;
        }
    const int row_len = d->N + 2;  // s = 0 .. N, and N + 1 for the row's last reader
    const int n_root = (d->N + 1) * (d->N + 1) / 4 + 1, n_delta = d->M * row_len;
    const int at_binom = n_root + (n_delta + 1) / 2;  // in 8-byte words
    std::vector<double> tab((size_t)at_binom + binom.size(), 0.0);
    uint32_t* delta = (uint32_t*)(tab.data() + n_root);
    for (int i = 1; i < d->M; ++i)
        for (int s = 1; s <= d->N; ++s) delta[(size_t)i * row_len + s] = (uint32_t)binom[(s + i - 2) * BINOM_N + s - 1];
    for (int k = 0; k < n_root; ++k) tab[k] = std::sqrt((double)k);
    std::memcpy(tab.data() + at_binom, binom.data(), binom.size() * 8);
    std::vector<uint64_t> keys((size_t)D);
    uint64_t x = (d->N >= 64) ? ~0ull : ((1ull << d->N) - 1);
    for (int64_t r = 0; r < D; ++r) {
        keys[r] = x;
        const uint64_t c = x & (~x + 1), rr = x + c;  // Gosper's hack
        x = c ? (((rr ^ x) >> 2) / c) | rr : 0;
    }
    if ((e = d->basis.alloc(D)) != hipSuccess) return bad("basis", e);
    if ((e = d->rot.alloc(D)) != hipSuccess) return bad("rotations", e);
    if ((e = d->tab.alloc(tab.size())) != hipSuccess) return bad("tables", e);
    if ((e = d->scal.alloc(8 * MAXR)) != hipSuccess) return bad("scalars", e);
    if ((e = hipHostMalloc((void**)&d->h_scal, 8 * MAXR * sizeof(double), hipHostMallocDefault)) != hipSuccess)
        return bad("pinned scalars", e);
    if ((e = hipMemcpy(d->basis.p, keys.data(), D * 8, hipMemcpyHostToDevice)) != hipSuccess) return bad("basis upload", e);
    if ((e = hipMemcpy(d->tab.p, tab.data(), tab.size() * 8, hipMemcpyHostToDevice)) != hipSuccess)
        return bad("table upload", e);
    dense_rotations_kernel<<<ceil_div(D, DT), DT, 0, d->stream>>>(d->basis.p, D, d->B,
                                                                  (const int64_t*)(d->tab.p + at_binom), d->rot.p);
    if ((e = hipGetLastError()) != hipSuccess) return bad("rotations", e);
    if ((e = hipStreamSynchronize(d->stream)) != hipSuccess) return bad("rotations", e);
    *out = d;
    return RIMU_OK;
}

int rimu_dense_destroy(rimu_dense* d) {
    if (!d) return RIMU_OK;
    if (d->stream) (void)hipStreamSynchronize(d->stream);
    d->basis.release(); d->rot.release(); d->tab.release(); d->x.release(); d->y.release(); d->z.release(); d->hist.release();
    d->partials.release(); d->scal.release();
    if (d->h_scal) (void)hipHostFree(d->h_scal);
    if (d->stream) (void)hipStreamDestroy(d->stream);
    delete d;
    return RIMU_OK;
}

int rimu_dense_dim(rimu_dense* d, int64_t* dim) {
    if (!d || !dim) return fail(RIMU_ERR_ARG, "null argument");
    *dim = d->D;
    return RIMU_OK;
}

int rimu_dense_basis(rimu_dense* d, uint64_t* keys) {
    if (!d || !keys) return fail(RIMU_ERR_ARG, "null argument");
    HIP_TRY(hipMemcpy(keys, d->basis.p, d->D * 8, hipMemcpyDeviceToHost));
    return RIMU_OK;
}

int rimu_dense_apply(rimu_dense* d, const double* a, const double* b, const double* v, double* w) {
    if (!d || !a || !b || !v || !w) return fail(RIMU_ERR_ARG, "null argument");
    const size_t bytes = (size_t)d->D * d->R * 8;
    HIP_TRY(d->x.alloc((size_t)d->D * d->R));
    HIP_TRY(d->y.alloc((size_t)d->D * d->R));
    HIP_TRY(hipMemcpyAsync(d->x.p, v, bytes, hipMemcpyHostToDevice, d->stream));
    if (int rc = apply(d, params(d, a, b), d->x.p, d->y.p)) return rc;
    HIP_TRY(hipMemcpyAsync(w, d->y.p, bytes, hipMemcpyDeviceToHost, d->stream));
    HIP_TRY(hipStreamSynchronize(d->stream));
    return RIMU_OK;
}

int rimu_dense_pullback(rimu_dense* d, const double* a, const double* b, const double* v,
                        const double* ybar, double* vbar, double* ubar, double* tbar) {
    if (!d || !a || !b || !v || !ybar || !vbar) return fail(RIMU_ERR_ARG, "null argument");
    const size_t n = (size_t)d->D * d->R, bytes = n * 8;
    HIP_TRY(d->x.alloc(n));
    HIP_TRY(d->y.alloc(n));
    HIP_TRY(d->z.alloc(n));
    HIP_TRY(hipMemcpyAsync(d->x.p, v, bytes, hipMemcpyHostToDevice, d->stream));
    HIP_TRY(hipMemcpyAsync(d->y.p, ybar, bytes, hipMemcpyHostToDevice, d->stream));
    if (int rc = pullback(d, params(d, a, b), d->x.p, d->y.p, d->z.p, d->scal.p, 0)) return rc;
    HIP_TRY(hipMemcpyAsync(vbar, d->z.p, bytes, hipMemcpyDeviceToHost, d->stream));
    HIP_TRY(hipMemcpyAsync(d->h_scal, d->scal.p, 2 * d->R * 8, hipMemcpyDeviceToHost, d->stream));
    HIP_TRY(hipStreamSynchronize(d->stream));
    for (int i = 0; i < d->R; ++i) {
        if (ubar) ubar[i] = d->h_scal[i];
        if (tbar) tbar[i] = d->h_scal[d->R + i];
    }
    return RIMU_OK;
}

int rimu_dense_projector(rimu_dense* d, int64_t K, double dtau, const double* shift, int64_t ckpt,
                         const double* v0, double* energy, double* grad_u, double* grad_t,
                         double* hf_u, double* hf_t, double* v_final) {
    if (!d || !shift || !v0) return fail(RIMU_ERR_ARG, "null argument");
    if (K < 0 || ckpt < 1 || !(dtau > 0)) return fail(RIMU_ERR_ARG, "need K >= 0, ckpt >= 1, dtau > 0");
    const int R = d->R;
    const size_t n = (size_t)d->D * R;
    const int64_t nseg = K == 0 ? 0 : ceil_div(K, ckpt);
    double a_t[MAXR], b_t[MAXR], a_h[MAXR], b_h[MAXR];
    for (int i = 0; i < R; ++i) {
        a_t[i] = 1 + dtau * shift[i];  // T = 1 + dt (S - H)
        b_t[i] = -dtau;
        a_h[i] = 0;                    // H itself
        b_h[i] = 1;
    }
    const DenseParams pT = params(d, a_t, b_t), pH = params(d, a_h, b_h);
    // the vectors between checkpoints and the two that every call needs stay with the handle
    // (d->x, d->y, d->z); the checkpoints, which grow with K, are given back
    DevBuf<double> ck, seg, lam, lam2;
    auto cleanup = [&]() { ck.release(); seg.release(); lam.release(); lam2.release(); };
    auto run = [&]() -> int {
        const int64_t last0 = nseg > 0 ? (nseg - 1) * ckpt : 0;  // first step of the last segment
        HIP_TRY(ck.alloc(std::max<int64_t>(nseg, 1) * n));
        HIP_TRY(seg.alloc((size_t)std::min<int64_t>(ckpt, std::max<int64_t>(K, 1)) * n));
        HIP_TRY(d->x.alloc(n));
        HIP_TRY(d->y.alloc(n));
        HIP_TRY(d->z.alloc(n));
        HIP_TRY(lam.alloc(n));
        HIP_TRY(lam2.alloc(n));
        double* cur = d->x.p;  // the final vector
        double* hv = d->y.p;
        HIP_TRY(hipMemcpyAsync(K > 0 ? ck.p : cur, v0, n * 8, hipMemcpyHostToDevice, d->stream));
        // vector j of the segment that starts at step s * ckpt: its checkpoint, then seg
        auto in_segment = [&](int64_t s, int64_t j) { return j == 0 ? ck.p + s * n : seg.p + j * n; };
        // forward sweep: every product writes where its result stays (checkpoints, and the last
        // segment, which the reverse sweep takes first) or alternates between two vectors
        const double* src = ck.p;
        for (int64_t k = 0; k < K; ++k) {
            const int64_t k1 = k + 1;
            double* dst = k1 == K             ? cur
                          : k1 % ckpt == 0    ? ck.p + (k1 / ckpt) * n
                          : k1 > last0        ? in_segment(nseg - 1, k1 - last0)
                          : (k & 1)           ? d->y.p
                                              : d->z.p;
            if (int rc = apply(d, pT, src, dst)) return rc;
            src = dst;
        }
        // energy: scal[0:R] = <v|v>, scal[R:2R] = <v|Hv>; HF: scal[2R:4R] = <v|D|v>, <v|K|v>
        if (int rc = apply(d, pH, cur, hv, d->scal.p + R)) return rc;
        if (int rc = dot(d, cur, cur, d->scal.p)) return rc;
        {
            double one[MAXR], unit_b[MAXR];
            for (int i = 0; i < R; ++i) { one[i] = 0; unit_b[i] = 1; }
            // pullback with ybar = v, b = 1 gives <v|D|v> and <v|K|v>; vbar is discarded
            if (int rc = pullback(d, params(d, one, unit_b), cur, cur, lam2.p, d->scal.p + 2 * R, 0)) return rc;
        }
        // cotangent of the Rayleigh quotient, and the (u, t) accumulators start at zero
        if (int rc = rq_gradient(d, cur, hv, d->scal.p, lam.p)) return rc;
        HIP_TRY(hipMemsetAsync(d->scal.p + 4 * R, 0, 2 * R * 8, d->stream));
        // reverse sweep: recompute each segment but the last from its checkpoint, then pull back
        for (int64_t s = nseg - 1; s >= 0; --s) {
            const int64_t len = std::min(K, (s + 1) * ckpt) - s * ckpt;
            for (int64_t j = 1; s < nseg - 1 && j < len; ++j)
                if (int rc = apply(d, pT, in_segment(s, j - 1), in_segment(s, j))) return rc;
            for (int64_t j = len - 1; j >= 0; --j) {
                if (int rc = pullback(d, pT, in_segment(s, j), lam.p, lam2.p, d->scal.p + 4 * R, 1)) return rc;
                std::swap(lam.p, lam2.p);
            }
        }
        HIP_TRY(hipMemcpyAsync(d->h_scal, d->scal.p, 6 * R * 8, hipMemcpyDeviceToHost, d->stream));
        if (v_final) HIP_TRY(hipMemcpyAsync(v_final, cur, n * 8, hipMemcpyDeviceToHost, d->stream));
        HIP_TRY(hipStreamSynchronize(d->stream));
        const double* h = d->h_scal;
        for (int i = 0; i < R; ++i) {
            const double vv = h[i], e = h[R + i] / vv;
            const double du = h[2 * R + i] / vv, dt = h[3 * R + i] / vv;
            if (energy) energy[i] = e;
            if (hf_u) hf_u[i] = du;
            if (hf_t) hf_t[i] = dt;
            // direct dependence of the final Rayleigh quotient plus the projection steps
            if (grad_u) grad_u[i] = du + h[4 * R + i];
            if (grad_t) grad_t[i] = dt + h[5 * R + i];
        }
        return RIMU_OK;
    };
    const int rc = run();
    cleanup();
    return rc;
}

int rimu_dense_ground_state(rimu_dense* d, const double* v0, int64_t max_iters, double tol,
                            double* energy, int64_t* iters) {
    if (!d || !v0 || !energy) return fail(RIMU_ERR_ARG, "null argument");
    if (max_iters < 1 || !(tol > 0)) return fail(RIMU_ERR_ARG, "need max_iters >= 1 and tol > 0");
    const int R = d->R;
    const size_t n = (size_t)d->D * R;
    const int64_t cap = std::min<int64_t>(max_iters, d->D);
    constexpr int64_t CHECK = 16;
    // beta^2 at or below this ends a right-hand side's Krylov space (rounding leaves
    // beta ~ 1e-14 |H| there; a true beta this small would move the Ritz value by ~beta^2)
    constexpr double FLOOR2 = 1e-20;
    double a_h[MAXR], b_h[MAXR];
    for (int i = 0; i < R; ++i) { a_h[i] = 0; b_h[i] = 1; }
    const DenseParams pH = params(d, a_h, b_h);
    DevBuf<double>&x = d->x, &y = d->y, &w = d->z, &hist = d->hist;  // kept with the handle
    // hist: alpha [cap][R], then |v0|^2 [R], then beta^2 [cap + 1][R] (beta^2[0] = 0 in the
    // tridiagonal matrix, its place holds one, x2 of the first iteration), then <x|Hx> [R]
    auto run = [&]() -> int {
        HIP_TRY(x.alloc(n));
        HIP_TRY(y.alloc(n));
        HIP_TRY(w.alloc(n));
        HIP_TRY(hist.alloc((size_t)(2 * cap + 3) * R));
        double* alpha = hist.p;
        double* n0 = hist.p + cap * R;
        double* beta2 = n0 + R;
        double* xw = beta2 + (cap + 1) * R;
        HIP_TRY(hipMemcpyAsync(x.p, v0, n * 8, hipMemcpyHostToDevice, d->stream));
        if (int rc = dot(d, x.p, x.p, n0)) return rc;
        lanczos_start_kernel<<<ceil_div(d->D, DT), DT, 0, d->stream>>>(x.p, d->D, R, n0, beta2);
        HIP_TRY(hipGetLastError());
        std::vector<double> h_a, h_n, last(R, INFINITY), cur(R);
        std::vector<int64_t> m_eff(R, -1);
        int64_t j = 0;
        for (; j < cap; ++j) {
            // x: the unnormalised v_j of squared norm beta2[j], y: that of v_{j-1}
            if (int rc = apply(d, pH, x.p, w.p, xw)) return rc;
            if (int rc = lanczos_update(d, w.p, x.p, y.p, xw, beta2 + j * R, beta2 + (j > 0 ? j - 1 : 0) * R,
                                        j > 0 ? FLOOR2 : 0.0, j > 1 ? FLOOR2 : 0.0, j == 0, alpha + j * R,
                                        beta2 + (j + 1) * R)) return rc;
            std::swap(y, x);
            std::swap(x, w);
            const bool last_iter = j + 1 == cap;
            if ((j + 1) % CHECK != 0 && !last_iter) continue;
            const int64_t m = j + 1;
            h_a.resize((size_t)m * R);
            h_n.resize((size_t)(m + 2) * R);  // |v0|^2, then beta^2
            HIP_TRY(hipMemcpyAsync(h_a.data(), alpha, (size_t)m * R * 8, hipMemcpyDeviceToHost, d->stream));
            HIP_TRY(hipMemcpyAsync(h_n.data(), n0, (size_t)(m + 2) * R * 8, hipMemcpyDeviceToHost, d->stream));
            HIP_TRY(hipStreamSynchronize(d->stream));
            const double* h_b2 = h_n.data() + R;
            bool done = true;
            std::vector<double> a(m), b2(m + 1);
            for (int i = 0; i < R; ++i) {
                if (!(h_n[i] > 0)) return fail(RIMU_ERR_ARG, "start vector is zero");
                int64_t mi = m;
                for (int64_t k = 1; k <= m; ++k) {
                    if (!(h_b2[k * R + i] > FLOOR2)) { mi = k; break; }  // exhausted after k vectors
                }
                for (int64_t k = 0; k < mi; ++k) {
                    a[k] = h_a[k * R + i];
                    b2[k] = h_b2[k * R + i];
                }
                cur[i] = tridiag_lowest(a.data(), b2.data(), mi);
                const bool exhausted = !(h_b2[mi * R + i] > FLOOR2);
                const bool conv = exhausted || std::fabs(cur[i] - last[i]) <= tol * std::max(1.0, std::fabs(cur[i]));
                if (!conv) done = false;
                last[i] = cur[i];
            }
            if (done) { ++j; break; }
        }
        for (int i = 0; i < R; ++i) energy[i] = cur[i];
        if (iters) *iters = j;
        return RIMU_OK;
    };
    return run();
}

}  // extern "C"
