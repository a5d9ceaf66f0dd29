// Additive Schwarz preconditioner (simulation_toolbox/src/fem/schwarz_precond.rs:134-342):
// P = sum_s R_s^T B_s^+ R_s + sum_untreated 1 / J_ii, with B_s the restriction of J to the
// subdomain's DOFs and B_s^+ = V diag(1 / max(|lambda|, 1e-12 max|lambda|)) V^T.
//
// Per update: (1) gather every B_s from J (precomputed slots) and (2) invert it by batched FP64 Gauss-Jordan
// in LDS, one work-group per block, accepted where it certifies that B_s is positive
// definite with kappa_2 < 1e11 (then the eigenvalue clamp is inactive and B_s^+ = B_s^-1),
// (3) for the remaining blocks, symmetric eigen-decomposition by parallel (round-robin) Jacobi
// in LDS and recomposition of B_s^+, (4) color-ordered gather of the blocks into P's row
// blocks, (5) reciprocal diagonal for untreated nodes.
#include <algorithm>
#include <cmath>

#include "host_threads.hpp"
#include "internal.hpp"

namespace hoefem {

// the partial sums per norm of a block above 96 x 96 (k_bgj_norm)
constexpr int BGJ_NORM_SPLIT = 32;

void schwarz_setup(Schwarz& s, Model& m, int64_t nsub, const int64_t* off, const int32_t* nodes, int64_t nunt,
                   const int32_t* unt) {
    s.model = &m;
    s.nsub = nsub;
    s.off.assign(off, off + nsub + 1);
    if (s.off[0] != 0) throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "subdomain offsets must start at 0");
    for (int64_t k = 0; k < nsub; ++k)
        if (s.off[k + 1] < s.off[k]) throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "subdomain offsets must be sorted");
    s.nodes.assign(nodes, nodes + s.off[nsub]);
    s.untreated.assign(unt, unt + nunt);
    for (int32_t v : s.nodes)
        if (v < 0 || v >= m.nv) throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "subdomain node out of range");
    s.colors = greedy_coloring(nsub, s.off.data(), s.nodes.data());
    build_node_pattern(m.nv, nsub, s.off.data(), s.nodes.data(), s.untreated, s.P);
    s.scatter.build(s.P, nsub, s.off.data(), s.nodes.data(), &s.colors, 1);
    // slots of every block entry in J's (model) pattern. SchwarzElementAssembler gathers with
    // csr_row.get(col).expect(..) (schwarz_precond.rs:304-320), which panics on a node pair that J
    // does not couple; here such entries are the zeros they are in J (-1 slot), so subdomains may be
    // any node sets, e.g. patches of many elements.
    s.jslot.resize(s.scatter.slot.size());
    s.small_max_dim = s.large_max_dim = 0;
    s.large.clear();
    std::vector<int64_t> panel_off;
    int64_t panel_total = 0;
    const int nt = thread_count((int64_t)s.jslot.size(), SETUP_ENTRIES);
    run_on_threads(nt, [&](int t) {
        std::vector<int32_t> pos(m.nv, -1);
        s.scatter.slots_in(m.pattern, s.off.data(), s.nodes.data(), t * m.nv / nt, (t + 1) * m.nv / nt, pos, s.jslot.data());
    });
    for (int64_t b = 0; b < nsub; ++b) {
        const int mb = (int)(s.off[b + 1] - s.off[b]);
        if (3 * mb > SCHWARZ_SMALL_DIM) {
            s.large.push_back((int32_t)b);
            s.large_max_dim = std::max(s.large_max_dim, 3 * mb);
            panel_off.push_back(panel_total);
            panel_total += ((int64_t)3 * mb + 63) / 64 * 64 * 64;  // 64 x 64 tiles
        } else {
            s.small_max_dim = std::max(s.small_max_dim, 3 * mb);
        }
    }
    if (s.large_max_dim > 4096) throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "Schwarz subdomain above 4096 DOFs");
    for (int32_t v : s.untreated)
        if (v < 0 || v >= m.nv || !s.P.diag_only[v])
            throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "untreated node must not belong to a subdomain");
    s.P.upload(m.stream);
    s.grid.build(m.pattern, &s.P, grid_device_cus(), m.stream);
    s.scatter.upload(m.stream);
    s.pack.add(s.jslot, s.d_jslot);
    s.pack.add(s.untreated, s.d_untreated);
    s.pack.add(s.off, s.d_off);
    s.pack.add(s.nodes, s.d_nodes);
    s.pack.upload(m.stream);
    if (s.fp32) {
        s.d_vals32.ensure(std::max<int64_t>(s.P.nnz(), 1));
        HIP_CHECK(hipMemsetAsync(s.d_vals32.get(), 0, sizeof(float) * s.d_vals32.n, m.stream));
    } else {
        s.d_vals.ensure(std::max<int64_t>(s.P.nnz(), 1));
        HIP_CHECK(hipMemsetAsync(s.d_vals.get(), 0, sizeof(double) * s.d_vals.n, m.stream));
    }
    s.d_blocks.ensure(std::max<int64_t>(s.scatter.val_off[nsub], 1));
    s.d_fallback.ensure(std::max<int64_t>(nsub, 1));
    if (!s.large.empty()) {
        s.d_large.upload(s.large, m.stream);
        s.d_panel_off.upload(panel_off, m.stream);
        s.d_piv.ensure(s.large.size() * 64 * 64);
        s.d_panels.ensure((size_t)2 * panel_total);
        const size_t nt = ((size_t)s.large_max_dim + 63) / 64;
        s.d_lnorm.ensure(s.large.size() * (BGJ_NORM_SPLIT + nt * (nt + 1) / 2));
    }
}

// B_s(r, c) = J[3 g_a + i, 3 g_c + j] of the blocks above 96 x 96 (listed in large), row-major (3m)^2, always
// FP64 (the smaller ones are gathered where they are inverted). Work-group (s, y) gathers
// entries [y SG_CHUNK, (y + 1) SG_CHUNK) of the s-th such block, so a block of hundreds of DOFs (the 64-element
// patches) is spread over many work-groups instead of walking its entries on one.
constexpr int SG_CHUNK = 2048;
template <class VJ>
__global__ void k_schwarz_gather(const int32_t* __restrict__ large, const int32_t* __restrict__ msz,
                                 const int64_t* __restrict__ val_off, const int64_t* __restrict__ slot_off, const int64_t* __restrict__ noff,
                                 const int32_t* __restrict__ nodes, const int32_t* __restrict__ jslot,
                                 const int32_t* __restrict__ jrowptr, const VJ* __restrict__ J,
                                 double* __restrict__ blocks) {
    const int64_t b = large[blockIdx.x];
    const int mb = msz[b], dim = 3 * mb;
    const int c0 = (int)blockIdx.y * SG_CHUNK;
    if (c0 >= dim * dim) return;
    const int c1 = min(dim * dim, c0 + SG_CHUNK);
    const int32_t* g = nodes + noff[b];
    double* out = blocks + val_off[b];
    for (int idx = c0 + (int)threadIdx.x; idx < c1; idx += blockDim.x) {
        const int r = idx / dim, c = idx % dim;
        const int a = r / 3, i = r % 3, cb = c / 3, j = c % 3;
        const int k = jslot[slot_off[b] + (int64_t)a * mb + cb];
        out[idx] = k < 0 ? 0.0 : (double)J[(int64_t)jrowptr[3 * (int64_t)g[a] + i] + 3 * k + j];
    }
}

// Parallel cyclic Jacobi (Brent-Luk round-robin ordering) on a symmetric dim x dim block in
// LDS, then B^+ = V diag(f(lambda)) V^T with f = 1/max(|lambda|, 1e-12 max|lambda|)
// (invert_element_block, schwarz_precond.rs:329-342). Rotations follow Golub & Van Loan,
// "Matrix Computations", sym.schur2.
constexpr int EIG_THREADS = 256;
// kappa_2 bound below which the eigenvalue clamp max(|lambda|, 1e-12 max|lambda|) is provably
// inactive, with a 2x margin for the rounding of the computed inverse (relative error ~kappa eps)
constexpr double SPD_COND_LIMIT = 5e11;

__device__ inline double block_max(double v, double* s_red) {
    const int t = threadIdx.x;
    s_red[t] = v;
    __syncthreads();
    for (int s = EIG_THREADS / 2; s > 0; s >>= 1) {
        if (t < s) s_red[t] = fmax(s_red[t], s_red[t + s]);
        __syncthreads();
    }
    const double r = s_red[0];
    __syncthreads();
    return r;
}

__device__ inline double block_sum(double v, double* s_red) {
    const int t = threadIdx.x;
    s_red[t] = v;
    __syncthreads();
    for (int s = EIG_THREADS / 2; s > 0; s >>= 1) {
        if (t < s) s_red[t] += s_red[t + s];
        __syncthreads();
    }
    const double r = s_red[0];
    __syncthreads();
    return r;
}

typedef double sgj_double4 __attribute__((ext_vector_type(4)));

// v of lane p of each row of 16 lanes, in all of the row's lanes
template <int P>
__device__ inline double row_lane(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + P, 0xf, 0xf, false);  // row_newbcast
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + P, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double lane_value(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(4 * lane, (int)b), hi = __builtin_amdgcn_ds_bpermute(4 * lane, (int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// One pivot of the in-register inversion of a 16 x 16 tile by a wavefront (lane l: column l % 16, rows
// 4 (l / 16) .. + 3 in a[4]); false if the pivot is not positive, uniformly.
template <int P>
__device__ inline bool gj_pivot(double (&a)[4], int l) {
    constexpr int G = P / 4, M = P % 4;
    const long long pb = __double_as_longlong(a[M]);
    const int plo = __builtin_amdgcn_readlane((int)pb, 16 * G + P), phi = __builtin_amdgcn_readlane((int)(pb >> 32), 16 * G + P);
    const double piv = __longlong_as_double(((long long)phi << 32) | (unsigned)plo);
    if (!(piv > 0.0) || !isfinite(piv)) return false;
    const double ip = 1.0 / piv;
    const int j = l & 15, g = l >> 4;
    const double row = lane_value(a[M], 16 * G + j);  // a(P, j)
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const double col = row_lane<P>(a[m]);  // a(i, P), i = 4 g + m
        const bool ip_row = g == G && m == M, ip_col = j == P;
        a[m] = ip_row ? (ip_col ? ip : row * ip) : (ip_col ? -col * ip : a[m] - col * row * ip);
    }
    return true;
}
template <int P>
__device__ inline bool gj_pivots(double (&a)[4], int l) {
    if constexpr (P == 16)
        return true;
    else
        return gj_pivot<P>(a, l) && gj_pivots<P + 1>(a, l);
}

// The elimination of k_spd_inverse_mf, in place on the NT x NT tiles in s_a (row stride 16 NT + 1; rows and
// columns past dim are the identity's), by the NW wavefronts of a work-group. s_bad: LDS, 0. Ends with a
// barrier; false if a pivot is not positive.
template <int NT, int NW>
__device__ inline bool gj_tiles(double* s_a, int dim, int& s_bad) {
    constexpr int LD = 16 * NT + 1;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    // C = (neg ? -1 : 1) X Y (+ Cin), 16 x 16 tiles at (xr, xc), (yr, yc) of s_a
    auto tile_mul = [&](int xr, int xc, int yr, int yc, bool neg, sgj_double4 acc) {
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
            const double x = s_a[(xr + (l & 15)) * LD + xc + 4 * s4 + (l >> 4)];
            const double y = s_a[(yr + 4 * s4 + (l >> 4)) * LD + yc + (l & 15)];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(neg ? -x : x, y, acc, 0, 0, 0);
        }
        return acc;
    };
    auto tile_store = [&](int r0, int c0, const sgj_double4& acc) {
#pragma unroll
        for (int v = 0; v < 4; ++v) s_a[(r0 + 4 * v + (l >> 4)) * LD + c0 + (l & 15)] = acc[v];
    };
    auto tile_load = [&](int r0, int c0) {
        sgj_double4 acc;
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = s_a[(r0 + 4 * v + (l >> 4)) * LD + c0 + (l & 15)];
        return acc;
    };
    const sgj_double4 zero = {0.0, 0.0, 0.0, 0.0};
    const int O = (dim + 15) / 16 - 1;  // tiles of dim other than kt
#pragma unroll 1
    for (int kt = 0; kt <= O; ++kt) {
        const int K = 16 * kt;
        auto other = [&](int n) { return 16 * (n < kt ? n : n + 1); };
        if (w == 0) {  // D = A_kk^-1 in one wavefront's registers
            double a[4];
            double* src = s_a + (K + 4 * (l >> 4)) * LD + K + (l & 15);
#pragma unroll
            for (int m = 0; m < 4; ++m) a[m] = src[m * LD];
            if (gj_pivots<0>(a, l)) {
#pragma unroll
                for (int m = 0; m < 4; ++m) src[m * LD] = a[m];
            } else if (l == 0) {
                s_bad = 1;
            }
        }
        __syncthreads();
        if (s_bad) return false;  // the same in every thread
        // row panel A_kj = D A_kj: the tile's old values are read (by its wavefront) before it is written
#pragma unroll 1
        for (int n = w; n < O; n += NW) tile_store(K, other(n), tile_mul(K, K, K, other(n), false, zero));
        __syncthreads();
#pragma unroll 1
        for (int n = w; n < O * O; n += NW) {
            const int i = other(n / O), j = other(n % O);
            tile_store(i, j, tile_mul(i, K, K, j, true, tile_load(i, j)));
        }
        __syncthreads();
#pragma unroll 1
        for (int n = w; n < O; n += NW) tile_store(other(n), K, tile_mul(other(n), K, K, K, true, zero));
        __syncthreads();
    }
    return true;
}

// Inverse of each small symmetric block B_s(r, c) = J[3 g_a + i, 3 g_c + j], without pivoting, on the matrix cores:
// in-place blocked Gauss-Jordan over tiles of 16 x 16 (dim <= 16 NT; the padding is the identity), one
// work-group of NW wavefronts per block, the block gathered from J into LDS (row stride LD = 16 NT + 1). For
// each diagonal tile k:
//   D = A_kk^-1        wavefront 0, in registers, pivot by pivot
//   A_kj = D A_kj      (j != k)
//   A_ij -= A_ik A_kj  (i, j != k; the new A_kj, the old A_ik)
//   A_ik = -A_ik D     (i != k);  A_kk = D
// The tile products run on v_mfma_f64_16x16x4 (lane l: A operand X(l % 16, 4 s + l / 16), B operand
// Y(4 s + l / 16, l % 16), result item v = (4 v + l / 16, l % 16)), the tiles of each step dealt to
// the wavefronts in turn. Every pivot is a diagonal entry of a Schur complement, so all are positive iff B
// is positive definite. Results per block (fallback[b]):
//   0  pivots positive and min(|B|_F |B^-1|_F, |B|_inf |B^-1|_inf) < SPD_COND_LIMIT (both upper
//      bounds of kappa_2(B) for symmetric B): the clamp of the pseudo-inverse is inactive, so
//      B^+ = B^-1, and the symmetrized inverse is the block's result;
//   2  pivots positive, the cheap bound too loose: the inverse is stored and
//      k_spd_power_certify decides with a sharper bound;
//   1  a pivot not positive: B itself is stored for the eigen path.
// A block's time is its serial chain (16 pivots per tile, about 200 cycles each, and three rounds of tile
// products), hidden behind the other blocks of its CU. Blocks of one or two tiles (Tet4, Hex8, Tet10) take a
// wavefront each: their rounds have one tile product. 1472 blocks of 81 x 81 took 252 us in 6 x 6 register tiles
// on the vector units with two barriers per pivot, and 65 us to be gathered into memory first; now 190 us
// together.
template <class VJ, int NT, int NW>
__global__ __launch_bounds__(64 * NW) void k_spd_inverse_mf(
    const int32_t* __restrict__ msz, const int64_t* __restrict__ val_off, const int64_t* __restrict__ slot_off,
    const int64_t* __restrict__ noff, const int32_t* __restrict__ nodes, const int32_t* __restrict__ jslot,
    const int32_t* __restrict__ jrowptr, const VJ* __restrict__ J, double* __restrict__ blocks,
    int* __restrict__ fallback) {
    constexpr int PD = 16 * NT, LD = PD + 1, THREADS = 64 * NW;
    extern __shared__ double s_a[];  // [PD][LD]
    __shared__ double s_red[2][NW];
    __shared__ int s_bad;
    const int64_t b = blockIdx.x;
    const int mb = msz[b], dim = 3 * mb;
    if (dim > SCHWARZ_SMALL_DIM || dim > PD) {  // handled by the blocked path in global memory
        if (threadIdx.x == 0) fallback[b] = 4;
        return;
    }
    const int t = threadIdx.x;
    double* blk = blocks + val_off[b];
    const int32_t *g = nodes + noff[b], *slot = jslot + slot_off[b];
    // out[r * ld + c] = B(r, c), a node pair per lane
    auto gather = [&](double* out, int ld) {
        for (int p = t; p < mb * mb; p += THREADS) {
            const int a = p / mb, c = p % mb, k = slot[p];
            double* o = out + 3 * a * ld + 3 * c;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const VJ* row = J + (k < 0 ? 0 : (int64_t)jrowptr[3 * (int64_t)g[a] + i] + 3 * k);
#pragma unroll
                for (int j = 0; j < 3; ++j) o[i * ld + j] = k < 0 ? 0.0 : (double)row[j];
            }
        }
    };
    gather(s_a, LD);
    for (int idx = t; idx < PD * PD; idx += THREADS) {
        const int i = idx / PD, j = idx % PD;
        if (i >= dim || j >= dim) s_a[i * LD + j] = i == j ? 1.0 : 0.0;
    }
    if (t == 0) s_bad = 0;
    __syncthreads();
    // |.|_F^2 and |.|_inf of the block's dim x dim part, a row per lane; ends with a barrier
    auto norms = [&](double& f2, double& finf) {
        double loc = 0.0, row = 0.0;
        for (int r = t; r < dim; r += THREADS) {
            double sum = 0.0;
            for (int j = 0; j < dim; ++j) {
                const double x = s_a[r * LD + j];
                loc += x * x;
                sum += fabs(x);
            }
            row = fmax(row, sum);
        }
        for (int off = 32; off > 0; off >>= 1) {
            loc += __shfl_xor(loc, off, 64);
            row = fmax(row, __shfl_xor(row, off, 64));
        }
        if ((t & 63) == 0) {
            s_red[0][t >> 6] = loc;
            s_red[1][t >> 6] = row;
        }
        __syncthreads();
        f2 = finf = 0.0;
        for (int w = 0; w < NW; ++w) {
            f2 += s_red[0][w];
            finf = fmax(finf, s_red[1][w]);
        }
        __syncthreads();
    };
    double nb2, nbinf;
    norms(nb2, nbinf);
    if (!gj_tiles<NT, NW>(s_a, dim, s_bad)) {  // the same in every thread: uniform exit
        gather(blk, dim);
        if (t == 0) fallback[b] = 1;
        return;
    }
    double ni2, niinf;
    norms(ni2, niinf);
    const double cert = fmin(sqrt(nb2) * sqrt(ni2), nbinf * niinf);
    for (int idx = t; idx < dim * dim; idx += THREADS) {
        const int i = idx / dim, j = idx % dim;
        blk[(int64_t)i * dim + j] = 0.5 * (s_a[i * LD + j] + s_a[j * LD + i]);
    }
    if (t == 0) fallback[b] = cert < SPD_COND_LIMIT ? 0 : 2;
}

// Positive semi-definiteness certificate of each symmetric block: Cholesky of B + delta I in LDS
// with delta = 1e-11 |B|_F. When every pivot is positive, lambda_min(B) > -delta, so clamping the
// eigenvalues at zero would move B by less than sqrt(dim) delta (the order of the eigensolver's
// own rounding): need[b] = 0 and the block is kept. Otherwise need[b] = 1 and the block goes to
// the eigen path.
__global__ __launch_bounds__(EIG_THREADS) void k_psd_certify(const int32_t* __restrict__ msz,
                                                             const int64_t* __restrict__ val_off,
                                                             const double* __restrict__ blocks, int* __restrict__ need,
                                                             int ldpad) {
    extern __shared__ double lds[];
    __shared__ double s_red[EIG_THREADS];
    const int64_t b = blockIdx.x;
    const int dim = 3 * msz[b];
    const int ld = ldpad;
    double* A = lds;
    const double* blk = blocks + val_off[b];
    const int t = threadIdx.x;
    double loc = 0.0;
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
        const double v = blk[idx];
        A[(idx / dim) * ld + idx % dim] = v;
        loc += v * v;
    }
    const double delta = 1e-11 * sqrt(block_sum(loc, s_red));  // block_sum synchronizes
    for (int i = t; i < dim; i += EIG_THREADS) A[i * ld + i] += delta;
    __syncthreads();
    // right-looking Cholesky on the lower triangle
    for (int k = 0; k < dim; ++k) {
        const double piv = A[k * ld + k];
        if (!(piv > 0.0)) {  // uniform: every thread reads the same LDS value
            if (t == 0) need[b] = 1;
            return;
        }
        const double d = sqrt(piv);
        __syncthreads();
        for (int i = k + 1 + t; i < dim; i += EIG_THREADS) A[i * ld + k] /= d;
        __syncthreads();
        const int m = dim - k - 1;
        for (int idx = t; idx < m * m; idx += EIG_THREADS) {
            const int i = k + 1 + idx / m, j = k + 1 + idx % m;
            if (j <= i) A[i * ld + j] -= A[i * ld + k] * A[j * ld + k];
        }
        __syncthreads();
    }
    if (t == 0) need[b] = 0;
}

// Positive semi-definite projection P = (B + B sign(B)) / 2 of each flagged symmetric block by the
// Newton-Schulz iteration for the matrix sign, X_0 = B / |B|_F, X_{k+1} = X_k (3 I - X_k^2) / 2
// (Higham, "Functions of Matrices", SIAM 2008, sec. 5.3). Every X_k is a polynomial in B, so the
// eigenvectors are B's and each eigenvalue x follows the scalar map: x in (0, 1] goes to 1, x < 0
// to -1, x = 0 stays. PSD_NS_ITERS steps settle every eigenvalue with |lambda| >= 1.5^-59 |B|_F
// (~4e-11 |B|_F); smaller ones contribute at most |lambda| to the error.
constexpr int PSD_NS_ITERS = 64;

__device__ inline void tile_gemm(const double* __restrict__ X, const double* __restrict__ Y, int dp, int ld, int ti,
                                 int tj, double (&acc)[4][4]) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[a][c] = 0.0;
    for (int k = 0; k < dp; ++k) {
        double x[4], y[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) x[a] = X[(4 * ti + a) * ld + k];
#pragma unroll
        for (int c = 0; c < 4; ++c) y[c] = Y[k * ld + 4 * tj + c];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[a][c] += x[a] * y[c];
    }
}

// One block per work-group of four wavefronts, X and T in LDS as NT x NT tiles of 16 x 16 (dim <= 16 NT, zero
// padding), the products on v_mfma_f64_16x16x4 (lane layout as in k_spd_inverse_mf). X, X^2 and
// X (3 I - X^2) / 2 are symmetric, so an iteration computes the tiles on and below the diagonal and
// mirrors their lower triangle; X and T are exactly symmetric, as their reads along rows for both operands need (an
// antisymmetric part would double with every iteration): 2 NT (NT + 1) / 2 tiles of 4 NT instructions, dealt to the wavefronts in turn. Bound by the
// matrix cores (64 cycles per instruction and SIMD): 3840 blocks of 60 x 60 are 79M instructions, 2.0 ms at the
// peak rate. 560 blocks of 60 x 60 take 918 us; 3307 us with 4 x 4 register tiles on the vector units, 1804 us with the
// products' operands read down columns.
template <int NT>
__global__ __launch_bounds__(EIG_THREADS) void k_psd_newton_schulz(const int32_t* __restrict__ msz,
                                                                   const int64_t* __restrict__ val_off,
                                                                   double* __restrict__ blocks,
                                                                   const int* __restrict__ need) {
    if (need[blockIdx.x] == 0) return;
    constexpr int PD = 16 * NT, LD = PD + 1, LOWER = NT * (NT + 1) / 2, PER = (LOWER + 3) / 4;
    extern __shared__ double lds[];
    __shared__ double s_red[EIG_THREADS];
    const int64_t b = blockIdx.x;
    const int dim = 3 * msz[b];
    double* X = lds;
    double* T = lds + PD * LD;
    double* blk = blocks + val_off[b];
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    double loc = 0.0;
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
        const double v = blk[idx];
        loc += v * v;
    }
    const double nrm = sqrt(block_sum(loc, s_red));
    if (nrm == 0.0) return;  // uniform
    const double inv = 1.0 / nrm;
    // dst = s (B + B^T) / 2
    auto load = [&](double* dst, double s) {
        for (int idx = t; idx < PD * PD; idx += EIG_THREADS) {
            const int r = idx / PD, c = idx % PD;
            dst[r * LD + c] = (r < dim && c < dim) ? 0.5 * (blk[r * dim + c] + blk[c * dim + r]) * s : 0.0;
        }
    };
    load(X, inv);  // symmetric: both sums of two commute
    __syncthreads();
    // tile (ti, tj) of A B for a symmetric A, whose operand A(r, k) is read as A(k, r), along a row as B's is
    auto product = [&](const double* A, const double* B, int ti, int tj) {
        sgj_double4 acc = {0.0, 0.0, 0.0, 0.0};
        const double* pa = A + (l >> 4) * LD + 16 * ti + (l & 15);
        const double* pb = B + (l >> 4) * LD + 16 * tj + (l & 15);
#pragma unroll
        for (int ks = 0; ks < 4 * NT; ++ks)  // entries past dim are zero
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[4 * ks * LD], pb[4 * ks * LD], acc, 0, 0, 0);
        return acc;
    };
    // the tiles on and below the diagonal, tile n = ti (ti + 1) / 2 + tj to wavefront n % 4
    auto each_tile = [&](auto f) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int n = 4 * q + w;
            if (n >= LOWER) break;  // uniform over the wavefront
            int ti = 0;
            while ((ti + 1) * (ti + 2) / 2 <= n) ++ti;
            f(q, ti, n - ti * (ti + 1) / 2);
        }
    };
    sgj_double4 acc[PER];
    for (int it = 0; it < PSD_NS_ITERS; ++it) {
        // T = X X
        each_tile([&](int, int ti, int tj) {
            const sgj_double4 d = product(X, X, ti, tj);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * ti + 4 * v + (l >> 4), c = 16 * tj + (l & 15);
                if (ti != tj || r >= c) T[r * LD + c] = T[c * LD + r] = d[v];
            }
        });
        __syncthreads();
        // X <- 1.5 X - 0.5 X T, stored once every product has read X
        each_tile([&](int q, int ti, int tj) { acc[q] = product(X, T, ti, tj); });
        __syncthreads();
        each_tile([&](int q, int ti, int tj) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * ti + 4 * v + (l >> 4), c = 16 * tj + (l & 15);
                if (ti != tj || r >= c) X[r * LD + c] = X[c * LD + r] = 1.5 * X[r * LD + c] - 0.5 * acc[q][v];
            }
        });
        __syncthreads();
    }
    // P = (B + B S) / 2: B back into T, B S into the block, then symmetrized (B S is symmetric in exact arithmetic)
    load(T, 1.0);
    __syncthreads();
    for (int n = w; n < NT * NT; n += 4) {
        const int ti = n / NT, tj = n % NT;
        const sgj_double4 d = product(T, X, ti, tj);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * ti + 4 * v + (l >> 4), c = 16 * tj + (l & 15);
            if (r < dim && c < dim) blk[r * dim + c] = 0.5 * (T[r * LD + c] + d[v]);
        }
    }
    __syncthreads();  // the work-group's stores are visible to it
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) X[(idx / dim) * LD + idx % dim] = blk[idx];
    __syncthreads();
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
        const int r = idx / dim, c = idx % dim;
        blk[idx] = 0.5 * (X[r * LD + c] + X[c * LD + r]);
    }
}

// Sharper certificate for the blocks k_spd_inverse_mf marked 2. For symmetric X with eigenvalues
// lambda, |X^8|_F = (sum lambda^16)^(1/2) >= max|lambda|^8, so
//     |X|_2 <= s |(X / s)^8|_F^(1/8),  s = |X|_F,
// an upper bound within a factor dim^(1/16) (<= 1.33) of |X|_2 instead of the factor up to dim of
// the norms above. Three squarings in LDS for B (gathered again from J) and for the inverse now in
// the block; kappa_2(B) <= |B|_2 |B^-1|_2 < SPD_COND_LIMIT accepts the inverse, otherwise B goes
// back into the block for the eigen path.
template <class VJ>
__global__ __launch_bounds__(EIG_THREADS) void k_spd_power_certify(
    const int32_t* __restrict__ msz, const int64_t* __restrict__ val_off, const int64_t* __restrict__ slot_off,
    const int64_t* __restrict__ noff, const int32_t* __restrict__ nodes, const int32_t* __restrict__ jslot,
    const int32_t* __restrict__ jrowptr, const VJ* __restrict__ J, double* __restrict__ blocks,
    int* __restrict__ fallback, int ldpad) {
    if (fallback[blockIdx.x] != 2) return;
    extern __shared__ double lds[];
    __shared__ double s_red[EIG_THREADS];
    const int64_t b = blockIdx.x;
    const int mb = msz[b], dim = 3 * mb, dp = (dim + 3) & ~3, ld = ldpad;
    if (dim > SCHWARZ_SMALL_DIM) return;
    double* X = lds;
    double* Y = lds + (size_t)dp * ld;
    double* blk = blocks + val_off[b];
    const int32_t* g = nodes + noff[b];
    const int t = threadIdx.x;
    auto entry = [&](int r, int c) -> double {  // B(r, c) = J[3 g_a + i, 3 g_cb + j]
        const int a = r / 3, i = r % 3, cb = c / 3, j = c % 3;
        const int k = jslot[slot_off[b] + (int64_t)a * mb + cb];
        return k < 0 ? 0.0 : (double)J[(int64_t)jrowptr[3 * (int64_t)g[a] + i] + 3 * k + j];
    };
    auto bound = [&]() -> double {  // spectral-norm bound of the symmetric matrix in X
        double loc = 0.0;
        for (int idx = t; idx < dp * dp; idx += EIG_THREADS) {
            const double v = X[(idx / dp) * ld + idx % dp];
            loc += v * v;
        }
        const double s = sqrt(block_sum(loc, s_red));  // synchronizes
        if (!(s > 0.0)) return 0.0;                    // uniform
        const double is = 1.0 / s;
        for (int idx = t; idx < dp * dp; idx += EIG_THREADS) X[(idx / dp) * ld + idx % dp] *= is;
        __syncthreads();
        const int nt = dp / 4;
        double* src = X;
        double* dst = Y;
        for (int sq = 0; sq < 3; ++sq) {
            for (int tile = t; tile < nt * nt; tile += EIG_THREADS) {
                const int ti = tile / nt, tj = tile % nt;
                double acc[4][4];
                tile_gemm(src, src, dp, ld, ti, tj, acc);
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int c = 0; c < 4; ++c) dst[(4 * ti + a) * ld + 4 * tj + c] = acc[a][c];
            }
            __syncthreads();
            double* tmp = src;
            src = dst;
            dst = tmp;
        }
        loc = 0.0;
        for (int idx = t; idx < dp * dp; idx += EIG_THREADS) {
            const double v = src[(idx / dp) * ld + idx % dp];
            loc += v * v;
        }
        const double n8 = sqrt(block_sum(loc, s_red));
        return s * sqrt(sqrt(sqrt(n8)));
    };
    for (int idx = t; idx < dp * dp; idx += EIG_THREADS) {
        const int r = idx / dp, c = idx % dp;
        X[r * ld + c] = (r < dim && c < dim) ? entry(r, c) : 0.0;
    }
    __syncthreads();
    const double nb = bound();
    for (int idx = t; idx < dp * dp; idx += EIG_THREADS) {
        const int r = idx / dp, c = idx % dp;
        X[r * ld + c] = (r < dim && c < dim) ? blk[(int64_t)r * dim + c] : 0.0;
    }
    __syncthreads();
    const double ni = bound();
    if (nb * ni < SPD_COND_LIMIT) {
        if (t == 0) fallback[b] = 0;
        return;
    }
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) blk[idx] = entry(idx / dim, idx % dim);
    if (t == 0) fallback[b] = 1;
}

// Cyclic Jacobi eigen-decomposition of each symmetric block in LDS, then the block is replaced by
// V f(lambda) V^T: project == 0, invert_element_block's clamped inverse (schwarz_precond.rs:329-342);
// project == 1, the positive semi-definite projection max(lambda, 0) of DefaultSemidefiniteProjection
// (fenris/src/assembly.rs:552-564).
__global__ __launch_bounds__(EIG_THREADS) void k_jacobi_inverse(const int32_t* __restrict__ msz,
                                                                const int64_t* __restrict__ val_off,
                                                                double* __restrict__ blocks,
                                                                const int* __restrict__ fallback, int ldpad,
                                                                int project) {
    if (fallback && (fallback[blockIdx.x] == 0 || fallback[blockIdx.x] >= 4)) return;
    extern __shared__ double lds[];
    const int64_t b = blockIdx.x;
    const int dim = 3 * msz[b];
    if (fallback && dim > SCHWARZ_SMALL_DIM) return;  // the LDS is sized for the small blocks
    const int nn = dim + (dim & 1);  // even number of players (one idle index when dim is odd)
    const int ld = ldpad;            // row stride (>= nn + 1)
    double* A = lds;
    double* V = lds + (size_t)nn * ld;
    double* cs = V + (size_t)nn * ld;  // [nn/2][2]
    int* perm = (int*)(cs + nn);
    __shared__ double s_red[EIG_THREADS];
    __shared__ int s_done;
    double* blk = blocks + val_off[b];
    const int t = threadIdx.x;
    for (int idx = t; idx < nn * nn; idx += EIG_THREADS) {
        const int r = idx / nn, c = idx % nn;
        A[r * ld + c] = (r < dim && c < dim) ? blk[r * dim + c] : 0.0;
        V[r * ld + c] = (r == c) ? 1.0 : 0.0;
    }
    for (int k = t; k < nn; k += EIG_THREADS) perm[k] = k;
    __syncthreads();
    // total Frobenius norm^2 for the stopping rule
    double loc = 0.0;
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
        const double v = A[(idx / dim) * ld + idx % dim];
        loc += v * v;
    }
    s_red[t] = loc;
    __syncthreads();
    for (int s = EIG_THREADS / 2; s > 0; s >>= 1) {
        if (t < s) s_red[t] += s_red[t + s];
        __syncthreads();
    }
    const double total = s_red[0];
    __syncthreads();
    const int half = nn / 2;
    for (int sweep = 0; sweep < 40; ++sweep) {
        // off-diagonal norm^2
        loc = 0.0;
        for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
            const int r = idx / dim, c = idx % dim;
            if (r != c) {
                const double v = A[r * ld + c];
                loc += v * v;
            }
        }
        s_red[t] = loc;
        __syncthreads();
        for (int s = EIG_THREADS / 2; s > 0; s >>= 1) {
            if (t < s) s_red[t] += s_red[t + s];
            __syncthreads();
        }
        if (t == 0) s_done = (s_red[0] <= 1e-32 * total || s_red[0] == 0.0) ? 1 : 0;
        __syncthreads();
        if (s_done) break;
        for (int round = 0; round < nn - 1; ++round) {
            // rotation parameters for each disjoint pair
            for (int k = t; k < half; k += EIG_THREADS) {
                int p = perm[k], q = perm[nn - 1 - k];
                if (p > q) { const int tmp = p; p = q; q = tmp; }
                double c = 1.0, s = 0.0;
                if (q < dim) {
                    const double apq = A[p * ld + q];
                    if (apq != 0.0) {
                        const double app = A[p * ld + p], aqq = A[q * ld + q];
                        const double theta = (aqq - app) / (2.0 * apq);
                        const double tt = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                        c = 1.0 / sqrt(tt * tt + 1.0);
                        s = tt * c;
                    }
                }
                cs[2 * k] = c;
                cs[2 * k + 1] = s;
            }
            __syncthreads();
            // columns: A <- A R, V <- V R
            for (int idx = t; idx < half * nn; idx += EIG_THREADS) {
                const int k = idx / nn, r = idx % nn;
                int p = perm[k], q = perm[nn - 1 - k];
                if (p > q) { const int tmp = p; p = q; q = tmp; }
                const double c = cs[2 * k], s = cs[2 * k + 1];
                if (s == 0.0) continue;
                const double arp = A[r * ld + p], arq = A[r * ld + q];
                A[r * ld + p] = c * arp - s * arq;
                A[r * ld + q] = s * arp + c * arq;
                const double vrp = V[r * ld + p], vrq = V[r * ld + q];
                V[r * ld + p] = c * vrp - s * vrq;
                V[r * ld + q] = s * vrp + c * vrq;
            }
            __syncthreads();
            // rows: A <- R^T A
            for (int idx = t; idx < half * nn; idx += EIG_THREADS) {
                const int k = idx / nn, r = idx % nn;
                int p = perm[k], q = perm[nn - 1 - k];
                if (p > q) { const int tmp = p; p = q; q = tmp; }
                const double c = cs[2 * k], s = cs[2 * k + 1];
                if (s == 0.0) continue;
                const double apr = A[p * ld + r], aqr = A[q * ld + r];
                A[p * ld + r] = c * apr - s * aqr;
                A[q * ld + r] = s * apr + c * aqr;
            }
            __syncthreads();
            for (int k = t; k < half; k += EIG_THREADS) {
                int p = perm[k], q = perm[nn - 1 - k];
                if (cs[2 * k + 1] != 0.0) {
                    A[p * ld + q] = 0.0;
                    A[q * ld + p] = 0.0;
                }
            }
            __syncthreads();
            // round-robin: keep perm[0], rotate perm[1..nn-1]
            if (t == 0) {
                const int last = perm[nn - 1];
                for (int k = nn - 1; k > 1; --k) perm[k] = perm[k - 1];
                perm[1] = last;
            }
            __syncthreads();
        }
    }
    // eigenvalues on the diagonal; f(lambda) into cs[0..dim)
    loc = 0.0;
    for (int k = t; k < dim; k += EIG_THREADS) loc = fmax(loc, fabs(A[k * ld + k]));
    s_red[t] = loc;
    __syncthreads();
    for (int s = EIG_THREADS / 2; s > 0; s >>= 1) {
        if (t < s) s_red[t] = fmax(s_red[t], s_red[t + s]);
        __syncthreads();
    }
    const double lower = 1e-12 * s_red[0];
    __syncthreads();
    for (int k = t; k < dim; k += EIG_THREADS) {
        if (project) {
            cs[k] = fmax(A[k * ld + k], 0.0);
        } else {
            const double ev = fabs(A[k * ld + k]);
            cs[k] = ev >= lower ? 1.0 / ev : 1.0 / lower;
        }
    }
    __syncthreads();
    for (int idx = t; idx < dim * dim; idx += EIG_THREADS) {
        const int r = idx / dim, c = idx % dim;
        double s = 0.0;
        for (int k = 0; k < dim; ++k) s += V[r * ld + k] * cs[k] * V[c * ld + k];
        blk[idx] = s;
    }
}

// ------------------------------------------------------------------ blocks above 96 x 96
// Blocked Gauss-Jordan inversion in global memory, 64 x 64 tiles, all large blocks of an update
// together. The block and every intermediate matrix are known from their lower triangles: with S the panels
// eliminated so far, M_ij is symmetric between tiles that are both in S or both not, and
// M_ji = -M_ij^T between one in S and one not. So only tiles on and below the diagonal are read and written.
// For panel k:
//   (1) P = A_kk^-1 in LDS (gj_tiles: unpivoted; every pivot is a diagonal entry of a Schur complement,
//       positive iff the block is positive definite);
//   (2) for every tile t != k: C_t = A_tk (t > k as stored; t < k, already eliminated: -A_kt^T) and
//       R_t = M_kt = s_t P C_t^T, s_t = 1 for t > k and -1 for t < k; stored as M_tk = -R_t^T (t > k) or
//       M_kt = R_t (t < k), M_kk = P, and C and R as panels for (3);
//   (3) M_ij = A_ij - C_i R_j for tiles i >= j other than k.
// The products run on v_mfma_f64_16x16x4. (3) is bound by memory: it reads and writes half a block once per
// panel, 51 blocks of 570 x 570 (132 MB, held by the Infinity Cache) in 9 panels; 32 x 32 tiles over whole blocks
// moved four times as much (18 panels; 64 us per panel, 2.1 ms per update).
// The inverse is accepted when |B|_F |B^-1|_F < SPD_COND_LIMIT (an upper bound of kappa_2): the
// eigenvalue clamp is then inactive and B^+ = B^-1. A block without that certificate (indefinite or too
// ill-conditioned) raises KERR_SCHWARZ: large blocks have no eigen fallback.
constexpr int BT = 64, BTP = 65;  // tile size, LDS row stride

// |B|_F^2 of every large block in BGJ_NORM_SPLIT partial sums: work-group (l, y) sums the y-th contiguous
// chunk of block l's entries into out[y] of the block's partials; k_bgj_check adds the partials in order.
__global__ __launch_bounds__(EIG_THREADS) void k_bgj_norm(const int32_t* __restrict__ large,
                                                          const int32_t* __restrict__ msz,
                                                          const int64_t* __restrict__ val_off,
                                                          const double* __restrict__ blocks, double* __restrict__ out,
                                                          int stride) {
    __shared__ double s_red[EIG_THREADS];
    const int b = large[blockIdx.x];
    const int dim = 3 * msz[b];
    const int64_t n = (int64_t)dim * dim;
    const int64_t chunk = (n + BGJ_NORM_SPLIT - 1) / BGJ_NORM_SPLIT;
    const int64_t c0 = blockIdx.y * chunk, c1 = min(n, c0 + chunk);
    const double* blk = blocks + val_off[b];
    double loc = 0.0;
    for (int64_t idx = c0 + threadIdx.x; idx < c1; idx += EIG_THREADS) loc += blk[idx] * blk[idx];
    const double tot = block_sum(loc, s_red);
    if (threadIdx.x == 0) out[(int64_t)blockIdx.x * stride + blockIdx.y] = tot;
}

// (1) P = A_kk^-1 by a work-group whose s_a (stride BTP) holds A_kk (bk x bk, its lower triangle mirrored,
// the padding the identity); false, in every thread, and an error if the block is not positive definite
__device__ inline bool bgj_invert(double* s_a, int bk, int& s_bad, double* out, int* err) {
    if (threadIdx.x == 0) s_bad = 0;
    __syncthreads();
    if (!gj_tiles<BT / 16, 4>(s_a, bk, s_bad)) {
        if (threadIdx.x == 0) atomicOr(err, KERR_SCHWARZ);
        return false;
    }
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT;
        out[idx] = 0.5 * (s_a[r * BTP + c] + s_a[c * BTP + r]);
    }
    return true;
}

// panel 0's pivot tile of every large block; the others' are inverted where the update finishes them
__global__ __launch_bounds__(EIG_THREADS) void k_bgj_pivot(const int32_t* __restrict__ large,
                                                           const int32_t* __restrict__ msz,
                                                           const int64_t* __restrict__ val_off,
                                                           const double* __restrict__ blocks, double* __restrict__ piv,
                                                           int* __restrict__ fallback, int* err) {
    __shared__ double s_a[BT * BTP];
    __shared__ int s_bad;
    const int lb = blockIdx.x, b = large[lb];
    const int dim = 3 * msz[b];
    if (fallback[b] != 4) return;
    const int bk = min(BT, dim);
    const double* blk = blocks + val_off[b];
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT;
        const int i = max(r, c), j = min(r, c);  // the lower triangle's entry
        s_a[r * BTP + c] = i < bk ? blk[(int64_t)i * dim + j] : (r == c ? 1.0 : 0.0);
    }
    if (!bgj_invert(s_a, bk, s_bad, piv + (int64_t)lb * BT * BT, err) && threadIdx.x == 0) fallback[b] = 5;
}

// acc[2 a + c] += the 16 x 16 tiles (2 si + a, 2 sj + c) of A B (64 x 64 in LDS): a wavefront's 32 x 32 quarter
__device__ inline void bgj_mfma(sgj_double4 (&acc)[4], const double* A, const double* B, int si, int sj) {
    const int l = threadIdx.x & 63;
    const double* pa = A + (32 * si + (l & 15)) * BTP + (l >> 4);
    const double* pb = B + (l >> 4) * BTP + 32 * sj + (l & 15);
#pragma unroll 4
    for (int ks = 0; ks < BT / 4; ++ks) {
        const double a0 = pa[4 * ks], a1 = pa[16 * BTP + 4 * ks];
        const double b0 = pb[4 * ks * BTP], b1 = pb[4 * ks * BTP + 16];
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[2], 0, 0, 0);
        acc[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[3], 0, 0, 0);
    }
}

// f(row, column, acc item) over the wavefront's quarter of a 64 x 64 tile
template <class F>
__device__ inline void bgj_each(int si, int sj, F f) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) f(32 * si + 16 * (q >> 1) + 4 * v + (l >> 4), 32 * sj + 16 * (q & 1) + (l & 15), q, v);
}

// (2) the panels C_t and R_t of tile t and the block's new tile; colp and rowp hold 64 x 64 tiles, zero past dim
__global__ __launch_bounds__(EIG_THREADS) void k_bgj_panel(const int32_t* __restrict__ large,
                                                           const int32_t* __restrict__ msz,
                                                           const int64_t* __restrict__ val_off,
                                                           double* __restrict__ blocks, const double* __restrict__ piv,
                                                           double* __restrict__ colp, double* __restrict__ rowp,
                                                           const int64_t* __restrict__ panel_off,
                                                           const int* __restrict__ fallback, int k) {
    extern __shared__ double lds[];
    double *sP = lds, *sC = lds + BT * BTP;  // sC: C_t^T
    const int lb = blockIdx.x, b = large[lb], t = blockIdx.y;
    const int dim = 3 * msz[b];
    const int nt = (dim + BT - 1) / BT;
    if (BT * k >= dim || t >= nt || fallback[b] != 4) return;
    double* blk = blocks + val_off[b];
    const double* P = piv + (int64_t)lb * BT * BT;
    if (t == k) {
        for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
            const int r = BT * k + idx / BT, c = BT * k + idx % BT;
            if (r < dim && c < dim) blk[(int64_t)r * dim + c] = P[idx];
        }
        return;
    }
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT;
        sP[r * BTP + c] = P[idx];
        // the stored tile: rows of the larger tile index
        const int gr = BT * max(t, k) + r, gc = BT * min(t, k) + c;
        const double v = gr < dim && gc < dim ? blk[(int64_t)gr * dim + gc] : 0.0;
        if (t > k)
            sC[c * BTP + r] = v;
        else
            sC[r * BTP + c] = -v;
    }
    __syncthreads();
    double* C = colp + panel_off[lb] + (int64_t)t * BT * BT;
    double* R = rowp + panel_off[lb] + (int64_t)t * BT * BT;
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) C[idx] = sC[(idx % BT) * BTP + idx / BT];
    const int w = threadIdx.x >> 6, si = w >> 1, sj = w & 1;
    sgj_double4 acc[4] = {};
    bgj_mfma(acc, sP, sC, si, sj);
    const double sign = t > k ? 1.0 : -1.0;
    bgj_each(si, sj, [&](int r, int c, int q, int v) {
        const double x = sign * acc[q][v];
        R[r * BT + c] = x;
        if (t < k && BT * k + r < dim && BT * t + c < dim) blk[(int64_t)(BT * k + r) * dim + BT * t + c] = x;
    });
    if (t < k) return;
    __syncthreads();  // M_tk = -R_t^T by way of sC, so that its rows are stored contiguously
    bgj_each(si, sj, [&](int r, int c, int q, int v) { sC[c * BTP + r] = -acc[q][v]; });
    __syncthreads();
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = BT * t + idx / BT, c = BT * k + idx % BT;
        if (r < dim && c < dim) blk[(int64_t)r * dim + c] = sC[(idx / BT) * BTP + idx % BT];
    }
}

// tile pair of index n among those on and below the diagonal
__device__ inline void bgj_lower(int n, int& i, int& j) {
    i = (int)((sqrtf(8.0f * (float)n + 1.0f) - 1.0f) * 0.5f);
    while ((i + 1) * (i + 2) / 2 <= n) ++i;
    while (i * (i + 1) / 2 > n) --i;
    j = n - i * (i + 1) / 2;
}

// (3) M_ij = A_ij - C_i R_j, tiles i >= j other than k. The work-group of tile (k + 1, k + 1), among the first to
// start, goes on to invert it: the next panel's pivot, 28 us (41 us one pivot at a time through LDS), runs beside the
// other tiles' updates. Two work-groups per CU by their LDS, so its registers cost the others nothing.
__global__ __launch_bounds__(EIG_THREADS) void k_bgj_update(const int32_t* __restrict__ large,
                                                            const int32_t* __restrict__ msz,
                                                            const int64_t* __restrict__ val_off,
                                                            double* __restrict__ blocks, const double* __restrict__ colp,
                                                            const double* __restrict__ rowp,
                                                            const int64_t* __restrict__ panel_off,
                                                            double* __restrict__ piv, const int* __restrict__ fallback,
                                                            int* err, int k) {
    extern __shared__ double lds[];
    __shared__ int s_bad;
    double *sA = lds, *sB = lds + BT * BTP;
    const int lb = blockIdx.x, b = large[lb];
    const int dim = 3 * msz[b];
    int ti, tj, n = (int)blockIdx.y;
    const int next = (k + 1) * (k + 2) / 2 + k + 1;  // tile (k + 1, k + 1), swapped with tile 0
    if (next < (int)gridDim.y && (n == 0 || n == next)) n = next - n;
    bgj_lower(n, ti, tj);
    if (BT * k >= dim || BT * ti >= dim || ti == k || tj == k || fallback[b] != 4) return;
    double* blk = blocks + val_off[b];
    const int w = threadIdx.x >> 6, si = w >> 1, sj = w & 1;
    const double* C = colp + panel_off[lb] + (int64_t)ti * BT * BT;
    const double* R = rowp + panel_off[lb] + (int64_t)tj * BT * BT;
    sgj_double4 acc[4];
    bgj_each(si, sj, [&](int r, int c, int q, int v) {
        const int gr = BT * ti + r, gc = BT * tj + c;
        acc[q][v] = gr < dim && gc < dim ? blk[(int64_t)gr * dim + gc] : 0.0;
    });
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT;
        sA[r * BTP + c] = -C[idx];
        sB[r * BTP + c] = R[idx];
    }
    __syncthreads();
    bgj_mfma(acc, sA, sB, si, sj);
    bgj_each(si, sj, [&](int r, int c, int q, int v) {
        const int gr = BT * ti + r, gc = BT * tj + c;
        if (gr < dim && gc < dim) blk[(int64_t)gr * dim + gc] = acc[q][v];
    });
    if (n != next) return;
    const int bk = min(BT, dim - BT * (k + 1));
    __syncthreads();  // sA has been read
    bgj_each(si, sj, [&](int r, int c, int q, int v) {
        if (r < c) return;
        const double x = r < bk ? acc[q][v] : (r == c ? 1.0 : 0.0);
        sA[r * BTP + c] = x;
        sA[c * BTP + r] = x;
    });
    bgj_invert(sA, bk, s_bad, piv + (int64_t)lb * BT * BT, err);
}

// The inverse's upper triangle from its lower one (the diagonal tiles averaged with their transposes), and
// the tile pair's share of |B^-1|_F^2 into the block's partials after the BGJ_NORM_SPLIT of |B|_F^2
__global__ __launch_bounds__(EIG_THREADS) void k_bgj_mirror(const int32_t* __restrict__ large,
                                                            const int32_t* __restrict__ msz,
                                                            const int64_t* __restrict__ val_off,
                                                            double* __restrict__ blocks, double* __restrict__ lnorm,
                                                            const int* __restrict__ fallback, int stride) {
    __shared__ double sA[BT * BTP];
    __shared__ double s_red[EIG_THREADS];
    const int lb = blockIdx.x, b = large[lb];
    const int dim = 3 * msz[b];
    int ti, tj;
    bgj_lower((int)blockIdx.y, ti, tj);
    if (BT * ti >= dim || fallback[b] != 4) return;
    double* blk = blocks + val_off[b];
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT, gr = BT * ti + r, gc = BT * tj + c;
        sA[r * BTP + c] = gr < dim && gc < dim ? blk[(int64_t)gr * dim + gc] : 0.0;
    }
    __syncthreads();
    double loc = 0.0;
    for (int idx = threadIdx.x; idx < BT * BT; idx += EIG_THREADS) {
        const int r = idx / BT, c = idx % BT, gr = BT * tj + r, gc = BT * ti + c;  // entry (r, c) of tile (tj, ti)
        const double x = ti == tj ? 0.5 * (sA[r * BTP + c] + sA[c * BTP + r]) : sA[c * BTP + r];
        loc += x * x;
        if (gr < dim && gc < dim) blk[(int64_t)gr * dim + gc] = x;
    }
    const double tot = block_sum(loc, s_red);
    if (threadIdx.x == 0) lnorm[(int64_t)lb * stride + BGJ_NORM_SPLIT + blockIdx.y] = ti == tj ? tot : 2.0 * tot;
}

// the certificate of every large block from its norms' partial sums
__global__ __launch_bounds__(64) void k_bgj_check(const int32_t* __restrict__ large, const int32_t* __restrict__ msz,
                                                  const double* __restrict__ lnorm, const int* __restrict__ fallback,
                                                  int* err, int stride) {
    const int lb = blockIdx.x, b = large[lb];
    if (fallback[b] != 4) return;
    const int nt = (3 * msz[b] + BT - 1) / BT, parts = nt * (nt + 1) / 2;
    const double* n2 = lnorm + (int64_t)lb * stride;
    double nb = 0.0, ni = 0.0;
    for (int y = threadIdx.x; y < BGJ_NORM_SPLIT; y += 64) nb += n2[y];
    for (int y = threadIdx.x; y < parts; y += 64) ni += n2[BGJ_NORM_SPLIT + y];
    for (int off = 32; off > 0; off >>= 1) {
        nb += __shfl_xor(nb, off, 64);
        ni += __shfl_xor(ni, off, 64);
    }
    if (threadIdx.x == 0 && !(sqrt(nb) * sqrt(ni) < SPD_COND_LIMIT)) atomicOr(err, KERR_SCHWARZ);
}

static void schwarz_update_large(Schwarz& s) {
    Model& m = *s.model;
    const hipStream_t st = m.stream;
    const unsigned nl = (unsigned)s.large.size();
    const int ntm = (s.large_max_dim + BT - 1) / BT, lower = ntm * (ntm + 1) / 2;
    const int stride = BGJ_NORM_SPLIT + lower;
    const int32_t* lg = s.d_large.get();
    const int32_t* msz = s.scatter.d_m.get();
    const int64_t* vo = s.scatter.d_val_off.get();
    const int64_t* po = s.d_panel_off.get();
    const int* fb = s.d_fallback.get();
    double* colp = s.d_panels.get();
    double* rowp = colp + s.d_panels.n / 2;
    const size_t lds = (size_t)2 * BT * BTP * sizeof(double);
    raise_lds_limit((const void*)k_bgj_panel, lds);
    raise_lds_limit((const void*)k_bgj_update, lds);
    hipLaunchKernelGGL(k_bgj_norm, dim3(nl, BGJ_NORM_SPLIT), dim3(EIG_THREADS), 0, st, lg, msz, vo,
                       (const double*)s.d_blocks.get(), s.d_lnorm.get(), stride);
    hipLaunchKernelGGL(k_bgj_pivot, dim3(nl), dim3(EIG_THREADS), 0, st, lg, msz, vo, (const double*)s.d_blocks.get(),
                       s.d_piv.get(), s.d_fallback.get(), m.d_err.get());
    for (int k = 0; k < ntm; ++k) {
        hipLaunchKernelGGL(k_bgj_panel, dim3(nl, (unsigned)ntm), dim3(EIG_THREADS), lds, st, lg, msz, vo,
                           s.d_blocks.get(), (const double*)s.d_piv.get(), colp, rowp, po, fb, k);
        hipLaunchKernelGGL(k_bgj_update, dim3(nl, (unsigned)lower), dim3(EIG_THREADS), lds, st, lg, msz, vo,
                           s.d_blocks.get(), (const double*)colp, (const double*)rowp, po, s.d_piv.get(),
                           s.d_fallback.get(), m.d_err.get(), k);
    }
    hipLaunchKernelGGL(k_bgj_mirror, dim3(nl, (unsigned)lower), dim3(EIG_THREADS), 0, st, lg, msz, vo,
                       s.d_blocks.get(), s.d_lnorm.get(), fb, stride);
    hipLaunchKernelGGL(k_bgj_check, dim3(nl), dim3(64), 0, st, lg, msz, (const double*)s.d_lnorm.get(), fb,
                       m.d_err.get(), stride);
    check_launch("blocked Gauss-Jordan");
}

// untreated nodes: P_ii = 1 / J_ii (schwarz_precond.rs:195-213)
template <class VJ, class VP>
__global__ void k_schwarz_untreated(int64_t nunt, const int32_t* __restrict__ unt, const int32_t* __restrict__ prowptr,
                                    const int32_t* __restrict__ jdiag, const VJ* __restrict__ J,
                                    VP* __restrict__ P, int* err) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= 3 * nunt) return;
    const int64_t row = 3 * (int64_t)unt[idx / 3] + idx % 3;
    const int32_t dp = jdiag[row];
    const double entry = dp >= 0 ? (double)J[dp] : 0.0;
    if (entry != 0.0)
        P[prowptr[row]] = (VP)(1.0 / entry);
    else
        atomicOr(err, KERR_ZERO_DIAG);
}

template <class VJ>
static void schwarz_update_t(Schwarz& s, const VJ* J) {
    Model& m = *s.model;
    const hipStream_t st = m.stream;
    if (s.nsub > 0) {
        if (!s.large.empty()) {
            const int64_t gmax = s.large_max_dim;
            const unsigned chunks = (unsigned)((gmax * gmax + SG_CHUNK - 1) / SG_CHUNK);
            k_schwarz_gather<VJ><<<dim3((unsigned)s.large.size(), chunks), dim3(256), 0, st>>>(
                s.d_large.get(), s.scatter.d_m.get(), s.scatter.d_val_off.get(), s.scatter.d_slot_off.get(), s.d_off.get(),
                s.d_nodes.get(), s.d_jslot.get(), m.pattern.d_rowptr.get(), J, s.d_blocks.get());
            check_launch("k_schwarz_gather");
        }
        const int dim = std::max(3, s.small_max_dim);
        // Gauss-Jordan fast path (blocks up to 96 x 96; it marks the larger ones 4), the sharper
        // certificate for the blocks it could not accept, then the eigen path for the rest; blocks
        // above 96 x 96 go through the blocked path
        auto run = [&](auto kernel, int nt, int nw) {
            const size_t lds = (size_t)16 * nt * (16 * nt + 1) * sizeof(double);
            raise_lds_limit((const void*)kernel, lds);
            hipLaunchKernelGGL(kernel, dim3((unsigned)s.nsub), dim3(64 * nw), lds, st, s.scatter.d_m.get(),
                               s.scatter.d_val_off.get(), s.scatter.d_slot_off.get(), s.d_off.get(), s.d_nodes.get(),
                               s.d_jslot.get(), m.pattern.d_rowptr.get(), J, s.d_blocks.get(), s.d_fallback.get());
            check_launch("k_spd_inverse_mf");
        };
        if (dim <= 16)
            run(&k_spd_inverse_mf<VJ, 1, 1>, 1, 1);
        else if (dim <= 32)
            run(&k_spd_inverse_mf<VJ, 2, 1>, 2, 1);
        else if (dim <= 64)
            run(&k_spd_inverse_mf<VJ, 4, 4>, 4, 4);
        else
            run(&k_spd_inverse_mf<VJ, 6, 8>, 6, 8);
        const int dp = (dim + 3) & ~3;
        const int ld_pc = dp + 1;
        const size_t lds_pc = (size_t)2 * dp * ld_pc * sizeof(double);  // 149 KB at dim 96
        raise_lds_limit((const void*)k_spd_power_certify<VJ>, lds_pc);
        hipLaunchKernelGGL(k_spd_power_certify<VJ>, dim3((unsigned)s.nsub), dim3(EIG_THREADS), lds_pc, st,
                           s.scatter.d_m.get(), s.scatter.d_val_off.get(), s.scatter.d_slot_off.get(), s.d_off.get(),
                           s.d_nodes.get(), s.d_jslot.get(), m.pattern.d_rowptr.get(), J, s.d_blocks.get(),
                           s.d_fallback.get(), ld_pc);
        check_launch("k_spd_power_certify");
        const int nn = dim + (dim & 1);
        const int ld = nn + 1;
        const size_t lds = (size_t)2 * nn * ld * sizeof(double) + (size_t)nn * sizeof(double) + (size_t)nn * sizeof(int);
        // at least the size of this launch (147 KB for 96 x 96 blocks), raised monotonically
        raise_lds_limit((const void*)k_jacobi_inverse, lds);
        hipLaunchKernelGGL(k_jacobi_inverse, dim3((unsigned)s.nsub), dim3(EIG_THREADS), lds, st, s.scatter.d_m.get(),
                           s.scatter.d_val_off.get(), s.d_blocks.get(), (const int*)s.d_fallback.get(), ld, 0);
        check_launch("k_jacobi_inverse");
        if (!s.large.empty()) schwarz_update_large(s);
        if (s.fp32)
            launch_block_gather(s.P, s.scatter, s.d_blocks.get(), s.d_vals32.get(), 0, 0.0, nullptr, true, st);
        else
            launch_block_gather(s.P, s.scatter, s.d_blocks.get(), s.d_vals.get(), 0, 0.0, nullptr, true, st);
    }
    if (!s.untreated.empty()) {
        const int64_t n = 3 * (int64_t)s.untreated.size();
        const unsigned g = (unsigned)((n + 255) / 256);
        if (s.fp32)
            k_schwarz_untreated<VJ, float><<<dim3(g), dim3(256), 0, st>>>(
                (int64_t)s.untreated.size(), s.d_untreated.get(), s.P.d_rowptr.get(), m.pattern.d_diag_pos.get(), J,
                s.d_vals32.get(), m.d_err.get());
        else
            k_schwarz_untreated<VJ, double><<<dim3(g), dim3(256), 0, st>>>(
                (int64_t)s.untreated.size(), s.d_untreated.get(), s.P.d_rowptr.get(), m.pattern.d_diag_pos.get(), J,
                s.d_vals.get(), m.d_err.get());
        check_launch("k_schwarz_untreated");
    }
}

// DefaultSemidefiniteProjection of every element matrix in m.d_ke (row-major (3n)^2 per element),
// in place: a Cholesky certificate keeps the blocks that are positive semi-definite to within
// rounding, the Newton-Schulz sign iteration (one work-group per element) projects the rest.
void launch_element_psd_projection(Model& m) {
    if (m.ne == 0) return;
    if (m.d_elem_m.n != (size_t)m.ne || m.d_elem_m.p == nullptr) {
        std::vector<int32_t> msz((size_t)m.ne, m.n);
        std::vector<int64_t> off((size_t)m.ne);
        for (int64_t e = 0; e < m.ne; ++e) off[e] = e * 9 * (int64_t)m.n * m.n;
        m.d_elem_m.upload(msz, m.stream);
        m.d_elem_off.upload(off, m.stream);
    }
    const int dim = 3 * m.n;
    m.d_elem_need.ensure((size_t)m.ne);
    const int ld_c = dim + 1;
    const size_t lds_c = (size_t)dim * ld_c * sizeof(double);
    raise_lds_limit((const void*)k_psd_certify, 120 * 1024);
    hipLaunchKernelGGL(k_psd_certify, dim3((unsigned)m.ne), dim3(EIG_THREADS), lds_c, m.stream, m.d_elem_m.get(),
                       m.d_elem_off.get(), (const double*)m.d_ke.get(), m.d_elem_need.get(), ld_c);
    check_launch("k_psd_certify");
    const int nt = (dim + 15) / 16;
    const size_t lds_ns = (size_t)2 * 16 * nt * (16 * nt + 1) * sizeof(double);  // 149 KB at 81 x 81
    auto run = [&](auto kernel) {
        raise_lds_limit((const void*)kernel, lds_ns);
        hipLaunchKernelGGL(kernel, dim3((unsigned)m.ne), dim3(EIG_THREADS), lds_ns, m.stream, m.d_elem_m.get(),
                           m.d_elem_off.get(), m.d_ke.get(), (const int*)m.d_elem_need.get());
    };
    switch (nt) {
        case 1: run(&k_psd_newton_schulz<1>); break;
        case 2: run(&k_psd_newton_schulz<2>); break;
        case 4: run(&k_psd_newton_schulz<4>); break;
        case 6: run(&k_psd_newton_schulz<6>); break;
        default: throw Error(HOEFEM_ERROR_INVALID_ARGUMENT, "element matrix size without a projection kernel");
    }
    check_launch("k_psd_newton_schulz");
}

void schwarz_update(Schwarz& s, const double* J) { schwarz_update_t<double>(s, J); }
void schwarz_update(Schwarz& s, const float* J) { schwarz_update_t<float>(s, J); }

void schwarz_apply(Schwarz& s, const double* x, double* y) {
    if (s.fp32)
        launch_spmv(s.P, s.d_vals32.get(), 0.0, y, 1.0, x, s.model->stream);
    else
        launch_spmv(s.P, s.d_vals.get(), 0.0, y, 1.0, x, s.model->stream);
}

}  // namespace hoefem
