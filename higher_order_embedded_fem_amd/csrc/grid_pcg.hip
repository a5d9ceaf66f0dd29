// Preconditioned conjugate gradient (fenris/src/cg.rs:377-482) as one resident grid: the whole solve of
// a system that fits the chip's register files and L2s runs in one launch (in chunks of iterations), its
// work-groups exchanging vectors and dot products through memory instead of through kernel boundaries.
//
// Why. The two-kernel iteration of solver.hip costs 5-9 us per kernel on the smallest systems (launch,
// descriptor, status, partial sums, row entries, columns and gathered vectors: a chain of dependent memory
// reads that starts anew in every kernel) and reads every matrix value from the Infinity Cache in every
// iteration on the larger ones. Here the matrix values, the columns and the vectors of a work-group's rows
// stay in its registers and LDS between iterations; an iteration moves one vector entry per node and
// phase, and its chain is: store own entries, post a partial sum, poll the others', load the neighbours'.
//
// Split. Work-group b owns a contiguous range of nodes and their rows of A and P, at most 170 nodes (one
// vector component per thread). Thread t holds a run of consecutive 3x3 blocks of those rows (sA of A, then
// sP of P), so every thread has the same work whatever the row lengths are; where a run leaves a row it
// writes the row's partial sum to LDS, and the thread of each row component adds its row's partials in
// order. The first N blocks of a thread stay in registers, the rest is re-read in every iteration from a
// work-group-private, coalesced copy (L2-resident up to about 30 MB).
//
// Iteration k (z, p, r: own entries in registers, own and neighbour entries in LDS):
//   A  p <- z + beta p for own and neighbour nodes (every work-group computes its neighbours' p itself, so
//      only z is exchanged); Ap = A p; publish Ap; exchange p.Ap
//   B  x += alpha p, r <- r - alpha Ap (neighbours' r likewise); z = P r; publish z; exchange z.r, |r|^2
// The stopping tests and their order are those of the two-kernel path.
//
// Exchange. Vector entries and partial sums are stored and loaded with agent scope (write-through stores,
// loads past the L2), so no cache is written back or invalidated, and every value is its own flag: an entry
// holds a sentinel (a signalling NaN, which no arithmetic yields) until its owner stores it, and its
// readers poll it. A phase thus costs one trip of a store and one of a load, the vector entries' beside the
// partial sums'. Every work-group adds all partial sums in the same order, so all agree on alpha, beta and
// the stopping tests bit for bit. Four sets of entries are used in turn. A work-group stores its entries of
// phase m and the sentinel into those of phase m + 2: their previous use, phase m - 2, has been read by all
// (they posted phase m - 1 after it), and the sentinel is in memory before the work-group posts phase m + 1
// (its waves wait for their older stores, s_waitcnt vmcnt(0), before the stores of a phase), so
// before anyone can poll phase m + 2.
//
// Residency. The work-groups wait for each other, so all of a launch's must be resident: launches are
// admitted in order against the CUs of every XCD (GridSlots below), one work-group per CU. Every wait is
// bounded (GRID_POLL_LIMIT polls); a launch that cannot make progress, because another process holds CUs, ends with
// an error status, the caller falls back to the two-kernel path, and so do its next solves (GridRest).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>

#include "grid_pcg.hpp"
#include "host_threads.hpp"

namespace hoefem {

namespace {

constexpr unsigned long long GRID_EMPTY = 0x7ff4deadbeef0001ull;  // slot sentinel
constexpr int GRID_POLL_LIMIT = 1 << 21;                           // about 2 s of polling
constexpr int GRID_WAVES = GRID_THREADS / 64;
// copies of the partial sums, each read by an eighth of the work-groups: 256 work-groups polling one array
// queue at its few memory channels (an exchange of partial sums alone takes 1.5 us at 8 work-groups, 2.3 at 256 with 8
// copies and 3.1 with one)
constexpr int GRID_COPIES = 8;

__device__ inline double agent_load(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void agent_store(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// the sum over the wavefront's lanes, the same in every lane (register lane shifts, no LDS)
__device__ inline double wave_total(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of each row of 16 holds the row's sum
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3: lane 63 holds the total
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ inline float fmav(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fmav(double a, double b, double c) { return __builtin_fma(a, b, c); }

// f(0), f(1), .. f(N - 1) with compile-time indices (register arrays stay in registers)
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (N > 0) {
        unrolled<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

__device__ inline bool is_empty(double v) { return (unsigned long long)__double_as_longlong(v) == GRID_EMPTY; }

// A barrier that orders LDS accesses only: global stores and loads in flight are not waited for
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A thread's run of consecutive blocks of its work-group's rows: the block (node, j) it stands at
struct Run {
    int node, j, k, left;
    int64_t base;
};

}  // namespace

// N blocks of a thread in registers: 10 of FP64 (180 of the 256 registers that two waves per SIMD leave a
// thread) or 16 of FP32, the next S.nlds in LDS; pairs of register blocks share one uniform test and have
// their LDS reads in flight together.
// K systems in one launch (descriptors in the kernel arguments), their work-groups one after the other.
template <class VT, int N, int K>
__global__ __launch_bounds__(GRID_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_grid_pcg(
    const GridSegs<VT, K> all) {
#pragma clang fp contract(off)
#define INLINE __attribute__((always_inline))
    extern __shared__ double lds[];
    __shared__ double s_w[GRID_WAVES][2];
    __shared__ double s_tot[2];
    __shared__ int s_bad;
    __shared__ double s_x[GRID_THREADS], s_v[GRID_THREADS], s_d[GRID_THREADS];  // own x; Ap or z; diagonal entries
    __shared__ uint32_t s_rows[2][GRID_THREADS];  // own component's partial sums: first | count << 16
    int b = (int)blockIdx.x, seg = 0;
    while (seg + 1 < K && b >= all.seg[seg].W) b -= all.seg[seg++].W;  // uniform
    const GridSeg<VT>& S = all.seg[seg];
    const int W = S.W;
    const GridWg g = S.wg[b];
    int sA = __builtin_amdgcn_readfirstlane(g.sA), nS = __builtin_amdgcn_readfirstlane(g.sA + g.sP);
    const int nR = N + S.nlds;
    double* s_p = lds;                          // p: own nodes, then A's halo
    double* s_r = s_p + 3 * (g.nown + g.nhA);   // r: own nodes, then P's halo
    double* s_part = s_r + 3 * (g.nown + g.nhP);
    VT* s_blk = reinterpret_cast<VT*>(lds + S.blk_off);  // the LDS-held blocks, [block][entry][thread]
    int t = threadIdx.x;

    // ---- the thread's blocks: values, packed columns, and the mask of blocks that end a row or the run
    static_assert(N % 2 == 0, "blocks are taken in pairs");
    VT v[N][9];
    constexpr int NL = GRID_LDS_SLOTS, NC = (N + NL) / 2;  // columns of the register and LDS blocks, in pairs
    uint32_t cp[NC];
#pragma unroll
    for (int s = 0; s < NC; ++s) cp[s] = 0;
    uint32_t mask = 0, pos;  // pos: the run's first partial sum of A | of P << 16
    {
        const uint16_t* col = S.col + g.col_off;
        VT* ws = S.ws + g.ws_off;
        const int64_t th = (int64_t)b * GRID_THREADS + t;
        const GridStart stA = S.start[2 * th], stP = S.start[2 * th + 1];
        pos = (uint32_t)stA.pos | (uint32_t)stP.pos << 16;
        Run R;
        const int32_t *nptr, *rowptr;
        const uint8_t* single;
        const VT* vals;
        auto open = [&](const GridStart& st, int slots, int blocks, const int32_t* np, const int32_t* rp,
                        const uint8_t* dg, const VT* va) INLINE {
            nptr = np;
            rowptr = rp;
            single = dg;
            vals = va;
            R.node = st.node;
            R.j = st.j;
            R.left = min(slots, max(0, blocks - t * slots));
            R.k = 0;
            if (R.left > 0) {
                R.k = nptr[R.node + 1] - nptr[R.node];
                R.base = rowptr[3 * (int64_t)R.node];
            }
        };
        // the run's next block into u[9] (zeros past its end); true where it ends a row or the run
        auto next = [&](VT* u) INLINE -> bool {
            if (R.left <= 0) {
#pragma unroll
                for (int c = 0; c < 9; ++c) u[c] = VT(0);
                return false;
            }
            const VT* src = vals + R.base + 3 * R.j;
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int c = 0; c < 3; ++c) u[3 * i + c] = src[3 * (int64_t)R.k * i + c];
            R.left -= 1;
            R.j += 1;
            const bool end = R.j == R.k;
            if (end && R.left > 0) {
                R.j = 0;
                do {
                    R.node += 1;
                    R.k = single && single[R.node] ? 0 : nptr[R.node + 1] - nptr[R.node];
                } while (R.k == 0);
                R.base = rowptr[3 * (int64_t)R.node];
            }
            return end || R.left == 0;
        };
        open(stA, sA, g.nbA, S.jnptr, S.jrowptr, nullptr, S.A);
        unrolled<N>([&](auto I) INLINE {
            constexpr int s = I;
            if (s < nS) {
                if (s == sA) open(stP, g.sP, g.nbP, S.pnptr, S.prowptr, S.pdiag, S.P);
                if (next(v[s])) mask |= 1u << s;
                cp[s / 2] |= (uint32_t)col[s * GRID_THREADS + t] << (16 * (s & 1));
            } else {
#pragma unroll
                for (int c = 0; c < 9; ++c) v[s][c] = VT(0);
            }
        });
        for (int s = N; s < nS; ++s) {
            if (s == sA) open(stP, g.sP, g.nbP, S.pnptr, S.prowptr, S.pdiag, S.P);
            VT u[9];
            if (next(u)) mask |= 1u << s;
            VT* dst = s < nR ? s_blk + (s - N) * 9 * GRID_THREADS : ws + (int64_t)(s - nR) * 9 * GRID_THREADS;
#pragma unroll
            for (int c = 0; c < 9; ++c) dst[c * GRID_THREADS + t] = u[c];
        }
        unrolled<NL>([&](auto I) INLINE {
            constexpr int s = N + I;
            if (s < nR && s < nS) cp[s / 2] |= (uint32_t)col[s * GRID_THREADS + t] << (16 * (s & 1));
        });
    }
    // ---- own component: the partial sums of its rows, the entry of a diagonal row of the preconditioner
    constexpr uint32_t DIAG = 0xffffffffu;
    if (t < 3 * g.nown) {
        const uint16_t* rp = S.rp + g.rp_off + t / 3;
        s_rows[0][t] = (uint32_t)rp[0] | (uint32_t)(rp[1] - rp[0]) << 16;
        s_rows[1][t] = (uint32_t)rp[g.nown + 1] | (uint32_t)(rp[g.nown + 2] - rp[g.nown + 1]) << 16;
        const int64_t node = g.node0 + t / 3;
        const int64_t dof = 3 * (int64_t)g.node0 + t;
        if (S.dinv) {
            s_rows[1][t] = DIAG;
            s_d[t] = S.dinv[dof];
        } else if (S.pdiag[node]) {
            s_rows[1][t] = DIAG;
            s_d[t] = (double)S.P[S.prowptr[3 * node + t % 3]];
        }
        s_x[t] = S.x[dof];
    }
    if (t == 0) s_bad = 0;

    // s_part <- partial row sums of the blocks [s0, s1) times the vector sx. In FP32 a block's row is summed in FP32
    // and the blocks in FP64: one FP32 chain over a thread's run of a row (up to 32 blocks,
    // 96 roundings) had 1.1 to 1.25 times the error of the two-kernel path's short ones on 18 to 90 thousand DOFs; this
    // has 0.62 to 0.7 times (3.0e-8 against 4.8e-8) and takes 0.5 % more of a step.
    auto products = [&](int s0, int s1, const double* sx, int at) INLINE {
        double y0 = 0.0, y1 = 0.0, y2 = 0.0;
        auto flush = [&](int s) INLINE {
            if ((mask >> s) & 1u) {
                double* d = s_part + 3 * at;
                d[0] = y0;
                d[1] = y1;
                d[2] = y2;
                ++at;
                y0 = y1 = y2 = 0.0;
            }
        };
        auto add = [&](const VT* u, VT c0, VT c1, VT c2) INLINE {
            if constexpr (sizeof(VT) == sizeof(double)) {
                y0 = fmav(u[2], c2, fmav(u[1], c1, fmav(u[0], c0, y0)));
                y1 = fmav(u[5], c2, fmav(u[4], c1, fmav(u[3], c0, y1)));
                y2 = fmav(u[8], c2, fmav(u[7], c1, fmav(u[6], c0, y2)));
            } else {
                y0 += (double)fmav(u[2], c2, fmav(u[1], c1, u[0] * c0));
                y1 += (double)fmav(u[5], c2, fmav(u[4], c1, u[3] * c0));
                y2 += (double)fmav(u[8], c2, fmav(u[7], c1, u[6] * c0));
            }
        };
        unrolled<N / 2>([&](auto I) INLINE {
            constexpr int s = 2 * I;
            if (s + 2 <= s0 || s >= s1) return;  // uniform
            const double* xa = sx + (cp[s / 2] & 0xffffu);
            const double* xb = sx + (cp[s / 2] >> 16);
            const bool ina = s >= s0, inb = s + 1 < s1;
            // a slot of the other phase may hold a column past this phase's vector: read entry 0 instead
            if (!ina) xa = sx;
            if (!inb) xb = sx;
            const VT c0 = VT(xa[0]), c1 = VT(xa[1]), c2 = VT(xa[2]);
            const VT e0 = VT(xb[0]), e1 = VT(xb[1]), e2 = VT(xb[2]);
            if (ina) {
                add(v[s], c0, c1, c2);
                flush(s);
            }
            if (inb) {
                add(v[s + 1], e0, e1, e2);
                flush(s + 1);
            }
        });
        unrolled<NL>([&](auto I) INLINE {
            constexpr int s = N + I;
            if (s < s0 || s >= s1 || s >= nR) return;  // uniform
            const double* xx = sx + (s & 1 ? cp[s / 2] >> 16 : cp[s / 2] & 0xffffu);
            VT u[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) u[c] = s_blk[(I * 9 + c) * GRID_THREADS + t];
            add(u, VT(xx[0]), VT(xx[1]), VT(xx[2]));
            flush(s);
        });
        if (s1 > nR) {
            const uint16_t* col = S.col + g.col_off;
            const VT* ws = S.ws + g.ws_off;
            for (int s = max(nR, s0); s < s1; ++s) {
                const double* xx = sx + col[s * GRID_THREADS + t];
                VT u[9];
#pragma unroll
                for (int c = 0; c < 9; ++c) u[c] = ws[((s - nR) * 9 + c) * GRID_THREADS + t];
                add(u, VT(xx[0]), VT(xx[1]), VT(xx[2]));
                flush(s);
            }
        }
    };
    // the own component's row sum: its partials in order, eight in flight (reads past them stay in s_part,
    // which has GRID_SPARE entries more)
    auto row_sum = [&](uint32_t rows) INLINE {
        const double* d = s_part + 3 * (rows & 0xffffu) + t % 3;
        double s = 0.0;
        for (int n = (int)(rows >> 16); n > 0; n -= 8, d += 24) {
            double e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = d[3 * i];
#pragma unroll
            for (int i = 0; i < 8; ++i) s += i < n ? e[i] : 0.0;
        }
        return s;
    };
    uint32_t phase = S.phase;
    constexpr int H = 4;  // halo entries of a thread taken in during the exchange
    double hq[H];
    // Publishes the own components (val; sets of the phase), the work-group's sums v0 (and v1), and takes in
    // the totals over all work-groups and the thread's first H halo components of off[0..n). False if
    // a value did not arrive in time. Begins with all stores of the previous phase complete and ends
    // with a barrier.
    auto exchange = [&](double val, double v0, double v1, int nv, const int32_t* off, int n, double& t0,
                        double& t1) INLINE -> bool {
        double* vec = S.vec + (int64_t)(phase & 3u) * S.ndof;
        {
            double* clean = S.vec + (int64_t)((phase + 2) & 3u) * S.ndof;
            const uint32_t dof = 3 * (uint32_t)g.node0 + t;
            if (t < 3 * g.nown) {
                agent_store(vec + dof, val);
                agent_store(clean + dof, __longlong_as_double((long long)GRID_EMPTY));
            }
            if (t < 2 * GRID_COPIES)
                agent_store((double*)&S.slots[(((phase + 2) & 3u) * 2 * GRID_COPIES + t) * W + b],
                            __longlong_as_double((long long)GRID_EMPTY));
        }
        const int wid = t >> 6, lane = t & 63;
        v0 = wave_total(v0);
        if (nv > 1) v1 = wave_total(v1);
        if (lane == 0) {
            s_w[wid][0] = v0;
            s_w[wid][1] = v1;
        }
        lds_barrier();
        bool missing = true;
        if (wid < nv) {  // wave w: value w
            unsigned long long* sl = S.slots + ((phase & 3u) * 2 + wid) * GRID_COPIES * W;
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < GRID_WAVES; ++w) s += s_w[w][wid];
            if (lane < GRID_COPIES) agent_store((double*)&sl[lane * W + b], s);
            sl += (b % GRID_COPIES) * W;
            double got[GRID_MAX_WG / 64] = {};
            for (int i = 0; missing && i < S.polls; ++i) {
                missing = false;
#pragma unroll
                for (int q = 0; q < GRID_MAX_WG / 64; ++q) {
                    const int w = lane + 64 * q;
                    got[q] = 0.0;
                    if (w < W) got[q] = agent_load((const double*)&sl[w]);
                }
#pragma unroll
                for (int q = 0; q < GRID_MAX_WG / 64; ++q) missing |= is_empty(got[q]);
                missing = __any(missing);
            }
            s = 0.0;
#pragma unroll
            for (int q = 0; q < GRID_MAX_WG / 64; ++q) s += got[q];
            s = wave_total(s);
            if (lane == 0) {
                s_tot[wid] = s;
                if (missing) s_bad = 1;
            }
        }
        missing = true;
        for (int i = 0; missing && i < S.polls; ++i) {
            missing = false;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const int j = t + h * GRID_THREADS;
                if (j < n) hq[h] = agent_load(vec + off[j]);
            }
#pragma unroll
            for (int h = 0; h < H; ++h) missing |= t + h * GRID_THREADS < n && is_empty(hq[h]);
        }
        if (missing) s_bad = 1;
        lds_barrier();
        t0 = s_tot[0];
        t1 = s_tot[1];
        ++phase;
        return s_bad == 0;
    };
    // dst[j] <- fn(dst[j], halo component j): the first H of a thread from hq, the others from the phase's vector
    auto take = [&](double* dst, const int32_t* off, int n, auto fn) INLINE {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int j = t + h * GRID_THREADS;
            if (j < n) dst[j] = fn(dst[j], hq[h]);
        }
        const double* vec = S.vec + (int64_t)((phase - 1) & 3u) * S.ndof;
        for (int j = t + H * GRID_THREADS; j < n; j += GRID_THREADS) {
            double q = agent_load(vec + off[j]);
            for (int i = 0; is_empty(q) && i < S.polls; ++i) q = agent_load(vec + off[j]);
            if (is_empty(q)) s_bad = 1;
            dst[j] = fn(dst[j], q);
        }
    };
    const int32_t* haloA = S.halo + g.halo_off;
    const int32_t* haloP = haloA + 3 * g.nhA;
    double* hp = s_p + 3 * g.nown;
    double* hr = s_r + 3 * g.nown;
    int status = GRID_RUNNING;
    bool alive = true;
    double zTr = 0.0, rr = 0.0, zprev = 1.0, bnorm = 0.0;
    int64_t k = 0;
    bool first = !S.resume;  // the preamble: r = b - A x, z = P r, by the loop's own products and exchanges
    {
        const int64_t dof = 3 * (int64_t)g.node0 + t;
        if (first) {
            if (t < 3 * g.nown) s_p[t] = s_x[t];
            for (int j = t; j < 3 * g.nhA; j += GRID_THREADS) hp[j] = S.x[haloA[j]];
        } else {
            const GridState st = *S.state;
            zTr = st.zTr;
            rr = st.rr;
            zprev = st.zprev;
            bnorm = st.bnorm;
            k = st.k;
            // p <- z + beta p is the loop's first update: its halo z by way of hq and, past H, of p itself
            const double beta = k == 0 ? 0.0 : zTr / zprev;
            const double *zs = S.save, *rs = zs + S.ndof, *ps = rs + S.ndof;
            for (int j = t; j < 3 * g.nhA; j += GRID_THREADS) hp[j] = fmav(beta, ps[haloA[j]], zs[haloA[j]]);
            for (int j = t; j < 3 * g.nhP; j += GRID_THREADS) hr[j] = rs[haloP[j]];
            if (t < 3 * g.nown) {
                s_r[t] = rs[dof];
                s_p[t] = ps[dof];
                s_v[t] = zs[dof];
            }
        }
    }
    bool resumed = !first;
    const int64_t k_end = k + S.chunk;
    // What is formed from these (LDS addresses, tests of the mask's bits) is formed where it is used, not kept in
    // registers over the loop, which the blocks fill
    auto opaque = [&]() INLINE {
        asm volatile("" : "+v"(t), "+v"(mask), "+v"(pos), "+s"(sA), "+s"(nS));
#pragma unroll
        for (int s = 0; s < NC; ++s) asm volatile("" : "+v"(cp[s]));
    };
    while (true) {
        opaque();
        const bool own = t < 3 * g.nown;
        if (!first) {
            // the stopping tests on r_k
            if (bnorm == 0.0)
                status = GRID_ZERO_RHS;
            else if (sqrt(rr) <= S.tol * bnorm)
                status = GRID_CONVERGED;
            else if (S.max_iter >= 0 && k >= S.max_iter)
                status = HOEFEM_ERROR_CG_MAX_ITERATIONS;
            if (status != GRID_RUNNING || (k == k_end && !resumed)) break;
            const double beta = k == 0 ? 0.0 : zTr / zprev;
            if (!resumed) take(hp, haloA, 3 * g.nhA, [&](double d, double q) INLINE { return fmav(beta, d, q); });
            if (own) s_p[t] = fmav(beta, s_p[t], s_v[t]);
            resumed = false;
        }
        lds_barrier();
        products(0, sA, s_p, pos & 0xffffu);
        lds_barrier();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the previous phase's stores
        double ap = 0.0, v0 = 0.0, v1 = 0.0, pAp, none;
        if (own) {
            ap = row_sum(s_rows[0][t]);
            v0 = s_p[t] * ap;
            if (first) {
                const double rhs = S.b[3 * (uint32_t)g.node0 + t];
                ap = rhs - ap;
                s_r[t] = ap;
                v0 = rhs * rhs;
            }
            s_v[t] = ap;
        }
        alive = exchange(ap, v0, 0.0, 1, haloP, 3 * g.nhP, pAp, none);
        if (!alive) break;
        if (first) {
            bnorm = sqrt(pAp);
            take(hr, haloP, 3 * g.nhP, [](double, double q) INLINE { return q; });
            for (int j = t; j < 3 * g.nhA; j += GRID_THREADS) hp[j] = 0.0;
            if (own) s_p[t] = 0.0;
        } else {
            if (pAp <= 0.0)
                status = HOEFEM_ERROR_CG_INDEFINITE_OPERATOR;
            else if (zTr <= 0.0)
                status = HOEFEM_ERROR_CG_INDEFINITE_PRECONDITIONER;
            if (status != GRID_RUNNING) break;
            const double alpha = zTr / pAp;
            take(hr, haloP, 3 * g.nhP, [&](double d, double q) INLINE { return fmav(-alpha, q, d); });
            if (own) {
                s_x[t] = fmav(alpha, s_p[t], s_x[t]);
                s_r[t] = fmav(-alpha, s_v[t], s_r[t]);
            }
            zprev = zTr;
            ++k;
        }
        opaque();
        lds_barrier();
        products(sA, nS, s_r, pos >> 16);
        lds_barrier();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        double z = 0.0;
        v0 = v1 = 0.0;
        if (own) {
            const double r = s_r[t];
            const uint32_t rows = s_rows[1][t];
            if (rows != DIAG)
                z = row_sum(rows);
            else
                z = S.dinv ? s_d[t] * r : (double)(VT(s_d[t]) * VT(r));
            s_v[t] = z;
            v0 = z * r;
            v1 = r * r;
        }
        alive = exchange(z, v0, v1, 2, haloA, 3 * g.nhA, zTr, rr);
        if (!alive) break;
        first = false;
    }
    if (!alive) {  // x keeps its last saved value
        if (t == 0) S.host->failed = 1;
        return;
    }
    if (t < 3 * g.nown) {
        const int64_t dof = 3 * (int64_t)g.node0 + t;
        S.x[dof] = status == GRID_ZERO_RHS ? 0.0 : s_x[t];
        if (status == GRID_RUNNING) {
            S.save[dof] = s_v[t];
            S.save[dof + S.ndof] = s_r[t];
            S.save[dof + 2 * S.ndof] = s_p[t];
        }
    }
    if (b == 0 && t == 0) {
        *S.state = GridState{zTr, rr, zprev, bnorm, k};
        S.host->iters = k;
        S.host->phase = phase;
        S.host->status = status;
    }
#undef INLINE
}

// ------------------------------------------------------------------ plan
// W: an exchange with its vector entries takes 2.6 us at 8 work-groups, 2.9 at 80 and 3.9 at 216 to 240 (5.1 where it
// waits for work-groups whose halo is past the entries taken in meanwhile), the two phases' products together 2.0, 2.4 and 3.5 us with
// 4, 7 and 13 blocks per thread, and both grow or shrink with W, so small systems take few work-groups: enough for
// GRID_BLOCKS_PER_THREAD blocks per thread, at least 8. Past GRID_WIDE work-groups the two balance over a wide
// range of W, and a system takes no more than what still keeps its blocks on the chip
// (GRID_BLOCKS_ON_CHIP per thread): alone it is as fast (48 to 74 thousand DOFs: -4 to +2.5 %), and two of a
// batch fit the CUs side by side (eight scenes of 2 to 30 thousand DOFs: 139 -> 100 ms per batch step).
constexpr int GRID_BLOCKS_PER_THREAD = 6, GRID_BLOCKS_ON_CHIP = 12, GRID_WIDE = 128;
constexpr int GRID_MAX_SLOTS = 32;                 // bits of a thread's row-end mask
constexpr size_t GRID_MAX_LDS = 143 * 1024;  // beside 16.3 KiB of fixed arrays
constexpr int GRID_MAX_NODES = GRID_THREADS / 3;   // per work-group
constexpr int64_t GRID_SETUP_BLOCKS = 1 << 16;     // blocks worth a host thread (about 0.3 ms of one)
constexpr int GRID_SPARE = 8;                      // spare partial sums (row_sum)
constexpr int64_t GRID_STATE_WORDS = (sizeof(GridState) + 255) / 256 * 32;

void GridPlan::build(const NodePattern& J, const NodePattern* P, int cus, hipStream_t s) {
    W = 0;
    matrix = J.id;
    const int64_t nn = J.num_nodes;
    if (nn == 0 || cus < 8) return;
    auto ka = [&](int64_t v) { return J.nptr[v + 1] - J.nptr[v]; };
    auto kp = [&](int64_t v) { return !P || P->diag_only[v] ? 0 : P->nptr[v + 1] - P->nptr[v]; };
    std::vector<int64_t> psum(nn + 1, 0);  // P's blocks before each node; A's are J.nptr
    for (int64_t v = 0; v < nn; ++v) psum[v + 1] = psum[v] + kp(v);
    const int64_t total = J.nptr[nn] + psum[nn];
    const int wmax = std::min(cus, GRID_MAX_WG);
    if (nn > (int64_t)wmax * GRID_MAX_NODES || total > (int64_t)wmax * GRID_THREADS * GRID_MAX_SLOTS) return;
    auto share = [&](int64_t blocks) { return (total + GRID_THREADS * blocks - 1) / (GRID_THREADS * blocks); };
    int64_t w = std::max(share(GRID_BLOCKS_ON_CHIP), std::min<int64_t>(share(GRID_BLOCKS_PER_THREAD), GRID_WIDE));
    w = std::max<int64_t>(w, (nn + GRID_MAX_NODES - 1) / GRID_MAX_NODES);
    w = std::min<int64_t>(std::max<int64_t>((w + 7) / 8 * 8, 8), wmax);
    w = std::min(w, nn);
    // Contiguous node ranges: the fewest blocks per thread that w ranges allow, then the evenest ranges (blocks,
    // and a few blocks' worth per node) with that many. Both by filling range after range up to a cap, a range's end
    // by bisection.
    std::vector<int64_t> cut;
    auto fill = [&](int64_t slots, int64_t cap) -> bool {
        cut.assign(1, 0);
        auto fits = [&](int64_t c, int64_t v) {  // the nodes [c, v) in one range
            const int64_t a = J.nptr[v] - J.nptr[c], p = psum[v] - psum[c];
            return a + p + 4 * (v - c) <= cap &&
                   (a + GRID_THREADS - 1) / GRID_THREADS + (p + GRID_THREADS - 1) / GRID_THREADS <= slots;
        };
        if (!fits(0, 1)) return false;
        for (int64_t c = 0; c < nn; c = cut.back()) {
            if ((int64_t)cut.size() > w) return false;
            int64_t lo = c + 1, hi = std::min(nn, c + GRID_MAX_NODES);  // a node by itself is a range in any case
            while (lo < hi) {
                const int64_t mid = (lo + hi + 1) / 2;
                if (fits(c, mid))
                    lo = mid;
                else
                    hi = mid - 1;
            }
            cut.push_back(lo);
        }
        return true;
    };
    int64_t slots = std::max<int64_t>(1, total / (w * GRID_THREADS));
    while (slots <= GRID_MAX_SLOTS && !fill(slots, INT64_MAX)) ++slots;
    if (slots > GRID_MAX_SLOTS) return;
    int64_t lo = (total + 4 * nn) / w, hi = total + 4 * nn;  // hi fits
    while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (fill(slots, mid))
            hi = mid;
        else
            lo = mid + 1;
    }
    fill(slots, hi);
    w = (int64_t)cut.size() - 1;
    std::vector<GridWg> wg(w);
    std::vector<GridStart> start((size_t)2 * w * GRID_THREADS);
    struct Part {  // of one work-group
        std::vector<int32_t> halo;
        std::vector<uint16_t> col, rp;
        int parts = 0;
        bool fits = true;
    };
    std::vector<Part> part(w);
    auto work = [&](int64_t b0, int64_t step) {
        std::vector<int32_t> local(nn, -1), list;
        for (int64_t b = b0; b < w; b += step) {
            GridWg& g = wg[b];
            Part& o = part[b];
            g = GridWg{};
            const int64_t n0 = cut[b], n1 = cut[b + 1];
            g.node0 = (int32_t)n0;
            g.nown = (int32_t)(n1 - n0);
            o.fits = g.nown <= GRID_MAX_NODES;
            for (int ph = 0; ph < 2 && o.fits; ++ph) {
                const NodePattern* pat = ph == 0 ? &J : P;
                auto kk = [&](int64_t v) { return ph == 0 ? ka(v) : kp(v); };
                list.clear();
                int64_t nb = 0;
                for (int64_t v = n0; v < n1; ++v) {
                    const int k = kk(v);
                    const int32_t* nc = k ? pat->ncol.data() + pat->nptr[v] : nullptr;
                    nb += k;
                    for (int j = 0; j < k; ++j) {
                        const int32_t c = nc[j];
                        if (local[c] < 0 && (c < n0 || c >= n1)) {
                            local[c] = 0;
                            list.push_back(c);
                        }
                    }
                }
                std::sort(list.begin(), list.end());
                for (size_t i = 0; i < list.size(); ++i) {
                    local[list[i]] = g.nown + (int32_t)i;
                    for (int c = 0; c < 3; ++c) o.halo.push_back(3 * list[i] + c);
                }
                const int slots = (int)((nb + GRID_THREADS - 1) / GRID_THREADS);
                o.fits = slots <= GRID_MAX_SLOTS && 3 * (g.nown + (int64_t)list.size()) <= 65535;
                int np = 0;  // partial sums so far
                if (o.fits) {
                    const size_t c0 = o.col.size();
                    o.col.resize(c0 + (size_t)slots * GRID_THREADS, 0);
                    int th = 0, sl = 0;  // the block's thread and its place in the thread's run
                    for (int64_t v = n0; v < n1; ++v) {
                        o.rp.push_back((uint16_t)np);
                        const int k = kk(v);
                        const int32_t* nc = k ? pat->ncol.data() + pat->nptr[v] : nullptr;
                        for (int j = 0; j < k; ++j) {
                            if (sl == 0) start[2 * (b * GRID_THREADS + th) + ph] = GridStart{(int32_t)v, j, np, 0};
                            const int32_t c = nc[j];
                            const int32_t l = c >= n0 && c < n1 ? (int32_t)(c - n0) : local[c];
                            o.col[c0 + (size_t)sl * GRID_THREADS + th] = (uint16_t)(3 * l);
                            if (j + 1 == k || sl + 1 == slots) ++np;
                            if (++sl == slots) {
                                sl = 0;
                                ++th;
                            }
                        }
                    }
                    o.rp.push_back((uint16_t)np);
                }
                o.parts = std::max(o.parts, np);
                for (int32_t c : list) local[c] = -1;
                (ph == 0 ? g.nhA : g.nhP) = (int32_t)list.size();
                (ph == 0 ? g.sA : g.sP) = slots;
                (ph == 0 ? g.nbA : g.nbP) = (int32_t)nb;
            }
        }
    };
    // large patterns on a few host threads
    const int nt = thread_count(total, GRID_SETUP_BLOCKS);
    run_on_threads(nt, [&](int i) { work(i, nt); });
    size_t nhalo = 0, ncol = 0, nrp = 0;
    lds_bytes = 0;
    max_slots = 0;
    ws = 0;
    for (int64_t b = 0; b < w; ++b) {
        GridWg& g = wg[b];
        const Part& o = part[b];
        max_slots = std::max(max_slots, g.sA + g.sP);
        if (!o.fits || max_slots > GRID_MAX_SLOTS) return;
        g.halo_off = (int64_t)nhalo;
        g.rp_off = (int64_t)nrp;
        g.col_off = (int64_t)ncol;
        nhalo += o.halo.size();
        nrp += o.rp.size();
        ncol += o.col.size();
        lds_bytes = std::max(lds_bytes, sizeof(double) * (size_t)(3 * (2 * g.nown + g.nhA + g.nhP) + 3 * (o.parts + GRID_SPARE)));
    }
    if (lds_bytes > GRID_MAX_LDS) return;
    // blocks past the registers: in the LDS that is left, then in memory (sized for FP64)
    constexpr size_t SLOT = sizeof(double) * 9 * GRID_THREADS;
    blk_off = (int)((lds_bytes / sizeof(double) + 1) / 2 * 2);
    const int over = std::max(0, max_slots - GRID_REG_F64);
    nlds = (int)std::min<size_t>((size_t)std::min(over, GRID_LDS_SLOTS), (GRID_MAX_LDS - std::min(GRID_MAX_LDS, sizeof(double) * blk_off)) / SLOT);
    lds_bytes = sizeof(double) * blk_off + SLOT * nlds;
    for (GridWg& g : wg) {
        g.ws_off = (int64_t)ws;
        ws += (size_t)std::max(0, g.sA + g.sP - GRID_REG_F64 - nlds) * 9 * GRID_THREADS;
    }
    // one upload of everything (an allocation and a copy each would be half a small model's setup)
    const size_t at_start = wg.size() * sizeof(GridWg), at_halo = at_start + start.size() * sizeof(GridStart);
    const size_t at_col = at_halo + nhalo * sizeof(int32_t), at_rp = at_col + ncol * sizeof(uint16_t);
    const size_t bytes = at_rp + nrp * sizeof(uint16_t);
    std::unique_ptr<char[]> all(new char[bytes]);
    std::memcpy(all.get(), wg.data(), at_start);
    std::memcpy(all.get() + at_start, start.data(), at_halo - at_start);
    for (int64_t b = 0; b < w; ++b) {
        const Part& o = part[b];
        std::copy(o.halo.begin(), o.halo.end(), reinterpret_cast<int32_t*>(all.get() + at_halo) + wg[b].halo_off);
        std::copy(o.col.begin(), o.col.end(), reinterpret_cast<uint16_t*>(all.get() + at_col) + wg[b].col_off);
        std::copy(o.rp.begin(), o.rp.end(), reinterpret_cast<uint16_t*>(all.get() + at_rp) + wg[b].rp_off);
    }
    d_all.upload(all.get(), bytes, s);
    d_wg = reinterpret_cast<const GridWg*>(d_all.get());
    d_start = reinterpret_cast<const GridStart*>(d_all.get() + at_start);
    d_halo = reinterpret_cast<const int32_t*>(d_all.get() + at_halo);
    d_col = reinterpret_cast<const uint16_t*>(d_all.get() + at_col);
    d_rp = reinterpret_cast<const uint16_t*>(d_all.get() + at_rp);
    ndof = 3 * nn;
    W = (int)w;
    if (exchange() + saved() + GRID_STATE_WORDS + (int64_t)ws > GRID_SCRATCH) d_spill.ensure(ws);
}

int64_t GridPlan::exchange() const { return (int64_t)8 * GRID_COPIES * W + 4 * ndof; }

void GridWork::ensure(const GridPlan& g) {
    if (W_ != g.W || ndof_ != g.ndof) {
        d_slots_.ensure((size_t)g.exchange());
        d_save_.ensure((size_t)g.saved());
        W_ = g.W;
        ndof_ = g.ndof;
        cleared = false;
    }
    d_ws_.ensure(g.ws);
    d_state_.ensure(1);
    if (!host_) host_.reset(new PinnedBuf<GridResult>(1, hipHostMallocCoherent));
    slots = d_slots_.get();
    save = d_save_.get();
    ws = d_ws_.get();
    state = d_state_.get();
    result = host_->p;
}

GridBuffers grid_scratch_buffers(const GridPlan& g, double* scratch, GridResult* result) {
    GridBuffers w;
    w.slots = reinterpret_cast<unsigned long long*>(scratch);
    w.save = scratch + g.exchange();
    w.state = reinterpret_cast<GridState*>(w.save + g.saved());
    w.ws = g.d_spill.n ? g.d_spill.get() : w.save + g.saved() + GRID_STATE_WORDS;
    w.result = result;
    return w;
}

__global__ void k_grid_clear(int64_t n, unsigned long long* __restrict__ p) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = GRID_EMPTY;
}

void grid_clear(const GridPlan& g, GridBuffers& w, hipStream_t s) {
    if (w.cleared) return;
    const int64_t n = g.exchange();
    k_grid_clear<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(n, w.slots);
    check_launch("k_grid_clear");
    w.phase = 0;
    w.cleared = true;
}

// ------------------------------------------------------------------ admission
// A launch is admitted when its work-groups (one per CU at most) fit beside those of the process's launches in
// flight on the device, so admitted grids are all resident and make progress.
namespace {
CuLine& device_line() {
    static std::mutex mu;
    static std::map<int, CuLine> lines;
    int d = 0;
    HIP_CHECK(hipGetDevice(&d));
    std::lock_guard<std::mutex> lock(mu);
    auto it = lines.find(d);
    if (it == lines.end()) {
        int n = 0;
        HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, d));
        it = lines.try_emplace(d, n / CuLine::XCDS * CuLine::XCDS).first;
    }
    return it->second;
}
}  // namespace

int grid_device_cus() { return device_line().cus(); }

bool GridSlots::acquire(int wgs, bool wait) {
    const int n = CuLine::charge(wgs);
    if (!place_) {
        release();
        line_ = &device_line();
        if (n > line_->cus()) return false;
        place_ = line_->enter();
    }
    if (!line_->take(place_, n, wait)) return false;
    place_ = 0;
    n_ = n;
    return true;
}

bool GridSlots::grow(int wgs) {
    const int n = CuLine::charge(wgs);
    if (n > n_ && !line_->take_more(n - n_)) return false;
    n_ = n;
    return true;
}

void GridSlots::release() {
    if (place_) line_->leave(place_);
    if (n_) line_->give(n_);
    place_ = 0;
    n_ = 0;
}

// ------------------------------------------------------------------ launches
template <class VT>
GridSeg<VT> grid_segment(const GridPlan& g, const GridBuffers& w, Model& m, const VT* A, const Schwarz* P,
                         const double* dinv, const double* b, double* x, double tol, int64_t max_iter) {
    GridSeg<VT> S{};
    S.wg = g.d_wg;
    S.halo = g.d_halo;
    S.col = g.d_col;
    S.rp = g.d_rp;
    S.start = g.d_start;
    S.jnptr = m.pattern.d_nptr.get();
    S.jrowptr = m.pattern.d_rowptr.get();
    S.A = A;
    if (P) {
        S.pnptr = P->P.d_nptr.get();
        S.prowptr = P->P.d_rowptr.get();
        S.pdiag = P->P.d_diag_only.get();
        if constexpr (sizeof(VT) == sizeof(double))
            S.P = P->d_vals.get();
        else
            S.P = P->d_vals32.get();
    } else {
        S.dinv = dinv;
    }
    S.b = b;
    S.x = x;
    S.vec = reinterpret_cast<double*>(w.slots + (size_t)8 * GRID_COPIES * g.W);
    S.save = w.save;
    S.ndof = g.ndof;
    S.ws = reinterpret_cast<VT*>(w.ws);
    S.slots = w.slots;
    S.state = w.state;
    S.host = w.result;
    S.W = g.W;
    S.phase = w.phase;
    S.polls = m.grid_polls < 0 ? GRID_POLL_LIMIT : m.grid_polls;
    S.nlds = g.nlds;
    S.blk_off = g.blk_off;
    S.tol = tol;
    S.max_iter = max_iter;
    return S;
}
template GridSeg<double> grid_segment<double>(const GridPlan&, const GridBuffers&, Model&, const double*, const Schwarz*, const double*,
                                              const double*, double*, double, int64_t);
template GridSeg<float> grid_segment<float>(const GridPlan&, const GridBuffers&, Model&, const float*, const Schwarz*, const double*,
                                            const double*, double*, double, int64_t);

template <class VT>
constexpr int grid_reg() {
    return sizeof(VT) == sizeof(double) ? GRID_REG_F64 : GRID_REG_F32;
}

template <class VT, int K>
void grid_launch(const GridSegs<VT, K>& all, int wgs, size_t lds, hipStream_t s) {
    auto* k = &k_grid_pcg<VT, grid_reg<VT>(), K>;
    raise_lds_limit((const void*)k, lds);
    k<<<dim3((unsigned)wgs), dim3(GRID_THREADS), lds, s>>>(all);
    check_launch("k_grid_pcg");
}
template void grid_launch<double, GRID_SEGS>(const GridSegs<double, GRID_SEGS>&, int, size_t, hipStream_t);
template void grid_launch<float, GRID_SEGS>(const GridSegs<float, GRID_SEGS>&, int, size_t, hipStream_t);

template <class VT>
bool grid_solve(const GridPlan& g, GridBuffers& w, GridRest& rest, Model& m, const VT* A, const Schwarz* P,
                const double* dinv, const double* b, double* x, double tol, int64_t max_iter, int64_t* iterations,
                hoefem_status* status) {
    if (rest.resting()) {
        rest.pass();
        return false;
    }
    GridSegs<VT, 1> all;
    GridSeg<VT>& S = all.seg[0];
    grid_clear(g, w, m.stream);
    S = grid_segment<VT>(g, w, m, A, P, dinv, b, x, tol, max_iter);
    S.chunk = GRID_CHUNK;
    while (true) {
        volatile GridResult* h = w.result;
        h->status = GRID_RUNNING;
        h->failed = 0;
        {
            GridSlots slots;
            if (!slots.acquire(g.W, true)) return false;
            grid_launch(all, g.W, g.lds_bytes, m.stream);
            HIP_CHECK(hipStreamSynchronize(m.stream));
        }
        if (h->failed) {
            w.cleared = false;
            rest.ended(false);
            m.grid_failures += 1;
            return false;
        }
        w.phase = S.phase = h->phase;
        *iterations = h->iters;
        if (h->status != GRID_RUNNING) break;
        S.resume = 1;
    }
    rest.ended(true);
    m.grid_solves += 1;
    const int st = w.result->status;
    *status = st == GRID_CONVERGED || st == GRID_ZERO_RHS ? HOEFEM_OK : (hoefem_status)st;
    return true;
}
template bool grid_solve<double>(const GridPlan&, GridBuffers&, GridRest&, Model&, const double*, const Schwarz*,
                                 const double*, const double*, double*, double, int64_t, int64_t*, hoefem_status*);
template bool grid_solve<float>(const GridPlan&, GridBuffers&, GridRest&, Model&, const float*, const Schwarz*,
                                const double*, const double*, double*, double, int64_t, int64_t*, hoefem_status*);

// ------------------------------------------------------------------ many systems
GridBatch::~GridBatch() {
    for (Lane& l : lanes) {
        if (l.s) (void)hipStreamSynchronize(l.s);
        if (l.done) (void)hipEventDestroy(l.done);
        if (l.s) (void)hipStreamDestroy(l.s);
    }
}

namespace {
// The resident-grid solves of a batch. Waiting systems are launched together, in the order they came, as far
// as their work-groups fit the free CUs, for GRID_BATCH_CHUNK iterations (so that CUs of systems that end
// soon come free); launches go to a few lanes (streams), so systems that come later run beside the earlier
// ones. A system that is not done goes on in a later launch; its arithmetic does not depend on where its launches
// are cut, so x, iteration count and status equal a solve by itself bit for bit.
template <class VT>
struct GridPoolT final : CgPool {
    struct Item {
        CgBatchSystem q;
        const GridPlan* g;
        GridWork* w;
        GridSeg<VT> seg;
    };
    GridBatch& B;
    std::vector<Item> items;
    std::vector<int> waiting;
    GridSlots slots[GRID_LANES];
    std::vector<int> running[GRID_LANES];

    explicit GridPoolT(GridBatch& b) : B(b) {
        for (GridBatch::Lane& l : B.lanes)
            if (!l.s) {
                HIP_CHECK(hipStreamCreateWithFlags(&l.s, hipStreamNonBlocking));
                HIP_CHECK(hipEventCreateWithFlags(&l.done, hipEventDisableTiming));
            }
    }
    ~GridPoolT() override {
        for (int l = 0; l < GRID_LANES; ++l)
            if (!running[l].empty()) (void)hipStreamSynchronize(B.lanes[l].s);
    }
    int join(const CgBatchSystem& q) override {
        Item it{q, q.P ? &q.P->grid : &q.m->grid, &q.w->grid, {}};
        it.w->ensure(*it.g);
        it.q.iterations = 0;
        it.q.status = HOEFEM_OK;
        it.seg = grid_segment<VT>(*it.g, *it.w, *q.m, (const VT*)q.A, q.P, q.P ? nullptr : q.w->diag_inv.get(), q.b, q.x,
                                  q.tol, q.max_iter);
        it.seg.chunk = GRID_BATCH_CHUNK;
        items.push_back(it);
        waiting.push_back((int)items.size() - 1);
        return (int)items.size() - 1;
    }
    const CgBatchSystem& system(int id) const override { return items[id].q; }
    bool idle() const override {
        for (const auto& r : running)
            if (!r.empty()) return false;
        return waiting.empty();
    }
    void ended_launch(int lane, std::vector<int>& ended) {
        slots[lane].release();
        std::vector<int> again;
        for (int id : running[lane]) {
            Item& it = items[id];
            volatile GridResult* h = it.w->result;
            if (h->failed) {  // solved from the start by the two kernels
                it.w->cleared = false;
                it.w->rest.ended(false);
                it.q.m->grid_failures += 1;
                HIP_CHECK(hipMemsetAsync(it.q.x, 0, sizeof(double) * it.g->ndof, it.q.m->stream));
                it.q.status = pcg_solve(*it.q.m, *it.q.w, (const VT*)it.q.A, it.q.P, it.q.b, it.q.x, it.q.tol,
                                        it.q.max_iter, &it.q.iterations, true);
                HIP_CHECK(hipStreamSynchronize(it.q.m->stream));
                ended.push_back(id);
                continue;
            }
            it.w->phase = h->phase;
            if (h->status == GRID_RUNNING) {
                it.seg.resume = 1;
                again.push_back(id);
                continue;
            }
            it.w->rest.ended(true);
            it.q.m->grid_solves += 1;
            it.q.iterations = h->iters;
            it.q.status = h->status == GRID_CONVERGED || h->status == GRID_ZERO_RHS ? HOEFEM_OK : (hoefem_status)h->status;
            ended.push_back(id);
        }
        running[lane].clear();
        waiting.insert(waiting.begin(), again.begin(), again.end());
    }
    void progress(std::vector<int>& ended) override {
        for (int l = 0; l < GRID_LANES; ++l)
            if (!running[l].empty()) {
                const hipError_t e = hipEventQuery(B.lanes[l].done);
                if (e == hipErrorNotReady) continue;
                HIP_CHECK(e);
                ended_launch(l, ended);
            }
        while (!waiting.empty()) {
            int l = -1;  // an idle lane, the one with a place in the line first
            for (int i = 0; i < GRID_LANES; ++i)
                if (running[i].empty() && (l < 0 || slots[i].waiting())) l = i;
            if (l < 0) break;
            // as many waiting systems as fit, at least the first
            int wgs = items[waiting[0]].g->W, n = 1;
            if (!slots[l].acquire(wgs, false)) break;
            while (n < (int)waiting.size() && n < GRID_SEGS && slots[l].grow(wgs + items[waiting[n]].g->W))
                wgs += items[waiting[n++]].g->W;
            GridSegs<VT, GRID_SEGS> all{};
            size_t lds = 0;
            const hipStream_t s = B.lanes[l].s;
            for (int k = 0; k < n; ++k) {
                Item& it = items[waiting[k]];
                volatile GridResult* h = it.w->result;
                h->status = GRID_RUNNING;
                h->failed = 0;
                if (!it.seg.resume) HIP_CHECK(hipMemsetAsync(it.q.x, 0, sizeof(double) * it.g->ndof, s));
                grid_clear(*it.g, *it.w, s);
                it.seg.phase = it.w->phase;
                all.seg[k] = it.seg;
                lds = std::max(lds, it.g->lds_bytes);
                running[l].push_back(waiting[k]);
            }
            waiting.erase(waiting.begin(), waiting.begin() + n);
            grid_launch(all, wgs, lds, s);
            HIP_CHECK(hipEventRecord(B.lanes[l].done, s));
        }
    }
};
}  // namespace

std::unique_ptr<CgPool> make_grid_pool(GridBatch& B, bool fp32) {
    if (fp32) return std::unique_ptr<CgPool>(new GridPoolT<float>(B));
    return std::unique_ptr<CgPool>(new GridPoolT<double>(B));
}

}  // namespace hoefem
