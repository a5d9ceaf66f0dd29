// The resident-grid PCG (grid_pcg.hip): plan of a system, its launch descriptor and entry points.
#pragma once

#include "cu_line.hpp"
#include "internal.hpp"

namespace hoefem {

constexpr int GRID_THREADS = 512;
constexpr int GRID_MAX_WG = 256;
constexpr int GRID_REG_F64 = 10, GRID_REG_F32 = 16;  // blocks of a thread held in registers,
constexpr int GRID_LDS_SLOTS = 4;                    // and at most so many more in LDS
constexpr int GRID_CHUNK = 1024;   // iterations per launch of a single solve
constexpr int GRID_BATCH_CHUNK = 128;
enum : int { GRID_RUNNING = 0, GRID_CONVERGED = 100, GRID_ZERO_RHS = 101 };

// one launch's descriptor of a system
template <class VT>
struct GridSeg {
    const GridWg* wg;
    const int32_t* halo;
    const uint16_t *col, *rp;
    const GridStart* start;
    const int32_t *jnptr, *jrowptr, *pnptr, *prowptr;
    const uint8_t* pdiag;
    const VT *A, *P;
    const double* dinv;  // Jacobi: the reciprocal diagonal (no P)
    const double* b;
    double* x;
    double* vec;      // four sets of exchanged vectors (z, Ap and the first residual)
    double* save;     // z, r and p between launches
    int64_t ndof;
    VT* ws;
    unsigned long long* slots;
    GridState* state;
    GridResult* host;
    int W;            // work-groups
    uint32_t phase;   // exchanges done so far (the sets in use)
    int resume;
    int polls;        // of a value before the launch is given up
    int nlds, blk_off;  // blocks of a thread in LDS, and their offset there (doubles)
    int64_t chunk, max_iter;
    double tol;
};

constexpr int GRID_SEGS = 16;  // systems of one launch (their descriptors fit the 4 KiB of kernel arguments)
template <class VT, int K>
struct GridSegs {
    GridSeg<VT> seg[K];
};
static_assert(sizeof(GridSegs<double, GRID_SEGS>) <= 4096, "kernel arguments");

// CUs held for a launch of resident grids on the current device
class GridSlots {
public:
    GridSlots() = default;
    GridSlots(const GridSlots&) = delete;
    GridSlots& operator=(const GridSlots&) = delete;
    ~GridSlots() { release(); }
    // false: not yet its turn, its place in the line kept (wait: the device never has so many)
    bool acquire(int wgs, bool wait);
    bool grow(int wgs);  // to wgs in all; false: not free, or others wait
    bool waiting() const { return place_ != 0; }
    void release();

private:
    CuLine* line_ = nullptr;
    uint64_t place_ = 0;
    int n_ = 0;
};

template <class VT>
GridSeg<VT> grid_segment(const GridPlan& g, const GridBuffers& w, Model& m, const VT* A, const Schwarz* P,
                         const double* dinv, const double* b, double* x, double tol, int64_t max_iter);
// One launch; the systems' buffers must be clear (grid_clear) before it on the same stream
template <class VT, int K>
void grid_launch(const GridSegs<VT, K>& all, int wgs, size_t lds, hipStream_t s);
void grid_clear(const GridPlan& g, GridBuffers& w, hipStream_t s);
// Solves A x = b on the model stream; false: the grid rests (rest) or could not run (x is a valid guess for
// another solver)
template <class VT>
bool grid_solve(const GridPlan& g, GridBuffers& w, GridRest& rest, Model& m, const VT* A, const Schwarz* P, const double* dinv,
                const double* b, double* x, double tol, int64_t max_iter, int64_t* iterations, hoefem_status* status);

// Buffers of allocation-free solves in a scratch of GRID_SCRATCH doubles
constexpr int64_t GRID_SCRATCH = 8 * 262144;
GridBuffers grid_scratch_buffers(const GridPlan& g, double* scratch, GridResult* result);

}  // namespace hoefem
