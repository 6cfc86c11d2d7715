// Host-side launch interface of the explicit-path kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "bx_internal.h"
#include "bx_mail.h"
#include "bx_physics.h"

namespace bx {

// A run to a stop time launches steps before it knows that the last one is
// not the final one.  The step that reaches the stop time writes its number to
// *last, and every kernel of a later step ends at once.
struct StepGate
{
    long long *last = nullptr; // null: never
    long long  step = 0;       // the step (from 1) this launch belongs to
    __device__ __forceinline__ bool closed() const { return last && *last < step; }
};

// The time loop's state, advanced by the sweeps themselves.  A step's first
// sweep forms its dt from the wave speed that the step before has reduced
// (every block for itself; block 0 stores it for the step's other sweeps), its
// last one adds the dt to the time.  What a launch reads no block of the same
// launch writes: the speeds go round MAX_SLOTS accumulators (a step reads slot
// n, reduces into n + 1 and clears n + 2, mod MAX_SLOTS), the time round two.
constexpr int MAX_SLOTS = 4, MAX_SLOT_WORDS = 16; // a 128-byte line each
struct StepCtl
{
    const unsigned long long *max_in    = nullptr; // first sweep: the speed (null: dt is read)
    unsigned long long       *max_clear = nullptr;
    double                   *dt        = nullptr;
    const double             *time_in   = nullptr;
    double                   *time_out  = nullptr; // last sweep: the new time
    double                    dx[3]     = { 0, 0, 0 };
    double                    cfl       = 0;
    double                    stop_time = -1;
    StepGate                  gate;
    Mail                     *mail = nullptr; // with gate.last: the new time, message seq
    unsigned long long        seq  = 0;
};

// x sweep: an item is B consecutive positions of a box plane (B = block
// size, at most X_LDS_STRIDE), of which B - 4 are updated; the block
// exchanges neighbour values through three LDS buffers (U, high-side half
// state, face flux) of NC rows of X_LDS_STRIDE doubles, allocated
// dynamically.  The compile-time row stride keeps every LDS address an
// immediate offset from the thread's own.
constexpr int X_LDS_STRIDE = 256;
constexpr int x_item_step(int B) { return B - 4; }
constexpr int x_lds_bytes(int NC) { return 3 * NC * X_LDS_STRIDE * 8; }
// most consecutive x-sweep items a block takes before the next block's turn
// (a power of two; x_chunk_shift() takes fewer where the level has few items)
constexpr int X_CHUNK = 8;

// log2 of the chunk length for a grid of that many blocks: the longest chunk
// that still leaves every block 8 turns, so that the blocks' item counts
// differ by at most 1/8.  Chunks save the box lookup of all but their first
// item, which a level with many items per block wants (4096^2: 68 items per
// block, chunks of 8); with few, a chunk idles the other CUs: 256^2 in
// chunks of 8 occupied 35 of 256 CUs and took 25.7 us, single items 8.0 us.
inline int x_chunk_shift(long long nitems, int grid)
{
    int sh = 0;
    while ((2 << sh) <= X_CHUNK && (nitems >> (sh + 1)) >= 8LL * grid)
        ++sh;
    return sh;
}

struct SweepLaunch
{
    const double       *Uin;
    double             *Uout;
    const DevBox       *boxes;
    const long long    *item_begin;
    const int          *xbox = nullptr; // x sweep: box of each chunk's first item
    int                 xsh  = 0;       // x sweep: log2 of the chunk length
    int                 nbox;
    long long           nitems;
    int                 ng;
    int                 K; // cells per lane segment (y/z sweeps)
    const double       *d_dt;
    double              dx;
    EulerParm           pm;
    LimTable            lt;
    unsigned long long *d_maxbits; // nullable: fused CFL reduction target
    StepCtl             ctl;
    PushList            push; // the ghost cells of the next direction's sweep
    int                 grid;
    int                 block;
    hipStream_t         stream;
};

// scheme: SCH_* (bx_physics.h), the BX_METHOD_* code
hipError_t  launch_sweep(int D, int dir, int scheme, int lim, int lv,
                         const SweepLaunch &L);
const void *sweep_kernel_ptr(int D, int dir);
// per-dimension instantiations (bx_explicit.hip, bx_sweep2d.hip, bx_sweep3d.hip)
hipError_t  launch_sweep_d1(int dir, int scheme, int lim, int lv, const SweepLaunch &L);
hipError_t  launch_sweep_d2(int dir, int scheme, int lim, int lv, const SweepLaunch &L);
hipError_t  launch_sweep_d3(int dir, int scheme, int lim, int lv, const SweepLaunch &L);
const void *sweep_kernel_ptr_d1(int dir);
const void *sweep_kernel_ptr_d2(int dir);
const void *sweep_kernel_ptr_d3(int dir);

hipError_t launch_fill_ghosts(int D, double *U, const GhostSeg *segs, int nseg, int grid,
                              const StepGate &gate, hipStream_t stream);

hipError_t launch_max_wave_speed(int D, const double *U, const DevBox *boxes,
                                 const long long *cbeg, int nbox,
                                 long long ncells, int ng, EulerParm pm,
                                 unsigned long long *d_maxbits, int grid, int chunk,
                                 hipStream_t stream);

hipError_t launch_compute_dt(unsigned long long *d_maxbits, double *d_dt,
                             const double *d_time, int D, const double dx[3],
                             double cfl, double stop_time, hipStream_t stream);

// the state of a time loop before its first step: the time, no last step, every
// speed accumulator zero
hipError_t launch_run_init(unsigned long long *d_maxbits, double *d_time, double time,
                           long long *d_last, hipStream_t stream);

hipError_t launch_set_u64(unsigned long long *p, unsigned long long v,
                          hipStream_t stream);

} // namespace bx
