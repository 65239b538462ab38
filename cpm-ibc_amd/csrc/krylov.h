// Launch interface of the batched BiCGStab kernels (krylov.hip).
#pragma once
#include "engine.h"

namespace cpmgpu {

// The segments of a fused kernel: the table and a block map, or the only
// segment by value.
template <typename T>
struct SegArg {
    const Seg<T>* segs;
    const int* bseg;
    Seg<T> one;
};

// The kernel of a launch's E gathers: every operator by shared-stencil tiles,
// every operator in the ELL format, some by tiles and the others by rows, or
// none by tiles (none built, or values too wide for their LDS).
enum GatherKind : int { GATHER_TILES, GATHER_ELL, GATHER_MIXED, GATHER_ROWS };

template <typename T>
struct LaunchCfg {
    const Seg<T>* segs;    // device segment table
    const Seg<T>* first;   // its first entry on the host
    const int* bseg;       // device block maps (segment | block << kSegBits), nblocks entries segment by
                           // segment, gblocks round-robin over the segments (the E gathers'), gblocks
                           // segment by segment (the refinement lanes' gathers'); not read where nseg = 1
    int nblocks;
    int gblocks;           // workgroups of an E gather
    GatherKind gather;     // decided once, where gblocks and the block maps are laid out for it: a choice
                           // made again at a launch could meet a grid that was laid out for another kernel
    int nseg;
    hipStream_t stream;
    int jacobi_sweeps;     // largest precond_iters over Jacobi-preconditioned segments (0: none)
    bool fold = false;     // the finalisers run inside the kernels that need them (Seg::sst set)
    bool fuse = false;     // ... and pupdate and supdate inside the gathers and lfinish, where those allow it
    bool fly = false;      // iterations form P^-1 where it is read (precond_fly; every gather by tiles)
};

// Whether the E gathers of an operator with ntiles shared-stencil tiles use
// them: there are some, the values' rows fit the tiles' LDS, and the
// environment does not say CPMGPU_GROUP_GATHER=none.
template <typename T, int NR>
bool grp_gather(int ntiles);
// Whether iterations that gather by tiles form y = P^-1 p and z = P^-1 s where
// they are read (CPMGPU_PRECOND_FLY=0 stores them instead).
bool precond_fly();

// Workspace vectors of one precision; every vector spans all segments
// (segment g occupies [off_g, off_g + D_g * NR)).
template <typename T>
struct Vecs {
    T *b, *x, *r, *r0, *p, *v, *s, *t, *y, *z, *tmp;
};

// FP64 vectors of a mixed-precision solve (same element layout as the FP32
// workspace), used by the FP32 iteration kernels for refinement steps.
struct MixVec {
    double* x64;          // solution
    double* r64;          // true residual b - A64 x64
    const double* b64;    // right-hand sides
    double* tmp64;        // E64 x64
};

template <typename T, int NR>
struct Launch {
    static void init(const LaunchCfg<T>& c, const T* b, T* x, T* r, T* r0, T* p, T* v);
    // n iterations; mixed: FP32 recurrence whose lanes take FP64 refinement steps in place
    // (mv holds the FP64 vectors); otherwise the reference's FP64 loop
    static void iterations(const LaunchCfg<T>& c, Vecs<T>& w, bool mixed, const MixVec& mv, int n);
    template <bool FOLD>
    static void iteration(const LaunchCfg<T>& c, Vecs<T>& w, bool mixed, const MixVec& mv, bool first);
    static void restart(const LaunchCfg<T>& c, Vecs<T>& w);
    // y = A x; lanes = status mask restricting the work to instances with such a lane (0: all)
    static void apply(const LaunchCfg<T>& c, const T* x, T* tmp, T* y, unsigned lanes = 0);
};

// Start of a mixed-precision solve: x64 = 0, r64 = b, then the FP32 vectors
// from the scaled residual (the segments of both precisions share one state
// array).
template <int NR>
struct MixedLaunch {
    static void start(const LaunchCfg<double>& c, const double* b, double* x64, double* r64);
    static void down(const LaunchCfg<double>& c, const double* r64, Vecs<float>& w);
};

// out = m x + n (L_ii x + L_off tmp) alone (the tail of an apply).
template <typename T>
void launch_lfinish_plain(const LaunchCfg<T>& c, const T* x, const T* tmp, T* out);

// Operators with shared-stencil tiles on callers' vectors (perm: the
// operator's row -> the caller's): y = A x (tmp: D doubles); y = E x
// (identity rows copy); an explicit step u <- E (u + coef Lfull u), identity
// rows <- g, of one field (heat) or of two with the Gray-Scott reaction (z:
// NR D doubles).  sg: the operator's segment, only D, op, m, n and nblocks
// are read.
void launch_apply_caller(const Seg<double>& sg, const int* perm, const double* x, double* tmp, double* y, hipStream_t st);
void launch_extend_caller(const Seg<double>& sg, const int* perm, const double* x, double* y, hipStream_t st);
struct HeldRows {   // Lfull rows of identity rows (Op::hrow ..)
    int64_t nh;
    int hw;
    const int *row, *col;
    const double* val;
};
template <int NR>
void launch_step_caller(const Seg<double>& sg, const HeldRows& h, const int* perm, double* const* u, const double* const* g,
                        const double* coef, double dt, double F, double k, double* z, hipStream_t st);

// E-gather alone (identity rows copy), for measurement; fly: of P^-1 x, as
// the iterations gather (where the launch uses shared-stencil tiles).
template <typename T, int NR>
void launch_egather(const LaunchCfg<T>& c, const T* x, T* out, bool fly = false);

// State reset before a (re)started solve: status, tolerance^2, iteration cap.
void launch_reset_states(KState* st, int n, double tol2, int max_it, double delta2, hipStream_t s);

}  // namespace cpmgpu
