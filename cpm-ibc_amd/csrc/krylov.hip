// Batched BiCGStab for the closest-point screened-Poisson operator.
//
// Restates the reference's right-preconditioned BiCGStab (src/BiCGStab.h:30-108)
// and its matrix-free operator (src/GeneralizedBiCGStabSystem.h:191-261) as
// bandwidth-bound kernels; one iteration is (B = BiCGStab.h,
// G = GeneralizedBiCGStabSystem.h)
//
//   pupdate   p = (p - w v) beta + r ; y = P^-1 p                 (B:73-77)
//   egather   tmp = E y          (identity rows copy)              (G:235-261)
//   lfinish   v = m y + n (Ld y + Loff tmp) ; partial (r0, v)       (G:93-115,166-189; B:78)
//   fin       alpha = rho / (r0, v)                                (B:79)
//   supdate   s = r - alpha v ; z = P^-1 s                         (B:81-83)
//   egather   tmp = E z
//   lfinish   t = m z + n (Ld z + Loff tmp) ; partials (t,t),(t,s)  (B:84-86)
//   fin       omega = (t, s) / (t, t)                              (B:87-94)
//   xrupdate  x += alpha y ; x += w z ; r = s - w t ; (r,r),(r0,r)  (B:96-98)
//   fin       loop test (B:59), rho (B:61), restart test (B:62), beta (B:73)
//
// Reductions: every workgroup writes its partial sums; a one-workgroup-per-
// instance "fin" kernel adds them in a fixed order and runs the scalar part
// of the recurrence on the device, so iterations need no host round trip and
// results are reproducible run to run.  Where a segment has few row blocks
// the fins are folded: every workgroup of the kernel that needs the scalars
// sums the partials itself, in the same order (fold_states), and workgroup 0
// of the segment writes the new states; one right-hand side's iterations then
// run as five kernels (k_fgather with pupdate or supdate formed where x is
// read, k_flfinish, k_fxrupdate).  (No device-scope fences: on the
// multi-XCD MI355X a release/acquire at agent scope writes back / invalidates
// L2 and costs more than the whole kernel.)
//
// One launch covers every instance of a batch: workgroups map to (instance,
// row block) through a segment table; finished instances are skipped.
// Right-hand sides of one operator are interleaved [row][rhs] so one read of
// an E slot serves all of them.  Each rhs lane has its own state; a kernel
// acts on the lanes whose status is in its mask.
//
// Precision CPM_FP32_REFINE: iterative refinement with FP32 BiCGStab inner
// solves, run as one continuous device-side recurrence.  The solution is
// accumulated in FP64; when the FP32 recurrence residual has dropped by
// delta (default 1e-2) since the last step, or meets the tolerance, or hits
// the rho-restart rule, the lane takes a refinement step inside the next
// iteration's kernels (no extra launches):
//
//   pupdate   x64 += x32 / scale ; x32 = 0
//   egather_upd  tmp64 = E64 x64   (a launch of its own after the FP32 gather)
//   lfinish   r64 = b - A64 x64 ; partial (r64, r64)
//   fin       converged on the true residual?  else scale = 1 / ||r64||
//   supdate   r32 = r64 scale ; r0 = r32 ; p = v = 0
//   lfinish   partial (r32, r32)
//   fin       rho = r0sq = (r32, r32) ; the lane rejoins the next iteration
//
// The FP64 vectors (x64, r64, b, tmp64) are lane-major within a segment,
// the FP32 ones interleave the lanes per row.
//
// (Keeping p across steps, as in reliable-update schemes for one operator,
// diverges here once the residual approaches the FP32 operator's own
// rounding: the FP32 and FP64 operators differ in the last bits.)
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "engine.h"
#include "krylov.h"

namespace cpmgpu {

// ---------------------------------------------------------------- helpers
template <typename T, int NR> struct VT { typedef T __attribute__((ext_vector_type(NR))) type; };
template <typename T> struct VT<T, 1> { typedef T type; };

// Every array lives in global memory, but pointers taken from the segment
// table reach the compiler as generic pointers and would be accessed with
// flat instructions; these helpers address them as global memory.
#define CPM_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T ldg(const T* p) {
    return *(const CPM_GLOBAL T*)p;
}
template <typename T>
__device__ __forceinline__ void stg(T* p, const T& v) {
    *(CPM_GLOBAL T*)p = v;
}
template <typename T, int NR>
__device__ __forceinline__ typename VT<T, NR>::type vload(const T* p) {
    return ldg(reinterpret_cast<const typename VT<T, NR>::type*>(p));
}
template <typename T, int NR>
__device__ __forceinline__ void vstore(T* p, const typename VT<T, NR>::type& v) {
    stg(reinterpret_cast<typename VT<T, NR>::type*>(p), v);
}
template <typename V> __device__ __forceinline__ auto lane(const V& v, int k) { return v[k]; }
__device__ __forceinline__ double lane(double v, int) { return v; }
__device__ __forceinline__ float lane(float v, int) { return v; }
template <typename V, typename S> __device__ __forceinline__ void setlane(V& v, int k, S s) { v[k] = s; }
__device__ __forceinline__ void setlane(double& v, int, double s) { v = s; }
__device__ __forceinline__ void setlane(float& v, int, float s) { v = s; }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Workgroup sums of NV*NR per-thread values.  Partials are stored
// component-major, part[c * nblocks + lb], so that the finaliser reads each
// component with coalesced loads.
// Wave sums of C = 2^L values per lane by a butterfly reduce-scatter: at step
// s (lane offset 32 >> s) a lane keeps the half of its values that its bit of
// the offset selects, summed with its partner's, so after L steps lane l holds
// component (l >> (6 - L)) & (C - 1) summed over 2^L lanes; the last 6 - L
// steps sum those groups.  2 (C - 1) + 6 - L exchanges instead of 6 C.
// Returns the lane's component total.
template <int C>
__device__ __forceinline__ double wave_reduce_scatter(double (&v)[C], int lanei, int& comp) {
    constexpr int L = C == 1 ? 0 : C == 2 ? 1 : C == 4 ? 2 : C == 8 ? 3 : 4;
    static_assert((1 << L) == C, "component count must be 1, 2, 4, 8 or 16");
#pragma unroll
    for (int st = 0; st < L; ++st) {
        const int o = 32 >> st, m = C >> st, h = m >> 1;
        const bool up = (lanei & o) != 0;
#pragma unroll
        for (int j = 0; j < h; ++j) {
            // both halves cross over and the lane selects its sum: a select
            // between two array elements would be folded into a dynamically
            // indexed load, and the array moved to LDS
            const double lo = v[j] + __shfl_xor(v[j], o, 64);
            const double hi = v[j + h] + __shfl_xor(v[j + h], o, 64);
            v[j] = up ? hi : lo;
        }
    }
    double w = v[0];
#pragma unroll
    for (int o = 32 >> L; o > 0; o >>= 1) w += __shfl_xor(w, o, 64);
    comp = (lanei >> (6 - L)) & (C - 1);
    return w;
}

template <int NV, int NR>
__device__ void block_partials(const double (&v)[NV][NR], double* part, int lb, int nblocks) {
    constexpr int C = NV * NR;
    __shared__ double red[kBlock / 64][C];
    const int lanei = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double flat[C];
#pragma unroll
    for (int a = 0; a < NV; ++a)
#pragma unroll
        for (int k = 0; k < NR; ++k) flat[a * NR + k] = v[a][k];
    int comp;
    const double w = wave_reduce_scatter<C>(flat, lanei, comp);
    if ((lanei & ((64 / C) - 1)) == 0) red[wave][comp] = w;
    __syncthreads();
    if (threadIdx.x < NV * NR) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) s += red[w][threadIdx.x];
        stg(&part[(size_t)threadIdx.x * nblocks + lb], s);
    }
}

constexpr int kXcdRun = CPMGPU_XCD_RUN;

template <typename T>
__device__ __forceinline__ const Seg<T>& seg_of(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, int& lb, int64_t& row) {
    // Workgroups are dispatched to the 8 XCDs round-robin (workgroup b to XCD
    // b mod 8).  Renumber them so that each XCD takes runs of kXcdRun
    // consecutive row blocks: the x rows a run's stencils gather then come
    // from that XCD's own L2 instead of every XCD fetching all of them, and
    // costly rows (interior-boundary rows sit together at the end) still
    // spread over all XCDs.  The tail that does not fill whole runs keeps
    // the plain order.
    const int b = (int)blockIdx.x, n = (int)gridDim.x;
    const int nfull = n / (8 * kXcdRun) * (8 * kXcdRun);
    int vb = b;
    if (b < nfull) {
        const int xcd = b % 8, k = b / 8;
        vb = ((k / kXcdRun) * 8 + xcd) * kXcdRun + k % kXcdRun;
    }
    if (!bseg) {   // one segment: no map (a dependent load less)
        lb = vb;
        row = (int64_t)lb * kBlock + threadIdx.x;
        return segs[0];
    }
    const int e = bseg[vb];
    lb = e >> kSegBits;
    row = (int64_t)lb * kBlock + threadIdx.x;
    return segs[e & (kMaxSegs - 1)];
}
// ... of a kernel that takes the only segment as an argument where the launch
// has one (ONE): the fields come with the kernel's arguments, one dependent
// load less than through the table.
template <bool ONE, typename T>
__device__ __forceinline__ const Seg<T>& seg_of(const SegArg<T>& a, int& lb, int64_t& row) {
    const Seg<T>& t = seg_of(a.segs, ONE ? nullptr : a.bseg, lb, row);
    return ONE ? a.one : t;
}

// Lane masks: bit s set = act on lanes whose status is s.
constexpr unsigned M_RUN = 1u << ST_RUN;
constexpr unsigned M_RESTART = 1u << ST_RESTART;
constexpr unsigned M_UPDATE = (1u << ST_UPDATE) | (1u << ST_UPDATE_MAXIT);
constexpr unsigned M_RESCALE = 1u << ST_RESCALE;
constexpr unsigned M_READY = 1u << ST_READY;
constexpr unsigned M_ALL = 0xffffffffu;
// The iteration's stages (the FP64 loop only ever has RUN lanes among these).
constexpr unsigned M_STAGE1 = M_RUN | M_UPDATE;    // pupdate .. fin alpha
constexpr unsigned M_STAGE2 = M_RUN | M_RESCALE;   // supdate, lfinish t .. fin omega
constexpr unsigned M_STAGE3 = M_RUN | M_READY;     // fin of the loop test

template <typename T>
__device__ __forceinline__ bool lane_in(const Seg<T>& sg, int k, unsigned mask) {
    return k < sg.nr && ((mask >> ldg(&sg.st[k].status)) & 1u);
}

// The FP64 vectors of mixed-precision segments are lane-major: lane k is a
// run of D values at off + k D, so a refinement step moves only the data of
// the lanes that refine and its gathers read with stride 1.
template <typename T>
__device__ __forceinline__ size_t lm_at(const Seg<T>& sg, int k, int64_t row) {
    return (size_t)(sg.off + (int64_t)k * sg.op.D + row);
}

template <typename T>
__device__ __forceinline__ bool seg_any(const Seg<T>& sg, unsigned mask) {
    bool a = false;
    for (int k = 0; k < sg.nr; ++k) a |= ((mask >> ldg(&sg.st[k].status)) & 1u) != 0;
    return a;
}

// The statuses of a segment's lanes, read once per kernel with all loads in
// flight together: a group always owns kMaxNR states, so every load is valid
// (testing lane by lane up to nr waits for each scalar load in turn, several
// microseconds before the first vector load of a kernel).  nr = 0: no lane.
template <int NR>
struct LaneStat {
    int s[NR];
    int nr;
    __device__ __forceinline__ unsigned of(unsigned mask) const {   // bit k: lane k's status is in mask
        unsigned b = 0;
#pragma unroll
        for (int k = 0; k < NR; ++k) b |= ((mask >> s[k]) & 1u) << k;
        return b & ((1u << nr) - 1u);
    }
};
template <int NR, typename T>
__device__ __forceinline__ LaneStat<NR> lane_stat(const Seg<T>& sg, bool valid = true, int copy = 0) {
    LaneStat<NR> L;
    const KState* st = sg.st + (int64_t)copy * sg.sst;
#pragma unroll
    for (int k = 0; k < NR; ++k) L.s[k] = valid ? ldg(&st[k].status) : 0;
    L.nr = valid ? sg.nr : 0;
    return L;
}
template <int NR>
__device__ __forceinline__ bool lane_in(const LaneStat<NR>& L, int k, unsigned mask) { return (L.of(mask) >> k) & 1u; }
template <int NR>
__device__ __forceinline__ bool seg_any(const LaneStat<NR>& L, unsigned mask) { return L.of(mask) != 0; }

// Diagonal_Inverse, GeneralizedBiCGStabSystem.h:303-338 (the branch the
// reference runs: Compute() is never called).  FP64 divides, as the
// reference does.  FP32 (a precision of this library's own, refined against
// FP64) multiplies by the segment's reciprocals of its trailing-row and (in
// the tensor-product format) its one plain diagonal value, formed once when
// the segment is set up: a division per value costs ~10 instructions where
// the gathers form P^-1 of every x row they load.
// TP: the operator is known to be in the tensor-product format.
// The diagonal of A = m I + n L at a row whose L_ii is ld.
template <typename T>
__device__ __forceinline__ T diag_denom(const Seg<T>& sg, T ld) { return (T)sg.m + ld * (T)sg.n; }

template <typename T, bool TP = false>
__device__ __forceinline__ T diag_inverse(const Seg<T>& sg, int64_t row, uint8_t f, T val) {
    constexpr bool kRecip = std::is_same<T, float>::value;
    const int64_t dof = sg.op.D - sg.op.nD;
    if (row >= dof) {   // :335-338 overwrite the trailing rows last
        if constexpr (kRecip) return val * sg.tinv;
        return val / (T)(sg.m - sg.n);
    }
    if (f & ROW_IDENTITY) return val;
    if (f & ROW_NODIAG) return val;
    if (TP || sg.op.fmt == OP_TP) {
        if constexpr (kRecip) return val * sg.dinv;
        return val / diag_denom(sg, sg.op.ldu);
    }
    return val / diag_denom(sg, ldg(&sg.op.ldiag[row]));
}

constexpr double kJacobiOmega = 2.0 / 3.0;   // GeneralizedBiCGStabSystem.h:364

// Precondition, GeneralizedBiCGStabSystem.h:350-385.  Jacobi: the first of the
// precond_iters damped sweeps from result = 0 (A 0 = 0), result = omega
// D^-1 x on the rows below dofs and 0 on the trailing nD rows; the further
// sweeps (k_jacobi) need an operator apply each.
template <typename T, bool TP = false>
__device__ __forceinline__ T precond_apply(const Seg<T>& sg, int64_t row, uint8_t f, T val) {
    if (sg.precond == 1 /*diagonal*/) return diag_inverse<T, TP>(sg, row, f, val);
    if (sg.precond == 2 /*jacobi*/) {
        if (sg.precond_iters <= 0 || row >= sg.op.D - sg.op.nD) return (T)0;
        return (T)kJacobiOmega * diag_inverse<T, TP>(sg, row, f, val);
    }
    return val;
}

// P^-1 of a row's NR values, lane by lane with precond_apply: the iteration
// forms y = P^-1 p and z = P^-1 s where it reads them (the gathers' LDS
// fills, lfinish, xrupdate) instead of storing them, with the same
// operations, so the results are those of stored vectors to the bit.
template <typename T, int NR, bool TP = false>
__device__ __forceinline__ typename VT<T, NR>::type precond_row(const Seg<T>& sg, int64_t row, uint8_t f,
                                                                const typename VT<T, NR>::type& v) {
    typename VT<T, NR>::type y;
#pragma unroll
    for (int k = 0; k < NR; ++k) setlane(y, k, precond_apply<T, TP>(sg, row, f, lane(v, k)));
    return y;
}

// P^-1 of one row as factors its lanes share, found once per row: y = c ((v
// / dd) mul), or 0 where `zero`.  A division by 1 and products with 1 change
// no value, so for every preconditioner, row class and format this performs
// precond_apply's operations in its order (the vector kernels' form of it:
// precond_apply's branches and scalar loads, taken for each of a row's
// lanes, made up two thirds of their instructions).  div: whether the
// segment's rows divide (FP64, or FP32 in the ELL format), uniform per
// segment.
template <typename T>
struct PRow {
    T dd, mul, c;
    bool zero;
    __device__ __forceinline__ T apply(T v, bool div) const {
        T q = div ? v / dd : v;
        q = q * mul;
        q = c * q;
        return zero ? (T)0 : q;
    }
};
template <typename T>
__device__ __forceinline__ bool prow_div(const Seg<T>& sg) {
    return !std::is_same<T, float>::value || sg.op.fmt != OP_TP;
}
template <typename T>
__device__ __forceinline__ PRow<T> prow_of(const Seg<T>& sg, int64_t row, uint8_t f) {
    constexpr bool kRecip = std::is_same<T, float>::value;
    PRow<T> p{(T)1, (T)1, (T)1, false};
    if (sg.precond != 1 && sg.precond != 2) return p;   // none: y = v
    const bool trail = row >= sg.op.D - sg.op.nD;
    if (sg.precond == 2) {   // Jacobi's first sweep: omega D^-1 v, 0 on the trailing rows
        p.c = (T)kJacobiOmega;
        p.zero = sg.precond_iters <= 0 || trail;
    }
    if (trail) {
        if constexpr (kRecip) p.mul = sg.tinv;
        else p.dd = (T)(sg.m - sg.n);
    } else if (!(f & (ROW_IDENTITY | ROW_NODIAG))) {
        if (sg.op.fmt == OP_TP) {
            if constexpr (kRecip) p.mul = sg.dinv;
            else p.dd = diag_denom(sg, sg.op.ldu);
        } else {
            p.dd = diag_denom(sg, ldg(&sg.op.ldiag[row]));
        }
    }
    return p;
}
template <typename T, int NR>
__device__ __forceinline__ typename VT<T, NR>::type prow_apply(const PRow<T>& p, bool div, const typename VT<T, NR>::type& v) {
    typename VT<T, NR>::type y;
#pragma unroll
    for (int k = 0; k < NR; ++k) setlane(y, k, p.apply(lane(v, k), div));
    return y;
}

// A shared-stencil list entry: the x row, and in bit 30 whether the row is an
// identity or no-diagonal row (its P^-1 leaves the value as it is).
constexpr int kListRowMask = (1 << 30) - 1;
constexpr int kListPlainBit = 30;

// E row of the tensor-product format: slot (i, j, k) in the reference's
// order, value (wz[k] wy[j]) wx[i] formed exactly as when E was built.  One
// stencil line (4 consecutive x rows) per step, two steps in flight (fully
// unrolled, the 64 NR-wide gathers would take every register).  A row whose
// columns an interior boundary moved runs the same loop with the line's four
// columns read from its exception record.  Both loops are kept free of
// branches: a conditional load inside the loop costs twice its time even
// when never taken.  `stride` = elements between consecutive rows of xb.
template <typename T, typename V, int W, bool EXC>
__device__ __forceinline__ void egather_tp_lines(const OpView<T>& op, int64_t row, const T* xb, int stride, int e,
                                                 V& acc) {
    typedef int I4 __attribute__((ext_vector_type(4)));
    const int64_t D = op.D;
    T wz[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) wz[q] = ldg(&op.tpw[(8 + q) * D + row]);
    const I4* ex = reinterpret_cast<const I4*>(op.ecx) + (size_t)e * 16;
#pragma unroll 2
    for (int l = 0; l < 16; ++l) {
        const T wx = ldg(&op.tpw[(l >> 2) * D + row]);
        const T wy = ldg(&op.tpw[(4 + (l & 3)) * D + row]);
        I4 c;
        if (EXC) {
            c = ldg(ex + l);
        } else {
            const int c0 = ldg(&op.tpc[l * D + row]);
            c = I4{c0, c0 + 1, c0 + 2, c0 + 3};
        }
        const V x0 = vload<T, W>(xb + (size_t)c.x * stride), x1 = vload<T, W>(xb + (size_t)c.y * stride),
                x2 = vload<T, W>(xb + (size_t)c.z * stride), x3 = vload<T, W>(xb + (size_t)c.w * stride);
        acc += ((wz[0] * wy) * wx) * x0;
        acc += ((wz[1] * wy) * wx) * x1;
        acc += ((wz[2] * wy) * wx) * x2;
        acc += ((wz[3] * wy) * wx) * x3;
    }
}

template <typename T, typename V, int W>
__device__ __forceinline__ void egather_tp(const OpView<T>& op, int64_t row, const T* xb, int stride, V& acc) {
    const int e = ldg(&op.exc[row]);
    if (e < 0) {
        egather_tp_lines<T, V, W, false>(op, row, xb, stride, 0, acc);
    } else {
        egather_tp_lines<T, V, W, true>(op, row, xb, stride, e, acc);
        const int xc = ldg(&op.xcol[e]);   // the extra entry after the stencil
        if (xc >= 0) acc += ldg(&op.xval[e]) * vload<T, W>(xb + (size_t)xc * stride);
    }
}

// LDS rows per tile for T x NR values per row (0: the list would not fit in
// kLdsBytes of LDS and every tile reads x directly).
template <typename T, int NR>
struct LdsTile {
    static constexpr int kRows = (kLdsRows * NR * (int)sizeof(T) <= kLdsBytes) ? kLdsRows : 0;
};

// LDS copy of a tile's x rows.  Rows of 32 bytes are kept as two planes of
// 16-byte halves (half h of row p at plane h, slot p): a ds_read_b128 of the
// lanes' rows then meets half the bank conflicts of 32-byte rows (measured on
// the torus-knot system; 8-byte planes were slower again).
template <typename V>
struct LdsRows {
    typedef int I4 __attribute__((ext_vector_type(4)));
    static constexpr bool kSplit = sizeof(V) == 32;
    V* base;
    int cap;
    __device__ __forceinline__ V load(int p) const {
        if constexpr (kSplit) {
            const I4* h = reinterpret_cast<const I4*>(base);
            const I4 a = h[p], b = h[cap + p];
            V v;
            __builtin_memcpy(reinterpret_cast<char*>(&v), &a, 16);
            __builtin_memcpy(reinterpret_cast<char*>(&v) + 16, &b, 16);
            return v;
        } else {
            return base[p];
        }
    }
    __device__ __forceinline__ void store(int p, const V& v) const {
        if constexpr (kSplit) {
            I4* h = reinterpret_cast<I4*>(base);
            I4 a, b;
            __builtin_memcpy(&a, reinterpret_cast<const char*>(&v), 16);
            __builtin_memcpy(&b, reinterpret_cast<const char*>(&v) + 16, 16);
            h[p] = a;
            h[cap + p] = b;
        } else {
            base[p] = v;
        }
    }
};

// A row's tensor-product metadata, loaded before the tile's x is in LDS so
// that its latency overlaps the fill.
template <typename T>
struct TpRow {
    T w[12];      // wx[4], wy[4], wz[4]
    int p[16];    // position of each line's first x row in the tile's list
};

template <typename T>
__device__ __forceinline__ void tp_row_load(const OpView<T>& op, int64_t row, TpRow<T>& m) {
    const int64_t D = op.D;
#pragma unroll
    for (int q = 0; q < 12; ++q) m.w[q] = ldg(&op.tpw[q * D + row]);
#pragma unroll
    for (int l = 0; l < 16; ++l) m.p[l] = ldg(&op.tpl[l * D + row]);
}

// E row of the tensor-product format from the tile's LDS copy of x: the same
// products in the same order as egather_tp_lines, so both paths agree to the
// bit.  lx.load(p) is the x row at position p of the tile's list.
template <typename T, typename V, int W>
__device__ __forceinline__ void egather_tp_lds(const TpRow<T>& m, const LdsRows<V>& lx, V& acc) {
#pragma unroll
    for (int l = 0; l < 16; ++l) {
        T wx = m.w[l >> 2], wy = m.w[4 + (l & 3)];
        // the empty asm (no instruction) holds each line's products to their
        // line: formed all together ahead of the LDS reads, the 64 products
        // take 64 (FP64: 128) registers, which halved the FP64 kernel's
        // occupancy once the row's weights were loaded with the tile's list
        asm volatile("" : "+v"(wx), "+v"(wy));
        const int q = m.p[l];
        const V x0 = lx.load(q), x1 = lx.load(q + 1), x2 = lx.load(q + 2), x3 = lx.load(q + 3);
        acc += ((m.w[8] * wy) * wx) * x0;
        acc += ((m.w[9] * wy) * wx) * x1;
        acc += ((m.w[10] * wy) * wx) * x2;
        acc += ((m.w[11] * wy) * wx) * x3;
    }
}

// An exception row's LDS positions (kExcPos int16 packed in pairs).
struct ExcRow {
    int pk[kExcPos / 2];
    __device__ __forceinline__ int pos(int s) const { return (int)(int16_t)(pk[s >> 1] >> (16 * (s & 1))); }
};

__device__ __forceinline__ void exc_row_load(const int16_t* tlx, int e, ExcRow& m) {
    typedef int I4 __attribute__((ext_vector_type(4)));
    const I4* src = reinterpret_cast<const I4*>(tlx + (size_t)e * kExcPos);
#pragma unroll
    for (int q = 0; q < kExcPos / 8; ++q) {
        const I4 v = ldg(src + q);
        m.pk[4 * q] = v.x;
        m.pk[4 * q + 1] = v.y;
        m.pk[4 * q + 2] = v.z;
        m.pk[4 * q + 3] = v.w;
    }
}

// An exception row (a row an interior boundary moved) from a tile's LDS copy
// of x, with its weights (wx[4], wy[4], wz[4]) and extra value loaded before
// the tile's fill: the slots and the extra entry of egather_tp's exception
// path, in its order.
template <typename T, typename V>
__device__ __forceinline__ void egather_grp_exc(const T (&w)[12], T xv, const ExcRow& m, const LdsRows<V>& lx, V& acc) {
#pragma unroll
    for (int l = 0; l < 16; ++l) {
        const T wx = w[l >> 2], wy = w[4 + (l & 3)];
        const V x0 = lx.load(m.pos(4 * l)), x1 = lx.load(m.pos(4 * l + 1)), x2 = lx.load(m.pos(4 * l + 2)),
                x3 = lx.load(m.pos(4 * l + 3));
        acc += ((w[8] * wy) * wx) * x0;
        acc += ((w[9] * wy) * wx) * x1;
        acc += ((w[10] * wy) * wx) * x2;
        acc += ((w[11] * wy) * wx) * x3;
    }
    // The extra entry's position, taken from its word only here: the empty
    // asm (no instruction) keeps the compiler from decoding it before the
    // tile's barrier, where it would wait for the record's load.
    int w64 = m.pk[32];
    asm volatile("" : "+v"(w64));
    const int xp = (int)(int16_t)w64;
    if (xp >= 0) acc += xv * lx.load(xp);
}

// A kind-0 item of a shared-stencil tile: up to kGrpRows rows with the same
// stencil block (absent rows have weight 0 and are not stored).
template <typename T>
struct GrpItem {
    T w[kGrpRows][12];   // wx[4], wy[4], wz[4] of each row
    int pp[8];           // positions of lines 2h and 2h + 1's first x rows in the tile's list (low, high 16 bits)
    int row[kGrpRows];
    __device__ __forceinline__ int p(int l) const { return (int)(((unsigned)pp[l >> 1] >> (16 * (l & 1))) & 0xffffu); }
};

// The rows and weights of the kGrpRows slots from s0 (slots past the last
// are read as the last: rows g >= n of an item are never used).  Loads with
// no condition, so that none waits on another; a slot's 12 weights are
// contiguous, read 16 bytes at a time.
template <typename T>
__device__ __forceinline__ void grp_item_load(const OpView<T>& op, int s0, GrpItem<T>& m) {
    constexpr int E = 16 / (int)sizeof(T);   // weights per 16-byte load
    typedef T V16 __attribute__((ext_vector_type(E)));
    const int64_t S = op.nslot;
#pragma unroll
    for (int g = 0; g < kGrpRows; ++g) {
        const int64_t sl = s0 + g < S ? s0 + g : S - 1;
        m.row[g] = ldg(&op.grow[sl]);
        const V16* src = reinterpret_cast<const V16*>(op.gw + sl * 12);
#pragma unroll
        for (int q = 0; q < 12 / E; ++q) {
            const V16 v = ldg(src + q);
#pragma unroll
            for (int e = 0; e < E; ++e) m.w[g][q * E + e] = v[e];
        }
    }
}

// The rows of a kind-0 item from the tile's LDS copy of x: every x row of the
// block is read once and used by all rows of the item; each row's products
// and sums are those of egather_tp_lds, in its order, so all paths agree to
// the bit.
template <typename T, typename V, int W>
__device__ __forceinline__ void egather_grp_lds(const GrpItem<T>& m, int n, const LdsRows<V>& lx, V (&acc)[kGrpRows]) {
#pragma unroll
    for (int l = 0; l < 16; ++l) {
        const int q = m.p(l);
        const V x0 = lx.load(q), x1 = lx.load(q + 1), x2 = lx.load(q + 2), x3 = lx.load(q + 3);
#pragma unroll
        for (int g = 0; g < kGrpRows; ++g) {
            if (g < n) {
                const T wx = m.w[g][l >> 2], wy = m.w[g][4 + (l & 3)];
                acc[g] += ((m.w[g][8] * wy) * wx) * x0;
                acc[g] += ((m.w[g][9] * wy) * wx) * x1;
                acc[g] += ((m.w[g][10] * wy) * wx) * x2;
                acc[g] += ((m.w[g][11] * wy) * wx) * x3;
            }
        }
    }
}

// A thread's entries of a tile's list of x rows (entry threadIdx.x + k kBlock).
template <int LR>
struct FillIdx {
    static constexpr int KF = LR > 0 ? (LR + kBlock - 1) / kBlock : 1;
    int src[KF];
    int nu;
};

// The list entries (lst of nu rows; lst[0] readable even when nu = 0), all
// loads in flight together: entries past the list read its last entry
// instead of branching (a load in a branch is waited for inside it).
template <int LR>
__device__ __forceinline__ void lds_fill_index(const int* lst, int nu, FillIdx<LR>& f) {
    f.nu = nu;
    const int last = nu > 0 ? nu - 1 : 0;
#pragma unroll
    for (int k = 0; k < FillIdx<LR>::KF; ++k) {
        const int u = (int)threadIdx.x + k * kBlock;
        f.src[k] = ldg(&lst[u < last ? u : last]);
    }
}

// The listed x rows into LDS, all loads in flight together, each row put
// through xform(row value, list entry) on its way, then a workgroup barrier.
template <typename T, int NR, int LR, typename V, typename F>
__device__ __forceinline__ void lds_fill_rows(const FillIdx<LR>& f, const T* xb, const LdsRows<V>& lrows, F&& xform) {
    constexpr int KF = FillIdx<LR>::KF;
    V buf[KF];
#pragma unroll
    for (int k = 0; k < KF; ++k)
        if ((int)threadIdx.x + k * kBlock < f.nu) buf[k] = vload<T, NR>(xb + (size_t)(f.src[k] & kListRowMask) * NR);
#pragma unroll
    for (int k = 0; k < KF; ++k) {
        const int u = (int)threadIdx.x + k * kBlock;
        if (u < f.nu) lrows.store(u, xform(buf[k], f.src[k]));
    }
    __syncthreads();
}

// Where a tile's x rows come from: load(row) issues a row's loads, value()
// forms the gathered row from them (ident: an identity or no-diagonal row).
// SrcPlain: x itself, or with FLY P^-1 x (x is p or s of an iteration that
// forms y and z where it reads them) with the preconditioner of segment *sg.
template <typename T, int NR, bool FLY>
struct SrcPlain {
    typedef typename VT<T, NR>::type V;
    typedef V Raw;
    const Seg<T>* sg;
    const T* x;
    __device__ __forceinline__ Raw load(int64_t row) const { return vload<T, NR>(x + (size_t)row * NR); }
    __device__ __forceinline__ V value(const Raw& v, int64_t row, bool ident) const {
        if constexpr (FLY) return precond_row<T, NR, true>(*sg, row, ident ? ROW_IDENTITY : 0, v);
        else return v;
    }
};
// P^-1 of the direction that pupdate would store: p = (p - w v) beta + r on
// the running lanes (the same operations, so the same bits).
template <typename T, int NR>
struct SrcP {
    typedef typename VT<T, NR>::type V;
    struct Raw { V p, v, r; };
    const Seg<T>* sg;
    const T *p, *v, *r;
    T beta[NR], w[NR];
    unsigned run;
    __device__ __forceinline__ Raw load(int64_t row) const {
        const size_t i = (size_t)row * NR;
        return Raw{vload<T, NR>(p + i), vload<T, NR>(v + i), vload<T, NR>(r + i)};
    }
    __device__ __forceinline__ V direction(const Raw& q) const {
        V pv = q.p;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const T pk = (-w[k] * lane(q.v, k) + lane(q.p, k)) * beta[k] + lane(q.r, k);
            if ((run >> k) & 1u) setlane(pv, k, pk);
        }
        return pv;
    }
    __device__ __forceinline__ V value(const Raw& q, int64_t row, bool ident) const {
        return precond_row<T, NR, true>(*sg, row, ident ? ROW_IDENTITY : 0, direction(q));
    }
};
// P^-1 of the residual that supdate would store: s = r - alpha v.
template <typename T, int NR>
struct SrcS {
    typedef typename VT<T, NR>::type V;
    struct Raw { V r, v; };
    const Seg<T>* sg;
    const T *r, *v;
    T alpha[NR];
    __device__ __forceinline__ Raw load(int64_t row) const {
        const size_t i = (size_t)row * NR;
        return Raw{vload<T, NR>(r + i), vload<T, NR>(v + i)};
    }
    __device__ __forceinline__ V residual(const Raw& q) const {
        V sv;
#pragma unroll
        for (int k = 0; k < NR; ++k) setlane(sv, k, -alpha[k] * lane(q.v, k) + lane(q.r, k));
        return sv;
    }
    __device__ __forceinline__ V value(const Raw& q, int64_t row, bool ident) const {
        return precond_row<T, NR, true>(*sg, row, ident ? ROW_IDENTITY : 0, residual(q));
    }
};
// A refinement lane's FP64 solution as pupdate would store it: x64 + x32 / scale.
template <int NR>
struct SrcX64 {
    typedef double V;
    struct Raw { double x; float d; };
    const double* x;
    const float* x32;
    double scale;
    __device__ __forceinline__ Raw load(int64_t row) const { return Raw{ldg(x + row), ldg(x32 + (size_t)row * NR)}; }
    __device__ __forceinline__ V value(const Raw& q, int64_t, bool) const { return q.x + (double)q.d / scale; }
};

// x of a caller's vector, whose row perm[r] the operator's row r is.
struct SrcPerm {
    typedef double V;
    typedef double Raw;
    const double* x;
    const int* perm;
    __device__ __forceinline__ Raw load(int64_t row) const { return ldg(x + ldg(perm + row)); }
    __device__ __forceinline__ V value(const Raw& v, int64_t, bool) const { return v; }
};

// Where a tile's rows go: to out, interleaved like x; or, DstPerm, to NR
// caller's vectors, identity rows taking the values of g (null: as gathered).
template <typename T, int NR>
struct DstPlain {
    static constexpr bool kSkipIdentity = false;
    T* out;
    __device__ __forceinline__ void store(int64_t row, const typename VT<T, NR>::type& v) const {
        vstore<T, NR>(out + (size_t)row * NR, v);
    }
    __device__ __forceinline__ void identity(int64_t) const {}
};
template <int NR, bool HELD>
struct DstPerm {
    static constexpr bool kSkipIdentity = HELD;
    double* out[NR];
    const double* g[NR];
    const int* perm;
    __device__ __forceinline__ void store(int64_t row, const typename VT<double, NR>::type& v) const {
        const int c = ldg(perm + row);
#pragma unroll
        for (int k = 0; k < NR; ++k) stg(out[k] + c, (double)lane(v, k));
    }
    __device__ __forceinline__ void identity(int64_t row) const {
        const int c = ldg(perm + row);
#pragma unroll
        for (int k = 0; k < NR; ++k) stg(out[k] + c, ldg(g[k] + c));
    }
};

// One shared-stencil tile of E x, (E x)_row to dst with x from src: thread
// t takes the item at place tile kBlock + t.  mid(src), called once the loads
// are under way, completes src (the scalars its values need) and says whether
// to go on (the same on every thread).
template <typename T, int NR, int LR, typename V, typename Src, typename Dst, typename Mid>
__device__ __forceinline__ void egather_grp_tile(const OpView<T>& op, int tile, Src& src, const Dst& dst, const LdsRows<V>& lrows,
                                                 Mid&& mid) {
    // Loads in two rounds, each issued as soon as the previous one's values
    // are in: the list entries (first: the x rows wait on them), the item's
    // offsets and line words, all at fixed places of the tile; then the x
    // rows and the item's data.
    constexpr int KF = FillIdx<LR>::KF;
    static_assert(KF * kBlock == LR && LR == kGrpLdsRows, "a tile's list places are read whole");
    int e[KF];
    const int nu = ldg(&op.gln[tile]);
#pragma unroll
    for (int k = 0; k < KF; ++k) e[k] = ldg(&op.glr[(size_t)tile * LR + threadIdx.x + k * kBlock]);
    const int64_t NI = op.nitem;
    const int item = tile * kBlock + (int)threadIdx.x;
    const int a = ldg(&op.gofs[item]), b = ldg(&op.gofs[item + 1]);
    GrpItem<T> m;
#pragma unroll
    for (int h = 0; h < 8; ++h) m.pp[h] = ldg(&op.gpl[h * NI + item]);
    const int s0 = a & kGrpOfsMask;
    const int kind = a >> kGrpKindShift;   // 3: an empty place
    const int n = (b & kGrpOfsMask) - s0;
    // The items' global loads are issued before the barrier: a load after it
    // holds its wave (and the workgroup's next tile) for a whole memory
    // latency.  kind 0: the rows' weights, line positions and rows; kind 1
    // (a row an interior boundary moved): its weights in m.w[0], its row,
    // positions and extra value.  kind 2 (identity rows, their rows in the
    // line words) reads its x values after the barrier: such items sit in
    // the last tiles only, and loads of them here reused registers that the
    // kind 1 loads then had to wait for.
    ExcRow mx;
    T xval = (T)0;
    if (kind == 1) {   // issued before the weights: they need only the line words
        const int x = m.pp[0];
        exc_row_load(op.glx, x, mx);
        xval = ldg(&op.xval[x]);
    }
    grp_item_load(op, s0, m);   // kinds 0 and 1 (kind 1: slot s0's row and weights)
    typename Src::Raw buf[KF];
#pragma unroll
    for (int k = 0; k < KF; ++k)
        if ((int)threadIdx.x + k * kBlock < nu) buf[k] = src.load(e[k] & kListRowMask);
    if (!mid(src)) return;
#pragma unroll
    for (int k = 0; k < KF; ++k) {
        const int u = (int)threadIdx.x + k * kBlock;
        if (u < nu) lrows.store(u, src.value(buf[k], e[k] & kListRowMask, (e[k] >> kListPlainBit) & 1));
    }
    __syncthreads();
    if (kind == 0) {
        V acc[kGrpRows];
#pragma unroll
        for (int g = 0; g < kGrpRows; ++g) acc[g] = (V)(T)0;
        egather_grp_lds<T, V, NR>(m, n, lrows, acc);
#pragma unroll
        for (int g = 0; g < kGrpRows; ++g)
            if (g < n) dst.store(m.row[g], acc[g]);
    } else if (kind == 1) {
        V acc = (V)(T)0;
        egather_grp_exc<T, V>(m.w[0], xval, mx, lrows, acc);
        dst.store(m.row[0], acc);
    } else if (kind == 2) {
#pragma unroll
        for (int g = 0; g < kGrpRows; ++g)
            if (g < n) {
                const int64_t r = m.pp[g];
                if (Dst::kSkipIdentity) dst.identity(r);
                else dst.store(r, src.value(src.load(r), r, ldg(&op.flag[r]) & (ROW_IDENTITY | ROW_NODIAG)));
            }
    }
}

// Slots s, s + 1, .. of an E row of the ELL format in rounds of U as long as
// whole ones are left, each round's columns, values and x loaded together.
template <int U, typename T, typename V, int W>
__device__ __forceinline__ int ell_rounds(const OpView<T>& op, int64_t row, const T* xb, int stride, int s, V& acc) {
    const int64_t D = op.D;
    const int* col = op.ecol + row;
    const T* val = op.eval + row;
    for (; s + U <= op.ew; s += U) {
        int c[U];
        T w[U];
        V x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) { c[u] = ldg(&col[(int64_t)(s + u) * D]); w[u] = ldg(&val[(int64_t)(s + u) * D]); }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = vload<T, W>(xb + (size_t)c[u] * stride);
#pragma unroll
        for (int u = 0; u < U; ++u) acc += w[u] * x[u];
    }
    return s;
}

// E row of the ELL format: a slot's x waits for its column, so a row's time is
// memory latencies, two for each round of slots, and a small operator has too
// few rows to hide them (18,855 rows of 64 slots are 74 workgroups). Rounds of
// U slots, then of 8, and what 8 does not divide slot by slot. 60 FP64 iterations with
// the remainder of 32 slot by slot and in rounds of 8: 27 slots a row, 91,741
// rows 4.1 and 2.9 ms; 125 slots, 50,970 rows 5.5 and 4.2 ms.
template <int U, typename T, typename V, int W>
__device__ __forceinline__ void egather_ell(const OpView<T>& op, int64_t row, const T* xb, int stride, V& acc) {
    int s = ell_rounds<U, T, V, W>(op, row, xb, stride, 0, acc);
    if constexpr (U > 8) s = ell_rounds<8, T, V, W>(op, row, xb, stride, s, acc);
    ell_rounds<1, T, V, W>(op, row, xb, stride, s, acc);
}

// (E x)_row for W consecutive values per row of xb.
template <typename T, int W>
__device__ __forceinline__ typename VT<T, W>::type erow(const OpView<T>& op, int64_t row, const T* xb, int stride) {
    typedef typename VT<T, W>::type V;
    V acc = (V)(T)0;
    if (ldg(&op.flag[row]) & ROW_IDENTITY) return vload<T, W>(xb + (size_t)row * stride);
    if (op.fmt == OP_TP) egather_tp<T, V, W>(op, row, xb, stride, acc);
    else egather_ell<8, T, V, W>(op, row, xb, stride, acc);
    return acc;
}

// (A x)_row = m x + n (Ld x + Loff tmp), identity rows x, trailing nD rows
// (m - n) x; xv = x_row, tb = tmp of the segment, W values per row.
template <typename T, int W>
__device__ __forceinline__ typename VT<T, W>::type arow(const OpView<T>& op, double m, double n, int64_t row,
                                                        const typename VT<T, W>::type& xv, const T* tb, int stride) {
    typedef typename VT<T, W>::type V;
    const int64_t D = op.D;
    if (row >= D - op.nD) return (T)(m - n) * xv;
    if (ldg(&op.flag[row]) & ROW_IDENTITY) return xv;
    V lo = (V)(T)0;
    T ld;
    if (op.fmt == OP_TP) {
        // a missing neighbour (-1) reads the row's own entry with weight 0:
        // no conditional load in the loop
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            const int c = ldg(&op.lcol[(int64_t)s * D + row]);
            const T wl = c >= 0 ? op.loff : (T)0;
            lo += wl * vload<T, W>(tb + (size_t)(c >= 0 ? c : row) * stride);
        }
        ld = op.ldu;
    } else {
        ld = ldg(&op.ldiag[row]);
        int s = 0;
        for (; s + 6 <= op.lw; s += 6) {   // six slots in flight (the Laplacian's neighbours)
            int c[6];
            T w[6];
#pragma unroll
            for (int u = 0; u < 6; ++u) {
                c[u] = ldg(&op.lcol[(int64_t)(s + u) * D + row]);
                w[u] = ldg(&op.lval[(int64_t)(s + u) * D + row]);
            }
#pragma unroll
            for (int u = 0; u < 6; ++u) lo += w[u] * vload<T, W>(tb + (size_t)c[u] * stride);
        }
        for (; s < op.lw; ++s) {
            const int c = ldg(&op.lcol[(int64_t)s * D + row]);
            lo += ldg(&op.lval[(int64_t)s * D + row]) * vload<T, W>(tb + (size_t)c * stride);
        }
    }
    return (T)m * xv + (T)n * (ld * xv + lo);
}

// arow of the tensor-product format with every load issued up front: the
// row's flag and L columns with x (and the caller's other loads), then the
// six neighbours' E x rows, then the products and sums of arow in its order,
// the trailing and identity rows taking their values by selection (a
// missing neighbour reads the row's own entry with weight 0).  pre: x goes
// through P^-1 first (x is p or s of an iteration that forms y and z where
// it reads them).
template <typename T, int W>
struct TpLRow {
    typename VT<T, W>::type xv;
    int c[6];
    uint8_t f;
};
template <typename T, int W>
__device__ __forceinline__ void arow_tp_load(const OpView<T>& op, int64_t row, const T* xr, TpLRow<T, W>& a) {
    const int64_t D = op.D;
    a.f = ldg(&op.flag[row]);
#pragma unroll
    for (int s = 0; s < 6; ++s) a.c[s] = ldg(&op.lcol[(int64_t)s * D + row]);
    a.xv = vload<T, W>(xr);
}
template <typename T, int W>
__device__ __forceinline__ typename VT<T, W>::type arow_tp(const Seg<T>& sg, int64_t row, TpLRow<T, W>& a, const T* tb,
                                                           int stride, bool pre) {
    typedef typename VT<T, W>::type V;
    const OpView<T>& op = sg.op;
    V nb[6];
#pragma unroll
    for (int s = 0; s < 6; ++s) nb[s] = vload<T, W>(tb + (size_t)(a.c[s] >= 0 ? a.c[s] : row) * stride);
    V xv = a.xv;
    if (pre) xv = prow_apply<T, W>(prow_of(sg, row, a.f), prow_div(sg), xv);
    V lo = (V)(T)0;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const T wl = a.c[s] >= 0 ? op.loff : (T)0;
        lo += wl * nb[s];
    }
    const T ld = op.ldu;
    V res = (T)sg.m * xv + (T)sg.n * (ld * xv + lo);
    if (a.f & ROW_IDENTITY) res = xv;
    if (row >= op.D - op.nD) res = (T)(sg.m - sg.n) * xv;
    return res;
}

// ---------------------------------------------------------------- finalisers
enum FinKind : int {
    FIN_INIT = 0, FIN_ALPHA, FIN_OMEGA, FIN_ITER64, FIN_RESTART64, FIN_MX_START, FIN_MX_INIT, FIN_ITER_MX
};

// Lanes each finaliser acts on (the producing kernel used the same mask) and
// the number of partial vectors it reads.
template <int KIND> struct FinTraits;
template <> struct FinTraits<FIN_INIT> { static constexpr int NV = 1; static constexpr unsigned M = M_ALL; };
template <> struct FinTraits<FIN_ALPHA> { static constexpr int NV = 1; static constexpr unsigned M = M_STAGE1; };
template <> struct FinTraits<FIN_OMEGA> { static constexpr int NV = 2; static constexpr unsigned M = M_STAGE2; };
template <> struct FinTraits<FIN_ITER64> { static constexpr int NV = 2; static constexpr unsigned M = M_STAGE3; };
template <> struct FinTraits<FIN_RESTART64> { static constexpr int NV = 1; static constexpr unsigned M = M_RESTART; };
template <> struct FinTraits<FIN_MX_START> { static constexpr int NV = 1; static constexpr unsigned M = M_ALL; };
template <> struct FinTraits<FIN_MX_INIT> { static constexpr int NV = 1; static constexpr unsigned M = M_RESCALE; };
template <> struct FinTraits<FIN_ITER_MX> { static constexpr int NV = 2; static constexpr unsigned M = M_STAGE3; };

constexpr double kEps = 2.220446049250313e-16;   // NumTraits<double>::epsilon (BiCGStab.h:56)

// FP32 recurrence (re)started from the scaled true residual.
// The scalar part of the recurrence for one (instance, rhs).
template <int KIND>
__device__ void fin_scalar(KState& s, const double* tot) {
    if (KIND == FIN_INIT) {   // BiCGStab.h:41-58 with x0 = 0: r = r0 = b
        const double bsq = tot[0];
        s.bsq = s.r0sq = s.rr = bsq;
        s.rho_old = s.alpha = s.omega = 1.0;
        s.iters = s.restarts = 0;
        if (!std::isfinite(bsq)) { s.status = ST_BREAKDOWN; return; }
        if (bsq == 0.0) { s.status = ST_ZERO_RHS; return; }
        if (!(bsq > s.tol2 * bsq)) { s.status = ST_CONVERGED; return; }   // tol >= 1
        if (s.max_it <= 0) { s.status = ST_MAXIT; return; }
        s.tol2 *= bsq;                 // tol2 held tol^2
        s.rho = bsq;                   // (r0, r) with r0 = r = b
        s.beta = s.rho;                // (rho / 1) * (1 / 1)
        s.status = ST_RUN;
    } else if (KIND == FIN_ALPHA) {
        if (s.status != ST_RUN) { mx_update(s, tot[0]); return; }
        s.alpha = s.rho / tot[0];                                      // BiCGStab.h:79
        if (!std::isfinite(s.alpha)) s.status = ST_BREAKDOWN;
    } else if (KIND == FIN_OMEGA) {
        if (s.status != ST_RUN) { mx_init(s, tot[0], ST_READY); return; }
        s.omega = tot[0] > 0.0 ? tot[1] / tot[0] : 0.0;                // BiCGStab.h:86-94
        if (!std::isfinite(s.omega)) s.status = ST_BREAKDOWN;
    } else if (KIND == FIN_ITER64) {
        ++s.iters;
        s.rr = tot[0];
        if (!(s.rr > s.tol2)) { s.status = std::isnan(s.rr) ? ST_BREAKDOWN : ST_CONVERGED; return; }   // BiCGStab.h:59
        if (s.iters >= s.max_it) { s.status = ST_MAXIT; return; }
        s.rho_old = s.rho;
        s.rho = tot[1];                                                // BiCGStab.h:61
        if (fabs(s.rho) < kEps * kEps * s.r0sq) { s.status = ST_RESTART; return; }   // BiCGStab.h:62
        s.beta = (s.rho / s.rho_old) * (s.alpha / s.omega);           // BiCGStab.h:73
        if (!std::isfinite(s.beta)) s.status = ST_BREAKDOWN;
    } else if (KIND == FIN_RESTART64) {                                // BiCGStab.h:62-71
        s.rho = s.r0sq = tot[0];
        if (s.restarts++ == 0) s.iters = 0;
        s.beta = (s.rho / s.rho_old) * (s.alpha / s.omega);
        s.status = std::isfinite(s.beta) ? ST_RUN : ST_BREAKDOWN;
    } else if (KIND == FIN_MX_START) {
        const double bsq = tot[0];
        s.bsq = s.rr_true = bsq;
        s.iters = s.restarts = s.updates = 0;
        if (!std::isfinite(bsq)) { s.status = ST_BREAKDOWN; return; }
        if (bsq == 0.0) { s.status = ST_ZERO_RHS; return; }
        if (!(bsq > s.tol2 * bsq)) { s.status = ST_CONVERGED; return; }
        if (s.max_it <= 0) { s.status = ST_MAXIT; return; }
        s.tol2 *= bsq;
        s.scale = 1.0 / sqrt(bsq);
        s.status = ST_RESCALE;
    } else if (KIND == FIN_MX_INIT) {
        mx_init(s, tot[0], ST_RUN);
    } else if (KIND == FIN_ITER_MX) {
        if (s.status == ST_READY) { s.status = ST_RUN; return; }
        ++s.iters;
        const double rr = tot[0];
        s.rr = rr;
        if (std::isnan(rr)) { s.status = ST_BREAKDOWN; return; }
        // scaled tolerance: ||r|| <= tol ||b|| with r scaled by `scale`
        s.judged = 0;
        if (!(rr > s.tol2 * s.scale * s.scale)) { s.judged = 2; s.status = ST_UPDATE; return; }
        if (s.iters >= s.max_it) { s.status = ST_UPDATE_MAXIT; return; }
        if (rr < s.delta2 * s.maxrr) { s.judged = 1; s.status = ST_UPDATE; return; }
        s.rho_old = s.rho;
        s.rho = tot[1];
        if (fabs(s.rho) < kEps * kEps * s.r0sq) { ++s.restarts; s.status = ST_UPDATE; return; }   // BiCGStab.h:62
        s.beta = (s.rho / s.rho_old) * (s.alpha / s.omega);
        if (!std::isfinite(s.beta)) { s.status = ST_BREAKDOWN; return; }
        if (rr > s.maxrr) s.maxrr = rr;
    }
}

// ---------------------------------------------------------------- folded finalisers
// A lane's components over all block partials of its segment, U blocks per
// thread in flight at once (the partials were just written by another
// kernel, so every round costs a full memory latency), then a workgroup sum
// in a fixed order: thread 0 holds the totals.
template <int NV, int NR, typename T>
__device__ __forceinline__ void part_totals(const Seg<T>& sg, const double* part, int k, double (*red)[kBlock / 64],
                                            double (&tot)[NV]) {
    constexpr int U = 8;
    const int lanei = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double acc[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) acc[a] = 0.0;
    for (int b0 = threadIdx.x; b0 < sg.nblocks; b0 += kBlock * U) {
        double v[NV][U];
#pragma unroll
        for (int a = 0; a < NV; ++a)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int b = b0 + kBlock * u;
                v[a][u] = b < sg.nblocks ? ldg(&part[(size_t)(a * NR + k) * sg.nblocks + b]) : 0.0;
            }
#pragma unroll
        for (int a = 0; a < NV; ++a)
#pragma unroll
            for (int u = 0; u < U; ++u) acc[a] += v[a][u];
    }
#pragma unroll
    for (int a = 0; a < NV; ++a) {
        const double t = wave_sum(acc[a]);
        if (lanei == 0) red[a][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int a = 0; a < NV; ++a) {
            double t = 0.0;
            for (int w = 0; w < kBlock / 64; ++w) t += red[a][w];
            tot[a] = t;
        }
}

// Partials of the kernel that leads to copy `in` of the states: xrupdate
// (copy 2) writes its own while workgroups still sum lfinish's.
template <int NR, typename T>
__device__ __forceinline__ double* part_of(const Seg<T>& sg, int copy) {
    return sg.part + (copy == 2 ? (size_t)2 * NR * sg.nblocks : 0);
}

// The finaliser KIND folded into the kernel that first needs its result: every
// workgroup of a segment sums the same partials in the same order and runs
// the same scalar update on its own copy of the lanes' states (in LDS), and
// the segment's first workgroup stores it for the kernels after it.  A
// finaliser of its own costs a launch (2.3-4 us with its gap, three an
// iteration); the sums cost each workgroup one round of loads that mostly
// hit the L2.  States live in three copies (Seg::sst apart): copy `in` is
// only read here while copy `out` is written, so no workgroup meets a state
// that another has already advanced.
template <int KIND, int NR>
struct LaneState {
    static constexpr int NV = FinTraits<KIND>::NV;
    KState s[NR];
    static constexpr int R = NV * NR <= 2 ? kBlock / 64 : 1;
    double red[NV * NR][R];   // the components' sums, of each wave or whole (FoldLoads::kAll)
};
// The loads of a fold, issued before the caller's own so that they overlap:
// the states' words and the first partials. With one lane every thread takes
// kFoldU partials of each component at a time (kAll): 4 x 256 loads a
// component in flight, which is what a sum over 2,000 partials waits for
// (before, a wave summed a component alone: plain solve of 42k / 117k / 181k
// rows 4.50 / 7.66 / 14.9 -> 4.30 / 7.12 / 13.7 ms). With more lanes a wave
// sums whole components, as all of them in turn cost more than they gain
// (6 surfaces x 3 right-hand sides of 8k rows: 5.35 against 5.85 ms).
constexpr int kFoldU = 4;
template <int C>
struct FoldLoads {
    static constexpr bool kAll = C <= 2;
    static constexpr int P = kAll ? C : 1;
    double v[P][kFoldU];
    int w0, w1;
};
// kFoldU partials at b0, b0 + STEP, .. of the P components from part on
template <int P, int STEP>
__device__ __forceinline__ void fold_load(const double* part, int nblocks, int b0, double (&v)[P][kFoldU]) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int u = 0; u < kFoldU; ++u) {
            const int b = b0 + STEP * u;
            v[p][u] = b < nblocks ? ldg(&part[(size_t)p * nblocks + b]) : 0.0;
        }
}
template <int KIND, int NR, typename T>
__device__ __forceinline__ void fold_begin(const Seg<T>& sg, int in, FoldLoads<FinTraits<KIND>::NV * NR>& f) {
    constexpr int C = FinTraits<KIND>::NV * NR;
    constexpr int W = (int)(sizeof(KState) / 4) * NR;   // a group owns kMaxNR states: every load is valid
    static_assert(W <= 2 * kBlock, "a thread copies at most two words");
    const int t = (int)threadIdx.x, wave = t >> 6;
    const int* src = reinterpret_cast<const int*>(sg.st + (int64_t)in * sg.sst);
    f.w0 = t < W ? ldg(&src[t]) : 0;
    f.w1 = W > kBlock && t + kBlock < W ? ldg(&src[t + kBlock]) : 0;
    const double* part = part_of<NR>(sg, in);
    if constexpr (FoldLoads<C>::kAll)
        fold_load<FoldLoads<C>::P, kBlock>(part, sg.nblocks, t, f.v);
    else
        fold_load<1, 64>(part + (size_t)(wave < C ? wave : 0) * sg.nblocks, sg.nblocks, t & 63, f.v);
}
// Each component's sum in part_totals' order: its lane l of wave w adds
// partials 64 w + l, 64 w + l + kBlock, .., and the waves' sums are added in
// order (the sums of lanes that are not in the finaliser's mask are formed and
// not used).
template <int KIND, int NR, typename T>
__device__ __forceinline__ LaneStat<NR> fold_end(const Seg<T>& sg, int in, int out, bool writer,
                                                 const FoldLoads<FinTraits<KIND>::NV * NR>& f, LaneState<KIND, NR>& sh) {
    constexpr int NV = FinTraits<KIND>::NV, C = NV * NR, NW = kBlock / 64;
    constexpr int W = (int)(sizeof(KState) / 4) * NR;
    const int t = (int)threadIdx.x, lanei = t & 63, wave = t >> 6;
    int* lds = reinterpret_cast<int*>(sh.s);
    if (t < W) lds[t] = f.w0;
    if (W > kBlock && t + kBlock < W) lds[t + kBlock] = f.w1;
    const double* part = part_of<NR>(sg, in);
    if constexpr (FoldLoads<C>::kAll) {
        double acc[C], v[C][kFoldU];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            acc[c] = 0.0;
#pragma unroll
            for (int u = 0; u < kFoldU; ++u) acc[c] += f.v[c][u];
        }
        for (int b0 = kBlock * kFoldU; b0 < sg.nblocks; b0 += kBlock * kFoldU) {
            fold_load<C, kBlock>(part, sg.nblocks, b0 + t, v);
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int u = 0; u < kFoldU; ++u) acc[c] += v[c][u];
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const double sum = wave_sum(acc[c]);
            if (lanei == 0) sh.red[c][wave] = sum;
        }
    } else {
        static_assert(kFoldU == NW, "a wave's load is one partial of every wave of part_totals");
        for (int c = wave; c < C; c += NW) {
            const double* pc = part + (size_t)c * sg.nblocks;
            double acc[NW], v[2][1][kFoldU];
            int b0 = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) acc[w] = 0.0;
            if (c == wave) {
#pragma unroll
                for (int w = 0; w < NW; ++w) acc[w] += f.v[0][w];
                b0 = kBlock;
            }
            for (; b0 < sg.nblocks; b0 += 2 * kBlock) {
                fold_load<1, 64>(pc, sg.nblocks, b0 + lanei, v[0]);
                fold_load<1, 64>(pc, sg.nblocks, b0 + kBlock + lanei, v[1]);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int w = 0; w < NW; ++w) acc[w] += v[u][0][w];
            }
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < NW; ++w) sum += wave_sum(acc[w]);
            if (lanei == 0) sh.red[c][0] = sum;
        }
    }
    __syncthreads();
    if (t < NR && t < sg.nr && ((FinTraits<KIND>::M >> sh.s[t].status) & 1u)) {
        double tot[NV];
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            double sum = 0.0;
            for (int w = 0; w < LaneState<KIND, NR>::R; ++w) sum += sh.red[a * NR + t][w];
            tot[a] = sum;
        }
        fin_scalar<KIND>(sh.s[t], tot);
    }
    __syncthreads();
    if (writer) {
        int* dst = reinterpret_cast<int*>(sg.st + (int64_t)out * sg.sst);
        for (int k = t; k < W; k += kBlock) stg(&dst[k], lds[k]);
    }
    LaneStat<NR> L;
#pragma unroll
    for (int k = 0; k < NR; ++k) L.s[k] = sh.s[k].status;
    L.nr = sg.nr;
    return L;
}
template <int KIND, int NR, typename T>
__device__ __forceinline__ LaneStat<NR> fold_states(const Seg<T>& sg, int in, int out, bool writer, LaneState<KIND, NR>& sh) {
    FoldLoads<FinTraits<KIND>::NV * NR> f;
    fold_begin<KIND, NR>(sg, in, f);
    return fold_end<KIND, NR>(sg, in, out, writer, f, sh);
}

// The states of a kernel that folds finaliser FOLD (copy IN to copy OUT), or
// of copy 0 where FOLD < 0: L their statuses, ST(k, f) field f of lane k.
#define FOLDED_STATES(FOLD, IN, OUT)                                                                      \
    __shared__ LaneState<(FOLD >= 0 ? FOLD : 0), (FOLD >= 0 ? NR : 1)> lst;                               \
    LaneStat<NR> L;                                                                                       \
    if constexpr (FOLD >= 0) L = fold_states<FOLD, NR>(sg, IN, OUT, lb == 0, lst);                        \
    else L = lane_stat<NR>(sg)
#define ST(k, f) (FOLD >= 0 ? lst.s[FOLD >= 0 ? (k) : 0].f : ldg(&sg.st[k].f))

template <typename T, int NR>
__global__ __launch_bounds__(kBlock) void k_init(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* b, T* x, T* r,
                                                 T* r0, T* p, T* v) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    double pv[1][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) pv[0][k] = 0.0;
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        auto bv = vload<T, NR>(b + i);
        typename VT<T, NR>::type zero = (typename VT<T, NR>::type)(T)0;
        vstore<T, NR>(r + i, bv);
        vstore<T, NR>(r0 + i, bv);
        vstore<T, NR>(x + i, zero);
        vstore<T, NR>(p + i, zero);
        vstore<T, NR>(v + i, zero);
#pragma unroll
        for (int k = 0; k < NR; ++k) pv[0][k] = (double)lane(bv, k) * (double)lane(bv, k);
    }
    block_partials<1, NR>(pv, sg.part, lb, sg.nblocks);
}

// RUN lanes: p = (p - w v) beta + r ; y = P^-1 p (fly: y is formed where it is read).
// UPDATE lanes (mixed): x64 += x32 / scale ; x32 = 0.
template <typename T, int NR, int FOLD>
__global__ __launch_bounds__(kBlock) void k_pupdate(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, T* p, const T* v,
                                                    const T* r, T* y, T* x, MixVec mv, int fly) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    FOLDED_STATES(FOLD, 2, 0);   // the loop test of the last iteration
    if (row >= sg.op.D || !seg_any(L, M_STAGE1)) return;
    const size_t i = (size_t)(sg.off + row * NR);
    if (seg_any(L, M_RUN)) {
        const uint8_t f = ldg(&sg.op.flag[row]);
        auto pv = vload<T, NR>(p + i);
        auto vv = vload<T, NR>(v + i);
        auto rv = vload<T, NR>(r + i);
        const unsigned run = L.of(M_RUN);
#pragma unroll
        for (int k = 0; k < NR; ++k) {   // a group owns kMaxNR states: every lane's load is valid
            const T beta = (T)ST(k, beta), w = (T)ST(k, omega);
            const T pk = (-w * lane(vv, k) + lane(pv, k)) * beta + lane(rv, k);   // p.Copy(-w,v,p); p*=beta; p+=r
            if ((run >> k) & 1u) setlane(pv, k, pk);
        }
        vstore<T, NR>(p + i, pv);
        if (!fly) vstore<T, NR>(y + i, prow_apply<T, NR>(prow_of(sg, row, f), prow_div(sg), pv));
    }
    if (std::is_same<T, float>::value && seg_any(L, M_UPDATE)) {
        auto xv = vload<T, NR>(x + i);
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (lane_in(L, k, M_UPDATE)) {
                double* xd = mv.x64 + lm_at(sg, k, row);
                stg(xd, ldg(xd) + (double)lane(xv, k) / ST(k, scale));
                setlane(xv, k, (T)0);
            }
        vstore<T, NR>(x + i, xv);
    }
}

// tmp = E x.  Rows are independent; a thread owns one row and all NR rhs.
// UPDATE lanes (mixed, first gather of the iteration): tmp64 = E64 x64.
// E x for the instance segments.  Tiles with an LDS list copy their x rows
// into LDS once and gather every stencil line from there; the other tiles
// (lists longer than the LDS, or operators without tiles) read x directly.
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) void k_egather(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* x, T* out,
                                                    unsigned lanes, MixVec mv, int copy) {
    typedef typename VT<T, NR>::type V;
    constexpr int LR = LdsTile<T, NR>::kRows;
    __shared__ V lx[LR > 0 ? LR : 1];
    const LdsRows<V> lrows{lx, LR > 0 ? LR : 1};
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    if (lb >= sg.nblocks) return;   // a launch with more tiles (k_egather_upd's) than row blocks
    const auto L = lane_stat<NR>(sg, lanes != 0, copy);
    if (lanes && !seg_any(L, lanes)) return;               // uniform per workgroup
    const bool main = !lanes || seg_any(L, lanes & ~M_UPDATE);
    const size_t i = (size_t)(sg.off + row * NR);
    const T* xb = x + sg.off;
    const int nu = (LR > 0 && main && sg.op.fmt == OP_TP && sg.op.tln) ? ldg(&sg.op.tln[lb]) : -1;
    if (nu >= 0 && nu <= LR) {
        // Loads in two rounds, each issued as soon as the previous one's
        // values are in: the tile's list entries with the row's flag,
        // exception record and weights (rows past the end read the last
        // row's, unused), all unconditional; then the listed x rows with the
        // row's LDS positions (a plain row's 16 line positions, or a moved
        // row's exception record and extra value, in one register array) or
        // an identity row's own x.  Then the LDS copy, the barrier and every
        // stencil line from LDS.
        FillIdx<LR> f;
        lds_fill_index<LR>(sg.op.tlr + ldg(&sg.op.tlo[lb]), nu, f);
        const bool act = row < sg.op.D;
        const int64_t rr = act ? row : sg.op.D - 1;
        const int64_t D = sg.op.D;
        const int e = ldg(&sg.op.exc[rr]);
        const uint8_t fl = ldg(&sg.op.flag[rr]);
        TpRow<T> m;
#pragma unroll
        for (int q = 0; q < 12; ++q) m.w[q] = ldg(&sg.op.tpw[q * D + rr]);
        const int kind = act ? ((fl & ROW_IDENTITY) ? 2 : (e < 0 ? 0 : 1)) : 3;
        ExcRow mx;   // kind 0: words 0..15 are the line positions; kind 1: the exception record
        T xval = (T)0;
        V xi = (V)(T)0;
        if (kind == 0) {
#pragma unroll
            for (int l = 0; l < 16; ++l) mx.pk[l] = ldg(&sg.op.tpl[l * D + row]);
        } else if (kind == 1) {   // rows an interior boundary moved
            exc_row_load(sg.op.tlx, e, mx);
            xval = ldg(&sg.op.xval[e]);
        } else if (kind == 2) {
            xi = vload<T, NR>(xb + (size_t)row * NR);
        }
        lds_fill_rows<T, NR, LR>(f, xb, lrows, [](const V& v, int) { return v; });
        if (act) {
            V acc = (V)(T)0;
#pragma unroll
            for (int l = 0; l < 16; ++l) m.p[l] = mx.pk[l];
            if (kind == 2) acc = xi;
            else if (kind == 0) egather_tp_lds<T, V, NR>(m, lrows, acc);
            else egather_grp_exc<T, V>(m.w, xval, mx, lrows, acc);
            vstore<T, NR>(out + i, acc);
        }
    } else if (main && row < sg.op.D) {
        vstore<T, NR>(out + i, erow<T, NR>(sg.op, row, xb, NR));
    }
}

// E x for launches whose every segment is in the ELL format: no LDS, and only
// this loop's registers. amdgpu_waves_per_eu(1, 2) lets the compiler keep a
// round's slots in registers (144 for one FP64 value, 107 for one FP32 value,
// 98 and 168 for four and eight FP64 values); left alone it schedules for eight
// waves a SIMD (68, 61, 60, 64 registers) and waits inside the rounds. 60
// iterations, milliseconds, with it and without: 64 slots a row, 41,870 rows,
// mixed x 1 2.63 and 3.17, FP64 x 8 6.15 and 7.31; 260,062 rows FP64 x 4 14.4
// and 15.9, x 8 24.2 and 34.2 (14.5 and 27.4 in k_egather); FP64 x 1 the same
// with both. 16 slots a round for two values: within 3% either way.
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_egather_ell(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* x,
                                                        T* out, unsigned lanes, MixVec, int copy) {
    typedef typename VT<T, NR>::type V;
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg, lanes != 0, copy);
    if (row >= sg.op.D || (lanes && !seg_any(L, lanes & ~M_UPDATE))) return;
    const T* xb = x + sg.off;
    V acc = (V)(T)0;
    if (ldg(&sg.op.flag[row]) & ROW_IDENTITY) acc = vload<T, NR>(xb + (size_t)row * NR);
    else egather_ell<NR == 1 ? 32 : 8, T, V, NR>(sg.op, row, xb, NR, acc);
    vstore<T, NR>(out + (size_t)(sg.off + row * NR), acc);
}

// FP64 gathers of the refinement lanes of FP32 segments: tmp64 = E64 x64 for
// every lane in an UPDATE status (a launch of its own beside the FP32
// gather, which then carries only FP32 work).  A lane's FP64 vectors are a
// run of D values, the one-right-hand-side layout, so block lb gathers tile
// lb of the operator's shared-stencil tiles for each such lane in turn;
// operators without tiles read x64 directly, a row per thread.
// x32: the solutions' FP32 parts are still to be added (fused iterations),
// null: pupdate has added them.
template <int NR>
__global__ __launch_bounds__(kBlock) void k_egather_upd(const Seg<float>* __restrict__ segs, const int* __restrict__ bseg,
                                                        MixVec mv, const float* x32) {
    constexpr int LR = GrpTile<double, 1>::kRows;
    static_assert(LR > 0, "FP64 shared-stencil tiles fit the LDS");
    __shared__ double lx[LR];
    const LdsRows<double> lrows{lx, LR};
    int lb;
    int64_t row;
    const Seg<float>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg);
    if (!seg_any(L, M_UPDATE)) return;   // uniform per workgroup
    if (sg.op64.ngt > 0) {
        if (lb >= sg.op64.ngt) return;
        bool first = true;
        for (int k = 0; k < sg.nr; ++k)
            if (lane_in(L, k, M_UPDATE)) {
                if (!first) __syncthreads();   // the previous lane's LDS reads are done
                first = false;
                const DstPlain<double, 1> ob{mv.tmp64 + lm_at(sg, k, 0)};
                if (x32) {
                    SrcX64<NR> src{mv.x64 + lm_at(sg, k, 0), x32 + sg.off + k, ldg(&sg.st[k].scale)};
                    egather_grp_tile<double, 1, LR>(sg.op64, lb, src, ob, lrows, [](auto&) { return true; });
                } else {
                    SrcPlain<double, 1, false> src{nullptr, mv.x64 + lm_at(sg, k, 0)};
                    egather_grp_tile<double, 1, LR>(sg.op64, lb, src, ob, lrows, [](auto&) { return true; });
                }
            }
        return;
    }
    if (row >= sg.op.D) return;
    for (int k = 0; k < sg.nr; ++k)
        if (lane_in(L, k, M_UPDATE))
            stg(&mv.tmp64[lm_at(sg, k, row)], erow<double, 1>(sg.op64, row, mv.x64 + lm_at(sg, k, 0), 1));
}

// E x for launches whose every segment has shared-stencil tiles: block lb of
// a segment takes its tile lb.  32 KB of LDS and at most 128 VGPRs, so four
// workgroups share a CU (a direct-read path for other segments, even out of
// line, made the FP32 x 8 kernel spill).
// FLY: x is p (or s) and the launch gathers y = P^-1 p (z = P^-1 s).
template <typename T, int NR, int WPE, bool FLY>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(WPE))) void k_egather_grp(
    const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* x, T* out, unsigned lanes, MixVec mv,
    int copy) {
    typedef typename VT<T, NR>::type V;
    constexpr int LR = GrpTile<T, NR>::kRows;
    static_assert(LR > 0, "shared-stencil tiles do not fit this value size");
    __shared__ V lx[LR];
    const LdsRows<V> lrows{lx, LR};
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg, lanes != 0, copy);
    if (lanes && !seg_any(L, lanes)) return;               // uniform per workgroup
    const bool main = !lanes || seg_any(L, lanes & ~M_UPDATE);
    if (!main || lb >= sg.op.ngt) return;
    SrcPlain<T, NR, FLY> src{&sg, x + sg.off};
    egather_grp_tile<T, NR, LR>(sg.op, lb, src, DstPlain<T, NR>{out + sg.off}, lrows, [](auto&) { return true; });
}

// E x for launches over operators of which some have shared-stencil tiles:
// those by their tiles, a row a thread of the others. 60 FP64 iterations of 3
// right-hand sides of an ELL operator of 19,021 rows and two others of 41,870
// and 41,185 / of 51,765, 115,734 and 113,404 rows: 4.6 / 7.2 ms; in a kernel
// each, which run one after the other, 5.5 / 7.9; every operator's rows read
// directly 5.5 / 9.7, tensor-product ones through row tiles 5.0 / 8.6.
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(CPMGPU_GROUP_WAVES_WIDE))) void k_egather_mixed(
    const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* x, T* out, unsigned lanes, MixVec, int copy) {
    typedef typename VT<T, NR>::type V;
    constexpr int LR = GrpTile<T, NR>::kRows;
    __shared__ V lx[LR];
    const LdsRows<V> lrows{lx, LR};
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg, lanes != 0, copy);
    if (lanes && !seg_any(L, lanes & ~M_UPDATE)) return;   // uniform per workgroup
    if (sg.op.ngt > 0) {
        if (lb >= sg.op.ngt) return;
        SrcPlain<T, NR, false> src{&sg, x + sg.off};
        egather_grp_tile<T, NR, LR>(sg.op, lb, src, DstPlain<T, NR>{out + sg.off}, lrows, [](auto&) { return true; });
    } else if (row < sg.op.D) {
        vstore<T, NR>(out + (size_t)(sg.off + row * NR), erow<T, NR>(sg.op, row, x + sg.off, NR));
    }
}

// out = A x from tmp = E x.  RED = 0: no reduction; 1: partial (other, out);
// 2: partials (out, out), (out, other).
// Mixed, RED = 1: UPDATE lanes r64 = b - A64 x64, partial (r64, r64).
// Mixed, RED = 2: RESCALE lanes partial (r32, r32) (rv32 = r32).
template <typename T, int NR, int RED>
__global__ __launch_bounds__(kBlock) void k_lfinish(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* x,
                                                    const T* tmp, T* out, const T* other, const T* rv32,
                                                    unsigned lanes, MixVec mv, int fly, int copy) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg, lanes != 0, copy);
    if (lanes && !seg_any(L, lanes)) return;   // uniform per segment
    constexpr int NV = RED == 2 ? 2 : 1;
    double pv[NV][NR];
#pragma unroll
    for (int a = 0; a < NV; ++a)
#pragma unroll
        for (int k = 0; k < NR; ++k) pv[a][k] = 0.0;
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        if (!lanes || seg_any(L, lanes & ~(M_UPDATE | M_RESCALE))) {
            typename VT<T, NR>::type res, ov;
            if (sg.op.fmt == OP_TP) {   // every load that waits on no other in one round
                TpLRow<T, NR> a;
                arow_tp_load<T, NR>(sg.op, row, x + i, a);
                if (RED > 0) ov = vload<T, NR>(other + i);
                res = arow_tp<T, NR>(sg, row, a, tmp + sg.off, NR, fly);   // fly: x is p or s
            } else {
                auto xv = vload<T, NR>(x + i);
                if (RED > 0) ov = vload<T, NR>(other + i);
                if (fly) xv = precond_row<T, NR>(sg, row, ldg(&sg.op.flag[row]), xv);
                res = arow<T, NR>(sg.op, sg.m, sg.n, row, xv, tmp + sg.off, NR);
            }
            vstore<T, NR>(out + i, res);
            if (RED > 0) {
#pragma unroll
                for (int k = 0; k < NR; ++k) {
                    const double rk = (double)lane(res, k);
                    if (RED == 1) {
                        pv[0][k] = (double)lane(ov, k) * rk;
                    } else {
                        pv[0][k] = rk * rk;
                        pv[NV - 1][k] = rk * (double)lane(ov, k);
                    }
                }
            }
        }
        if (std::is_same<T, float>::value && RED == 1 && seg_any(L, M_UPDATE)) {
#pragma unroll
            for (int k = 0; k < NR; ++k)   // constant indices keep pv in registers
                if (k < sg.nr && lane_in(L, k, M_UPDATE)) {
                    const size_t j = lm_at(sg, k, row);
                    const double ax =
                        arow<double, 1>(sg.op64, sg.m, sg.n, row, ldg(&mv.x64[j]), mv.tmp64 + lm_at(sg, k, 0), 1);
                    const double rk = ldg(&mv.b64[j]) - ax;
                    stg(&mv.r64[j], rk);
                    pv[0][k] = rk * rk;
                }
        }
        if (std::is_same<T, float>::value && RED == 2 && seg_any(L, M_RESCALE)) {
            auto rr = vload<T, NR>(rv32 + i);
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (lane_in(L, k, M_RESCALE)) {
                    const double rk = (double)lane(rr, k);
                    pv[0][k] = rk * rk;
                    pv[NV - 1][k] = 0.0;
                }
        }
    }
    if (RED > 0) block_partials<NV, NR>(pv, sg.part, lb, sg.nblocks);
}

// RUN lanes: s = r - alpha v ; z = P^-1 s (fly: z is formed where it is read).
// RESCALE lanes (mixed): r32 = r64 scale ; r0 = r32 ; p = v = 0.
template <typename T, int NR, int FOLD>
__global__ __launch_bounds__(kBlock) void k_supdate(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, T* r, T* v, T* s, T* z,
                                                    T* r0, T* p, MixVec mv, int fly) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    FOLDED_STATES(FOLD, 0, 1);   // alpha
    if (row >= sg.op.D || !seg_any(L, M_STAGE2)) return;
    const size_t i = (size_t)(sg.off + row * NR);
    const uint8_t f = ldg(&sg.op.flag[row]);
    auto rv = vload<T, NR>(r + i);
    auto vv = vload<T, NR>(v + i);
    if (seg_any(L, M_RUN)) {
        typename VT<T, NR>::type sv;
#pragma unroll
        for (int k = 0; k < NR; ++k) {   // a group owns kMaxNR states: every lane's load is valid
            const T a = (T)ST(k, alpha);
            setlane(sv, k, -a * lane(vv, k) + lane(rv, k));   // s.Copy(-alpha, v, r)
        }
        vstore<T, NR>(s + i, sv);
        if (!fly) vstore<T, NR>(z + i, prow_apply<T, NR>(prow_of(sg, row, f), prow_div(sg), sv));
    }
    if (std::is_same<T, float>::value && seg_any(L, M_RESCALE)) {
        auto r0v = vload<T, NR>(r0 + i);
        auto pv = vload<T, NR>(p + i);
#pragma unroll
        for (int k = 0; k < NR; ++k)
            if (lane_in(L, k, M_RESCALE)) {
                const T rk = (T)(ldg(&mv.r64[lm_at(sg, k, row)]) * ST(k, scale));
                setlane(rv, k, rk);
                setlane(r0v, k, rk);
                setlane(pv, k, (T)0);
                setlane(vv, k, (T)0);
            }
        vstore<T, NR>(r + i, rv);
        vstore<T, NR>(r0 + i, r0v);
        vstore<T, NR>(p + i, pv);
        vstore<T, NR>(v + i, vv);
    }
}

// Jacobi sweep `sweep` (>= 1) of RUN lanes: y += omega D^-1 (x - A y) on the
// rows below dofs, A y from tmp = E y (GeneralizedBiCGStabSystem.h:366-378).
// A y is formed here rather than stored by a launch of lfinish: a sweep is
// launch-bound on the geodesic problems that use it (10,906 rows, 2,000
// sweeps an application).
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) void k_jacobi(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg,
                                                   const T* x, const T* tmp, T* y, int sweep, int copy) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg, true, copy);
    if (sg.precond != 2 || sweep >= sg.precond_iters) return;
    if (row >= sg.op.D - sg.op.nD || !seg_any(L, M_RUN)) return;
    const size_t i = (size_t)(sg.off + row * NR);
    const uint8_t f = ldg(&sg.op.flag[row]);
    auto xv = vload<T, NR>(x + i);
    typename VT<T, NR>::type yv, av;
    if (sg.op.fmt == OP_TP) {
        TpLRow<T, NR> a;
        arow_tp_load<T, NR>(sg.op, row, y + i, a);
        yv = a.xv;
        av = arow_tp<T, NR>(sg, row, a, tmp + sg.off, NR, false);
    } else {
        yv = vload<T, NR>(y + i);
        av = arow<T, NR>(sg.op, sg.m, sg.n, row, yv, tmp + sg.off, NR);
    }
#pragma unroll
    for (int k = 0; k < NR; ++k)
        if (lane_in(L, k, M_RUN))
            setlane(yv, k, lane(yv, k) + (T)kJacobiOmega * diag_inverse(sg, row, f, (T)(lane(xv, k) - lane(av, k))));
    vstore<T, NR>(y + i, yv);
}

template <typename T, int NR, int FOLD>
__global__ __launch_bounds__(kBlock) void k_xrupdate(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, T* x, const T* y,
                                                     const T* z, T* r, const T* s, const T* t, const T* r0, int fly) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    FOLDED_STATES(FOLD, 1, 2);   // omega
    if (!seg_any(L, M_RUN)) return;
    double pv[2][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) { pv[0][k] = 0.0; pv[1][k] = 0.0; }
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        auto xv = vload<T, NR>(x + i);
        auto yv = vload<T, NR>(y + i);   // fly: p
        auto sv = vload<T, NR>(s + i);
        auto tv = vload<T, NR>(t + i);
        auto r0v = vload<T, NR>(r0 + i);
        const uint8_t f = ldg(&sg.op.flag[row]);
        // r is rewritten on every RUN lane: read only to keep the others
        const unsigned run = L.of(M_RUN);
        const bool all_run = run == (1u << NR) - 1u;
        typename VT<T, NR>::type rv = all_run ? (typename VT<T, NR>::type)(T)0 : vload<T, NR>(r + i);
        typename VT<T, NR>::type zv;
        if (fly) {   // y = P^-1 p, z = P^-1 s
            const PRow<T> pr = prow_of(sg, row, f);
            const bool div = prow_div(sg);
            yv = prow_apply<T, NR>(pr, div, yv);
            zv = prow_apply<T, NR>(pr, div, sv);
        } else {
            zv = vload<T, NR>(z + i);
        }
#pragma unroll
        for (int k = 0; k < NR; ++k) {   // a group owns kMaxNR states: every lane's load is valid
            if (!((run >> k) & 1u)) continue;
            const T a = (T)ST(k, alpha), w = (T)ST(k, omega);
            T xk = a * lane(yv, k) + lane(xv, k);   // x.Copy(alpha, y, x)
            xk = w * lane(zv, k) + xk;               // x.Copy(w, z, x)
            T rk = -w * lane(tv, k) + lane(sv, k);   // r.Copy(-w, t, s)
            setlane(xv, k, xk);
            setlane(rv, k, rk);
            pv[0][k] = (double)rk * (double)rk;
            pv[1][k] = (double)lane(r0v, k) * (double)rk;
        }
        vstore<T, NR>(x + i, xv);
        vstore<T, NR>(r + i, rv);
    }
    block_partials<2, NR>(pv, part_of<NR>(sg, FOLD >= 0 ? 2 : 0), lb, sg.nblocks);
}

// ---------------------------------------------------------------- fused iterations
// Iterations of launches whose gathers fill LDS from shared-stencil tiles and
// whose preconditioner is pointwise, with folded finalisers, in five launches
// instead of ten: pupdate and supdate have no launch of their own.
//
//   fgather<1>   (loop test) p formed in the LDS fill ; tmp = E P^-1 p
//   flfinish<1>  p formed again and stored ; v = A P^-1 p from tmp ; (r0, v)
//   fgather<2>   (alpha) s formed in the LDS fill ; tmp = E P^-1 s
//   flfinish<2>  s formed again ; t = A P^-1 s ; (t, t), (t, s)
//   fxrupdate    (omega) s formed again ; x, r ; (r, r), (r0, r)
//
// s is never stored.  A row's values are formed by the same operations
// wherever they are needed, so the results are the separate kernels' to the
// bit.  Every tile lists a row's neighbours too, so the fills read p, v and r
// (1.5 rows each per row) where the separate kernels read one vector: more
// bytes, fewer launches, which pays while an iteration is bound by its
// launches and their dependent loads rather than by its bytes (folding,
// capi.hip).  Refinement (mixed) lanes: x64 += x32 / scale is formed in
// k_egather_upd's fill and stored by flfinish<1>, the rescaled residual is
// stored by flfinish<2>.

// A finished segment of a launch over several: whether no lane's status in
// copy `in` is in mask, read before the kernel's own loads are issued. Its
// first workgroup still runs the finaliser and hands the states on. (Without
// it a finished system streams its vectors until the last one ends: eight FP64
// systems of 260,062 rows that end after 8 to 340 iterations took 75.0 ms.)
// The only segment of a launch is not looked at: its status would cost a
// memory latency before the first load.
template <int FOLD, int NR, typename T, typename LST>
__device__ __forceinline__ bool segment_done(const Seg<T>& sg, int in, int out, int lb, unsigned mask, LST& lst) {
    if (seg_any(lane_stat<NR>(sg, true, in), mask)) return false;
    if constexpr (FOLD >= 0)
        if (lb == 0) fold_states<FOLD, NR>(sg, in, out, true, lst);
    return true;
}

// PH 1: tmp = E P^-1 p, after the loop test (FOLD) ; PH 2: tmp = E P^-1 s, after alpha.
template <typename T, int NR, bool ONE, int WPE, int PH, int FOLD>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(WPE))) void k_fgather(
    const SegArg<T> segs, Vecs<T> w) {
    typedef typename VT<T, NR>::type V;
    constexpr int LR = GrpTile<T, NR>::kRows;
    __shared__ V lx[LR];
    __shared__ LaneState<(FOLD >= 0 ? FOLD : 0), (FOLD >= 0 ? NR : 1)> lst;
    const LdsRows<V> lrows{lx, LR};
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of<ONE>(segs, lb, row);
    if (lb >= sg.op.ngt) return;
    constexpr int in = PH == 1 && FOLD >= 0 ? 2 : 0, out = PH == 1 ? 0 : 1;
    if (!ONE && segment_done<FOLD, NR>(sg, in, out, lb, M_STAGE3, lst)) return;   // before the loop test: RUN or READY
    FoldLoads<FinTraits<(FOLD >= 0 ? FOLD : 0)>::NV * NR> f;
    if constexpr (FOLD >= 0) fold_begin<(FOLD >= 0 ? FOLD : 0), NR>(sg, in, f);
    typename std::conditional<PH == 1, SrcP<T, NR>, SrcS<T, NR>>::type src;
    src.sg = &sg;
    src.v = w.v + sg.off;
    src.r = w.r + sg.off;
    if constexpr (PH == 1) src.p = w.p + sg.off;
    egather_grp_tile<T, NR, LR>(sg.op, lb, src, DstPlain<T, NR>{w.tmp + sg.off}, lrows, [&](auto& q) {
        LaneStat<NR> L;
        if constexpr (FOLD >= 0) L = fold_end<(FOLD >= 0 ? FOLD : 0), NR>(sg, in, out, lb == 0, f, lst);
        else L = lane_stat<NR>(sg);
        if (!seg_any(L, M_RUN)) return false;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if constexpr (PH == 1) {
                q.beta[k] = (T)ST(k, beta);
                q.w[k] = (T)ST(k, omega);
            } else {
                q.alpha[k] = (T)ST(k, alpha);
            }
        }
        if constexpr (PH == 1) q.run = L.of(M_RUN);
        return true;
    });
}

template <typename T, int NR, bool ONE, int PH>
__global__ __launch_bounds__(kBlock) void k_flfinish(const SegArg<T> segs, Vecs<T> w,
                                                     MixVec mv) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of<ONE>(segs, lb, row);
    const KState* st = sg.st + (PH == 1 ? 0 : sg.sst);
    const auto L = lane_stat<NR>(sg, true, PH == 1 ? 0 : 1);
    if (!seg_any(L, PH == 1 ? M_STAGE1 : M_STAGE2)) return;   // uniform per segment
    constexpr int NV = PH;
    double pv[NV][NR];
#pragma unroll
    for (int a = 0; a < NV; ++a)
#pragma unroll
        for (int k = 0; k < NR; ++k) pv[a][k] = 0.0;
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        if (seg_any(L, M_RUN)) {
            TpLRow<T, NR> a;
            typename VT<T, NR>::type ov;   // r0 ; s
            if constexpr (PH == 1) {
                SrcP<T, NR> src;
                src.p = w.p;
                src.v = w.v;
                src.r = w.r;
                src.run = L.of(M_RUN);
#pragma unroll
                for (int k = 0; k < NR; ++k) {
                    src.beta[k] = (T)ldg(&st[k].beta);
                    src.w[k] = (T)ldg(&st[k].omega);
                }
                arow_tp_load<T, NR>(sg.op, row, w.r0 + i, a);
                const typename SrcP<T, NR>::Raw q{vload<T, NR>(w.p + i), vload<T, NR>(w.v + i), vload<T, NR>(w.r + i)};
                ov = a.xv;
                a.xv = src.direction(q);
                vstore<T, NR>(w.p + i, a.xv);
            } else {
                SrcS<T, NR> src;
#pragma unroll
                for (int k = 0; k < NR; ++k) src.alpha[k] = (T)ldg(&st[k].alpha);
                arow_tp_load<T, NR>(sg.op, row, w.r + i, a);
                const typename SrcS<T, NR>::Raw q{a.xv, vload<T, NR>(w.v + i)};
                ov = a.xv = src.residual(q);
            }
            const typename VT<T, NR>::type res = arow_tp<T, NR>(sg, row, a, w.tmp + sg.off, NR, true);
            vstore<T, NR>((PH == 1 ? w.v : w.t) + i, res);
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                const double rk = (double)lane(res, k);
                if (PH == 1) {
                    pv[0][k] = (double)lane(ov, k) * rk;
                } else {
                    pv[0][k] = rk * rk;
                    pv[NV - 1][k] = rk * (double)lane(ov, k);
                }
            }
        }
        if (std::is_same<T, float>::value && PH == 1 && seg_any(L, M_UPDATE)) {
            auto xv = vload<T, NR>(w.x + i);
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (lane_in(L, k, M_UPDATE)) {
                    const size_t j = lm_at(sg, k, row);
                    const double xd = ldg(&mv.x64[j]) + (double)lane(xv, k) / ldg(&st[k].scale);
                    stg(&mv.x64[j], xd);
                    setlane(xv, k, (T)0);
                    const double ax = arow<double, 1>(sg.op64, sg.m, sg.n, row, xd, mv.tmp64 + lm_at(sg, k, 0), 1);
                    const double rk = ldg(&mv.b64[j]) - ax;
                    stg(&mv.r64[j], rk);
                    pv[0][k] = rk * rk;
                }
            vstore<T, NR>(w.x + i, xv);
        }
        if (std::is_same<T, float>::value && PH == 2 && seg_any(L, M_RESCALE)) {
            auto rv = vload<T, NR>(w.r + i), r0v = vload<T, NR>(w.r0 + i), p = vload<T, NR>(w.p + i), v = vload<T, NR>(w.v + i);
#pragma unroll
            for (int k = 0; k < NR; ++k)
                if (lane_in(L, k, M_RESCALE)) {
                    const T rk = (T)(ldg(&mv.r64[lm_at(sg, k, row)]) * ldg(&st[k].scale));
                    setlane(rv, k, rk);
                    setlane(r0v, k, rk);
                    setlane(p, k, (T)0);
                    setlane(v, k, (T)0);
                    pv[0][k] = (double)rk * (double)rk;
                    pv[NV - 1][k] = 0.0;
                }
            vstore<T, NR>(w.r + i, rv);
            vstore<T, NR>(w.r0 + i, r0v);
            vstore<T, NR>(w.p + i, p);
            vstore<T, NR>(w.v + i, v);
        }
    }
    block_partials<NV, NR>(pv, sg.part, lb, sg.nblocks);
}

template <typename T, int NR, bool ONE>
__global__ __launch_bounds__(kBlock) void k_fxrupdate(const SegArg<T> segs, Vecs<T> w) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of<ONE>(segs, lb, row);
    __shared__ LaneState<FIN_OMEGA, NR> lst;
    if (!ONE && segment_done<FIN_OMEGA, NR>(sg, 1, 2, lb, M_RUN, lst)) return;
    FoldLoads<FinTraits<FIN_OMEGA>::NV * NR> f;
    fold_begin<FIN_OMEGA, NR>(sg, 1, f);
    typedef typename VT<T, NR>::type V;
    const bool in = row < sg.op.D;
    const size_t i = (size_t)(sg.off + (in ? row : 0) * NR);
    V xv = vload<T, NR>(w.x + i);
    const V pp = vload<T, NR>(w.p + i), vv = vload<T, NR>(w.v + i), tv = vload<T, NR>(w.t + i), r0v = vload<T, NR>(w.r0 + i);
    V rv = vload<T, NR>(w.r + i);
    const uint8_t fl = ldg(&sg.op.flag[in ? row : 0]);
    const auto L = fold_end<FIN_OMEGA, NR>(sg, 1, 2, lb == 0, f, lst);
    if (!seg_any(L, M_RUN)) return;
    double pv[2][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) { pv[0][k] = 0.0; pv[1][k] = 0.0; }
    if (in) {
        const unsigned run = L.of(M_RUN);
        const PRow<T> pr = prow_of(sg, row, fl);
        const bool div = prow_div(sg);
        V sv;
#pragma unroll
        for (int k = 0; k < NR; ++k) setlane(sv, k, -(T)lst.s[k].alpha * lane(vv, k) + lane(rv, k));
        const V yv = prow_apply<T, NR>(pr, div, pp), zv = prow_apply<T, NR>(pr, div, sv);   // y = P^-1 p, z = P^-1 s
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (!((run >> k) & 1u)) continue;
            const T a = (T)lst.s[k].alpha, om = (T)lst.s[k].omega;
            T xk = a * lane(yv, k) + lane(xv, k);
            xk = om * lane(zv, k) + xk;
            const T rk = -om * lane(tv, k) + lane(sv, k);
            setlane(xv, k, xk);
            setlane(rv, k, rk);
            pv[0][k] = (double)rk * (double)rk;
            pv[1][k] = (double)lane(r0v, k) * (double)rk;
        }
        vstore<T, NR>(w.x + i, xv);
        vstore<T, NR>(w.r + i, rv);
    }
    block_partials<2, NR>(pv, part_of<NR>(sg, 2), lb, sg.nblocks);
}

// ---------------------------------------------------------------- applies on callers' vectors
// An apply or an explicit step of a shared-stencil operator reads and writes
// the caller's vectors in place through the row permutation, its segment an
// argument of the launch: no packing launches before and after, no tables to
// copy.  (An apply of 1.05 M rows: two packs of 10 us beside a gather of 29
// and an lfinish of 11; of 10,906 rows: launches and copies.)

// Gather through a permutation: x and y in the caller's order, or tmp in the operator's.
template <int NR, typename Src, typename Dst>
__global__ __launch_bounds__(kBlock) void k_gather_caller(const SegArg<double> a, Src src, const Dst dst) {
    typedef typename VT<double, NR>::type V;
    constexpr int LR = GrpTile<double, NR>::kRows;
    __shared__ V lx[LR];
    const LdsRows<V> lrows{lx, LR};
    int lb;
    int64_t row;
    const Seg<double>& sg = seg_of<true>(a, lb, row);
    if (lb >= sg.op.ngt) return;
    egather_grp_tile<double, NR, LR>(sg.op, lb, src, dst, lrows, [](auto&) { return true; });
}

// y = m x + n (L_ii x + L_off tmp), x and y in the caller's order.
__global__ __launch_bounds__(kBlock) void k_lfinish_caller(const SegArg<double> a, const int* perm, const double* x,
                                                           const double* tmp, double* y) {
    int lb;
    int64_t row;
    const Seg<double>& sg = seg_of<true>(a, lb, row);
    if (row >= sg.op.D) return;
    const int c = ldg(perm + row);
    TpLRow<double, 1> r;
    arow_tp_load<double, 1>(sg.op, row, x + c, r);
    stg(y + c, arow_tp<double, 1>(sg, row, r, tmp, 1, false));
}

// Explicit diffusion of NR fields, z = x + c (Lfull x) (m = 1, n = c[k]), and
// for two fields the Gray-Scott reaction (ReactionDiffusionWithIBC.cpp:89-93)
// of their old values: fields in the caller's order, z interleaved in the
// operator's.  Identity rows take their Lfull rows from k_diffuse_held.
struct StepArg {
    const int* perm;
    const double* x[2];
    double c[2];
    double dt, F, k;
    double* z;
};
template <int NR>
__device__ __forceinline__ void diffuse_store(const StepArg& s, int64_t row, const double (&x)[NR], const double (&d)[NR]) {
    double z[NR];
#pragma unroll
    for (int f = 0; f < NR; ++f) z[f] = x[f] + s.c[f] * d[f];
    if constexpr (NR == 2) {
        z[0] += s.dt * (-x[0] * x[1] * x[1] + s.F * (1.0 - x[0]));
        z[1] += s.dt * (x[0] * x[1] * x[1] - (s.F + s.k) * x[1]);
    }
    typename VT<double, NR>::type v;
#pragma unroll
    for (int f = 0; f < NR; ++f) setlane(v, f, z[f]);
    vstore<double, NR>(s.z + (size_t)row * NR, v);
}
template <int NR>
__global__ __launch_bounds__(kBlock) void k_diffuse(const SegArg<double> a, const StepArg s) {
    int lb;
    int64_t row;
    const Seg<double>& sg = seg_of<true>(a, lb, row);
    const OpView<double>& op = sg.op;
    if (row >= op.D || (ldg(&op.flag[row]) & ROW_IDENTITY)) return;
    int c[7];
#pragma unroll
    for (int q = 0; q < 6; ++q) c[q] = ldg(&op.lcol[(int64_t)q * op.D + row]);
    c[6] = ldg(s.perm + row);
    double x[NR], d[NR];
#pragma unroll
    for (int f = 0; f < NR; ++f) x[f] = ldg(s.x[f] + c[6]);
#pragma unroll
    for (int q = 0; q < 6; ++q) c[q] = c[q] >= 0 ? ldg(s.perm + c[q]) : -1;
#pragma unroll
    for (int f = 0; f < NR; ++f) {
        double lo = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q) lo += (c[q] >= 0 ? op.loff : 0.0) * ldg(s.x[f] + (c[q] >= 0 ? c[q] : c[6]));
        d[f] = op.ldu * x[f] + lo;
    }
    diffuse_store<NR>(s, row, x, d);
}
template <int NR>
__global__ void k_diffuse_held(int64_t nh, int hw, const int* hrow, const int* hcol, const double* hval, const uint8_t* flag,
                               const StepArg s) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nh) return;
    const int r = hrow[k];
    if (!(flag[r] & ROW_IDENTITY)) return;
    double x[NR], d[NR];
    const int c = s.perm[r];
#pragma unroll
    for (int f = 0; f < NR; ++f) {
        x[f] = s.x[f][c];
        d[f] = 0.0;
    }
    for (int q = 0; q < hw; ++q) {
        const double v = hval[(int64_t)q * nh + k];
        const int h = s.perm[hcol[(int64_t)q * nh + k]];
#pragma unroll
        for (int f = 0; f < NR; ++f) d[f] += v * s.x[f][h];
    }
    diffuse_store<NR>(s, r, x, d);
}

// FP64 restart, BiCGStab.h:62-71: r = b - A x (A x already in ax), r0 = r; partial (r, r).
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) void k_restart(const Seg<T>* __restrict__ segs, const int* __restrict__ bseg, const T* b,
                                                    const T* ax, T* r, T* r0) {
    int lb;
    int64_t row;
    const Seg<T>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg);
    if (!seg_any(L, M_RESTART)) return;
    double pv[1][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) pv[0][k] = 0.0;
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        auto bv = vload<T, NR>(b + i);
        auto av = vload<T, NR>(ax + i);
        auto rv = vload<T, NR>(r + i);
        auto r0v = vload<T, NR>(r0 + i);
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (!lane_in(L, k, M_RESTART)) continue;
            T rk = lane(bv, k) - lane(av, k);
            setlane(rv, k, rk);
            setlane(r0v, k, rk);
            pv[0][k] = (double)rk * (double)rk;
        }
        vstore<T, NR>(r + i, rv);
        vstore<T, NR>(r0 + i, r0v);
    }
    block_partials<1, NR>(pv, sg.part, lb, sg.nblocks);
}

// ---------------------------------------------------------------- mixed precision start
// x64 = 0, r64 = b ; partial (b, b)
template <int NR>
__global__ __launch_bounds__(kBlock) void k_mx_start(const Seg<double>* __restrict__ segs, const int* __restrict__ bseg, const double* b,
                                                     double* x, double* r) {
    int lb;
    int64_t row;
    const Seg<double>& sg = seg_of(segs, bseg, lb, row);
    double pv[1][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) pv[0][k] = 0.0;
    if (row < sg.op.D) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const size_t j = lm_at(sg, k, row);
            const double bk = b[j];
            r[j] = bk;
            x[j] = 0.0;
            pv[0][k] = bk * bk;
        }
    }
    block_partials<1, NR>(pv, sg.part, lb, sg.nblocks);
}

// FP32 start of the lanes in ST_RESCALE: r32 = r64 * scale, r0 = r32,
// p = v = x32 = 0 ; partial (r32, r32).
template <int NR>
__global__ __launch_bounds__(kBlock) void k_mx_down(const Seg<double>* __restrict__ segs, const int* __restrict__ bseg, const double* r64,
                                                    float* r, float* r0, float* p, float* v, float* x) {
    int lb;
    int64_t row;
    const Seg<double>& sg = seg_of(segs, bseg, lb, row);
    const auto L = lane_stat<NR>(sg);
    if (!seg_any(L, M_RESCALE)) return;
    double pv[1][NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) pv[0][k] = 0.0;
    if (row < sg.op.D) {
        const size_t i = (size_t)(sg.off + row * NR);
        auto ro = vload<float, NR>(r + i);
        auto r0o = vload<float, NR>(r0 + i);
        auto po = vload<float, NR>(p + i);
        auto vo = vload<float, NR>(v + i);
        auto xo = vload<float, NR>(x + i);
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (!lane_in(L, k, M_RESCALE)) continue;
            const float rk = (float)(r64[lm_at(sg, k, row)] * ldg(&sg.st[k].scale));
            setlane(ro, k, rk);
            setlane(r0o, k, rk);
            setlane(po, k, 0.0f);
            setlane(vo, k, 0.0f);
            setlane(xo, k, 0.0f);
            pv[0][k] = (double)rk * (double)rk;
        }
        vstore<float, NR>(r + i, ro);
        vstore<float, NR>(r0 + i, r0o);
        vstore<float, NR>(p + i, po);
        vstore<float, NR>(v + i, vo);
        vstore<float, NR>(x + i, xo);
    }
    block_partials<1, NR>(pv, sg.part, lb, sg.nblocks);
}

// One workgroup per (segment, rhs lane): the sums of the producing kernel's
// partials, then the lane's scalar update; copy `in` of the states to copy
// `out` (the same where they are kept once).
template <typename T, int NR, int KIND>
__global__ __launch_bounds__(kBlock) void k_fin(const Seg<T>* __restrict__ segs, int in, int out) {
    constexpr int NV = FinTraits<KIND>::NV;
    constexpr unsigned M = FinTraits<KIND>::M;
    const Seg<T>& sg = segs[blockIdx.x / NR];
    const int k = (int)(blockIdx.x % NR);
    if (k >= sg.nr) return;
    const KState* src = sg.st + (int64_t)in * sg.sst + k;
    KState* dst = sg.st + (int64_t)out * sg.sst + k;
    __shared__ double red[NV][kBlock / 64];
    __shared__ KState s;
    double tot[NV];
    // the state's words, loaded with its status and the partials (loaded
    // after the sums they cost the launch another memory latency)
    constexpr int W = (int)(sizeof(KState) / 4);
    const int t = (int)threadIdx.x;
    const int word = t < W ? ldg(reinterpret_cast<const int*>(src) + t) : 0;
    const bool act = (M >> ldg(&src->status)) & 1u;   // same test the producer used
    if (!act && src == dst) return;
    if (t < W) reinterpret_cast<int*>(&s)[t] = word;
    if (act) part_totals<NV, NR>(sg, part_of<NR>(sg, in), k, red, tot);
    if (act && t == 0) fin_scalar<KIND>(s, tot);
    __syncthreads();
    if (t < W) stg(reinterpret_cast<int*>(dst) + t, reinterpret_cast<const int*>(&s)[t]);
}

__global__ void k_reset_states(KState* st, int n, double tol2, int max_it, double delta2) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    KState z = {};
    z.tol2 = tol2;
    z.max_it = max_it;
    z.delta2 = delta2;
    z.status = ST_RUN;
    st[i] = z;
}

void launch_reset_states(KState* st, int n, double tol2, int max_it, double delta2, hipStream_t s) {
    hipLaunchKernelGGL(k_reset_states, dim3((n + 255) / 256), dim3(256), 0, s, st, n, tol2, max_it, delta2);
}

// ---------------------------------------------------------------- launchers
#define LAUNCH(kern, ...) \
    hipLaunchKernelGGL(kern, dim3(c.nblocks), dim3(kBlock), 0, c.stream, c.segs, c.nseg == 1 ? nullptr : c.bseg, __VA_ARGS__)
// The refinement lanes' gathers run the same workgroups segment by segment.
#define LAUNCH_UPD(kern, ...)                                                                            \
    hipLaunchKernelGGL(kern, dim3(c.gblocks), dim3(kBlock), 0, c.stream, c.segs,                        \
                       c.nseg == 1 ? nullptr : c.bseg + c.nblocks + c.gblocks, __VA_ARGS__)
#define FIN_COPY(T, NR, KIND, IN, OUT) \
    hipLaunchKernelGGL((k_fin<T, NR, KIND>), dim3(c.nseg * NR), dim3(kBlock), 0, c.stream, c.segs, IN, OUT)
#define FIN(T, NR, KIND) FIN_COPY(T, NR, KIND, 0, 0)

// Waves per SIMD the shared-stencil gather is compiled for: four (128 VGPRs)
// where that does not spill, two (256 VGPRs) for FP32 x 4 and the FP64 shapes.
template <typename T, int NR>
struct GrpWaves {
    static constexpr int kWaves = (sizeof(T) == 4 && NR != 4) ? 4 : CPMGPU_GROUP_WAVES_WIDE;
};

// E gathers of launch c; fly: of P^-1 x (only by tiles).
template <typename T, int NR>
static void egather(const LaunchCfg<T>& c, bool fly, const T* x, T* out, unsigned lanes, const MixVec& mv, int copy) {
    const int* map = c.nseg == 1 ? nullptr : c.bseg + c.nblocks;   // the round-robin block map
    auto run = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(c.gblocks), dim3(kBlock), 0, c.stream, c.segs, map, x, out, lanes, mv, copy); };
    if constexpr (GrpTile<T, NR>::kRows > 0) {
        constexpr int W = GrpWaves<T, NR>::kWaves;
        if (c.gather == GATHER_TILES) return fly ? run(k_egather_grp<T, NR, W, true>) : run(k_egather_grp<T, NR, W, false>);
        if (c.gather == GATHER_MIXED) return run(k_egather_mixed<T, NR>);
    }
    if (c.gather == GATHER_ELL) return run(k_egather_ell<T, NR>);
    run(k_egather<T, NR>);
}

bool precond_fly() {
    const char* e = std::getenv("CPMGPU_PRECOND_FLY");
    return !(e && std::string(e) == "0");
}

template <typename T, int NR>
bool grp_gather(int ntiles) {
    if (GrpTile<T, NR>::kRows == 0 || ntiles <= 0) return false;
    const char* e = std::getenv("CPMGPU_GROUP_GATHER");
    return !(e && std::string(e) == "none");
}

template <typename T, int NR>
void Launch<T, NR>::init(const LaunchCfg<T>& c, const T* b, T* x, T* r, T* r0, T* p, T* v) {
    LAUNCH((k_init<T, NR>), b, x, r, r0, p, v);
    FIN(T, NR, FIN_INIT);
}
template <typename T, int NR>
template <bool FOLD>
void Launch<T, NR>::iteration(const LaunchCfg<T>& c, Vecs<T>& w, bool mixed, const MixVec& mv, bool first) {
    // fly: y = P^-1 p and z = P^-1 s are formed where they are read (the
    // gathers' LDS fills, lfinish, xrupdate) rather than stored: launches
    // whose gathers fill LDS from shared-stencil tiles and whose
    // preconditioner is pointwise (no Jacobi sweeps after the first)
    const bool fly = c.fly && c.jacobi_sweeps <= 1;
    const int fl = fly ? 1 : 0;
    const T* yp = fly ? w.p : w.y;   // the vector the first gather and lfinish read
    const T* zs = fly ? w.s : w.z;   // ... the second
    constexpr int kIter = std::is_same<T, float>::value ? FIN_ITER_MX : FIN_ITER64;
    constexpr int A = FOLD ? FIN_ALPHA : -1, O = FOLD ? FIN_OMEGA : -1, I = FOLD ? kIter : -1;
    const int s1 = FOLD ? 1 : 0;   // copy of the states after alpha
    if (FOLD && !first) LAUNCH((k_pupdate<T, NR, I>), w.p, w.v, w.r, w.y, w.x, mv, fl);
    else LAUNCH((k_pupdate<T, NR, -1>), w.p, w.v, w.r, w.y, w.x, mv, fl);
    for (int sw = 1; sw < c.jacobi_sweeps; ++sw) {   // y = P^-1 p, Jacobi sweeps after the first
        egather<T, NR>(c, false, w.y, w.tmp, M_RUN, MixVec{}, 0);
        LAUNCH((k_jacobi<T, NR>), w.p, w.tmp, w.y, sw, 0);
    }
    if constexpr (std::is_same<T, float>::value) {
        if (mixed) {   // FP32 lanes in the gather, refinement lanes' FP64 gathers in a launch of their own
            egather<T, NR>(c, fly, yp, w.tmp, M_RUN, mv, 0);
            LAUNCH_UPD((k_egather_upd<NR>), mv, (const float*)nullptr);
        } else {
            egather<T, NR>(c, fly, yp, w.tmp, M_STAGE1, mv, 0);
        }
    } else {
        egather<T, NR>(c, fly, yp, w.tmp, M_STAGE1, mv, 0);
    }
    LAUNCH((k_lfinish<T, NR, 1>), yp, w.tmp, w.v, w.r0, (const T*)nullptr, M_STAGE1, mv, fl, 0);
    if (!FOLD) FIN(T, NR, FIN_ALPHA);
    LAUNCH((k_supdate<T, NR, A>), w.r, w.v, w.s, w.z, w.r0, w.p, mv, fl);
    for (int sw = 1; sw < c.jacobi_sweeps; ++sw) {   // z = P^-1 s
        egather<T, NR>(c, false, w.z, w.tmp, M_RUN, MixVec{}, s1);
        LAUNCH((k_jacobi<T, NR>), w.s, w.tmp, w.z, sw, s1);
    }
    egather<T, NR>(c, fly, zs, w.tmp, M_RUN, mv, s1);
    LAUNCH((k_lfinish<T, NR, 2>), zs, w.tmp, w.t, w.s, (const T*)w.r, M_STAGE2, mv, fl, s1);
    if (!FOLD) FIN(T, NR, FIN_OMEGA);
    LAUNCH((k_xrupdate<T, NR, O>), w.x, yp, w.z, w.r, w.s, w.t, w.r0, fl);
    if (!FOLD) {
        if (mixed) FIN(T, NR, FIN_ITER_MX);
        else FIN(T, NR, FIN_ITER64);
    }
}
template <typename T, int NR>
void Launch<T, NR>::iterations(const LaunchCfg<T>& c, Vecs<T>& w, bool mixed, const MixVec& mv, int n) {
    if (!c.fold) {
        for (int i = 0; i < n; ++i) iteration<false>(c, w, mixed, mv, false);
        return;
    }
    bool fused = false;
    if constexpr (NR == 1) {
        fused = c.fuse && c.fly && c.jacobi_sweeps <= 1;
        constexpr int kIter = std::is_same<T, float>::value ? FIN_ITER_MX : FIN_ITER64;
        // waves per SIMD that the fused gathers are compiled for: as many as do not spill
        constexpr int WPE = sizeof(T) == 4 ? 4 : 2;
        auto run = [&](auto one) {
            constexpr bool ONE = decltype(one)::value;
            const SegArg<T> rows{c.segs, c.bseg, *c.first}, tiles{c.segs, c.bseg + c.nblocks, *c.first};
            const dim3 gb(c.gblocks), nb(c.nblocks), tb(kBlock);
            for (int i = 0; i < n; ++i) {
                if (i == 0) hipLaunchKernelGGL((k_fgather<T, NR, ONE, WPE, 1, -1>), gb, tb, 0, c.stream, tiles, w);
                else hipLaunchKernelGGL((k_fgather<T, NR, ONE, WPE, 1, kIter>), gb, tb, 0, c.stream, tiles, w);
                if constexpr (std::is_same<T, float>::value)
                    if (mixed) LAUNCH_UPD((k_egather_upd<NR>), mv, (const float*)w.x);
                hipLaunchKernelGGL((k_flfinish<T, NR, ONE, 1>), nb, tb, 0, c.stream, rows, w, mv);
                hipLaunchKernelGGL((k_fgather<T, NR, ONE, WPE, 2, FIN_ALPHA>), gb, tb, 0, c.stream, tiles, w);
                hipLaunchKernelGGL((k_flfinish<T, NR, ONE, 2>), nb, tb, 0, c.stream, rows, w, mv);
                hipLaunchKernelGGL((k_fxrupdate<T, NR, ONE>), nb, tb, 0, c.stream, rows, w);
            }
        };
        if (fused && c.nseg == 1) run(std::true_type{});
        else if (fused) run(std::false_type{});
    }
    for (int i = 0; !fused && i < n; ++i) iteration<true>(c, w, mixed, mv, i == 0);
    // the loop test of the last iteration, so that copy 0 is current
    if (mixed) FIN_COPY(T, NR, FIN_ITER_MX, 2, 0);
    else FIN_COPY(T, NR, FIN_ITER64, 2, 0);
}
template <typename T, int NR>
void Launch<T, NR>::restart(const LaunchCfg<T>& c, Vecs<T>& w) {
    const MixVec none{};
    egather<T, NR>(c, false, w.x, w.tmp, M_RESTART, none, 0);
    LAUNCH((k_lfinish<T, NR, 0>), w.x, w.tmp, w.t, (const T*)nullptr, (const T*)nullptr, M_RESTART, none, 0, 0);
    LAUNCH((k_restart<T, NR>), w.b, w.t, w.r, w.r0);
    FIN(T, NR, FIN_RESTART64);
}
template <typename T, int NR>
void Launch<T, NR>::apply(const LaunchCfg<T>& c, const T* x, T* tmp, T* y, unsigned lanes) {
    const MixVec none{};
    egather<T, NR>(c, false, x, tmp, lanes, none, 0);
    LAUNCH((k_lfinish<T, NR, 0>), x, tmp, y, (const T*)nullptr, (const T*)nullptr, lanes, none, 0, 0);
}

template <typename T>
void launch_lfinish_plain(const LaunchCfg<T>& c, const T* x, const T* tmp, T* out) {
    const MixVec none{};
    LAUNCH((k_lfinish<T, 1, 0>), x, tmp, out, (const T*)nullptr, (const T*)nullptr, 0u, none, 0, 0);
}
template void launch_lfinish_plain<double>(const LaunchCfg<double>&, const double*, const double*, double*);

static SegArg<double> caller_arg(const Seg<double>& sg) { return SegArg<double>{nullptr, nullptr, sg}; }

void launch_apply_caller(const Seg<double>& sg, const int* perm, const double* x, double* tmp, double* y, hipStream_t st) {
    const SegArg<double> a = caller_arg(sg);
    hipLaunchKernelGGL((k_gather_caller<1, SrcPerm, DstPlain<double, 1>>), dim3(sg.op.ngt), dim3(kBlock), 0, st, a,
                       SrcPerm{x, perm}, DstPlain<double, 1>{tmp});
    hipLaunchKernelGGL(k_lfinish_caller, dim3(sg.nblocks), dim3(kBlock), 0, st, a, perm, x, tmp, y);
}

void launch_extend_caller(const Seg<double>& sg, const int* perm, const double* x, double* y, hipStream_t st) {
    hipLaunchKernelGGL((k_gather_caller<1, SrcPerm, DstPerm<1, false>>), dim3(sg.op.ngt), dim3(kBlock), 0, st, caller_arg(sg),
                       SrcPerm{x, perm}, DstPerm<1, false>{{y}, {nullptr}, perm});
}

template <int NR>
void launch_step_caller(const Seg<double>& sg, const HeldRows& h, const int* perm, double* const* u, const double* const* g,
                        const double* coef, double dt, double F, double k, double* z, hipStream_t st) {
    const SegArg<double> a = caller_arg(sg);
    StepArg s{perm, {u[0], NR > 1 ? u[NR - 1] : nullptr}, {coef[0], coef[NR - 1]}, dt, F, k, z};
    hipLaunchKernelGGL(k_diffuse<NR>, dim3(sg.nblocks), dim3(kBlock), 0, st, a, s);
    if (h.nh > 0)
        hipLaunchKernelGGL(k_diffuse_held<NR>, dim3((unsigned)((h.nh + 255) / 256)), dim3(256), 0, st, h.nh, h.hw, h.row, h.col,
                           h.val, sg.op.flag, s);
    DstPerm<NR, true> dst;
    for (int f = 0; f < NR; ++f) {
        dst.out[f] = u[f];
        dst.g[f] = g[f];
    }
    dst.perm = perm;
    hipLaunchKernelGGL((k_gather_caller<NR, SrcPlain<double, NR, false>, DstPerm<NR, true>>), dim3(sg.op.ngt), dim3(kBlock), 0, st,
                       a, (SrcPlain<double, NR, false>{nullptr, z}), dst);
}
template void launch_step_caller<1>(const Seg<double>&, const HeldRows&, const int*, double* const*, const double* const*,
                                    const double*, double, double, double, double*, hipStream_t);
template void launch_step_caller<2>(const Seg<double>&, const HeldRows&, const int*, double* const*, const double* const*,
                                    const double*, double, double, double, double*, hipStream_t);

template <typename T, int NR>
void launch_egather(const LaunchCfg<T>& c, const T* x, T* out, bool fly) {
    const MixVec none{};
    const bool fl = fly && c.fly;
    egather<T, NR>(c, fl, x, out, 0u, none, 0);
}

template <int NR>
void MixedLaunch<NR>::start(const LaunchCfg<double>& c, const double* b, double* x64, double* r64) {
    LAUNCH((k_mx_start<NR>), b, x64, r64);
    FIN(double, NR, FIN_MX_START);
}
template <int NR>
void MixedLaunch<NR>::down(const LaunchCfg<double>& c, const double* r64, Vecs<float>& w) {
    LAUNCH((k_mx_down<NR>), r64, w.r, w.r0, w.p, w.v, w.x);
    FIN(double, NR, FIN_MX_INIT);
}

#define CPM_INST(T, NR) template struct Launch<T, NR>; template bool grp_gather<T, NR>(int); template void launch_egather<T, NR>(const LaunchCfg<T>&, const T*, T*, bool);
CPM_INST(double, 1) CPM_INST(double, 2) CPM_INST(double, 4) CPM_INST(double, 8)
CPM_INST(float, 1) CPM_INST(float, 2) CPM_INST(float, 4) CPM_INST(float, 8)
template struct MixedLaunch<1>;
template struct MixedLaunch<2>;
template struct MixedLaunch<4>;
template struct MixedLaunch<8>;

}  // namespace cpmgpu
