// Tensor-product execution format of operators built on a tube.
//
// The reference stores E as a general sparse matrix: 64 (column, value)
// pairs per row for p = 3 (Interpolation.cpp:204-225), i.e. 768 bytes of
// FP64 per row, read twice per BiCGStab iteration.  Every E row is in fact
// the tensor product of three 1-D barycentric weight vectors over the 4x4x4
// grid nodes b + (i, j, k).  Once the tube's rows are renumbered in
// lexicographic grid order (z fastest), the nodes b + (i, j, 0..3) of a
// stencil line are four consecutive rows, so a row is described by 16 line
// starts and 12 weights (160 bytes in FP64, 112 in FP32).  Where an interior
// boundary moved some of a row's columns (PoissonWithIBC MoveToIBCColumns) or
// appended the Dirichlet identity column, an exception record lists the
// columns of all 64 slots and the extra entry.
//
// The builder derives the format from the reference-order ELL rows and the
// rows' query points, and accepts an operator only if every row is
// reproduced exactly: the same columns and bit-identical FP64 values
// (w_z w_y) w_x, the order of Interpolation.cpp:95-107.  Otherwise the caller
// keeps the ELL format.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <atomic>
#include <climits>
#include <mutex>
#include <thread>
#include <cstdlib>
#include <string>
#include <vector>

#include "tube.h"
#include "krylov.h"

namespace cpmgpu {

namespace {

constexpr int kS = 4;   // p = 3

__global__ void k_lex_count(const int32_t* gidx, int64_t G, int* bcount) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int32_t v = i < G ? gidx[i] : -1;
    const int occ = (v >= 0 && v < kCand) ? 1 : 0;
    const unsigned long long m = __ballot(occ);
    __shared__ int ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) bcount[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

// Tube nodes in linear grid order: lex[pos] = tube index, rlex[tube index] = pos.
__global__ void k_lex_emit(const int32_t* gidx, int64_t G, const int* boff, int64_t N, int32_t* lex, int32_t* rlex,
                           int* err) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int32_t v = i < G ? gidx[i] : -1;
    const int occ = (v >= 0 && v < kCand) ? 1 : 0;
    const unsigned long long m = __ballot(occ);
    __shared__ int ws[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) ws[w] = __popcll(m);
    __syncthreads();
    if (!occ) return;
    int pos = boff[blockIdx.x];
    for (int k = 0; k < w; ++k) pos += ws[k];
    pos += __popcll(m & ((1ull << lane) - 1ull));
    if (pos >= N || v >= N) { atomicOr(err, 1); return; }
    lex[pos] = v;
    rlex[v] = pos;
}

struct TpArgs {
    int64_t D, N;
    const int* ecol;
    const double* eval;
    int ew;
    const int* lcol;
    const double* lval;
    int lw;
    const double* ldiag;
    const uint8_t* flag;
    const double* qpts;
    const int32_t* gidx;
    GridDev g;
    const int32_t* lex;
    const int32_t* rlex;
    double loff, ldu;
};

__device__ __forceinline__ int64_t to_internal(const TpArgs& a, int64_t c) { return c < a.N ? a.rlex[c] : c; }
__device__ __forceinline__ int64_t to_reference(const TpArgs& a, int64_t r) { return r < a.N ? a.lex[r] : r; }

// Error bits of the builder (any bit: the operator keeps the ELL format).
enum : int {
    TP_STENCIL = 2, TP_OUTSIDE = 4, TP_GAP = 8, TP_VALUE = 16, TP_TAIL = 32, TP_LVAL = 64, TP_LDIAG = 128
};

// Pass 1, one thread per internal row: line starts, weights, L columns, the
// row's moved-slot mask and its exception counts.
__global__ void k_tp_rows(TpArgs a, int* tpc, double* tpw64, float* tpw32, int* lcol_out, uint8_t* flag_out,
                          unsigned long long* mask_out, int* n_exc, int* n_mov, int* err) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= a.D) return;
    const int64_t D = a.D;
    const int64_t R = to_reference(a, r);
    const uint8_t f = a.flag[R];
    flag_out[r] = f;
    mask_out[r] = 0;
    n_exc[r] = 0;
    n_mov[r] = 0;
    if (f & ROW_IDENTITY) {
        for (int l = 0; l < kS * kS; ++l) tpc[l * D + r] = 0;
        for (int q = 0; q < 3 * kS; ++q) { tpw64[q * D + r] = 0.0; tpw32[q * D + r] = 0.0f; }
        for (int s = 0; s < 6; ++s) lcol_out[s * D + r] = -1;
        return;
    }
    if (f & ROW_NODIAG) { atomicOr(err, TP_LDIAG); return; }
    int64_t b[3];
    double w[3][5];
    if (!stencil_weights(a.g, kS - 1, a.qpts + 3 * R, b, w)) { atomicOr(err, TP_STENCIL); return; }
    const int64_t N1 = a.g.N1d;
    // sign of the row (ghost rows of Dirichlet curves are negated)
    double sign = 0.0;
    for (int s = 0; s < kS * kS * kS && sign == 0.0; ++s) {
        const int i = s / 16, j = (s / 4) % 4, k = s % 4;
        const double v = w[2][k] * w[1][j] * w[0][i];
        if (v == 0.0) continue;
        const double e = a.eval[s * D + R];
        sign = e == v ? 1.0 : (e == -v ? -1.0 : 2.0);
    }
    if (sign != 1.0 && sign != -1.0) { atomicOr(err, TP_VALUE); return; }
    unsigned long long mask = 0;
    int moved = 0;
    for (int i = 0; i < kS; ++i)
        for (int j = 0; j < kS; ++j) {
            int64_t c0 = -1;
            for (int k = 0; k < kS; ++k) {
                const int s = (i * kS + j) * kS + k;
                const int32_t gv = a.gidx[((b[0] + i) * N1 + (b[1] + j)) * N1 + (b[2] + k)];
                if (!(gv >= 0 && gv < a.N)) { atomicOr(err, TP_OUTSIDE); return; }
                const int64_t ci = a.rlex[gv];
                if (k == 0) c0 = ci;
                else if (ci != c0 + k) { atomicOr(err, TP_GAP); return; }
                const double v = w[2][k] * w[1][j] * (sign * w[0][i]);
                if (!(a.eval[s * D + R] == v)) { atomicOr(err, TP_VALUE); return; }
                if (a.ecol[s * D + R] != gv) { mask |= 1ull << s; ++moved; }
            }
            tpc[(i * kS + j) * D + r] = (int)c0;
        }
    for (int q = 0; q < kS; ++q) {
        const double wx = sign * w[0][q];
        tpw64[q * D + r] = wx;
        tpw64[(kS + q) * D + r] = w[1][q];
        tpw64[(2 * kS + q) * D + r] = w[2][q];
        tpw32[q * D + r] = (float)wx;
        tpw32[(kS + q) * D + r] = (float)w[1][q];
        tpw32[(2 * kS + q) * D + r] = (float)w[2][q];
    }
    bool extra = false;
    for (int s = kS * kS * kS; s < a.ew; ++s) {
        const double v = a.eval[s * D + R];
        const int c = a.ecol[s * D + R];
        if (v == 0.0 && c == R) continue;                 // padding
        if (s == kS * kS * kS) { extra = true; continue; }
        atomicOr(err, TP_TAIL);
        return;
    }
    for (int s = 0; s < 6; ++s) {
        int out = -1;
        if (s < a.lw) {
            const double v = a.lval[s * D + R];
            const int c = a.lcol[s * D + R];
            if (!(v == 0.0 && c == R)) {
                if (!(v == a.loff)) { atomicOr(err, TP_LVAL); return; }
                out = (int)to_internal(a, c);
            }
        }
        lcol_out[s * D + r] = out;
    }
    if (!(a.ldiag[R] == a.ldu)) { atomicOr(err, TP_LDIAG); return; }
    mask_out[r] = mask;
    n_exc[r] = (moved > 0 || extra) ? 1 : 0;
    n_mov[r] = moved;
}

// Pass 2: exception records (n_exc now holds exclusive offsets): the
// internal column of every slot, and the extra entry.
__global__ void k_tp_exc(TpArgs a, const int* exc_off, int64_t nexc_total, int* exc, int* ecx, int* xcol,
                         double* xval64, float* xval32) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= a.D) return;
    const int64_t D = a.D;
    const int64_t R = to_reference(a, r);
    const int e = exc_off[r];
    const int e_next = r + 1 < a.D ? exc_off[r + 1] : (int)nexc_total;
    if (e_next == e || (a.flag[R] & ROW_IDENTITY)) { exc[r] = -1; return; }
    exc[r] = e;
    for (int s = 0; s < kS * kS * kS; ++s) ecx[(int64_t)e * 64 + s] = (int)to_internal(a, a.ecol[s * D + R]);
    xcol[e] = -1;
    xval64[e] = 0.0;
    xval32[e] = 0.0f;
    if (a.ew > kS * kS * kS) {
        const int s = kS * kS * kS;
        const double v = a.eval[s * D + R];
        const int c = a.ecol[s * D + R];
        if (!(v == 0.0 && c == R)) {
            xcol[e] = (int)to_internal(a, c);
            xval64[e] = v;
            xval32[e] = (float)v;
        }
    }
}

__global__ void k_perm_full(const int32_t* lex, int64_t N, int64_t D, int32_t* perm) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < D) perm[r] = r < N ? lex[r] : (int32_t)r;
}

inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// The tube's lexicographic order, computed on first use (on the calling
// context's stream; the lock keeps concurrent first uses apart).
static void ensure_lex(Tube& t, Ctx* ctx) {
    static std::mutex lock;
    std::lock_guard<std::mutex> g(lock);
    if (t.lex.p) return;
    const hipStream_t st = ctx->stream;
    const int64_t G = t.N1d * t.N1d * t.N1d;
    const int64_t nb = (G + 255) / 256;
    Buffer bcount((size_t)(nb + 1) * 4), flags(64);
    Buffer lex((size_t)t.N * 4), rlex((size_t)t.N * 4);
    int* total = bcount.as<int>() + nb;
    HIPCHK(hipMemsetAsync(flags.p, 0, 64, st));
    hipLaunchKernelGGL(k_lex_count, dim3((unsigned)nb), dim3(256), 0, st, t.gidx.as<int32_t>(), G, bcount.as<int>());
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(256), 0, st, bcount.as<int>(), nb, total);
    hipLaunchKernelGGL(k_lex_emit, dim3((unsigned)nb), dim3(256), 0, st, t.gidx.as<int32_t>(), G, bcount.as<int>(),
                       t.N, lex.as<int32_t>(), rlex.as<int32_t>(), flags.as<int>());
    HIPCHK(hipGetLastError());
    int h[2] = {0, 0};
    HIPCHK(hipMemcpyAsync(&h[0], total, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(&h[1], flags.p, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (h[0] != t.N || h[1]) throw std::logic_error("tube index grid is inconsistent with the node list");
    t.lex = std::move(lex);
    t.rlex = std::move(rlex);
}

// CPMGPU_LDS_TILES selects the LDS tiles built with tensor-product
// operators: unset or "1", shared-stencil tiles; "rows", row tiles; "0", none
// (every gather reads x directly).
static int lds_tile_mode() {
    const char* e = std::getenv("CPMGPU_LDS_TILES");
    if (!e) return 2;
    const std::string v(e);
    return v == "0" ? 0 : v == "rows" ? 1 : 2;
}

// The slots' weights in slot order (grouped copy of tpw).
template <typename T>
__global__ void k_slot_weights(const T* tpw, int64_t D, const int* grow, int64_t S, T* gw) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    const int64_t r = grow[s];
#pragma unroll
    for (int q = 0; q < 12; ++q) gw[s * 12 + q] = tpw[q * D + r];
}

// Tensor-product rows on the host, for the row tiles' builder.
struct HostTp {
    int64_t D = 0, ne = 0;
    std::vector<uint8_t> flag;
    std::vector<int> tpc, exc, ecx, xcol;   // [16][D], [D], [ne][64], [ne]
    HostTp(int64_t D_, int64_t ne_, const Buffer& tpc_, const Buffer& exc_, const Buffer& ecx_, const Buffer& xcol_,
           const Buffer& flag_)
        : D(D_), ne(ne_), flag((size_t)D_), tpc((size_t)16 * D_), exc((size_t)D_),
          ecx((size_t)std::max<int64_t>(ne_, 1) * 64), xcol((size_t)std::max<int64_t>(ne_, 1)) {
        HIPCHK(hipMemcpy(flag.data(), flag_.p, flag.size(), hipMemcpyDeviceToHost));
        HIPCHK(hipMemcpy(tpc.data(), tpc_.p, tpc.size() * 4, hipMemcpyDeviceToHost));
        HIPCHK(hipMemcpy(exc.data(), exc_.p, exc.size() * 4, hipMemcpyDeviceToHost));
        if (ne > 0) {
            HIPCHK(hipMemcpy(ecx.data(), ecx_.p, (size_t)ne * 64 * 4, hipMemcpyDeviceToHost));
            HIPCHK(hipMemcpy(xcol.data(), xcol_.p, (size_t)ne * 4, hipMemcpyDeviceToHost));
        }
    }
};

// ---------------------------------------------------------------- shared-stencil tiles
// Built on the device.  Rows are sorted by the place of their stencil block
// (the first node of line (0, 0)) along a Hilbert curve through the grid, so
// that consecutive rows read a compact patch of x rows; identity rows come
// last.  Plain rows of one block are cut into items of up to kGrpRows rows,
// exception rows are single items beside the plain rows of their block, and
// identity rows are items of up to kGrpRows rows.  A tile is a run of items
// whose list of distinct x rows fits kGrpLdsRows.
//
// In the lexicographic order of the blocks a tile of 256 items is a strip one
// grid column wide; along the curve it is a patch, whose stencils overlap in
// both directions of the surface: 2.47 -> 1.53 list rows per row on the
// h = 0.02 torus (Morton order: 1.54).

constexpr uint32_t kIdentKey = 0xffffffffu;
constexpr int kMinTileItems = 8;
static_assert(kMinTileItems * 65 <= kGrpLdsRows, "the lists of this few items always fit");
static_assert((kGrpLdsRows & (kGrpLdsRows - 1)) == 0, "the lists are sorted by a bitonic network");
constexpr int kHash = 4 * 1024;        // open-addressing table of a tile's x rows (LDS)

// Position of (x, y, z), each below 2^10, along the Hilbert curve of the 2^10
// cube (Skilling, "Programming the Hilbert curve", AIP Conf. Proc. 707, 2004:
// the axes' Gray-code transform, then their bits interleaved).
__host__ __device__ inline uint32_t hilbert_index(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t v[3] = {x, y, z};
    for (uint32_t q = 1u << 9; q > 1; q >>= 1) {
        const uint32_t low = q - 1;
        for (int i = 0; i < 3; ++i) {
            if (v[i] & q) {
                v[0] ^= low;
            } else {
                const uint32_t t = (v[0] ^ v[i]) & low;
                v[0] ^= t;
                v[i] ^= t;
            }
        }
    }
    v[1] ^= v[0];
    v[2] ^= v[1];
    uint32_t t = 0;
    for (uint32_t q = 1u << 9; q > 1; q >>= 1)
        if (v[2] & q) t ^= q - 1;
    uint32_t h = 0;
    for (int b = 9; b >= 0; --b)
        for (int i = 0; i < 3; ++i) h = (h << 1) | (((v[i] ^ t) >> b) & 1u);
    return h;
}

// Sort key of each row: twice the curve position of its block, plus one for
// exception rows; identity rows sort last.
__global__ void k_grp_keys(int64_t D, const uint8_t* flag, const int* tpc, const int* exc, const int32_t* lex,
                           const int64_t* rec, int64_t N1d, uint32_t* key, int* row) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= D) return;
    row[r] = (int)r;
    if (flag[r] & ROW_IDENTITY) { key[r] = kIdentKey; return; }
    const int64_t l = rec[lex[tpc[r]]];   // line (0, 0) starts at a tube node
    const uint32_t z = (uint32_t)(l % N1d), y = (uint32_t)((l / N1d) % N1d), x = (uint32_t)(l / (N1d * N1d));
    key[r] = 2u * hilbert_index(x, y, z) + (exc[r] >= 0 ? 1u : 0u);
}

// First position of each run of equal keys (0 elsewhere), for a maximum scan.
__global__ void k_grp_heads(int64_t D, const uint32_t* key, int* head) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < D) head[i] = (i == 0 || key[i] != key[i - 1]) ? (int)i : 0;
}

__device__ __forceinline__ bool grp_exc_key(uint32_t k) { return k != kIdentKey && (k & 1u); }

// 1 where an item starts.
__global__ void k_grp_starts(int64_t D, const uint32_t* key, const int* head, int* start) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < D) start[i] = grp_exc_key(key[i]) || ((int)i - head[i]) % kGrpRows == 0;
}

// pos: exclusive sums of start; ifirst[item] = its first sorted row, ifirst[nitem] = D;
// counts: items, plain items, exception rows, identity rows, identity items.
__global__ void k_grp_items(int64_t D, const uint32_t* key, const int* start, const int* pos, int* ifirst, int* counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < D;
    const bool st = in && start[i];
    const bool id = in && key[i] == kIdentKey, ex = in && grp_exc_key(key[i]);
    if (st) ifirst[pos[i]] = (int)i;
    if (in && i == D - 1) {
        const int n = pos[i] + start[i];
        ifirst[n] = (int)D;
        counts[0] = n;
    }
    const unsigned long long p = __ballot(st && !id && !ex), e = __ballot(ex), d = __ballot(id), di = __ballot(id && st);
    if ((threadIdx.x & 63) == 0) {
        if (p) atomicAdd(&counts[1], __popcll(p));
        if (e) atomicAdd(&counts[2], __popcll(e));
        if (d) atomicAdd(&counts[3], __popcll(d));
        if (di) atomicAdd(&counts[4], __popcll(di));
    }
}

struct GrpSrc {
    int64_t D;
    int nitem;
    const uint32_t* key;    // sorted
    const int* row;         // rows in sorted order
    const int* ifirst;      // [nitem + 1]
    const uint8_t* flag;
    const int* tpc;
    const int* exc;
    const int* ecx;
    const int* xcol;
};

// f(c) for the x rows that thread t's share of items [i0, i1) reads: 16
// threads an item, one stencil line each.
template <typename F>
__device__ __forceinline__ void grp_columns(const GrpSrc& s, int i0, int i1, F&& f) {
    for (int u = (int)threadIdx.x; u < (i1 - i0) * 16; u += (int)blockDim.x) {
        const int p = s.ifirst[i0 + (u >> 4)], l = u & 15;
        const uint32_t k = s.key[p];
        if (k == kIdentKey) continue;
        const int64_t r = s.row[p];
        if (grp_exc_key(k)) {
            const int e = s.exc[r];
            for (int q = 0; q < 4; ++q) f(s.ecx[(int64_t)e * 64 + 4 * l + q]);
            if (l == 0 && s.xcol[e] >= 0) f(s.xcol[e]);
        } else {
            const int c = s.tpc[(int64_t)l * s.D + r];
            for (int q = 0; q < 4; ++q) f(c + q);
        }
    }
}

// Distinct x rows of items [i0, i1) into the hash table `tab` (all -1 outside
// the entries); returns their number, or more than kGrpLdsRows when they do
// not fit (the table is then incomplete).  Threads stop inserting past the
// limit, so at most kGrpLdsRows + blockDim entries are ever taken.
__device__ int grp_collect(const GrpSrc& s, int i0, int i1, int* tab, int* count) {
    for (int k = (int)threadIdx.x; k < kHash; k += (int)blockDim.x) tab[k] = -1;
    if (threadIdx.x == 0) *count = 0;
    __syncthreads();
    grp_columns(s, i0, i1, [&](int c) {
        if (*(volatile int*)count > kGrpLdsRows) return;
        unsigned h = ((unsigned)c * 2654435761u) >> 20;
        for (;;) {
            const int old = atomicCAS(&tab[h & (kHash - 1)], -1, c);
            if (old == c) return;
            if (old == -1) { atomicAdd(count, 1); return; }
            ++h;
        }
    });
    __syncthreads();
    const int n = *count;
    __syncthreads();
    return n;
}
static_assert(kGrpLdsRows + 2 * kBlock < kHash, "the table always keeps empty entries, so every probe ends");

// One workgroup per run of `m` items: the number of equal parts (1, 2, 4 ..)
// the run is cut into so that every part's list fits.
__global__ __launch_bounds__(kBlock) void k_grp_count(GrpSrc s, int m, int* parts) {
    __shared__ int tab[kHash];
    __shared__ int count;
    const int i0 = (int)blockIdx.x * m, i1 = min(s.nitem, i0 + m);
    int sz = m;
    for (int a = i0; a < i1;) {
        const int n = grp_collect(s, a, min(i1, a + sz), tab, &count);
        if (n > kGrpLdsRows && sz > kMinTileItems) {   // start over with parts of half the size
            sz >>= 1;
            a = i0;
            continue;
        }
        a += sz;
    }
    if (threadIdx.x == 0) parts[blockIdx.x] = m / sz;
}

struct GrpOut {
    int64_t nip;            // item places
    int* gofs;
    int* grow;
    int* gpl;
    int* gln;
    int* glr;
    int16_t* glx;
    int* total_list;        // rows in all lists
    int* err;
};

// One workgroup per run: the tiles of its parts (first[run] is the first).
// A tile's items are placed by kind and row count (plain items with more rows
// first, then exception rows, then identity rows), so that a wave's threads
// take one path of the gather and end together; which thread takes an item
// changes no row's arithmetic.
__global__ __launch_bounds__(kBlock) void k_grp_tiles(GrpSrc s, GrpOut o, int m, const int* first, int nruns, int ntiles) {
    __shared__ int tab[kHash];
    __shared__ int list[kGrpLdsRows];
    __shared__ int count, used;
    __shared__ int place[kBlock];      // item at a place
    __shared__ int rows[kBlock];       // its rows, then their exclusive sums
    __shared__ int ccount[4][kGrpRows + 3];
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const int i0 = (int)blockIdx.x * m, i1 = min(s.nitem, i0 + m);
    const int t0 = first[blockIdx.x], t1 = (int)blockIdx.x + 1 < nruns ? first[blockIdx.x + 1] : ntiles;
    const int sz = m / (t1 - t0);
    for (int tile = t0; tile < t1; ++tile) {
        const int a = min(i1, i0 + (tile - t0) * sz), b = min(i1, a + sz), ni = b - a;
        const int nu = grp_collect(s, a, b, tab, &count);
        if (nu > kGrpLdsRows) {   // uniform (the parts were cut so that none is)
            if (t == 0) atomicOr(o.err, 1);
            return;
        }
        // the table's entries, sorted (unused places sort last)
        if (t == 0) used = 0;
        for (int k = t; k < kGrpLdsRows; k += kBlock) list[k] = INT_MAX;
        __syncthreads();
        for (int k = t; k < kHash; k += kBlock)
            if (tab[k] >= 0) list[atomicAdd(&used, 1)] = tab[k];
        __syncthreads();
        for (int w = 2; w <= kGrpLdsRows; w <<= 1)
            for (int h = w >> 1; h > 0; h >>= 1) {
                for (int k = t; k < kGrpLdsRows / 2; k += kBlock) {
                    const int p = 2 * k - (k & (h - 1)), q = p + h;
                    const int u = list[p], v = list[q];
                    if ((u > v) == ((p & w) == 0)) {
                        list[p] = v;
                        list[q] = u;
                    }
                }
                __syncthreads();
            }
        auto pos = [&](int c) {   // index of c in the list
            int lo = 0, hi = nu;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (list[mid] < c) lo = mid + 1;
                else hi = mid;
            }
            if (lo >= nu || list[lo] != c) atomicOr(o.err, 2);
            return lo;
        };
        // list entries, the unused places repeating the last (the gather reads every place without
        // a branch); bit 30: P^-1 leaves the row as it is (identity or no-diagonal row)
        for (int k = t; k < kGrpLdsRows; k += kBlock) {
            int c = nu > 0 ? list[min(k, nu - 1)] : 0;
            if (nu > 0 && (s.flag[c] & (ROW_IDENTITY | ROW_NODIAG))) c |= 1 << 30;
            o.glr[(int64_t)tile * kGrpLdsRows + k] = c;
        }
        if (t == 0) {
            o.gln[tile] = nu;
            atomicAdd(o.total_list, nu);
        }
        // places: a stable counting sort of the items by class
        int cls = -1, n = 0, p0 = 0;
        if (t < ni) {
            p0 = s.ifirst[a + t];
            n = s.ifirst[a + t + 1] - p0;
            const uint32_t k = s.key[p0];
            cls = k == kIdentKey ? kGrpRows + 1 : (k & 1u) ? kGrpRows : kGrpRows - n;
        }
        int before = 0;
        for (int c = 0; c < kGrpRows + 2; ++c) {
            const unsigned long long same = __ballot(cls == c);
            if (cls == c) before = __popcll(same & ((1ull << lane) - 1ull));
            if (lane == 0) ccount[wave][c] = __popcll(same);
        }
        rows[t] = 0;
        __syncthreads();
        if (t < ni) {
            for (int c = 0; c < cls; ++c)
                for (int w = 0; w < 4; ++w) before += ccount[w][c];
            for (int w = 0; w < wave; ++w) before += ccount[w][cls];
            place[before] = t;
            rows[before] = n;
        }
        __syncthreads();
        int sum = rows[t];   // inclusive sums
        for (int d = 1; d < kBlock; d <<= 1) {
            const int add = t >= d ? rows[t - d] : 0;
            __syncthreads();
            sum += add;
            rows[t] = sum;
            __syncthreads();
        }
        // the items in place order: slots, rows, positions
        const int64_t qp = (int64_t)tile * kBlock + t;
        const int base = s.ifirst[a];
        int word[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (t < ni) {
            const int it = a + place[t];
            const int q0 = s.ifirst[it], cnt = s.ifirst[it + 1] - q0;
            const int slot = base + rows[t] - cnt;
            const uint32_t k = s.key[q0];
            const int kind = k == kIdentKey ? 2 : (k & 1u) ? 1 : 0;
            o.gofs[qp] = slot | (kind << kGrpKindShift);
            const int64_t r = s.row[q0];
            for (int g = 0; g < cnt; ++g) o.grow[slot + g] = s.row[q0 + g];
            if (kind == 0) {
#pragma unroll
                for (int l = 0; l < 16; ++l) {
                    const int p = pos(s.tpc[(int64_t)l * s.D + r]);
                    if (p + 3 >= nu) atomicOr(o.err, 4);
                    word[l >> 1] |= (int)((unsigned)p << (16 * (l & 1)));
                }
            } else if (kind == 1) {
                const int e = s.exc[r];
                for (int q = 0; q < 64; ++q) o.glx[(int64_t)e * kExcPos + q] = (int16_t)pos(s.ecx[(int64_t)e * 64 + q]);
                const int xc = s.xcol[e];
                o.glx[(int64_t)e * kExcPos + 64] = xc >= 0 ? (int16_t)pos(xc) : (int16_t)-1;
                for (int q = 65; q < kExcPos; ++q) o.glx[(int64_t)e * kExcPos + q] = -1;
                word[0] = e;   // read with the line positions, a step before the record
            } else {
#pragma unroll
                for (int g = 0; g < kGrpRows; ++g) word[g] = g < cnt ? s.row[q0 + g] : -1;
            }
        } else {
            o.gofs[qp] = s.ifirst[b] | (3 << kGrpKindShift);   // an empty place
        }
#pragma unroll
        for (int h = 0; h < 8; ++h) o.gpl[(int64_t)h * o.nip + qp] = word[h];
        __syncthreads();
    }
    if (t1 == ntiles && t == 0) o.gofs[o.nip] = (int)s.D;
}

// Exclusive sums of the runs' parts (one workgroup; a few thousand runs at most per million rows).
__global__ void k_grp_first(const int* parts, int n, int* first, int* total) {
    __shared__ int sums[256];
    const int t = (int)threadIdx.x, per = (n + 255) / 256, b = min(n, t * per), e = min(n, b + per);
    int s = 0;
    for (int k = b; k < e; ++k) s += parts[k];
    sums[t] = s;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
        const int add = t >= d ? sums[t - d] : 0;
        __syncthreads();
        sums[t] += add;
        __syncthreads();
    }
    int run = sums[t] - s;
    for (int k = b; k < e; ++k) {
        first[k] = run;
        run += parts[k];
    }
    if (t == 255) *total = sums[255];
}

// Items per tile: 256, one per thread of a gather workgroup (the most x rows
// shared: 1.53 list rows per row, 1.90 with 128, 2.48 with 64), also where
// that leaves fewer workgroups than the GPU has CUs; 128 for operators of less
// than 64 such tiles.  Measured with 256 / 128 / 64 items: FP64 solve of
// 260,000 rows 20.5 / 23.2 / 26.2 ms, of 41,870 rows 4.38 / 4.33 / 4.39 ms,
// batch of six tubes of 57,000 rows in all 5.20 / 5.01 / 4.99 ms.  Small
// operators alone would take 64 (an apply of 10,906 rows 7.67 / 7.32 / 7.14 us,
// their solves the same), but their workgroups are three quarters empty, and
// many together pay for it: 60 iterations of 128 FP64 systems of 10,906 rows
// 10.1 / 11.1 / 13.7 ms (row tiles 11.5), of 240 of 3,190 6.2 / 7.0 / 7.9 (7.1).
static int group_tile_items(int nitem) {
    // CPMGPU_GROUP_ITEMS: items per tile, rounded down to a power of two (measurements); read once per process
    static const int forced = [] {
        const char* e = std::getenv("CPMGPU_GROUP_ITEMS");
        int m = kBlock;
        while (e && m > kMinTileItems && m > std::atoi(e)) m >>= 1;
        return e ? m : 0;
    }();
    if (forced) return forced;
    return nitem < kBlock * 64 ? kBlock / 2 : kBlock;
}

// Returns false (nothing built) for operators whose slots exceed gofs's bits.
static bool build_group_tiles(Op& op, const Tube& tube) {
    const int64_t D = op.D;
    if (D >= (int64_t)kGrpOfsMask) return false;
    const hipStream_t st = op.ctx->stream;
    const dim3 gb(nblk(D)), tb(256);
    Buffer key((size_t)D * 8), row((size_t)D * 8), head((size_t)D * 4), start((size_t)D * 4), pos((size_t)D * 4),
        ifirst((size_t)(D + 1) * 4), small(256);
    uint32_t *k0 = key.as<uint32_t>(), *k1 = k0 + D;
    int *r0 = row.as<int>(), *r1 = r0 + D;
    int* counts = small.as<int>();   // [0..4] items by kind, [5] list rows, [6] errors, [7] tiles
    HIPCHK(hipMemsetAsync(small.p, 0, 256, st));
    hipLaunchKernelGGL(k_grp_keys, gb, tb, 0, st, D, op.flag.as<uint8_t>(), op.tpc.as<int>(), op.exc.as<int>(),
                       tube.lex.as<int32_t>(), tube.rec.as<int64_t>(), tube.N1d, k0, r0);
    size_t sort_bytes = 0, max_bytes = 0, sum_bytes = 0;
    HIPCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, k0, k1, r0, r1, (int)D, 0, 32, st));
    HIPCHK(hipcub::DeviceScan::InclusiveScan(nullptr, max_bytes, head.as<int>(), head.as<int>(), hipcub::Max(), (int)D, st));
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, sum_bytes, start.as<int>(), pos.as<int>(), (int)D, st));
    Buffer tmp(std::max({sort_bytes, max_bytes, sum_bytes, (size_t)256}));
    HIPCHK(hipcub::DeviceRadixSort::SortPairs(tmp.p, sort_bytes, k0, k1, r0, r1, (int)D, 0, 32, st));
    hipLaunchKernelGGL(k_grp_heads, gb, tb, 0, st, D, k1, pos.as<int>());
    HIPCHK(hipcub::DeviceScan::InclusiveScan(tmp.p, max_bytes, pos.as<int>(), head.as<int>(), hipcub::Max(), (int)D, st));
    hipLaunchKernelGGL(k_grp_starts, gb, tb, 0, st, D, k1, head.as<int>(), start.as<int>());
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(tmp.p, sum_bytes, start.as<int>(), pos.as<int>(), (int)D, st));
    hipLaunchKernelGGL(k_grp_items, gb, tb, 0, st, D, k1, start.as<int>(), pos.as<int>(), ifirst.as<int>(), counts);
    HIPCHK(hipGetLastError());
    int h[8] = {0};
    HIPCHK(hipMemcpyAsync(h, counts, 32, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    const int nitem = h[0];
    const int m = group_tile_items(nitem);
    const int nruns = (nitem + m - 1) / m;
    GrpSrc src{D, nitem, k1, r1, ifirst.as<int>(), op.flag.as<uint8_t>(), op.tpc.as<int>(), op.exc.as<int>(),
               op.ecx.as<int>(), op.xcol.as<int>()};
    // start and pos are free again: parts of each run, first tile of each run
    hipLaunchKernelGGL(k_grp_count, dim3((unsigned)nruns), dim3(kBlock), 0, st, src, m, start.as<int>());
    hipLaunchKernelGGL(k_grp_first, dim3(1), dim3(256), 0, st, start.as<int>(), nruns, pos.as<int>(), counts + 7);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(h, counts, 32, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    const int64_t ngt = h[7], nip = ngt * kBlock;
    Buffer gofs((size_t)(nip + 1) * 4), grow((size_t)D * 4), gpl((size_t)8 * nip * 4), gln((size_t)ngt * 4),
        glr((size_t)ngt * kGrpLdsRows * 4), glx((size_t)std::max<int64_t>(op.nexc, 1) * kExcPos * 2),
        gw64((size_t)12 * D * 8), gw32((size_t)12 * D * 4);
    GrpOut out{nip, gofs.as<int>(), grow.as<int>(), gpl.as<int>(), gln.as<int>(), glr.as<int>(), glx.as<int16_t>(),
               counts + 5, counts + 6};
    hipLaunchKernelGGL(k_grp_tiles, dim3((unsigned)nruns), dim3(kBlock), 0, st, src, out, m, pos.as<int>(), nruns, (int)ngt);
    hipLaunchKernelGGL(k_slot_weights<double>, gb, tb, 0, st, op.tpw64.as<double>(), D, grow.as<int>(), D, gw64.as<double>());
    hipLaunchKernelGGL(k_slot_weights<float>, gb, tb, 0, st, op.tpw32.as<float>(), D, grow.as<int>(), D, gw32.as<float>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(h, counts, 32, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (h[6]) throw std::logic_error("shared-stencil tiles: a list or position is out of range");
    op.gofs = std::move(gofs);
    op.grow = std::move(grow);
    op.gpl = std::move(gpl);
    op.gln = std::move(gln);
    op.glr = std::move(glr);
    op.glx = std::move(glx);
    op.gw64 = std::move(gw64);
    op.gw32 = std::move(gw32);
    op.grp_items = nitem;
    op.grp_items0 = h[1];
    op.grp_exc = h[2];
    op.grp_ident = h[3];
    op.grp_ident_items = h[4];
    op.grp_rows0 = D - h[2] - h[3];
    op.grp_list = h[5];
    op.ngt = (int)ngt;
    op.nitem = (int)nip;
    op.nslot = D;
    return true;
}

// LDS tiles: for every block of kBlock internal rows, the sorted distinct x
// rows its E rows read, and for each stencil line the position of its first
// row in that list (the line's four rows are consecutive integers, hence
// consecutive in the list); rows with an exception record get the positions
// of their 64 columns and of the extra entry instead (tlx, kExcPos per
// record, -1 = no extra entry).  Tiles whose list would exceed kLdsRows keep
// reading x directly (tln = -1).
static void build_lds_tiles(Op& op, const HostTp& h) {
    const int64_t D = h.D, ne = h.ne;
    const std::vector<uint8_t>& hf = h.flag;
    const std::vector<int>&hc = h.tpc, &he = h.exc, &hx = h.ecx, &hxc = h.xcol;
    const int64_t ntiles = (D + kBlock - 1) / kBlock;
    std::vector<int> tln((size_t)ntiles), tlo((size_t)ntiles), tlr;
    std::vector<int16_t> tpl((size_t)kS * kS * D, 0), tlx((size_t)std::max<int64_t>(ne, 1) * kExcPos, -1);
    std::vector<std::vector<int>> lists((size_t)ntiles);
    // tiles are independent: host threads over contiguous tile ranges
    const int nth = (int)std::max<int64_t>(1, std::min<int64_t>({16, ntiles, (int64_t)std::max(1u, std::thread::hardware_concurrency())}));
    auto parallel = [&](auto&& body) {
        std::vector<std::thread> th;
        for (int w = 0; w < nth; ++w)
            th.emplace_back([&, w] {
                for (int64_t tile = ntiles * w / nth; tile < ntiles * (w + 1) / nth; ++tile) body(tile);
            });
        for (auto& x : th) x.join();
    };
    // 1. each tile's sorted distinct x rows
    parallel([&](int64_t tile) {
        const int64_t r0 = tile * kBlock, r1 = std::min<int64_t>(D, r0 + kBlock);
        std::vector<int>& u = lists[(size_t)tile];
        for (int64_t r = r0; r < r1; ++r) {
            const int e = he[(size_t)r];
            if (e >= 0) {
                for (int s = 0; s < 64; ++s) u.push_back(hx[(size_t)e * 64 + s]);
                if (hxc[(size_t)e] >= 0) u.push_back(hxc[(size_t)e]);
                continue;
            }
            for (int l = 0; l < kS * kS; ++l) {
                const int c0 = hc[(size_t)l * D + r];
                for (int k = 0; k < kS; ++k) u.push_back(c0 + k);
            }
        }
        std::sort(u.begin(), u.end());
        u.erase(std::unique(u.begin(), u.end()), u.end());
    });
    // 2. offsets, counts, the concatenated lists
    for (int64_t tile = 0; tile < ntiles; ++tile) {
        const int64_t r0 = tile * kBlock, r1 = std::min<int64_t>(D, r0 + kBlock);
        const std::vector<int>& u = lists[(size_t)tile];
        tlo[(size_t)tile] = (int)tlr.size();
        const bool fits = (int64_t)u.size() <= kLdsRows;
        for (int64_t r = r0; r < r1; ++r)
            if (!(hf[(size_t)r] & ROW_IDENTITY)) ++op.tile_rows[(fits ? 0 : 2) + (he[(size_t)r] >= 0 ? 1 : 0)];
        if (!fits) {
            tln[(size_t)tile] = -1;
            continue;
        }
        tln[(size_t)tile] = (int)u.size();
        op.tile_list += (int64_t)u.size();
        tlr.insert(tlr.end(), u.begin(), u.end());
    }
    // 3. positions of every line (or exception column) in its tile's list
    parallel([&](int64_t tile) {
        if (tln[(size_t)tile] < 0) return;
        const int64_t r0 = tile * kBlock, r1 = std::min<int64_t>(D, r0 + kBlock);
        const std::vector<int>& u = lists[(size_t)tile];
        auto pos = [&](int c) { return (int16_t)(std::lower_bound(u.begin(), u.end(), c) - u.begin()); };
        for (int64_t r = r0; r < r1; ++r) {
            const int e = he[(size_t)r];
            if (e >= 0) {
                for (int s = 0; s < 64; ++s) tlx[(size_t)e * kExcPos + s] = pos(hx[(size_t)e * 64 + s]);
                if (hxc[(size_t)e] >= 0) tlx[(size_t)e * kExcPos + 64] = pos(hxc[(size_t)e]);
                continue;
            }
            for (int l = 0; l < kS * kS; ++l) tpl[(size_t)l * D + r] = pos(hc[(size_t)l * D + r]);
        }
    });
    tlr.push_back(0);   // an entry at every tile's list offset: the gather clamps its list reads into the list
    auto up = [](Buffer& b, const void* p, size_t bytes) {
        b = Buffer(bytes);
        HIPCHK(hipMemcpy(b.p, p, bytes, hipMemcpyHostToDevice));
    };
    up(op.tln, tln.data(), tln.size() * 4);
    up(op.tlo, tlo.data(), tlo.size() * 4);
    up(op.tlr, tlr.data(), tlr.size() * 4);
    up(op.tpl, tpl.data(), tpl.size() * 2);
    up(op.tlx, tlx.data(), tlx.size() * 2);
}

bool op_build_tp(Op& op, Tube& t, const TpSource& src) {
    if (t.p != 3 || t.dim != 3 || src.ew < kS * kS * kS || src.lw > 6 || op.nD != 0) return false;
    if (src.D > (int64_t)INT32_MAX / 2) return false;
    ensure_lex(t, op.ctx);
    const hipStream_t st = op.ctx->stream;
    const int64_t D = src.D;
    TpArgs a{};
    a.D = D;
    a.N = src.N;
    a.ecol = src.ecol;
    a.eval = src.eval;
    a.ew = src.ew;
    a.lcol = src.lcol;
    a.lval = src.lval;
    a.lw = src.lw;
    a.ldiag = src.ldiag;
    a.flag = src.flag;
    a.qpts = src.qpts;
    a.gidx = t.gidx.as<int32_t>();
    a.g = GridDev{t.N1d, t.xstart, t.dx, t.r_t};
    a.lex = t.lex.as<int32_t>();
    a.rlex = t.rlex.as<int32_t>();
    a.loff = 1.0 / (t.dx * t.dx);          // FDMatrices.cpp:25-49: 1 / h^2 off the diagonal
    a.ldu = -6.0 / (t.dx * t.dx);          // -2 dim / h^2 on it

    Buffer tpc((size_t)16 * D * 4), tpw64((size_t)12 * D * 8), tpw32((size_t)12 * D * 4), lcol((size_t)6 * D * 4),
        flag((size_t)D), mask((size_t)D * 8), nexc((size_t)(D + 1) * 4), nmov((size_t)(D + 1) * 4), flags(64),
        perm((size_t)D * 4), exc((size_t)D * 4);
    HIPCHK(hipMemsetAsync(flags.p, 0, 64, st));
    int* tot = flags.as<int>() + 4;
    hipLaunchKernelGGL(k_tp_rows, dim3(nblk(D)), dim3(256), 0, st, a, tpc.as<int>(), tpw64.as<double>(),
                       tpw32.as<float>(), lcol.as<int>(), flag.as<uint8_t>(), mask.as<unsigned long long>(),
                       nexc.as<int>(), nmov.as<int>(), flags.as<int>());
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(256), 0, st, nexc.as<int>(), D, tot);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(256), 0, st, nmov.as<int>(), D, tot + 1);
    HIPCHK(hipGetLastError());
    int h[6] = {0};
    HIPCHK(hipMemcpyAsync(h, flags.p, 24, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (h[0]) return false;
    const int64_t ne = h[4], nm = h[5];
    Buffer ecx((size_t)std::max<int64_t>(ne, 1) * 64 * 4), xcol((size_t)std::max<int64_t>(ne, 1) * 4),
        xval64((size_t)std::max<int64_t>(ne, 1) * 8), xval32((size_t)std::max<int64_t>(ne, 1) * 4);
    hipLaunchKernelGGL(k_tp_exc, dim3(nblk(D)), dim3(256), 0, st, a, nexc.as<int>(), ne, exc.as<int>(), ecx.as<int>(),
                       xcol.as<int>(), xval64.as<double>(), xval32.as<float>());
    hipLaunchKernelGGL(k_perm_full, dim3(nblk(D)), dim3(256), 0, st, t.lex.as<int32_t>(), src.N, D, perm.as<int32_t>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));

    op.fmt = OP_TP;
    op.ew = kS * kS * kS;
    op.lw = 6;
    op.loff = a.loff;
    op.ldu = a.ldu;
    op.nexc = ne;
    op.nmoved = nm;
    op.tpc = std::move(tpc);
    op.tpw64 = std::move(tpw64);
    op.tpw32 = std::move(tpw32);
    op.lcol = std::move(lcol);
    op.flag = std::move(flag);
    op.perm = std::move(perm);
    op.exc = std::move(exc);
    op.ecx = std::move(ecx);
    op.xcol = std::move(xcol);
    op.xval64 = std::move(xval64);
    op.xval32 = std::move(xval32);
    op.ecol = Buffer();
    op.eval64 = Buffer();
    op.eval32 = Buffer();
    op.lval64 = Buffer();
    op.lval32 = Buffer();
    op.ldiag64 = Buffer();
    op.ldiag32 = Buffer();
    const int mode = lds_tile_mode();
    if (mode > 0 && !(mode == 2 && build_group_tiles(op, t))) op_ensure_row_tiles(op);
    return true;
}

void op_ensure_row_tiles(Op& op) {
    if (op.fmt != OP_TP || op.tln.p) return;
    build_lds_tiles(op, HostTp(op.D, op.nexc, op.tpc, op.exc, op.ecx, op.xcol, op.flag));
}

}  // namespace cpmgpu
