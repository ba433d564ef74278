// adjoint_kernels.h -- reverse-time (adjoint) step of the CPML time loop,
// for the FWI gradient with respect to fact = vel^2 dt^2.
//
// Forward step s (interior nodes, per absorbing side with layer index m
// of the node along the side's axis, m = q - off, off = 0 on the low side
// and n - halo - 2 on the high side; slab nodes are 1 <= m <= halo):
//   psi^s[e] = bKh[e] psi^{s-1}[e] + ah[e] (p^{s-1}[off+e+1] - p^{s-1}[off+e]) / d
//   xi^s[m-1] = bK[m-1] xi^{s-1}[m-1] + a[m-1] (d2 p^{s-1} + (psi^s[m] - psi^s[m-1]) / d)
//   p^s = 2 p^{s-1} - p^{s-2} + f (L p^{s-1} + sum (dpsi + xi^s)) + sources
// with traces^s = p^s at the receivers.  For a cotangent tbar of the
// traces, the adjoint variables (lam of p, alpha of psi, beta of xi) obey,
// for s = nt .. 1:
//   lam^s = R^T tbar^s + 2 lam^{s+1} - lam^{s+2} + L(f lam^{s+1})
//           + sum_sides [ (ah[m-1] alpha^{s+1}[m-1] - ah[m] alpha^{s+1}[m]) / d
//                         + D2(z) ],          z = a beta^{s+1} on slab nodes
//   beta^s   = f lam^s + bK beta^{s+1}                     (slab nodes)
//   alpha^{s+1}[e] = bKh[e] alpha^{s+2}[e] + (w[off+e] - w[off+e+1]) / d,
//            w = f lam^{s+1} + a beta^{s+1} on slab nodes, 0 elsewhere
//   fbar += lam^s * q^s,  q^s = L p^{s-1} + sum (dpsi + xi^s)
// (q^s is written by the forward kernel during the checkpoint replay).
// Dirichlet nodes are constants of the forward map, so lam stays zero on
// them.  alpha^{s+1} is recomputed where it is needed from alpha^{s+2} and
// the w values around the node, the same fusion the forward kernel uses
// for psi, so one launch per step reads lam^{s+1}, lam^{s+2} and q of
// every shot and writes lam^s; f and the gradient accumulator are read
// once per group of shots.  Every absorbing side touches the nodes
// 0 <= m <= halo+1 ("extended" range); the plan requires n >= 2 halo + 4
// on every absorbing axis so the two sides' ranges are disjoint.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "stencil_kernels.h"  // kTileX, logical_block

namespace awcpml {

template <typename T>
struct AdjSide {
    const T* al_rd;  // alpha^{s+2} (psi layout, halo+1 layers)
    T* al_wr;        // alpha^{s+1}
    const T* be_rd;  // beta^{s+1} (xi layout, halo layers)
    T* be_wr;        // beta^s
    const T* a;
    const T* bK;
    const T* ah;
    const T* bKh;
};

template <typename T>
struct AdjointArgs {
    int64_t n[3];             // n[2] = 1 in 2D
    int64_t px;
    int64_t halo;
    int64_t field_stride;     // elements between two shots' fields
    const T* lam1;            // lam^{s+1}
    const T* lam2;            // lam^{s+2}
    T* lam0;                  // lam^s (written)
    const T* fact;            // shared by the shots
    const T* q;               // q^s
    T* grad;                  // accumulators of fbar, one per shot group
    T inv_d[3];
    T inv_d2[3];
    AdjSide<T> side[3][2];
    int active[3][2];
    int64_t psi_stride[3];    // elements between two shots' alpha slabs
    int64_t xi_stride[3];
    int ndim;
    int nshots;
    int group[2];             // shots per thread (one gradient accumulator per group)
                              // outside and in the block classes with CPML nodes
    int tiles_x, tiles_y;     // 64-wide x tiles, row groups
    // block classes: per axis (x tiles, row groups, 3D planes) the tiles
    // none of whose nodes lies in the CPML range of an absorbing side,
    // [int_lo, int_hi) of ntiles; class c (bit a set: the tiles of axis a
    // outside that range).  Class 0 has blocks[0] blocks, classes 1 and up
    // blocks[1], class c from cls_start[c] on
    int ntiles[3], int_lo[3], int_hi[3];
    int cls_start[9];
    int blocks[2];
};

// Element index of layer L of axis a's slab at node (i, j, k) in a slab
// with `layers` layers along the axis (layouts as the forward's psi/xi).
__device__ __forceinline__ int64_t slab_index(int a, int64_t layers, int64_t L, int64_t i,
                                              int64_t j, int64_t k, int64_t px, int64_t ny) {
    if (a == 0) return L + layers * (j + ny * k);
    if (a == 1) return i + px * (L + layers * k);
    return i + px * (j + ny * L);
}

// CPML data of one node on one axis.  The node lies at m = c - off in the
// range 0 <= m <= halo+1 of at most one active side; v0/v1/v2 say whether
// the nodes m-1, m, m+1 are slab layers (1..halo), e_lo/e_hi whether the
// alpha edges m-1 and m exist, w_lo whether this node stores edge m-1
// (edge 0 of the low side, which no other node owns).
template <typename T>
struct AdjCoef {
    bool ext, v0, v1, v2, e_lo, e_hi, w_lo;
    int side, m;
    T a0, a1, a2;      // a of layers m-1, m, m+1
    T bK1;             // bK of layer m (the node's own beta)
    T bKh_lo, ah_lo;   // edge m-1
    T bKh_hi, ah_hi;   // edge m
};

// Layers m-2, m-1, m of 0..h-1 and edges m-1, m of 0..h, clamped so that every
// lane may load them; a value counts only where its flag in AdjCoef is set.
struct AdjLayers {
    int b0, b1, b2, lo, hi;
};

__device__ __forceinline__ AdjLayers adj_layers(int m, int h) {
    AdjLayers L;
    L.b0 = min(max(m - 2, 0), h - 1);
    L.b1 = min(max(m - 1, 0), h - 1);
    L.b2 = min(m, h - 1);
    L.lo = min(max(m - 1, 0), h);
    L.hi = min(m, h);
    return L;
}

template <typename T>
__device__ __forceinline__ AdjCoef<T> adj_coef(const AdjointArgs<T>& A, int a, int64_t c, AdjLayers& L) {
    AdjCoef<T> C;
    const int64_t h = A.halo;
    int64_t m = -1;
    int side = 0;
    if (A.active[a][0] && c <= h + 1) {
        m = c;
    } else if (A.active[a][1] && c >= A.n[a] - h - 2) {
        m = c - (A.n[a] - h - 2);
        side = 1;
    }
    C.ext = m >= 0 && m <= h + 1;
    C.side = side;
    C.m = C.ext ? (int)m : 0;
    L = adj_layers(C.m, (int)h);
    const T* av = side ? A.side[a][1].a : A.side[a][0].a;
    const T* bK = side ? A.side[a][1].bK : A.side[a][0].bK;
    const T* bKh = side ? A.side[a][1].bKh : A.side[a][0].bKh;
    const T* ah = side ? A.side[a][1].ah : A.side[a][0].ah;
    C.a0 = av[L.b0];
    C.a1 = av[L.b1];
    C.a2 = av[L.b2];
    C.bK1 = bK[L.b1];
    C.bKh_lo = bKh[L.lo];
    C.ah_lo = ah[L.lo];
    C.bKh_hi = bKh[L.hi];
    C.ah_hi = ah[L.hi];
    C.v0 = C.ext && m >= 2 && m - 1 <= h;
    C.v1 = C.ext && m >= 1 && m <= h;
    C.v2 = C.ext && m + 1 <= h;
    C.e_lo = C.ext && m >= 1;
    C.e_hi = C.ext && m <= h;
    C.w_lo = C.ext && m == 1 && side == 0;
    return C;
}

// The slab values one node reads on one axis: beta^{s+1} of layers m-1,
// m, m+1 and alpha^{s+2} of edges m-1, m.
template <typename T>
struct AdjVals {
    T b0, b1, b2, alo, ahi;
};

// One axis's slab terms of lam^s (added to acc) and its alpha^{s+1} stores
// (alo, ahi: where edges m-1 and m are kept).
// um/uc/up: f lam^{s+1} one node below, at and above the node on the axis.
template <typename T>
__device__ __forceinline__ void adj_term(const AdjCoef<T>& C, const AdjVals<T>& V, T um, T uc,
                                         T up, T inv_d, T inv_d2, T* alo, T* ahi, T& acc) {
    const T z0 = C.v0 ? C.a0 * V.b0 : T(0);
    const T z1 = C.v1 ? C.a1 * V.b1 : T(0);
    const T z2 = C.v2 ? C.a2 * V.b2 : T(0);
    const T w0 = C.v0 ? um + z0 : T(0);
    const T w1 = C.v1 ? uc + z1 : T(0);
    const T w2 = C.v2 ? up + z2 : T(0);
    T y_lo = T(0), y_hi = T(0);
    if (C.e_lo) {
        const T alv = C.bKh_lo * V.alo + (w0 - w1) * inv_d;
        y_lo = C.ah_lo * alv;
        if (C.w_lo) *alo = alv;
    }
    if (C.e_hi) {
        const T alv = C.bKh_hi * V.ahi + (w1 - w2) * inv_d;
        y_hi = C.ah_hi * alv;
        *ahi = alv;
    }
    acc += (y_lo - y_hi) * inv_d;
    acc += (z0 - T(2) * z1 + z2) * inv_d2;
}

// Everything one shot reads at one node outside the CPML ranges: lam^{s+1} at
// the node and its axis neighbours, lam^{s+2} and q^s.
template <typename T, int NDIM>
struct AdjShot {
    T lc, lm[NDIM], lp[NDIM], l2, q;
};

// Value at byte offset o; the base is the same for all lanes of a wave, so the
// load takes it from scalar registers and needs one offset register.
template <typename T, typename Off>
__device__ __forceinline__ T adj_at(const T* base, Off o) {
    return *(const T*)((const char*)base + o);
}

template <typename T, typename Off>
__device__ __forceinline__ T* adj_ptr(T* base, Off o) {
    return (T*)((char*)base + o);
}

// off: byte offset of the node
template <typename T, int NDIM, typename Off>
__device__ __forceinline__ void adj_load_shot(const AdjointArgs<T>& A, int g, Off off, const int64_t* so,
                                              AdjShot<T, NDIM>& S) {
    const int64_t fs = (int64_t)g * A.field_stride;
    const T* l1 = A.lam1 + fs;
    S.lc = adj_at(l1, off);
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        S.lm[a] = adj_at(l1 - so[a], off);
        S.lp[a] = adj_at(l1 + so[a], off);
    }
    S.l2 = adj_at(A.lam2 + fs, off);
    S.q = adj_at(A.q + fs, off);
}

// The plain part of lam^s; um/uc/up: f lam^{s+1} around the node.
template <typename T, int NDIM>
__device__ __forceinline__ T adj_plain(const AdjointArgs<T>& A, T fc, const T* fm, const T* fp,
                                       const AdjShot<T, NDIM>& S, T& uc, T* um, T* up) {
    uc = fc * S.lc;
    T acc = T(2) * S.lc - S.l2;
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        um[a] = fm[a] * S.lm[a];
        up[a] = fp[a] * S.lp[a];
        acc += (up[a] - T(2) * uc + um[a]) * A.inv_d2[a];
    }
    return acc;
}

// One shot of the three-slot pipeline: refill slot F with shot g+2's
// loads, then compute shot g from slot C (loaded two shots earlier): its
// lam^s is stored, its gradient term lam^s q^s added to gsum.
template <typename T, int NDIM, typename Off>
__device__ __forceinline__ void adj_pipe(const AdjointArgs<T>& A, int g, int g1, Off off, const int64_t* so,
                                         T fc, const T* fm, const T* fp, AdjShot<T, NDIM>& C,
                                         AdjShot<T, NDIM>& F, T& gsum) {
    if (g >= g1) return;
    if (g + 2 < g1) adj_load_shot<T, NDIM>(A, g + 2, off, so, F);
    // keep the later shots' loads ahead of this shot's arithmetic
    __builtin_amdgcn_sched_barrier(0);
    T uc, um[NDIM], up[NDIM];
    const T acc = adj_plain<T, NDIM>(A, fc, fm, fp, C, uc, um, up);
    *adj_ptr(A.lam0 + (int64_t)g * A.field_stride, off) = acc;
    gsum += acc * C.q;
}

// Tiles of axis a in block class c, and the u-th of them.
__device__ __forceinline__ int adj_class_tiles(int c, int n, int lo, int hi, int a) {
    return ((c >> a) & 1) ? n - (hi - lo) : hi - lo;
}
__device__ __forceinline__ int adj_class_tile(int c, int lo, int hi, int a, int u) {
    if (!((c >> a) & 1)) return lo + u;
    return u < lo ? u : hi + (u - lo);
}

// The node of a thread of a reverse step's launch.  Block (64, BY): lane -> x,
// threadIdx.y -> y row, plane k in 3D; a thread owns one interior node and walks
// the shots g0 .. g1-1 of its group.  Logical blocks within a class: x tile
// fastest, then row group, plane (3D), shot group, renumbered XCD-aware.
struct AdjNode {
    int cls, grp, g0, g1;
    int64_t i, j, k;
};

// lb: the block's number among those of class 0 (CP = false) or 1..7.
template <typename T, int NDIM, bool CP>
__device__ __forceinline__ bool adj_node(const AdjointArgs<T>& A, int lb, AdjNode& N) {
    if (lb >= A.blocks[CP]) return false;
    N.cls = 0;
    if (CP)
        for (int c = 1; c < 8; ++c)
            if (lb >= A.cls_start[c]) N.cls = c;
    int rest = CP ? lb - A.cls_start[N.cls] : lb;
    int t[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int na = adj_class_tiles(N.cls, A.ntiles[a], A.int_lo[a], A.int_hi[a], a);
        t[a] = adj_class_tile(N.cls, A.int_lo[a], A.int_hi[a], a, rest % na);
        rest /= na;
    }
    N.grp = rest;
    N.g0 = rest * A.group[CP];
    N.g1 = N.g0 + A.group[CP] < A.nshots ? N.g0 + A.group[CP] : A.nshots;
    N.k = NDIM == 3 ? 1 + t[2] : 0;
    N.i = (int64_t)t[0] * kTileX + threadIdx.x;
    // one row per wavefront: j (and the y axis's CPML data) is wave-uniform
    N.j = 1 + (int64_t)t[1] * blockDim.y + __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    return N.i >= 1 && N.i <= A.n[0] - 2 && N.j <= A.n[1] - 2;
}

// One reverse step of the nodes of block class 0 (no node of the block in a
// CPML range).  fact and the gradient accumulator of the node are read once per
// group of shots, whose gradient terms are summed in registers (one
// read-modify-write of the group's accumulator per step).  Shots run through a
// three-slot pipeline: the loads of shots g+1 and g+2 are in flight while shot g
// is computed.
template <typename T, int NDIM, typename Off>
__device__ __forceinline__ void adj_plain_block(const AdjointArgs<T>& A, int lb) {
    AdjNode N;
    if (!adj_node<T, NDIM, false>(A, lb, N)) return;
    const int64_t so[3] = {1, A.px, A.px * A.n[1]};
    const Off off = (Off)((N.i + A.px * N.j + so[2] * N.k) * (int64_t)sizeof(T));
    const T* f = A.fact;
    const T fc = adj_at(f, off);
    T fm[NDIM], fp[NDIM];
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        fm[a] = adj_at(f - so[a], off);
        fp[a] = adj_at(f + so[a], off);
    }
    const int g0 = N.g0, g1 = N.g1;
    T gsum = T(0);
    AdjShot<T, NDIM> s0, s1, s2;
    adj_load_shot<T, NDIM>(A, g0, off, so, s0);
    if (g0 + 1 < g1) adj_load_shot<T, NDIM>(A, g0 + 1, off, so, s1);
    for (int g = g0; g < g1; g += 3) {
        adj_pipe<T, NDIM>(A, g, g1, off, so, fc, fm, fp, s0, s2, gsum);
        adj_pipe<T, NDIM>(A, g + 1, g1, off, so, fc, fm, fp, s1, s0, gsum);
        adj_pipe<T, NDIM>(A, g + 2, g1, off, so, fc, fm, fp, s2, s1, gsum);
    }
    *adj_ptr(A.grad + (int64_t)N.grp * A.field_stride, off) += gsum;
}

// The same of the other block classes, whose tiles hold CPML nodes of the axes
// in the class's bits.  Shots one after the other, each axis's loads clamped
// instead of branched on: latency hides behind waves.  Three shots' loads in
// registers, as in the plain blocks, took 256 VGPRs in FP64 3D (one wave per
// SIMD) and 125 in FP32 2D: 81x73x69 FP64, 2 shots, 126 us per step, 45 so;
// 554x554 FP32, 32 shots, 38 us, 30 so.  The next shot's fields loaded early, or
// the accumulator, spill and lose it again.
template <typename T, int NDIM, typename Off>
__device__ __forceinline__ void adj_slab_block(const AdjointArgs<T>& A, int lb) {
    AdjNode N;
    if (!adj_node<T, NDIM, true>(A, lb, N)) return;
    const int64_t so[3] = {1, A.px, A.px * A.n[1]};
    const int64_t i = N.i, j = N.j, k = N.k, h = A.halo;
    const Off off = (Off)((i + A.px * j + so[2] * k) * (int64_t)sizeof(T));
    const Off offx = (Off)(i * (int64_t)sizeof(T));
    const T* f = A.fact;
    const T fc = adj_at(f, off);
    T fm[NDIM], fp[NDIM];
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        fm[a] = adj_at(f - so[a], off);
        fp[a] = adj_at(f + so[a], off);
    }
    // x: the side and layers differ from lane to lane, and its slabs hold the
    // layers of row (j, k) together.  y, z: one side and layer per wave, kept
    // as rows of nodes.
    AdjCoef<T> C[NDIM];
    AdjLayers L[NDIM];
    bool on[NDIM];
#pragma unroll
    for (int a = 0; a < NDIM; ++a) {
        on[a] = (N.cls >> a) & 1;
        if (!on[a]) continue;
        C[a] = adj_coef<T>(A, a, a == 0 ? i : (a == 1 ? j : k), L[a]);
        if (a) on[a] = C[a].ext;
    }
    auto row = [&](int a, int layers, int layer) -> int64_t {
        return a == 1 ? A.px * (layer + layers * k) : A.px * (j + A.n[1] * layer);
    };
    // x: fn(side, its slab row's offsets) for the lanes in a CPML range.  2D:
    // once per side that lanes of the wave lie in, from scalar bases; 3D: with
    // each lane's own (the scalar form spills: 81x73x69 FP64, 2 shots, 50 and
    // 56 us per step; 554x554 FP32, 32 shots, 34 and 30 us)
    const int64_t rx = j + A.n[1] * k;
    const bool extx = on[0] && C[0].ext, hix = extx && C[0].side;
    const bool anyhi = __any(hix), anylo = __any(extx && !hix);
    auto x_sides = [&](int g, auto fn) {
        const int64_t bx = g * A.xi_stride[0] + h * rx, ax = g * A.psi_stride[0] + (h + 1) * rx;
        const AdjSide<T>& D0 = A.side[0][0];
        const AdjSide<T>& D1 = A.side[0][1];
        if constexpr (NDIM == 2) {
            if (anylo && extx && !hix) fn(D0.be_rd + bx, D0.be_wr + bx, D0.al_rd + ax, D0.al_wr + ax);
            if (anyhi && hix) fn(D1.be_rd + bx, D1.be_wr + bx, D1.al_rd + ax, D1.al_wr + ax);
        } else if (extx) {
            fn((hix ? D1.be_rd : D0.be_rd) + bx, (hix ? D1.be_wr : D0.be_wr) + bx,
               (hix ? D1.al_rd : D0.al_rd) + ax, (hix ? D1.al_wr : D0.al_wr) + ax);
        }
    };
    const unsigned es = sizeof(T);
    T gsum = T(0);
    for (int g = N.g0; g < N.g1; ++g) {
        const int64_t fs = (int64_t)g * A.field_stride;
        AdjVals<T> V[NDIM];
        AdjShot<T, NDIM> S;
        adj_load_shot<T, NDIM>(A, g, off, so, S);
        x_sides(g, [&](const T* be, T*, const T* al, T*) {
            V[0].b0 = adj_at(be, es * L[0].b0);
            V[0].b1 = adj_at(be, es * L[0].b1);
            V[0].b2 = adj_at(be, es * L[0].b2);
            V[0].alo = adj_at(al, es * L[0].lo);
            V[0].ahi = adj_at(al, es * L[0].hi);
        });
#pragma unroll
        for (int a = 1; a < NDIM; ++a) {
            if (!on[a]) continue;
            const T* be = (C[a].side ? A.side[a][1].be_rd : A.side[a][0].be_rd) + g * A.xi_stride[a];
            const T* al = (C[a].side ? A.side[a][1].al_rd : A.side[a][0].al_rd) + g * A.psi_stride[a];
            V[a].b0 = adj_at(be + row(a, (int)h, L[a].b0), offx);
            V[a].b1 = adj_at(be + row(a, (int)h, L[a].b1), offx);
            V[a].b2 = adj_at(be + row(a, (int)h, L[a].b2), offx);
            V[a].alo = adj_at(al + row(a, (int)h + 1, L[a].lo), offx);
            V[a].ahi = adj_at(al + row(a, (int)h + 1, L[a].hi), offx);
        }
        T uc, um[NDIM], up[NDIM];
        T acc = adj_plain<T, NDIM>(A, fc, fm, fp, S, uc, um, up);
        x_sides(g, [&](const T*, T*, const T*, T* al) {
            adj_term(C[0], V[0], um[0], uc, up[0], A.inv_d[0], A.inv_d2[0], adj_ptr(al, es * L[0].lo),
                     adj_ptr(al, es * L[0].hi), acc);
        });
#pragma unroll
        for (int a = 1; a < NDIM; ++a) {
            if (!on[a]) continue;
            T* al = (C[a].side ? A.side[a][1].al_wr : A.side[a][0].al_wr) + g * A.psi_stride[a];
            adj_term(C[a], V[a], um[a], uc, up[a], A.inv_d[a], A.inv_d2[a],
                     adj_ptr(al + row(a, (int)h + 1, L[a].lo), offx),
                     adj_ptr(al + row(a, (int)h + 1, L[a].hi), offx), acc);
        }
        *adj_ptr(A.lam0 + fs, off) = acc;
        // beta^s = bK beta^{s+1} + f lam^s on every slab holding the node
        x_sides(g, [&](const T*, T* be, const T*, T*) {
            if (C[0].v1) *adj_ptr(be, es * L[0].b1) = C[0].bK1 * V[0].b1 + fc * acc;
        });
#pragma unroll
        for (int a = 1; a < NDIM; ++a) {
            if (!on[a] || !C[a].v1) continue;
            T* be = (C[a].side ? A.side[a][1].be_wr : A.side[a][0].be_wr) + g * A.xi_stride[a];
            *adj_ptr(be + row(a, (int)h, L[a].b1), offx) = C[a].bK1 * V[a].b1 + fc * acc;
        }
        gsum += acc * S.q;
    }
    *adj_ptr(A.grad + (int64_t)N.grp * A.field_stride, off) += gsum;
}

// One reverse step: of the blocks without CPML nodes (KIND 0), with (1), or both
// (2).  2D takes both in one launch: those with CPML nodes wait on their loads
// and keep the VALU busy, the others run at the memory's rate, and the two kinds
// take turns in proportion to their numbers, in groups of one block per XCD
// (554x554 FP32, 32 shots: 56 us per step in two launches, 52 in one).  In 3D the
// plain blocks lose more from the other kind's registers (110x100x98 FP64, 4
// shots, 60 steps' gradient: 21.5 and 23.6 ms).
template <typename T, int NDIM, typename Off, int KIND>
__global__ __launch_bounds__(256, (KIND == 0 ? 1 : (sizeof(T) == 8 ? 3 : (NDIM == 2 ? 5 : 4))))
void adjoint_step(const AdjointArgs<T> A) {
    const int xcd = (int)blockIdx.x % kNumXcd, q = (int)blockIdx.x / kNumXcd;
    const int all = (int)gridDim.x / kNumXcd;
    if constexpr (KIND == 0) {
        adj_plain_block<T, NDIM, Off>(A, xcd * all + q);
    } else if constexpr (KIND == 1) {
        adj_slab_block<T, NDIM, Off>(A, xcd * all + q);
    } else {
        const int slab = (A.blocks[1] + kNumXcd - 1) / kNumXcd;
        const int before = (int)((int64_t)q * slab / all);
        if ((int)((int64_t)(q + 1) * slab / all) > before)
            adj_slab_block<T, NDIM, Off>(A, xcd * slab + before);
        else
            adj_plain_block<T, NDIM, Off>(A, xcd * (all - slab) + (q - before));
    }
}

// Trace cotangent injection of step it0 (0-based) after adjoint_step:
// for each distinct interior receiver node of a shot, r = the sum of the
// cotangents of its receivers; lam^s += r, beta^s += f r on every
// absorbing slab holding the node (beta^s = f lam^s + ...), and r q^s,
// the node's extra gradient term, is added to the node's own entry of rq
// (entry u of the receiver node list), which fold_receivers adds to the
// gradient.  One block per shot; entries of different shots never share
// memory, so the shots run in parallel and the sums stay in a fixed order.
template <typename T>
struct AdjIoArgs {
    T* lam0;
    T* rq;                     // per receiver node entry: sum of r q^s
    const T* q;
    const T* fact;
    int64_t field_stride;
    const int64_t* node_lin;   // distinct interior receiver nodes, all shots
    const int* node_start;     // nshots+1 CSR offsets into node_lin
    const int* rec_start;      // per node: CSR offsets into rec_idx
    const int* rec_idx;        // receiver index (all shots) of each entry
    const T* tbar;             // nt values per receiver
    int64_t nt;
    int64_t n[3];
    int64_t px, halo;
    int ndim;
    AdjSide<T> side[3][2];
    int active[3][2];
    int64_t xi_stride[3];
};

template <typename T>
__global__ __launch_bounds__(256) void adjoint_inject(const AdjIoArgs<T> A, int64_t it0) {
    const int shot = blockIdx.x;
    const int u0 = A.node_start[shot], u1 = A.node_start[shot + 1];
    const int64_t fs = (int64_t)shot * A.field_stride;
    for (int u = u0 + threadIdx.x; u < u1; u += blockDim.x) {
        T r = T(0);
        for (int e = A.rec_start[u]; e < A.rec_start[u + 1]; ++e)
            r += A.tbar[(int64_t)A.rec_idx[e] * A.nt + it0];
        const int64_t lin = A.node_lin[u];
        A.lam0[fs + lin] += r;
        A.rq[u] += r * A.q[fs + lin];
        const T fr = A.fact[lin] * r;
        const int64_t ny = A.n[1];
        const int64_t c[3] = {lin % A.px, (lin / A.px) % ny, lin / (A.px * ny)};
        const int64_t h = A.halo;
        for (int a = 0; a < A.ndim; ++a)
            for (int s = 0; s < 2; ++s) {
                if (!A.active[a][s]) continue;
                const int64_t m = c[a] - (s ? A.n[a] - h - 2 : 0);
                if (m < 1 || m > h) continue;
                const int64_t idx = slab_index(a, h, m - 1, c[0], c[1], c[2], A.px, ny);
                A.side[a][s].be_wr[shot * A.xi_stride[a] + idx] += fr;
            }
    }
}

// Add the receiver gradient terms rq to the gradient total and clear them:
// for each distinct receiver node v over all shots, total[lin[v]] += the
// sum of its entries rq[idx[e]], start[v] <= e < start[v+1], in shot
// order.
template <typename T, typename A>
__global__ __launch_bounds__(256) void fold_receivers(T* rq, A* total, const int64_t* lin,
                                                      const int* start, const int* idx, int count) {
    const int v = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (v >= count) return;
    A acc = A(0);
    for (int e = start[v]; e < start[v + 1]; ++e) {
        acc += (A)rq[idx[e]];
        rq[idx[e]] = T(0);
    }
    total[lin[v]] += acc;
}

// Fold the shot groups' partial gradients of the last reverse steps into
// the FP64 total: total += sum over groups (in group order), partials = 0.
// The partial sums then run over at most one checkpoint segment and one
// group of shots in the plan's precision, and the long sum over time and
// groups is FP64.
template <typename T>
__global__ __launch_bounds__(256) void fold_gradient(T* grad, double* total, int64_t field_stride,
                                                     int ngroups) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= field_stride) return;
    double acc = total[t];
    for (int s = 0; s < ngroups; ++s) {
        T& g = grad[(int64_t)s * field_stride + t];
        acc += (double)g;
        g = T(0);
    }
    total[t] = acc;
}

// Sum of the shot groups' gradients into group 0's accumulator.
template <typename T>
__global__ __launch_bounds__(256) void sum_shots(T* grad, int64_t field_stride, int ngroups) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= field_stride) return;
    T acc = grad[t];
    for (int s = 1; s < ngroups; ++s) acc += grad[(int64_t)s * field_stride + t];
    grad[t] = acc;
}

}  // namespace awcpml
