// tile2d_kernels.h -- up to kTileSteps time steps of the 2D CPML stencil per
// launch, on tiles held in registers.
//
// A single-step launch moves three fields per node and step, and on small
// grids it costs a kernel launch for a fraction of a microsecond of work.  A
// block here loads a tile of 64 x (R*W) nodes -- p^{t-1}, p^t, fact and, in
// the CPML slabs, psi and xi -- once, takes n <= kTileSteps steps on it
// without touching memory, and stores p^{t+n-1}, p^{t+n}, psi and xi of the
// nodes it owns: those at least kTileHalo = kTileSteps nodes inside the tile,
// whose values do not depend on what lies outside (each step makes one more
// ring of the tile stale).  Lane -> x; a wave holds R consecutive rows, one
// node per lane and row, so y neighbours are registers, x neighbours DPP lane
// shifts, and only a wave's first and last row travel through LDS, once per
// step and with one barrier (the exchange buffer alternates).
//
// Sources are added inside the tile at every step, in source order, by every
// tile that holds their node; receivers are sampled by the owning tile
// through an LDS copy of the tile, made only in blocks that have receivers.
// So a launch replaces n stencil and n source/receiver launches.
//
// Measured (MI355X, HIP events around runs of 200 to 1000 steps with sources and
// receivers, single steps -> tiles): 1066^2 x 64 shots FP32, 238 -> 71 us per
// step; 298^2 FP64, one shot, 15.7 -> 2.1 us (latency: 133 blocks); 4097^2 FP64,
// 133 -> 25.6 us; 701x333 FP32, 7 shots, 17.1 -> 4.2 us.  What bounds the first:
// VALU issue.  Per launch of 8 steps the 26,880 plain blocks issue 200 M wave
// instructions, 14.5 a node and step, 781 k of the 759 k cycles of 332 us at 4 a
// SIMD; the 6,976 slab blocks 135 M, 527 k of 602 k cycles.  Memory is behind
// that: 1.32 GB past L2 at 4.0 TB/s, 0.46 GB at 1.9 TB/s.  44 % of a 64-row
// tile's nodes are its rings.
//
// The arithmetic of a node is the single-step kernel's, operation for
// operation (-ffp-contract=off), so the results equal n single-step launches
// (up to the sign of zeros).  Outputs go to buffers distinct from the inputs,
// which neighbouring tiles read.  As for the other multi-step kernels the
// host requires every field buffer to be zero on the Dirichlet nodes.
#pragma once

#include "stencil2_kernels.h"

namespace awcpml {

constexpr int kTileSteps = 8;            // most steps per launch
constexpr int kTileHalo = kTileSteps;    // stale rings a tile allows for
constexpr int kTileOwnX = kTileX - 2 * kTileHalo;
constexpr int kRecBand = 16;             // rows per receiver band

template <typename T>
struct TileArgs {
    // geometry, coefficients, pold = p^{t-1}, pcur = p^t; side[][].psi_rd and
    // .xi are the inputs, side[][].psi_wr receives psi after the last step
    StencilArgs<T> s;
    T* p1;                    // p^{t+steps-1}
    T* p2;                    // p^{t+steps}
    T* xi_out[2][2];          // xi after the last step
    // optional: d(pnew)/d(fact) of every step (StencilArgs::qout), q_step
    // elements apart; null = off
    T* q;
    int64_t q_step;
    int q_stream;             // 1: q is stored past the caches
    const int64_t* src_xy;    // source nodes of all shots (x | y << 32)
    const T* src_wav;         // nt values per source
    const int* src_start;     // nshots+1 CSR offsets
    // interior receivers of every shot, sorted into bands of kRecBand rows:
    // nodes, trace indices, and nshots*bands+1 CSR offsets
    const int64_t* rec_xy;
    const int* rec_idx;
    const int* rec_band;
    int bands;
    T* traces;                // nt values per receiver
    int64_t nt;
    int64_t it0;              // 0-based index of the first step
    int steps;
    int io;                   // 0: no sources, no receivers (timing)
    // tile (tx, ty) owns the kTileOwnX columns from tx*kTileOwnX - shift_x on and
    // the OY rows from 1 + ty*OY - shift_y on, as far as they are interior
    int tiles_x, tiles_y, shift_x, shift_y;
    // tiles [ix0, ix1) x [iy0, iy1) lie wholly inside the domain and outside
    // the CPML slabs; a launch takes those (CP = false), the others, or all
    // (the range is then empty)
    int ix0, ix1, iy0, iy1;
    int logical_blocks, grid_blocks;
};

// Tile (tx, ty) and shot of logical block lb: x fastest, then y, then shot.
template <typename T, bool CP>
__device__ __forceinline__ void tile_of(const TileArgs<T>& B, int lb, int* tx, int* ty, int* shot) {
    const int in = (B.ix1 - B.ix0) * (B.iy1 - B.iy0);
    const int per = CP ? B.tiles_x * B.tiles_y - in : in;
    *shot = lb / per;
    int u = lb % per;
    if (!CP) {
        *tx = B.ix0 + u % (B.ix1 - B.ix0);
        *ty = B.iy0 + u / (B.ix1 - B.ix0);
        return;
    }
    const int head = B.iy0 * B.tiles_x;                 // whole rows of tiles before the range
    const int side = B.tiles_x - (B.ix1 - B.ix0);       // tiles beside it in its rows
    const int mid = side * (B.iy1 - B.iy0);
    if (u < head || in == 0) {
        *tx = u % B.tiles_x;
        *ty = u / B.tiles_x;
    } else if (u < head + mid) {
        u -= head;
        const int c = u % side;
        *tx = c < B.ix0 ? c : c + (B.ix1 - B.ix0);
        *ty = B.iy0 + u / side;
    } else {
        u -= head + mid;
        *tx = u % B.tiles_x;
        *ty = B.iy1 + u / B.tiles_x;
    }
}

// The value of lane i-1 (below) or i+1; lanes at the wave's ends get 0.  With
// zero fill the compiler folds the shift into the FP32 add or subtract that
// uses it (no instruction of its own; the form that keeps the end lanes' own
// values cost two moves per shift, 15 instead of 11 VALU operations a node).
__device__ __forceinline__ int dpp_shift0(int v, bool below) {
    return below ? __builtin_amdgcn_update_dpp(0, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, true)
                 : __builtin_amdgcn_update_dpp(0, v, 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
}
__device__ __forceinline__ float shift0(float v, bool below) {
    return __builtin_bit_cast(float, dpp_shift0(__builtin_bit_cast(int, v), below));
}
__device__ __forceinline__ double shift0(double v, bool below) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = dpp_shift0((int)(unsigned)(u & 0xffffffffull), below);
    const int hi = dpp_shift0((int)(unsigned)(u >> 32), below);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// The psi edge of a node: the side it belongs to (-1: none) and its layer m,
// 0 <= m <= halo, the edge between the node (layer m) and the next one.  The
// slab nodes are those with m >= 1; layer 0's edge is kept by the node before
// the side's first slab node (x = 0 or x = n-halo-2).
__device__ __forceinline__ int edge_layer(int q, int n, int h, const int* active, int* m) {
    if (active[0] && q >= 0 && q <= h) {
        *m = q;
        return 0;
    }
    if (active[1] && q >= n - h - 2 && q <= n - 2) {
        *m = q - (n - h - 2);
        return 1;
    }
    return -1;
}

// What the tile kernels' paths have to cover.
enum TileKind {
    kTilePlain,    // tiles inside the domain and outside the slabs
    kTileSlabs,    // any tile; every axis has n >= 2*halo+3, so a node's psi[m-1]
                   // is the edge of the node before it (layer m-1, same side)
    kTileOverlap,  // any tile and grid: every slab node keeps both its edges
};

// Q: d(pnew)/d(fact) outputs (1), past the caches (2).
template <typename T, int R, int W, int KIND, int Q>
__global__ __launch_bounds__(64 * W, KIND == kTileOverlap ? 2 : sizeof(T) == 4 ? 8 : 4) void stencil2d_tile(const TileArgs<T> B) {
    constexpr int TY = R * W, OY = TY - 2 * kTileHalo;
    constexpr bool CP = KIND != kTilePlain, OV = KIND == kTileOverlap;
    constexpr int RC = CP ? R : 1, RO = OV ? R : 1;
    __shared__ T edge[2][2 * W][kTileX];   // waves' first and last rows, two steps
    __shared__ T rows[TY][kTileX];         // the tile for its receivers
    // y coefficients per row: bKh, ah of its edge, bK, a of its node, and (OV)
    // bKh, ah of the edge before it
    __shared__ __align__(16) T cy[CP ? TY : 1][OV ? 8 : 4];
    const StencilArgs<T>& A = B.s;
    const int lb = logical_block(blockIdx.x, B.grid_blocks);
    if (lb >= B.logical_blocks) return;  // whole block
    int tx, ty, shot;
    tile_of<T, CP>(B, lb, &tx, &ty, &shot);
    const int lane = (int)threadIdx.x;
    const int wy = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int nx = (int)A.nx, ny = (int)A.ny, h = (int)A.halo;
    const int xt = tx * kTileOwnX - B.shift_x - kTileHalo;   // first column of the tile
    const int x = xt + lane;
    const int yt = 1 + ty * OY - B.shift_y - kTileHalo;      // first row of the tile
    const int y0 = yt + wy * R;               // first row of the wave
    const bool inx = x >= 1 && x <= nx - 2;
    const int xc = x < 0 ? 0 : (x > nx - 1 ? nx - 1 : x);
    const int64_t fo = (int64_t)shot * A.field_stride;
    const uint32_t E = sizeof(T);
    const uint32_t pitch = (uint32_t)A.px * E, col = (uint32_t)xc * E;

    // p, o, f: pressure, previous pressure and fact of the lane's rows; nodes
    // outside the interior hold 0
    T p[R], o[R], f[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = y0 + r;
        const int jc = CP ? (j < 0 ? 0 : (j > ny - 1 ? ny - 1 : j)) : j;
        const uint32_t off = col + (uint32_t)jc * pitch;
        p[r] = ldg(A.pcur + fo, off);
        o[r] = ldg(A.pold + fo, off);
        f[r] = ldg(A.fact, off);
    }
    // CPML state of the lane's nodes: psi of the node's edge and xi of the
    // node, in x (xh, xx) and y (yh, yx); yl: psi of the edge before the
    // wave's first row.  OV: both edges of every slab node (xl, yl).
    T xh[RC], xx[RC], yh[RC], yx[RC], xl[RO], yl[RO];
    T cxh = T(0), cxah = T(0), cxl = T(0), cxal = T(0), cxb = T(0), cxa = T(0);
    T cyl = T(0), cyal = T(0);   // coefficients of the edge before the first row
    int sx = -1, mx = 0;
    bool nodex = false, anyx = false;   // the lane's nodes lie in an x slab; any x edge in the wave
    uint32_t ymask = 0;      // rows of the wave in a y slab
    uint32_t yedge = 0;      // rows of the wave with a y edge
    uint32_t imask = 0;      // rows of the wave in the interior
    if (CP) {
        if (OV) {
            sx = inx ? classify(x, nx, h, A.active[0], &mx) : -1;
            nodex = sx >= 0;
        } else {
            sx = edge_layer(x, nx, h, A.active[0], &mx);
            nodex = sx >= 0 && mx >= 1;
        }
        anyx = __any(sx >= 0);
        const CpmlSide<T>& X = A.side[0][sx == 1 ? 1 : 0];
        const T* xpsi = X.psi_rd + shot * A.psi_stride[0];
        const T* xxi = X.xi + shot * A.xi_stride[0];
        if (sx >= 0) {
            cxh = X.bKh[mx];
            cxah = X.ah[mx];
            if (nodex) {
                cxb = X.bK[mx - 1];
                cxa = X.a[mx - 1];
            }
            if (OV) {
                cxl = X.bKh[mx - 1];
                cxal = X.ah[mx - 1];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int j = y0 + r;
            const bool iny = j >= 1 && j <= ny - 2;
            if (iny) imask |= 1u << r;
            xh[r] = xx[r] = yh[r] = yx[r] = T(0);
            if (OV) xl[r] = yl[r] = T(0);
            if (sx >= 0 && iny) {
                const uint32_t op = (uint32_t)(mx + (h + 1) * j) * E;
                xh[r] = ldg(xpsi, op);
                if (OV) xl[r] = ldg(xpsi, op - E);
                if (nodex) xx[r] = ldg(xxi, (uint32_t)(mx - 1 + h * j) * E);
            }
            int my = 0;
            const int sy = OV ? (iny ? classify(j, ny, h, A.active[1], &my) : -1)
                              : edge_layer(j, ny, h, A.active[1], &my);
            if (sy >= 0) {
                const CpmlSide<T>& Y = A.side[1][sy];
                const T* ypsi = Y.psi_rd + shot * A.psi_stride[1];
                const bool node = OV || my >= 1;
                const uint32_t oy = col + (uint32_t)my * pitch;
                yedge |= 1u << r;
                yh[r] = ldg(ypsi, oy);
                if (OV) yl[r] = ldg(ypsi, oy - pitch);
                if (node) {
                    ymask |= 1u << r;
                    yx[r] = ldg((const T*)Y.xi + shot * A.xi_stride[1], oy - pitch);
                    if (!OV && r == 0) {
                        yl[0] = ldg(ypsi, oy - pitch);
                        cyl = Y.bKh[my - 1];
                        cyal = Y.ah[my - 1];
                    }
                }
                if (lane == 0) {
                    T* d = cy[wy * R + r];
                    d[0] = Y.bKh[my];
                    d[1] = Y.ah[my];
                    d[2] = node ? Y.bK[my - 1] : T(0);
                    d[3] = node ? Y.a[my - 1] : T(0);
                    if (OV) {
                        d[4] = Y.bKh[my - 1];
                        d[5] = Y.ah[my - 1];
                    }
                }
            }
            const bool in = inx && iny;
            p[r] = in ? p[r] : T(0);
            o[r] = in ? o[r] : T(0);
            f[r] = in ? f[r] : T(0);
        }
        if (!OV && !(ymask & 1u)) yl[0] = T(0);
    }

    // sources and receivers of the tile
    const int s0 = B.src_start[shot], s1 = B.io ? B.src_start[shot + 1] : s0;
    bool src = false;
    for (int e = s0; e < s1; ++e) {
        const int64_t xy = B.src_xy[e];
        const int dx = (int)(xy & 0xffffffff) - xt, dy = (int)(xy >> 32) - yt;
        src = src || (dx >= 0 && dx < kTileX && dy >= 0 && dy < TY);
    }
    const int ye = yt + kTileHalo + OY;
    const int oy0 = yt + kTileHalo > 1 ? yt + kTileHalo : 1, oy1 = ye < ny - 1 ? ye : ny - 1;  // owned rows
    const int q0 = B.rec_band[shot * B.bands + oy0 / kRecBand];
    const int q1 = B.io ? B.rec_band[shot * B.bands + (oy1 - 1) / kRecBand + 1] : q0;
    const int tid = wy * kTileX + lane;
    bool mine = false;
    for (int q = q0 + tid; q < q1; q += 64 * W) {
        const int64_t xy = B.rec_xy[q];
        const int rx = (int)(xy & 0xffffffff) - xt - kTileHalo, ry = (int)(xy >> 32);
        mine = mine || (rx >= 0 && rx < kTileOwnX && ry >= oy0 && ry < oy1);
    }
    const bool rec = __syncthreads_or(mine);

    const T two = T(2);
    const T i2a = A.inv_d2[0], i2m = A.inv_d2[1], ia = A.inv_d[0], im = A.inv_d[1];
    const bool ownx = lane >= kTileHalo && lane < kTileX - kTileHalo && (!CP || inx);
    for (int s = 0; s < B.steps; ++s) {
        T(*ex)[kTileX] = edge[s & 1];
        ex[2 * wy][lane] = p[0];
        ex[2 * wy + 1][lane] = p[R - 1];
        __syncthreads();
        // the rows above and below the wave (stale beyond the tile)
        const T up = ex[wy > 0 ? 2 * wy - 1 : 0][lane];
        const T dn = ex[wy < W - 1 ? 2 * wy + 2 : 2 * W - 1][lane];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T pc = p[r];
            const T pm = r == 0 ? up : o[r > 0 ? r - 1 : 0];  // o[r-1] is row r-1 before this step
            const T pp = r == R - 1 ? dn : p[r < R - 1 ? r + 1 : r];
            const T xp = shift0(pc, false);
            const T d2a = (xp - two * pc + shift0(pc, true)) * i2a;
            const T d2m = (pp - two * pc + pm) * i2m;
            const T lap = d2a + d2m;
            T v = two * pc - o[r] + f[r] * lap;
            T slab = T(0);
            if (CP) {
                T damp = T(0);
                if (anyx) {
                    // update_psi_x!, update_p!; lanes without an edge or node
                    // have zero coefficients and state
                    xh[r] = cxh * xh[r] + cxah * (xp - pc) * ia;
                    if (OV) xl[r] = cxl * xl[r] + cxal * (pc - shift0(pc, true)) * ia;
                    const T dpsi = (OV ? xh[r] - xl[OV ? r : 0] : xh[r] - shift0(xh[r], true)) * ia;
                    xx[r] = cxb * xx[r] + cxa * (d2a + dpsi);
                    const T t = nodex ? dpsi + xx[r] : T(0);
                    damp = f[r] * t;
                    slab = t;
                }
                if (yedge & (1u << r)) {
                    const T* d = cy[wy * R + r];
                    yh[r] = d[0] * yh[r] + d[1] * (pp - pc) * im;
                    if (ymask & (1u << r)) {
                        T lo;
                        if (r == 0 || OV) {
                            const T c0 = OV ? d[OV ? 4 : 0] : cyl, c1 = OV ? d[OV ? 5 : 1] : cyal;
                            yl[OV ? r : 0] = c0 * yl[OV ? r : 0] + c1 * (pc - pm) * im;
                            lo = yl[OV ? r : 0];
                        } else {
                            lo = yh[r > 0 ? r - 1 : 0];
                        }
                        const T dpsi = (yh[r] - lo) * im;
                        yx[r] = d[2] * yx[r] + d[3] * (d2m + dpsi);
                        const T t = dpsi + yx[r];
                        damp += f[r] * t;
                        slab += t;
                    }
                }
                v = v + damp;
                v = inx && (imask & (1u << r)) ? v : T(0);
            }
            o[r] = pc;
            p[r] = v;
            if (Q) {
                const int k = wy * R + r;
                if (ownx && k >= kTileHalo && k < TY - kTileHalo && (!CP || (imask & (1u << r)))) {
                    T* q = B.q + fo + s * B.q_step;
                    const uint32_t off = col + (uint32_t)(y0 + r) * pitch;
                    if constexpr (Q == 2) stg_stream(q, off, lap + slab);
                    else stg(q, off, lap + slab);
                }
            }
        }
        if (src) {
            // inject_sources!, in source order
            for (int e = s0; e < s1; ++e) {
                const int64_t xy = B.src_xy[e];
                const int dx = (int)(xy & 0xffffffff) - x, dy = (int)(xy >> 32) - y0;
                if (dy < 0 || dy >= R) continue;
                const T w = B.src_wav[(int64_t)e * B.nt + B.it0 + s];
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (dy == r && dx == 0) p[r] += w;
            }
        }
        if (rec) {
            // record_receivers!: the next write of `rows` comes after the
            // next step's barrier
#pragma unroll
            for (int r = 0; r < R; ++r) rows[wy * R + r][lane] = p[r];
            __syncthreads();
            for (int q = q0 + tid; q < q1; q += 64 * W) {
                const int64_t xy = B.rec_xy[q];
                const int rx = (int)(xy & 0xffffffff) - xt - kTileHalo, ry = (int)(xy >> 32);
                if (rx >= 0 && rx < kTileOwnX && ry >= oy0 && ry < oy1)
                    B.traces[(int64_t)B.rec_idx[q] * B.nt + B.it0 + s] = rows[ry - yt][rx + kTileHalo];
            }
        }
    }

    // the owned nodes; a side's first slab node also stores the edge before it
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = wy * R + r, j = y0 + r;
        T xlo = T(0);
        if (CP && anyx) xlo = OV ? xl[OV ? r : 0] : shift0(xh[r], true);
        if (k < kTileHalo || k >= TY - kTileHalo || (CP && !(imask & (1u << r)))) continue;
        if (!ownx) continue;
        const uint32_t off = col + (uint32_t)j * pitch;
        if constexpr (KIND == kTilePlain) {
            // large grids: next read in the following launch, and the tiles'
            // shared margins stay in L2 (2001x1501 FP64, 3 shots, 160 steps:
            // 2.87 ms, 2.71 so; 1066x1066 FP32, 64 shots, 400 steps: 33.0, 32.7)
            stg_stream(B.p1 + fo, off, o[r]);
            stg_stream(B.p2 + fo, off, p[r]);
        } else {
            stg(B.p1 + fo, off, o[r]);
            stg(B.p2 + fo, off, p[r]);
        }
        if (CP) {
            if (nodex) {
                T* pw = (sx ? A.side[0][1].psi_wr : A.side[0][0].psi_wr) + shot * A.psi_stride[0];
                T* xw = (sx ? B.xi_out[0][1] : B.xi_out[0][0]) + shot * A.xi_stride[0];
                const uint32_t op = (uint32_t)(mx + (h + 1) * j) * E;
                stg(pw, op, xh[r]);
                if (mx == (OV && sx ? right_first(nx, h) : 1)) stg(pw, op - E, xlo);
                stg(xw, (uint32_t)(mx - 1 + h * j) * E, xx[r]);
            }
            if (ymask & (1u << r)) {
                int my = 0;
                const int sy = OV ? classify(j, ny, h, A.active[1], &my)
                                  : edge_layer(j, ny, h, A.active[1], &my);
                T* pw = (sy == 1 ? A.side[1][1].psi_wr : A.side[1][0].psi_wr) + shot * A.psi_stride[1];
                T* xw = (sy == 1 ? B.xi_out[1][1] : B.xi_out[1][0]) + shot * A.xi_stride[1];
                const uint32_t oy = col + (uint32_t)my * pitch;
                stg(pw, oy, yh[r]);
                if (my == (OV && sy == 1 ? right_first(ny, h) : 1))
                    stg(pw, oy - pitch, r == 0 || OV ? yl[OV ? r : 0] : yh[r > 0 ? r - 1 : 0]);
                stg(xw, oy - pitch, yx[r]);
            }
        }
    }
}

}  // namespace awcpml
