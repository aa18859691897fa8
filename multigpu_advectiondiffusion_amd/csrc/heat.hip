// heat.hip -- the 3-D heat equation: several forward-Euler steps of the
// 7-point Laplacian in one pass (u' = u + dt*L7(u) on the Dirichlet interior,
// boundary copied; L7 is Compute_Laplace3d_O2, SingleGPU/Diffusion3d_
// baselineCode/kernels.cu:59-62, the update stage 1 of Compute_RK :130-132),
// the reference's 13-point SSP-RK3 step in one pass, and the 13-point
// operators of the drop-ins.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <tuple>
#include <type_traits>

#include "mgad_common.hpp"

namespace mgad {

// k_heat7_fe and k_heat13 march a 64 x TY tile of (x, y) columns through a chunk of
// z planes.  Wave w of the 256-thread block owns the tile rows w, w + 4, ...
// and keeps its columns' z neighbours in a register ring; each plane of the
// tile, with its x/y halo, passes through LDS once (double buffered, one
// barrier per plane), so every node comes from memory once per tile and the
// x/y neighbours are LDS reads.  Loads for the next plane are issued before
// the current one is computed, and every thread issues the same loads each
// plane (indices clamped into the grid), so the compiler's wait counts stay
// exact across the loop.  Tiles are ordered so that the blocks of one XCD
// take neighbouring tiles (their halos meet in that XCD's L2).
constexpr int kHeatTX = 64;

template <int N>
using Ic = std::integral_constant<int, N>;

using PlaneBuf = PlaneIo<double>;

// A halo entry of one thread: LDS (row, column) and the byte offset within a
// plane it is loaded from (clamped into the grid).
struct HaloSlot {
    int row = -1, col = 0;
    unsigned off = 0;
};

// The halo a thread loads, R nodes wide, for a tile of TY rows whose first
// node is (i0, j0): waves 0 and 1 the R rows below and above (R entries each),
// waves 2 and 3 the R columns left and right of every row.
template <int R, int TY>
__device__ __forceinline__ void heat_halo(HaloSlot (&h)[R], int w, int lane, int i0, int j0, int nx, int ny,
                                          int px) {
    constexpr int W = kHeatTX + 2 * R;
    static_assert(2 * R * TY <= 128, "x halo exceeds waves 2 and 3");
    if (w < 2) {
#pragma unroll
        for (int e = 0; e < R; e++) {
            const int jj = w == 0 ? max(j0 - R + e, 0) : min(j0 + TY + e, ny - 1);
            h[e].row = w == 0 ? e : TY + R + e;
            h[e].col = lane + R;
            h[e].off = 8u * static_cast<unsigned>(min(i0 + lane, nx - 1) + px * jj);
        }
    } else {
        const int t = (w - 2) * 64 + lane;
        if (t < 2 * R * TY) {
            const int c = t / TY, rr = t % TY;  // c: column 0..2R-1 left to right
            const int ii = c < R ? max(i0 - R + c, 0) : min(i0 + kHeatTX + c - R, nx - 1);
            h[0].row = rr + R;
            h[0].col = c < R ? c : W - 2 * R + c;
            h[0].off = 8u * static_cast<unsigned>(ii + px * min(j0 + rr, ny - 1));
        }
    }
}

// One forward-Euler step, u' = u + dt*L7(u) on the Dirichlet interior and
// u' = u on the boundary nodes.  L7 is Compute_Laplace3d_O2
// (Diffusion3d_baselineCode/kernels.cu:59-62) with 12*k as the source
// evaluates it, the update stage 1 of Compute_RK (:130-132); a step reads u
// once and writes u' once (16 B per node) instead of the reference's Lu
// round trip.
template <int TY>
__global__ __launch_bounds__(256) void k_heat7_fe(const double *__restrict__ u, double *__restrict__ v, int nx,
                                                  int ny, int nz, int ntx, int nty, int kchunk, double kx, double ky,
                                                  double kz, double dt) {
    constexpr int RPT = TY / 4, W = kHeatTX + 2;
    __shared__ double sp[2][TY + 2][W];
    const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tix = tile % ntx, tiy = (tile / ntx) % nty, tiz = tile / (ntx * nty);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i0 = tix * kHeatTX, j0 = tiy * TY, z0 = tiz * kchunk, z1 = min(z0 + kchunk, nz);
    const int i = i0 + lane;
    const size_t xy = static_cast<size_t>(nx) * ny;
    const unsigned pb = static_cast<unsigned>(xy * 8);
    unsigned lo[RPT], so[RPT];  // load and store offsets; so = pb drops the store
    bool keep[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int j = j0 + w + 4 * r;
        lo[r] = 8u * static_cast<unsigned>(min(i, nx - 1) + nx * min(j, ny - 1));
        so[r] = i < nx && j < ny ? lo[r] : pb;
        keep[r] = i == 0 || j == 0 || i == nx - 1 || j == ny - 1;
    }
    HaloSlot hs[1];
    heat_halo<1, TY>(hs, w, lane, i0, j0, nx, ny, nx);
    const bool hal = hs[0].row >= 0;
    const unsigned ho = hal ? hs[0].off : lo[0];  // lanes without a halo node repeat their own
    const double ckx = 12 * kx, cky = 12 * ky, ckz = 12 * kz;
    const int zl = min(z1, nz - 1);  // last plane this chunk reads
    // plane p of the own columns in slot (p - z0 + 1) & 3, of the halo in (p - z0) & 1
    double q[RPT][4] = {}, h[2] = {};
    {
        const PlaneBuf pa(u + xy * max(z0 - 1, 0), pb), pc(u + xy * z0, pb), pd(u + xy * min(z0 + 1, zl), pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            q[r][0] = pa.load(lo[r]);
            q[r][1] = pc.load(lo[r]);
            q[r][2] = pd.load(lo[r]);
        }
        h[0] = pc.load(ho);
    }
    int kb = z0;
    auto plane = [&](auto S) {
        constexpr int s = decltype(S)::value;
        const int k = kb + s;
        const PlaneBuf pn(u + xy * min(k + 2, zl), pb), ph(u + xy * min(k + 1, z1 - 1), pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) q[r][(s + 3) & 3] = pn.load(lo[r]);
        h[(s + 1) & 1] = ph.load(ho);
        double(*P)[W] = sp[s & 1];
#pragma unroll
        for (int r = 0; r < RPT; r++) P[w + 4 * r + 1][lane + 1] = q[r][(s + 1) & 3];
        if (hal) P[hs[0].row][hs[0].col] = h[s & 1];
        __syncthreads();
        const bool zb = k == 0 || k == nz - 1;
        const PlaneBuf pv(v + xy * k, pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            const int row = w + 4 * r + 1;
            const double cur = q[r][(s + 1) & 3], below = q[r][s & 3], above = q[r][(s + 2) & 3];
            // (u_e - 2 u_o) + u_w etc., the 2*u_o product exact
            const double Lu = ckx * (p2fma(-2.0, cur, P[row][lane + 2]) + P[row][lane]) +
                              cky * (p2fma(-2.0, cur, P[row + 1][lane + 1]) + P[row - 1][lane + 1]) +
                              ckz * (p2fma(-2.0, cur, above) + below);
            pv.store(so[r], (keep[r] || zb) ? cur : cur + dt * Lu);
        }
    };
    for (; kb < z1; kb += 4) {
        plane(Ic<0>{});
        if (kb + 1 >= z1) break;
        plane(Ic<1>{});
        if (kb + 2 >= z1) break;
        plane(Ic<2>{});
        if (kb + 3 >= z1) break;
        plane(Ic<3>{});
    }
}

// What k_heat13 writes: the 13-point operator itself (Call_Lu3d), the operator
// added to Lu over the Burgers viscous region (Call_Diff_), or stored there
// (the blocked heat code's Call_Lu3d).
enum : int { kHeatLu = 1, kHeatDiffB5 = 2, kHeatLuB5 = 3 };

// The 13-point operators of the drop-ins as a z-march.  Loads run D planes
// ahead of their first use: planes of the own columns sit in an 8-slot
// register ring (k-2..k+2 in use), the halo and Lu in 4-slot rings.
// MODE kHeatLu is Compute_Laplace3d (Diffusion3d_baselineCode/kernels.cu:
// 94-97): Lu on the interior 2..n-3 of every axis, with the
// CopyToConstantMemory coefficients.  MODE kHeatDiffB5 is
// Compute_Laplace_Async (SingleGPU/Burgers3d_WENO5/kernels.cu:444-494):
// nodes 3..n-4 in x and y, planes 3..nz-3, each axis's 4th-order difference
// summed from the low side (-u_{-2} + 16 u_{-1} ... instead of from the high
// side), added to Lu.  MODE kHeatLuB5 is Compute_Laplace3d_Async of
// SingleGPU/Diffusion3d_Blocking (kernels.cu:37-88, Call_Lu3d :187-191): the
// same region and sums, stored into Lu.
template <int TY, int D, int MODE>
__global__ __launch_bounds__(256) void k_heat13(const double *__restrict__ uin, double *Lu, int nx, int ny, int nz,
                                                int px, int ntx, int nty, int kchunk, double kx, double ky,
                                                double kz) {
    static_assert(D >= 1 && D <= 3, "prefetch distance");
    constexpr bool LU = MODE == kHeatLu || MODE == kHeatLuB5, B5 = MODE == kHeatDiffB5 || MODE == kHeatLuB5;
    constexpr int LO = B5 ? 3 : 2;  // first interior node of x and y (and z)
    constexpr int RPT = TY / 4, W = kHeatTX + 4;
    __shared__ double sp[2][TY + 4][W];
    const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tix = tile % ntx, tiy = (tile / ntx) % nty, tiz = tile / (ntx * nty);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i0 = LO + tix * kHeatTX, j0 = LO + tiy * TY, z0 = LO + tiz * kchunk, z1 = min(z0 + kchunk, nz - 2);
    const int i = i0 + lane;
    const size_t xy = static_cast<size_t>(px) * ny;
    const unsigned pb = static_cast<unsigned>(xy * 8);
    unsigned lo[RPT], so[RPT];  // load and store offsets; so = pb drops the store
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int j = j0 + w + 4 * r;
        lo[r] = 8u * static_cast<unsigned>(min(i, nx - 1) + px * min(j, ny - 1));
        so[r] = i < nx - LO && j < ny - LO ? lo[r] : pb;
    }
    HaloSlot hs[2];
    heat_halo<2, TY>(hs, w, lane, i0, j0, nx, ny, px);
    const unsigned ho0 = hs[0].row >= 0 ? hs[0].off : lo[0], ho1 = hs[1].row >= 0 ? hs[1].off : lo[0];
    // own plane p in slot (p - z0 + 2) & 7, halo and Lu plane p in (p - z0) & 3;
    // planes past the chunk's last read are clamped to it
    const int zq = z1 + 1, zh = z1 - 1;
    double q[RPT][8] = {}, h0[4] = {}, h1[4] = {}, o[RPT][4] = {};
#pragma unroll
    for (int t = 0; t < 4 + D; t++) {
        const PlaneBuf pq(uin + xy * min(z0 - 2 + t, zq), pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) q[r][t] = pq.load(lo[r]);
    }
#pragma unroll
    for (int t = 0; t < D; t++) {
        const PlaneBuf ph(uin + xy * min(z0 + t, zh), pb), po(Lu + xy * min(z0 + t, zh), pb);
        h0[t] = ph.load(ho0);
        h1[t] = ph.load(ho1);
        if (!LU) {
#pragma unroll
            for (int r = 0; r < RPT; r++) o[r][t] = po.load(lo[r]);
        }
    }
    int kb = z0;
    auto plane = [&](auto S) {
        constexpr int s = decltype(S)::value;
        const int k = kb + s;
        const PlaneBuf pn(uin + xy * min(k + 2 + D, zq), pb), ph(uin + xy * min(k + D, zh), pb),
            po(Lu + xy * min(k + D, zh), pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) q[r][(s + 4 + D) & 7] = pn.load(lo[r]);
        h0[(s + D) & 3] = ph.load(ho0);
        h1[(s + D) & 3] = ph.load(ho1);
        if (!LU) {
#pragma unroll
            for (int r = 0; r < RPT; r++) o[r][(s + D) & 3] = po.load(lo[r]);
        }
        double(*P)[W] = sp[s & 1];
#pragma unroll
        for (int r = 0; r < RPT; r++) P[w + 4 * r + 2][lane + 2] = q[r][(s + 2) & 7];
        if (hs[0].row >= 0) P[hs[0].row][hs[0].col] = h0[s & 3];
        if (hs[1].row >= 0) P[hs[1].row][hs[1].col] = h1[s & 3];
        __syncthreads();
        const PlaneBuf pv(Lu + xy * k, pb);
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            const int row = w + 4 * r + 2, x = lane + 2;
            const double c = q[r][(s + 2) & 7];
            double X, Y, Z;
            if (B5) {
                X = d4(P[row][x - 2], P[row][x - 1], c, P[row][x + 1], P[row][x + 2]);
                Y = d4(P[row - 2][x], P[row - 1][x], c, P[row + 1][x], P[row + 2][x]);
                Z = d4(q[r][s & 7], q[r][(s + 1) & 7], c, q[r][(s + 3) & 7], q[r][(s + 4) & 7]);
            } else {
                X = d4(P[row][x + 2], P[row][x + 1], c, P[row][x - 1], P[row][x - 2]);
                Y = d4(P[row + 2][x], P[row + 1][x], c, P[row - 1][x], P[row - 2][x]);
                Z = d4(q[r][(s + 4) & 7], q[r][(s + 3) & 7], c, q[r][(s + 1) & 7], q[r][s & 7]);
            }
            const double L = (kx * X + ky * Y) + kz * Z;
            pv.store(so[r], LU ? L : o[r][s & 3] + L);
        }
    };
    for (; kb < z1; kb += 8) {
        plane(Ic<0>{});
        if (kb + 1 >= z1) break;
        plane(Ic<1>{});
        if (kb + 2 >= z1) break;
        plane(Ic<2>{});
        if (kb + 3 >= z1) break;
        plane(Ic<3>{});
        if (kb + 4 >= z1) break;
        plane(Ic<4>{});
        if (kb + 5 >= z1) break;
        plane(Ic<5>{});
        if (kb + 6 >= z1) break;
        plane(Ic<6>{});
        if (kb + 7 >= z1) break;
        plane(Ic<7>{});
    }
}

// The value of the lane below (i - 1) or above (i + 1) in the wave, by a DPP
// wave shift (two 32-bit moves, no LDS).  Lane 0 (63) gets 0.
__device__ __forceinline__ double lane_below(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_above(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true));
}

// c ? a : b by halves, so that the compiler does not put the computation of
// b behind a branch per node (rows then could not overlap).
__device__ __forceinline__ double sel(bool c, double a, double b) {
    return __hiloint2double(c ? __double2hiint(a) : __double2hiint(b), c ? __double2loint(a) : __double2loint(b));
}

// The tile of one block of a fused step kernel: 64 columns (a wave's lanes) by
// E rows are loaded, and H nodes on each side that has a neighbouring tile are
// halo, computed again by that neighbour.  A side at the grid's edge has no
// halo: its boundary nodes are kept, so nothing from beyond them is used.
struct StepTile {
    int xs, ys;          // first column and row loaded
    int xo0, xo1;        // columns stored
    int yo0, yo1;        // rows stored
    int z0, z1;          // planes stored
};
template <int E, int H>
__device__ __forceinline__ StepTile step_tile(unsigned tile, int nx, int ny, int nz, int ntx, int nty, int kchunk) {
    const int tix = tile % ntx, tiy = (tile / ntx) % nty, tiz = tile / (ntx * nty);
    StepTile t;
    t.xs = tix * (64 - 2 * H);
    t.ys = tiy * (E - 2 * H);
    t.xo0 = tix == 0 ? 0 : t.xs + H;
    t.xo1 = tix == ntx - 1 ? nx : t.xs + 64 - H;
    t.yo0 = tiy == 0 ? 0 : t.ys + H;
    t.yo1 = tiy == nty - 1 ? ny : t.ys + E - H;
    t.z0 = tiz * kchunk;
    t.z1 = min(t.z0 + kchunk, nz);
    return t;
}

// One whole SSP-RK3 step of the reference heat equation (the 13-point operator
// of Compute_Laplace3d and the three stages of Compute_RK, Diffusion3d_
// baselineCode/kernels.cu:94-97, :127-140), v = step(u), in one launch: u is
// read once and v written once (16 B per node) where three stage launches move
// 64.  A block of W waves marches its tile up z, each wave owning R rows;
// at iteration k it loads plane k of u and computes stage 1 on plane k-2,
// stage 2 on plane k-4 and stage 3 on plane k-6, whose z neighbours sit in
// register rings (planes k-6..k of u, five planes of each stage).  x neighbours
// come by lane shifts; y neighbours outside the wave's own rows through LDS,
// one barrier per plane.  The boundary layers (two nodes) keep u at every
// stage and are stored too.  What bounds it: FP64 issue, about 29 slots a node
// and stage, on 1.8 times the nodes (6 halo nodes a side of 64 x 36), less the
// waves and planes that a stage does not need, which skip it (1.5 times is
// left).  One launch per stage was bound by memory: 161 us a step at
// 201x199x200 and 2021 at 512^3 (4.3 TB/s), now 66 and 920 us (146 Gpts/s).
template <int W, int R>
__global__ __launch_bounds__(64 * W) void k_heat13_step(const double *__restrict__ u, double *__restrict__ v, int nx,
                                                        int ny, int nz, int ntx, int nty, int kchunk, double kx,
                                                        double ky, double kz, double dt) {
    constexpr int H = 6, E = W * R;
    static_assert(R >= 2 && E > 2 * H, "tile");
    __shared__ double ex[2][3][W][R][64];  // the centre plane of each stage's input, every row
    const StepTile t = step_tile<E, H>(xcd_tile(blockIdx.x, gridDim.x), nx, ny, nz, ntx, nty, kchunk);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wb = max(w - 1, 0), wa = min(w + 1, W - 1);  // at the tile's ends: any rows, their values are not used
    const int i = t.xs + lane, jw = t.ys + w * R;
    const size_t xy = static_cast<size_t>(nx) * ny;
    const unsigned pb = static_cast<unsigned>(xy * 8);
    unsigned lo[R], so[R];  // load and store offsets; so = pb drops the store
    bool keep[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = jw + r;
        lo[r] = 8u * static_cast<unsigned>(min(i, nx - 1) + nx * min(j, ny - 1));
        so[r] = i >= t.xo0 && i < t.xo1 && j >= t.yo0 && j < t.yo1 ? lo[r] : pb;
        keep[r] = i < 2 || j < 2 || i >= nx - 2 || j >= ny - 2;
    }
    // rows of this wave that stage s needs: the stored rows and 2(3 - s) more
    auto rows_needed = [&](int s) { return jw + R > t.yo0 - 2 * (3 - s) && jw < t.yo1 + 2 * (3 - s) && jw < ny; };
    const bool need1 = rows_needed(1), need2 = rows_needed(2), need3 = rows_needed(3);
    // plane p of u in slot (p - ks) & 7, of the stages' results in (p - ks) & 3
    const int ks = max(t.z0 - H, 0), ke = t.z1 + H;
    double q0[R][8] = {}, q1[R][4] = {}, q2[R][4] = {}, nxt[R];
    {
        const PlaneBuf p(u + xy * ks, pb);
#pragma unroll
        for (int r = 0; r < R; r++) nxt[r] = p.load(lo[r]);
    }
    // -u_{+2} + 16 u_{+1} - 30 u + 16 u_{-1} - u_{-2} of each axis, with the
    // plane's values c[-2..R+1] of this column
    auto lap = [&](const double *c, int r, double up2, double up1, double dn1, double dn2) {
        const double m = c[r + 2];
        const double e1 = lane_above(m), w1 = lane_below(m);
        const double X = d4(lane_above(e1), e1, m, w1, lane_below(w1));
        const double Y = d4(c[r + 4], c[r + 3], m, c[r + 1], c[r]);
        const double Z = d4(up2, up1, m, dn1, dn2);
        return (kx * X + ky * Y) + kz * Z;
    };
    int kb = ks;
    auto plane = [&](auto S) {
        constexpr int s = decltype(S)::value, b = s & 1;
        const int k = kb + s;
#pragma unroll
        for (int r = 0; r < R; r++) q0[r][s & 7] = nxt[r];
        {
            const PlaneBuf p(u + xy * min(k + 1, nz - 1), pb);
#pragma unroll
            for (int r = 0; r < R; r++) nxt[r] = p.load(lo[r]);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            ex[b][0][w][r][lane] = q0[r][(s - 2) & 7];
            ex[b][1][w][r][lane] = q1[r][(s - 4) & 3];
            ex[b][2][w][r][lane] = q2[r][(s - 6) & 3];
        }
        __syncthreads();
        double n1[R], n2[R];
        const bool do1 = need1 && k >= max(t.z0 - 2, 2), do2 = need2 && k >= max(t.z0 + 2, 4),
                   do3 = need3 && k >= t.z0 + 6;
        if (do1) {
            const bool zb = k - 2 < 2 || k - 2 >= nz - 2;
            double c[R + 4];
            c[0] = ex[b][0][wb][R - 2][lane];
            c[1] = ex[b][0][wb][R - 1][lane];
            c[R + 2] = ex[b][0][wa][0][lane];
            c[R + 3] = ex[b][0][wa][1][lane];
#pragma unroll
            for (int r = 0; r < R; r++) c[r + 2] = q0[r][(s - 2) & 7];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const double L = lap(c, r, q0[r][s & 7], q0[r][(s - 1) & 7], q0[r][(s - 3) & 7], q0[r][(s - 4) & 7]);
                n1[r] = sel(keep[r] || zb, c[r + 2], c[r + 2] + dt * L);
            }
        }
        if (do2) {
            const bool zb = k - 4 < 2 || k - 4 >= nz - 2;
            double c[R + 4];
            c[0] = ex[b][1][wb][R - 2][lane];
            c[1] = ex[b][1][wb][R - 1][lane];
            c[R + 2] = ex[b][1][wa][0][lane];
            c[R + 3] = ex[b][1][wa][1][lane];
#pragma unroll
            for (int r = 0; r < R; r++) c[r + 2] = q1[r][(s - 4) & 3];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const double L = lap(c, r, n1[r], q1[r][(s - 3) & 3], q1[r][(s - 5) & 3], q1[r][(s - 6) & 3]);
                const double x = 0.75 * q0[r][(s - 4) & 7] + 0.25 * (c[r + 2] + dt * L);
                n2[r] = sel(keep[r] || zb, c[r + 2], x);
            }
        }
        if (do3) {
            const bool zb = k - 6 < 2 || k - 6 >= nz - 2;
            double c[R + 4];
            c[0] = ex[b][2][wb][R - 2][lane];
            c[1] = ex[b][2][wb][R - 1][lane];
            c[R + 2] = ex[b][2][wa][0][lane];
            c[R + 3] = ex[b][2][wa][1][lane];
#pragma unroll
            for (int r = 0; r < R; r++) c[r + 2] = q2[r][(s - 6) & 3];
            const PlaneBuf pv(v + xy * (k - 6), pb);
            // (uo + 2 (u + dt L)) / 3: the quotient of div_by where |a| is in
            // [2^-900, 2^1000), one range test on the high words for the rows
            constexpr unsigned lo32 = (1023u - 900u) << 20, hi32 = (1023u + 1000u) << 20;
            double a[R], x[R];
            unsigned m = 0u;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const double L = lap(c, r, n2[r], q2[r][(s - 5) & 3], q2[r][(s - 7) & 3], q2[r][(s - 8) & 3]);
                a[r] = p2fma(2.0, c[r + 2] + dt * L, q0[r][(s - 6) & 7]);
                const double q = a[r] * (1.0 / 3.0);
                x[r] = __builtin_fma(__builtin_fma(-3.0, q, a[r]), 1.0 / 3.0, q);
                m = max(m, (static_cast<unsigned>(__double2hiint(a[r])) & 0x7fffffffu) - lo32);
            }
            if (__builtin_expect(m >= hi32 - lo32, 0)) {
#pragma unroll
                for (int r = 0; r < R; r++) x[r] = a[r] / 3.0;
            }
#pragma unroll
            for (int r = 0; r < R; r++) pv.store(so[r], sel(keep[r] || zb, c[r + 2], x[r]));
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            q1[r][(s - 2) & 3] = n1[r];
            q2[r][(s - 4) & 3] = n2[r];
        }
    };
    for (; kb < ke; kb += 8) {
        plane(Ic<0>{});
        if (kb + 1 >= ke) break;
        plane(Ic<1>{});
        if (kb + 2 >= ke) break;
        plane(Ic<2>{});
        if (kb + 3 >= ke) break;
        plane(Ic<3>{});
        if (kb + 4 >= ke) break;
        plane(Ic<4>{});
        if (kb + 5 >= ke) break;
        plane(Ic<5>{});
        if (kb + 6 >= ke) break;
        plane(Ic<6>{});
        if (kb + 7 >= ke) break;
        plane(Ic<7>{});
    }
}

// T forward-Euler steps of k_heat7_fe in one launch, v = step^T(u): u is read
// once and v written once where T launches move 16 B a node each.  The march
// is that of k_heat13_step: at iteration k step l = 1..T is computed on plane
// k - l, whose z neighbours are the last two planes of step l - 1 in registers
// and the one just computed.  At 512^3 one step a launch is bound by memory
// (5.6 TB/s, 388 us a step); with 4 (174 us) the FP64 issue time is about 90
// us (16 slots a node and step on 64/(64-2T) * E/(E-2T) times the nodes) and
// the memory time 100 us, and the barrier of each plane keeps them from
// overlapping fully.  At 64^3 it is the launch and first-load latency, paid
// once for T steps (3.2 -> 2.4 us a step).
template <int T, int W, int R, int D>
__global__ __launch_bounds__(64 * W) void k_heat7_steps(const double *__restrict__ u, double *__restrict__ v, int nx,
                                                        int ny, int nz, int ntx, int nty, int kchunk, double kx,
                                                        double ky, double kz, double dt) {
    constexpr int H = T, E = W * R;
    static_assert(T >= 2 && E > 2 * H, "tile");
    __shared__ double ex[2][T][W][2][64];  // first and last row of each step's centre plane
    const StepTile t = step_tile<E, H>(xcd_tile(blockIdx.x, gridDim.x), nx, ny, nz, ntx, nty, kchunk);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wb = max(w - 1, 0), wa = min(w + 1, W - 1);  // at the tile's ends: any rows, their values are not used
    const int i = t.xs + lane, jw = t.ys + w * R;
    const size_t xy = static_cast<size_t>(nx) * ny;
    const unsigned pb = static_cast<unsigned>(xy * 8);
    unsigned lo[R], so[R];  // load and store offsets; so = pb drops the store
    bool keep[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = jw + r;
        lo[r] = 8u * static_cast<unsigned>(min(i, nx - 1) + nx * min(j, ny - 1));
        so[r] = i >= t.xo0 && i < t.xo1 && j >= t.yo0 && j < t.yo1 ? lo[r] : pb;
        keep[r] = i < 1 || j < 1 || i >= nx - 1 || j >= ny - 1;
    }
    const double ckx = 12 * kx, cky = 12 * ky, ckz = 12 * kz;
    const int ks = max(t.z0 - H, 0), ke = t.z1 + H;
    // q[l]: plane p of step l's result (l = 0: u) in slot (p - ks) & 1; nxt:
    // planes k..k+D-1 of u, plane p in slot (p - ks) % D
    double q[T][R][2] = {}, nxt[R][D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        const PlaneBuf p(u + xy * min(ks + d, nz - 1), pb);
#pragma unroll
        for (int r = 0; r < R; r++) nxt[r][d] = p.load(lo[r]);
    }
    int kb = ks;
    auto plane = [&](auto S) {
        constexpr int s = decltype(S)::value, b = s & 1;
        const int k = kb + s;
        double n[R];  // the newest plane of step l, k - l
#pragma unroll
        for (int r = 0; r < R; r++) n[r] = nxt[r][s % D];
        {
            const PlaneBuf p(u + xy * min(k + D, nz - 1), pb);
#pragma unroll
            for (int r = 0; r < R; r++) nxt[r][s % D] = p.load(lo[r]);
        }
#pragma unroll
        for (int l = 0; l < T; l++) {
            ex[b][l][w][0][lane] = q[l][0][(s + l + 1) & 1];
            ex[b][l][w][1][lane] = q[l][R - 1][(s + l + 1) & 1];
        }
        __syncthreads();
        double hb[T], ha[T];  // the rows below and above this wave's
#pragma unroll
        for (int l = 0; l < T; l++) {
            hb[l] = ex[b][l][wb][1][lane];
            ha[l] = ex[b][l][wa][0][lane];
        }
#pragma unroll
        for (int l = 0; l < T; l++) {
            // step l + 1 on plane k - l - 1, if this wave's rows and the plane need it
            const int p = k - l - 1, m = T - 1 - l;
            const bool go = jw + R > t.yo0 - m && jw < t.yo1 + m && jw < ny && p >= max(t.z0 - m, 0);
            double x[R];
            if (go) {
                const bool zb = p == 0 || p >= nz - 1;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const double c = q[l][r][(s + l + 1) & 1], dn = q[l][r][(s + l) & 1];
                    const double N = r + 1 < R ? q[l][r + 1][(s + l + 1) & 1] : ha[l];
                    const double Sv = r > 0 ? q[l][r - 1][(s + l + 1) & 1] : hb[l];
                    // (u_e - 2 u_o) + u_w etc., the 2*u_o product exact
                    const double Lu = ckx * (p2fma(-2.0, c, lane_above(c)) + lane_below(c)) +
                                      cky * (p2fma(-2.0, c, N) + Sv) + ckz * (p2fma(-2.0, c, n[r]) + dn);
                    x[r] = sel(keep[r] || zb, c, c + dt * Lu);
                }
                if (l == T - 1) {
                    const PlaneBuf pv(v + xy * p, pb);
#pragma unroll
                    for (int r = 0; r < R; r++) pv.store(so[r], x[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                q[l][r][(s + l) & 1] = n[r];
                n[r] = x[r];
            }
        }
    };
    static_assert(4 % D == 0, "slots of a march unrolled by 4");
    for (; kb < ke; kb += 4) {
        plane(Ic<0>{});
        if (kb + 1 >= ke) break;
        plane(Ic<1>{});
        if (kb + 2 >= ke) break;
        plane(Ic<2>{});
        if (kb + 3 >= ke) break;
        plane(Ic<3>{});
    }
}

// T forward-Euler steps in one launch for grids whose blocks fit one round:
// the same tiles as k_heat7_steps with 16 rows, one row a wave, but a thread
// holds all kCubeZ + 2T planes of its column in registers and takes the steps
// one after the other, the planes and rows needed shrinking by one a side.
// All loads are in flight at once and there is one barrier a step, where the
// march waits for each of its planes.  Of a launch's 8 us at 64^3 (4 steps;
// 9.7 by the march, 4 launches of one step 12.9) 2.4 are the launch, the rest
// is the serial work of a CU's one block, 3.8 times the nodes of the tile.
constexpr int kCubeRows = 16, kCubeZ = 2;

template <int T>
__global__ __launch_bounds__(64 * kCubeRows) void k_heat7_cube(const double *__restrict__ u, double *__restrict__ v,
                                                               int nx, int ny, int nz, int ntx, int nty, double kx,
                                                               double ky, double kz, double dt) {
    constexpr int H = T, E = kCubeRows, NP = kCubeZ + 2 * T;
    static_assert(E > 2 * H, "tile");
    // planes 1..NP-2 for the first step, 2..NP-3 for the second, and so on in turn
    __shared__ double ex0[E][NP - 2][64], ex1[E][NP - 4][64];
    const StepTile t = step_tile<E, H>(xcd_tile(blockIdx.x, gridDim.x), nx, ny, nz, ntx, nty, kCubeZ);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wb = max(w - 1, 0), wa = min(w + 1, E - 1);  // at the tile's ends: any rows, their values are not used
    const int i = t.xs + lane, j = t.ys + w;
    const size_t xy = static_cast<size_t>(nx) * ny;
    const unsigned pb = static_cast<unsigned>(xy * 8);
    const unsigned lo = 8u * static_cast<unsigned>(min(i, nx - 1) + nx * min(j, ny - 1));
    const unsigned so = i >= t.xo0 && i < t.xo1 && j >= t.yo0 && j < t.yo1 ? lo : pb;  // pb drops the store
    const bool keep = i < 1 || j < 1 || i >= nx - 1 || j >= ny - 1;
    const double ckx = 12 * kx, cky = 12 * ky, ckz = 12 * kz;
    double q[NP];  // plane z0 - T + p in q[p]
#pragma unroll
    for (int p = 0; p < NP; p++)
        q[p] = PlaneBuf(u + xy * min(max(t.z0 - T + p, 0), nz - 1), pb).load(lo);
#pragma unroll
    for (int l = 0; l < T; l++) {
        double(*const ex)[64] = l & 1 ? ex1[w] : ex0[w];
        const double(*const exb)[64] = l & 1 ? ex1[wb] : ex0[wb];
        const double(*const exa)[64] = l & 1 ? ex1[wa] : ex0[wa];
#pragma unroll
        for (int p = l + 1; p < NP - 1 - l; p++) ex[p - l - 1][lane] = q[p];
        __syncthreads();
        const int m = T - 1 - l;
        if (j + 1 > t.yo0 - m && j < t.yo1 + m && j < ny) {
            double dn = q[l];
#pragma unroll
            for (int p = l + 1; p < NP - 1 - l; p++) {
                const double c = q[p];
                const int k = t.z0 - T + p;
                // (u_e - 2 u_o) + u_w etc., the 2*u_o product exact
                const double Lu = ckx * (p2fma(-2.0, c, lane_above(c)) + lane_below(c)) +
                                  cky * (p2fma(-2.0, c, exa[p - l - 1][lane]) + exb[p - l - 1][lane]) +
                                  ckz * (p2fma(-2.0, c, q[p + 1]) + dn);
                q[p] = sel(keep || k <= 0 || k >= nz - 1, c, c + dt * Lu);
                dn = c;
            }
        }
    }
#pragma unroll
    for (int p = T; p < T + kCubeZ; p++)
        if (t.z0 - T + p < t.z1) PlaneBuf(v + xy * (t.z0 - T + p), pb).store(so, q[p]);
}

namespace {

// Tile heights and the 13-point kernel's prefetch distance, from sweeps at
// 512^3 (7-point: 16 rows 5.6 TB/s vs 32 rows 5.5; 13-point: 32 rows
// 4.9 TB/s vs 16 rows 4.0, distance 2 no faster than 1).
constexpr int kHeat7TY = 16, kHeat13TY = 32, kHeat13D = 1;

long device_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus;
}

struct HeatGrid {
    int ntx, nty, kc;
    unsigned blocks;
    long cost;  // step_grid's
};

HeatGrid heat_tiles(unsigned ex, unsigned ey, int ty) {
    HeatGrid g{};
    g.ntx = static_cast<int>((ex + kHeatTX - 1) / kHeatTX);
    g.nty = static_cast<int>((ey + ty - 1) / ty);
    return g;
}

// 7-point: z chunks as long as possible while the grid keeps >= 512 blocks
// (two per CU), down to one plane.
HeatGrid heat7_grid(unsigned nx, unsigned ny, unsigned nz) {
    HeatGrid g = heat_tiles(nx, ny, kHeat7TY);
    const long bxy = static_cast<long>(g.ntx) * g.nty;
    int kc = static_cast<int>(nz);
    while (kc > 1 && bxy * ((nz + kc - 1) / kc) < 512) kc = (kc + 1) / 2;
    g.kc = kc;
    g.blocks = static_cast<unsigned>(bxy * ((nz + kc - 1) / kc));
    return g;
}

// 13-point operators over the (ex, ey, ez) interior: the z chunk among 8..64 planes
// that minimises (rounds of resident blocks) x (planes each block reads,
// chunk + 4), so a small grid runs in one round of long chunks and a large
// one in a few rounds.
HeatGrid heat13_grid(unsigned ex, unsigned ey, unsigned ez) {
    HeatGrid g = heat_tiles(ex, ey, kHeat13TY);
    const long bxy = static_cast<long>(g.ntx) * g.nty;
    int dev = 0, cus = 0, per = 0;
    long cap = 256;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void *>(&k_heat13<kHeat13TY, kHeat13D, kHeatDiffB5>), 256, 0) == hipSuccess &&
        per > 0)
        cap = static_cast<long>(cus) * per;
    long best = -1;
    for (int kc : {8, 12, 16, 24, 32, 48, 64}) {
        const int k = std::min(kc, static_cast<int>(ez));
        const long blocks = bxy * ((ez + k - 1) / k);
        const long cost = ((blocks + cap - 1) / cap) * (k + 4);
        if (best < 0 || cost < best) {
            best = cost;
            g.kc = k;
            g.blocks = static_cast<unsigned>(blocks);
        }
    }
    return g;
}

// Tiles of `full` nodes that cover n with h halo nodes on each shared side
// (see StepTile).
int step_tiles(unsigned n, int full, int h) {
    const int m = static_cast<int>(n);
    return m <= full ? 1 : 1 + (m - full + full - 2 * h - 1) / (full - 2 * h);
}

// Grid of a fused step kernel whose block loads 64 columns by `e` rows with
// `h` halo nodes and computes `lev` stages (or steps), each needing 2h/lev more
// planes than the next: the z chunk that minimises (blocks a CU runs) x
// (planes a block computes, over all stages), the blocks taken by a CU one
// after the other or side by side at the same rate.
HeatGrid step_grid(unsigned nx, unsigned ny, unsigned nz, int e, int h, int lev) {
    HeatGrid g{};
    g.ntx = step_tiles(nx, 64, h);
    g.nty = step_tiles(ny, e, h);
    const long bxy = static_cast<long>(g.ntx) * g.nty, cus = device_cus();
    long best = -1;
    for (int n = 1; n <= static_cast<int>(nz); n++) {
        const int kc = (static_cast<int>(nz) + n - 1) / n;
        if (n > 1 && (n - 1) * kc >= static_cast<int>(nz)) continue;
        const long blocks = bxy * n;
        const long cost = ((blocks + cus - 1) / cus) * (static_cast<long>(lev) * kc + (lev - 1) * h + lev);
        if (best < 0 || cost < best) {
            best = g.cost = cost;
            g.kc = kc;
            g.blocks = static_cast<unsigned>(blocks);
        }
        if (blocks >= 8 * cus) break;
    }
    return g;
}

// Waves and rows per wave of a fused 13-point step's block: 3 waves a SIMD
// hide the FP64 latency that 2 do not (us a step, 201x199x200 / 512^3: 8 waves
// of 4 rows 82 / 966, of 5 rows 85 / 1006; 12 waves of 3 rows 74 / 915, of 4
// rows, which spill, 146 / 2007).
constexpr int kHeat13W = 12, kHeat13R = 3;

int enqueue_heat13(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, DiffCoef c, double dt, const double *u,
                   double *v) {
    const HeatGrid g = step_grid(nx, ny, nz, kHeat13W * kHeat13R, 6, 3);
    hipLaunchKernelGGL((k_heat13_step<kHeat13W, kHeat13R>), dim3(g.blocks), dim3(64 * kHeat13W), 0, s, u, v, (int)nx, (int)ny,
                       (int)nz, g.ntx, g.nty, g.kc, c.kx, c.ky, c.kz, dt);
    return check_launch();
}

template <int T, int W, int R, int D>
void launch_heat7(hipStream_t s, const HeatGrid &g, unsigned nx, unsigned ny, unsigned nz, double kx, double ky,
                  double kz, double dt, const double *u, double *v) {
    hipLaunchKernelGGL((k_heat7_steps<T, W, R, D>), dim3(g.blocks), dim3(64 * W), 0, s, u, v, (int)nx, (int)ny,
                       (int)nz, g.ntx, g.nty, g.kc, kx, ky, kz, dt);
}

// Grid of t forward-Euler steps in one launch: tiles of 36 rows (12 waves of 3
// rows) or of 16 (8 waves of 2), whichever gives a CU less work (rows x planes
// over the steps).  The low tile leaves more halo rows but fills the CUs at
// small grids: us a step, 4 steps a launch, low / tall: 64^3 2.43 / 3.17,
// 128^3 8.1 / 6.4, 201x199x200 18.2 / 14.2, 512^3 216 / 172.  Taller tiles (48
// rows, 6 a wave) and fewer waves of more rows (8 of 4) were no faster.
HeatGrid heat7_steps_grid(unsigned nx, unsigned ny, unsigned nz, int t, bool &tall) {
    const HeatGrid lo = step_grid(nx, ny, nz, 16, t, t), hi = step_grid(nx, ny, nz, 36, t, t);
    tall = t > 4 || 36 * hi.cost < 16 * lo.cost;
    return tall ? hi : lo;
}

// Grid of k_heat7_cube, or 0 blocks where it is not taken: t of 2..4, and one
// round of at most a block a CU.
HeatGrid heat7_cube_grid(unsigned nx, unsigned ny, unsigned nz, int t) {
    HeatGrid g{};
    if (t < 2 || t > 4) return g;
    g.ntx = step_tiles(nx, 64, t);
    g.nty = step_tiles(ny, kCubeRows, t);
    g.kc = kCubeZ;
    const long blocks = static_cast<long>(g.ntx) * g.nty * ((nz + kCubeZ - 1) / kCubeZ);
    g.blocks = blocks <= device_cus() ? static_cast<unsigned>(blocks) : 0u;
    return g;
}

// t forward-Euler steps u -> v in one launch (t <= 5).
int enqueue_heat7(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, double kx, double ky, double kz, double dt,
                  const double *u, double *v, int t) {
    if (t == 1) {
        const HeatGrid g = heat7_grid(nx, ny, nz);
        hipLaunchKernelGGL(k_heat7_fe<kHeat7TY>, dim3(g.blocks), dim3(256), 0, s, u, v, (int)nx, (int)ny, (int)nz,
                           g.ntx, g.nty, g.kc, kx, ky, kz, dt);
        return check_launch();
    }
    const HeatGrid cg = heat7_cube_grid(nx, ny, nz, t);
    if (cg.blocks) {
        auto go = [&](auto TT) {
            hipLaunchKernelGGL((k_heat7_cube<decltype(TT)::value>), dim3(cg.blocks), dim3(64 * kCubeRows), 0, s, u, v,
                               (int)nx, (int)ny, (int)nz, cg.ntx, cg.nty, kx, ky, kz, dt);
        };
        if (t == 2)
            go(Ic<2>{});
        else if (t == 3)
            go(Ic<3>{});
        else
            go(Ic<4>{});
        return check_launch();
    }
    bool tall;
    const HeatGrid g = heat7_steps_grid(nx, ny, nz, t, tall);
    auto go = [&](auto TT) {
        constexpr int T = decltype(TT)::value;
        if (tall)
            launch_heat7<T, 12, 3, T <= 4 ? 2 : 1>(s, g, nx, ny, nz, kx, ky, kz, dt, u, v);
        else
            launch_heat7<T, 8, 2, 2>(s, g, nx, ny, nz, kx, ky, kz, dt, u, v);
    };
    if (t == 2)
        go(Ic<2>{});
    else if (t == 3)
        go(Ic<3>{});
    else if (t == 4)
        go(Ic<4>{});
    else
        launch_heat7<5, 12, 3, 1>(s, g, nx, ny, nz, kx, ky, kz, dt, u, v);
    return check_launch();
}

// Most steps a launch takes: 4, or 5 where the tall tile is taken.  A
// fifth step costs the tall tile next to nothing (us a step with 1, 2, 3, 4, 5
// steps a launch: 512^3 388, 301, 185, 174, 177; 201x199x200 26.4, 16.9, 13.0,
// 12.4, 12.3) and saves launches that would only make their number even; the
// low tile loses more of its rows to the halo (64^3 by the march: 3.23, 2.59,
// 2.47, 2.43, 2.88).
int heat7_most_steps(unsigned nx, unsigned ny, unsigned nz) {
    bool tall;
    heat7_steps_grid(nx, ny, nz, 4, tall);
    return tall ? 5 : 4;
}

// nsteps steps as an even number of launches (u -> w -> u ...), as few as the
// most steps a launch takes allow and as equal as possible; a single step is
// copied back.
int enqueue_heat(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, double kx, double ky,
                 double kz, double dt, double *u, double *w, int nsteps) {
    const int tmax = heat7_most_steps(nx, ny, nz);
    int launches = (nsteps + tmax - 1) / tmax;
    if (launches < nsteps) launches += launches & 1;
    for (int it = 0, done = 0; it < launches; it++) {
        const int t = (nsteps - done + launches - it - 1) / (launches - it);
        const int st = enqueue_heat7(s, nx, ny, nz, kx, ky, kz, dt, (it & 1) ? w : u, (it & 1) ? u : w, t);
        if (st) return st;
        done += t;
    }
    if (launches & 1)
        return check_hip(hipMemcpyAsync(u, w, sizeof(double) * nx * ny * nz,
                                        hipMemcpyDeviceToDevice, s));
    return MGAD_OK;
}

}  // namespace

// Compute_Laplace3d (Diffusion3d_baselineCode/kernels.cu:94-97) into Lu on
// the interior 2..n-3 with the LDS z-march (Call_Lu3d):
// row pitch px, planes of px*ny < 2^29 values.
int heat13_lu_launch(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, unsigned px, const double *u,
                     double *Lu) {
    const HeatGrid g = heat13_grid(nx - 4, ny - 4, nz - 4);
    const DiffCoef c = diff_coef();
    const auto kern = k_heat13<kHeat13TY, kHeat13D, kHeatLu>;
    hipLaunchKernelGGL(kern, dim3(g.blocks), dim3(256), 0, s, u, Lu, (int)nx, (int)ny, (int)nz, (int)px, g.ntx,
                       g.nty, g.kc, c.kx, c.ky, c.kz);
    return check_launch();
}

// Compute_Laplace_Async (SingleGPU/Burgers3d_WENO5/kernels.cu:444-494,
// Call_Diff_): Lu += the 13-point operator on nodes 3..n-4 in x and y and
// planes 3..nz-3, with the same z-march; row pitch px, planes of
// px*ny < 2^29 values, nx, ny >= 7, nz >= 6.
int diff13_b5_launch(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, unsigned px, const double *u, double *Lu,
                     double kx, double ky, double kz) {
    const HeatGrid g = heat13_grid(nx - 6, ny - 6, nz - 5);
    const auto kern = k_heat13<kHeat13TY, kHeat13D, kHeatDiffB5>;
    hipLaunchKernelGGL(kern, dim3(g.blocks), dim3(256), 0, s, u, Lu, (int)nx, (int)ny, (int)nz, (int)px, g.ntx,
                       g.nty, g.kc, kx, ky, kz);
    return check_launch();
}

// Compute_Laplace3d_Async of SingleGPU/Diffusion3d_Blocking (kernels.cu:
// 37-88, launched by Call_Lu3d :187-191 with kstart 3, kstop nz-2): Lu = the
// 13-point operator on nodes 3..n-4 in x and y and planes 3..nz-3, summed
// as Call_Diff_'s operator; row pitch px, planes of px*ny < 2^29 values,
// nx, ny >= 7, nz >= 6.
int lu13_b5_launch(hipStream_t s, unsigned nx, unsigned ny, unsigned nz, unsigned px, const double *u, double *Lu) {
    const HeatGrid g = heat13_grid(nx - 6, ny - 6, nz - 5);
    const DiffCoef c = diff_coef();
    const auto kern = k_heat13<kHeat13TY, kHeat13D, kHeatLuB5>;
    hipLaunchKernelGGL(kern, dim3(g.blocks), dim3(256), 0, s, u, Lu, (int)nx, (int)ny, (int)nz, (int)px, g.ntx,
                       g.nty, g.kc, c.kx, c.ky, c.kz);
    return check_launch();
}

namespace {

struct HeatKey {
    hipStream_t s;
    unsigned nx, ny, nz;
    double kx, ky, kz, dt;
    double *u, *w;
    bool operator<(const HeatKey &o) const {
        return std::tie(s, nx, ny, nz, kx, ky, kz, dt, u, w) <
               std::tie(o.s, o.nx, o.ny, o.nz, o.kx, o.ky, o.kz, o.dt, o.u, o.w);
    }
};

}  // namespace
}  // namespace mgad

using namespace mgad;

extern "C" int mgad_heat7_fe_steps(hipStream_t stream, unsigned int nx, unsigned int ny,
                                   unsigned int nz, double kx, double ky, double kz, double dt,
                                   double *u, double *w, int nsteps, int use_graph) {
    if (nx < 3 || ny < 3 || nz < 3 || 1ull * nx * ny * nz >= (1ull << 31) || 1ull * nx * ny >= (1ull << 29) || !u ||
        !w || u == w || nsteps < 0) {
        set_error(MGAD_ERR_INVALID_ARG);
        return MGAD_ERR_INVALID_ARG;
    }
    if (!use_graph || stream == nullptr || nsteps == 0)
        return enqueue_heat(stream, nx, ny, nz, kx, ky, kz, dt, u, w, nsteps);
    std::lock_guard<std::recursive_mutex> lock(host_mutex());
    if (const int st = refuse_capture(stream)) return st;
    // whole graphs of 24 pairs of full launches, u -> w -> u, and the rest as a
    // call without a graph; where that would be less than two full launches it
    // gets a graph's steps too (launches of one step take twice the time a step)
    const int t = heat7_most_steps(nx, ny, nz), per = graph_steps(2), full = per * 2 * t;
    int graphs = nsteps / full;
    const int left = nsteps - graphs * full;
    if (graphs > 0 && left > 0 && left < 2 * t) graphs--;
    int st = MGAD_OK;
    if (graphs > 0) {
        static std::map<HeatKey, KeptGraph> cache;
        const HeatKey key{stream, nx, ny, nz, kx, ky, kz, dt, u, w};
        st = replay_steps(cache, 16, key, stream, graphs * per, per, [&] {
            const int r = enqueue_heat7(stream, nx, ny, nz, kx, ky, kz, dt, u, w, t);
            return r ? r : enqueue_heat7(stream, nx, ny, nz, kx, ky, kz, dt, w, u, t);
        });
    }
    return st ? st : enqueue_heat(stream, nx, ny, nz, kx, ky, kz, dt, u, w, nsteps - graphs * full);
}

// The reference's heat step fused (SingleGPU/Diffusion3d_baselineCode/
// main.cpp:108-121): per step uo <- u, then for rk = 1..3 Call_Lu3d and
// Call_RK3d(rk), as one launch per step; the two ghost layers keep u.
extern "C" int mgad_heat13_rk3_steps(hipStream_t stream, unsigned int nx, unsigned int ny, unsigned int nz, double dt,
                                     double *u, double *w1, double *w2, int nsteps, int use_graph) {
    if (nx < 5 || ny < 5 || nz < 5 || 1ull * nx * ny * nz >= (1ull << 31) || 1ull * nx * ny >= (1ull << 29) || !u ||
        !w1 || !w2 || u == w1 || u == w2 || w1 == w2 || nsteps < 0) {
        set_error(MGAD_ERR_INVALID_ARG);
        return MGAD_ERR_INVALID_ARG;
    }
    if (nsteps == 0) return MGAD_OK;
    const DiffCoef c = diff_coef();
    std::unique_lock<std::recursive_mutex> lock(host_mutex(), std::defer_lock);
    const bool graph = use_graph && stream != nullptr;
    if (graph) {
        lock.lock();
        if (const int st = refuse_capture(stream)) return st;
    }
    // a step goes u -> w1 or w1 -> u; an odd count's last one is copied back
    const int pairs = nsteps / 2;
    int st = MGAD_OK;
    auto pair = [&] {
        const int r = enqueue_heat13(stream, nx, ny, nz, c, dt, u, w1);
        return r ? r : enqueue_heat13(stream, nx, ny, nz, c, dt, w1, u);
    };
    if (!graph) {
        for (int s = 0; s < pairs && !st; s++) st = pair();
    } else {
        using Key = std::tuple<hipStream_t, unsigned, unsigned, unsigned, double, double, double, double, double *,
                               double *>;
        static std::map<Key, KeptGraph> cache;
        const Key key{stream, nx, ny, nz, c.kx, c.ky, c.kz, dt, u, w1};
        st = replay_steps(cache, 16, key, stream, pairs, graph_steps(2), pair);
    }
    if (!st && (nsteps & 1)) {
        st = enqueue_heat13(stream, nx, ny, nz, c, dt, u, w1);
        if (!st)
            st = check_hip(hipMemcpyAsync(u, w1, sizeof(double) * nx * ny * nz, hipMemcpyDeviceToDevice, stream));
    }
    return st;
}

