// burgers_ref.hip -- the reference's own Burgers step, fused: one launch per
// SSP-RK3 stage that gives the same u as the drop-in sequence
//   Call_Adv_x, Call_Adv_y, Call_Adv_z, [Call_Diff_], Call_sspRK
// (SingleGPU/Burgers3d_WENO5/main.cpp:139-149): local Lax-Friedrichs split
// (alpha = |u_i|), WENO5 faces, the optional 13-point viscous term with the
// CopyToConstantMemory coefficients, and the SSP-RK3 combine on the interior
// nodes 3..n-4 of every axis; the three ghost layers are never written.
//
// Per interior node the right-hand side is accumulated in the drop-ins' order
//   Lu = -(F_{i+1/2}-F_{i-1/2})/dx;  Lu -= (G..)/dy;  Lu -= (H..)/dz;
//   Lu += kx*(-u[i-2] + 16u[i-1] - 30u[i] + 16u[i+1] - u[i+2]) + ky*(..) + kz*(..)
// (kernels.cu:197-394, 474-476) and the stage is Compute_RK (kernels.cu:520-527).
// The tile / z-march structure is that of the periodic stage kernel, over the
// interior instead of the whole periodic grid: tiles start at node 3, the last
// ones may be partial (their extra columns load clamped, valid addresses and
// store nothing), and halos read the ghost layers instead of wrapping.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <tuple>
#include <type_traits>

#include "burgers_periodic.hpp"

namespace mgad {

struct RefArgs {
    int nx, ny, nz, kchunk, ntx, nty;
    double dx, dy, dz, rdx, rdy, rdz;
    // max|u| slots: [0] u^n, [1] u^(1), [2] u^(2) (interior values written by
    // the stages), [3] all of u at the call's start (covers the ghost layers,
    // which no stage writes)
    unsigned long long *amax;
};

template <int TX, int TY>
struct RefSmem {
    double2 P[TY + 6][TX + 6];  // (f+, f-) of the current plane, tile + 3-node halo
    double U[TY + 6][TX + 6];   // u of the same nodes (viscous term)
    double FX[TY][TX + 1];
    double FY[TY + 1][TX];
    double EX[TY], EY[TX];  // f- side of the low-edge faces, whose f+ side is in FX[.][0], FY[0][.]
    double UR[7][TX * TY];  // u of this thread's column, planes k-2 .. k+3 (viscous term)
    unsigned long long red[TX * TY / 64];
};

// One tile x z-chunk of one stage; returns the largest |u_out| bit pattern
// this thread stored.  FD: fast_division_ok<WENO>(max|u|, eps) holds for the
// stage's input (the weight divisions then take the shortened sequence).
template <int WENO, int P, bool VISC, int TX, int TY, bool FD>
__device__ __forceinline__ unsigned long long ref_stage_tile(const double *__restrict__ uin, const double *un,
                                                             double *uout, const RefArgs &g, int stage, double dt,
                                                             double eps_in, const DiffCoef &kc, RefSmem<TX, TY> &sm) {
    const double eps = fd_eps<FD>(eps_in);
    constexpr int NT = TX * TY;
    constexpr int NW = NT / 64;
    static_assert(NT % 64 == 0 && 6 * TX + 6 * TY <= NT && TX + TY <= 64, "tile shape");
    unsigned long long vmax = 0ull;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = tile % g.ntx, by = (tile / g.ntx) % g.nty, bz = tile / (g.ntx * g.nty);
    const int x0 = 3 + bx * TX, y0 = 3 + by * TY;
    const int z0 = 3 + bz * g.kchunk, z1 = min(z0 + g.kchunk, nz - 3);
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const bool active = x0 + tx < nx - 3 && y0 + ty < ny - 3;
    const unsigned plane = static_cast<unsigned>(nx) * static_cast<unsigned>(ny), pb = 8u * plane;
    // plane k of a field (nz >= 7 and fewer than 2^31 nodes: see PlaneIo)
    auto io = [&](const double *base, int k) { return PlaneIo<double>(base + static_cast<size_t>(plane) * k, pb); };
    auto cx = [&](int x) { return static_cast<unsigned>(min(x, nx - 1)); };
    auto cy = [&](int y) { return static_cast<unsigned>(min(y, ny - 1)); };
    const unsigned col = 8u * (cx(x0 + tx) + static_cast<unsigned>(nx) * cy(y0 + ty));
    const unsigned scol = active ? col : pb;  // byte offset stored to

    // halo node of this thread: 6*TY x-halo nodes, then 6*TX y-halo nodes
    int hl_r = 0, hl_c = 0;
    unsigned hcol = pb;  // byte offset; pb: no halo node, loads 0
    const bool has_halo = tid < 6 * TY + 6 * TX;
    if (tid < 6 * TY) {
        const int r = tid / 6, c = tid % 6;
        hl_r = r + 3;
        hl_c = c < 3 ? c : TX + c;
        hcol = 8u * (cx(x0 + hl_c - 3) + static_cast<unsigned>(nx) * cy(y0 + r));
    } else if (has_halo) {
        const int h = tid - 6 * TY, c = h % TX, q = h / TX;
        hl_r = q < 3 ? q : TY + q;
        hl_c = c + 3;
        hcol = 8u * (cx(x0 + c) + static_cast<unsigned>(nx) * cy(y0 + hl_r - 3));
    }

    // z rings, plane p in slot (p - z0 + a) % 7: at plane k = z0 + s (mod 7)
    // qp/qm[R(q)] are the split fluxes of plane k-3+q, uq[R(q)] u of plane
    // k-2+q (in LDS, this thread's own column, where the viscous term would
    // otherwise keep six more doubles in registers), sp/sn[R(q)] the 13/12
    // terms centred on plane k-1+q.  The march is unrolled by 7, so every slot
    // is a constant and no register moves shift the rings (1601x986x35: 6009
    // to 5813 us a call of 2 steps, spills 8 to 0; 512^3, on 32x32 tiles, unchanged:
    // they still spill 7 with WENO-Z and 3 with JS, in the viscous kernels).
    double qp[7], qm[7], uq[7], sp[7], sn[7];
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const double v = io(uin, z0 - 3 + q).load(col);
        lf_split_local(v, qp[q], qm[q]);
        if (q >= 1) {
            if (VISC)
                sm.UR[q - 1][tid] = v;
            else
                uq[q - 1] = v;
        }
    }
    const double sp0 = sterm<FD>(qp[0], qp[1], qp[2]);
#pragma unroll
    for (int q = 0; q < 3; q++) {
        sp[q] = sterm<FD>(qp[q + 1], qp[q + 2], qp[q + 3]);
        sn[q] = sterm<FD>(qm[q + 1], qm[q + 2], qm[q + 3]);
    }
    double fz_prev = weno_face_s<WENO, P, FD>(qp[0], qp[1], qp[2], qp[3], qp[4], qm[1], qm[2], qm[3], qm[4], qm[5],
                                              sp0, sp[0], sp[1], sn[0], sn[1], sn[2], eps);
    double own_next = io(uin, z0 + 3).load(col);
    double halo_next = io(uin, z0).load(hcol);
    double un_next = stage == 1 ? 0.0 : io(un, z0).load(col);

    int kb = z0;
    auto plane_step = [&](auto SC) {
        constexpr int s = decltype(SC)::value;
        auto R = [](int q) { return (s + q) % 7; };
        const int k = kb + s;
        const double own = own_next, halo = halo_next, unv = un_next;
        if (k + 1 < z1) {
            own_next = io(uin, k + 4).load(col);
            halo_next = io(uin, k + 1).load(hcol);
            if (stage != 1) un_next = io(un, k + 1).load(col);
        }
        lf_split_local(own, qp[R(6)], qm[R(6)]);
        if (VISC)
            sm.UR[R(5)][tid] = own;
        else
            uq[R(5)] = own;
        const double u0 = VISC ? sm.UR[R(2)][tid] : uq[R(2)];
        sp[R(3)] = sterm<FD>(qp[R(4)], qp[R(5)], qp[R(6)]);
        sn[R(3)] = sterm<FD>(qm[R(4)], qm[R(5)], qm[R(6)]);
        const double2 ctr = make_double2(qp[R(3)], qm[R(3)]);
        sm.P[ty + 3][tx + 3] = ctr;
        if (VISC) sm.U[ty + 3][tx + 3] = u0;
        if (has_halo) {
            double hp, hm;
            lf_split_local(halo, hp, hm);
            sm.P[hl_r][hl_c] = make_double2(hp, hm);
            if (VISC) sm.U[hl_r][hl_c] = halo;
        }
        __syncthreads();

        const double fz = weno_face_s<WENO, P, FD>(qp[R(1)], qp[R(2)], qp[R(3)], qp[R(4)], qp[R(5)], qm[R(2)],
                                                   qm[R(3)], qm[R(4)], qm[R(5)], qm[R(6)], sp[R(0)], sp[R(1)],
                                                   sp[R(2)], sn[R(1)], sn[R(2)], sn[R(3)], eps);
        {
            const double2 a0 = sm.P[ty + 3][tx + 1], a1 = sm.P[ty + 3][tx + 2], a2 = ctr, a3 = sm.P[ty + 3][tx + 4],
                          a4 = sm.P[ty + 3][tx + 5], a5 = sm.P[ty + 3][tx + 6];
            sm.FX[ty][tx + 1] =
                weno_face2<WENO, P, FD>(a0.x, a1.x, a2.x, a3.x, a4.x, a1.y, a2.y, a3.y, a4.y, a5.y, eps);
        }
        {
            const double2 a0 = sm.P[ty + 1][tx + 3], a1 = sm.P[ty + 2][tx + 3], a2 = ctr,
                          a3 = sm.P[ty + 4][tx + 3], a4 = sm.P[ty + 5][tx + 3], a5 = sm.P[ty + 6][tx + 3];
            sm.FY[ty + 1][tx] =
                weno_face2<WENO, P, FD>(a0.x, a1.x, a2.x, a3.x, a4.x, a1.y, a2.y, a3.y, a4.y, a5.y, eps);
        }
        // x and y part of the viscous term: U is read only between the two
        // barriers (the next plane overwrites it after the second), here and not
        // before the faces, where its values add to theirs (32x16: 17 spills)
        double XY = 0.0;
        if (VISC) {
            const double X = d4(sm.U[ty + 3][tx + 1], sm.U[ty + 3][tx + 2], u0, sm.U[ty + 3][tx + 4], sm.U[ty + 3][tx + 5]);
            const double Y = d4(sm.U[ty + 1][tx + 3], sm.U[ty + 2][tx + 3], u0, sm.U[ty + 4][tx + 3], sm.U[ty + 5][tx + 3]);
            XY = kc.kx * X + kc.ky * Y;
        }
        // the tile's low-edge faces, their f+ sides by one wave and their f-
        // sides by the next, rotating with k (as in the periodic stage)
        const int ew = (wave - k) & (NW - 1);
        if (ew < 2 && lane < TY + TX) {
            int e0 = lane < TY ? (lane + 3) * (TX + 6) : lane - TY + 3;
            int es = lane < TY ? 1 : TX + 6;
            asm volatile("" : "+v"(e0), "+v"(es));  // computed here, not kept in registers over the march
            const double2 *a = &sm.P[0][0] + e0;
            if (ew == 0) {
                const double f = weno_side<WENO, P, true, FD>(a[0].x, a[es].x, a[2 * es].x, a[3 * es].x, a[4 * es].x, eps);
                *(lane < TY ? &sm.FX[lane][0] : &sm.FY[0][lane - TY]) = f;
            } else {
                const double f =
                    weno_side<WENO, P, false, FD>(a[es].y, a[2 * es].y, a[3 * es].y, a[4 * es].y, a[5 * es].y, eps);
                *(lane < TY ? &sm.EX[lane] : &sm.EY[lane - TY]) = f;
            }
        }
        __syncthreads();

        double fx_lo = sm.FX[ty][tx], fy_lo = sm.FY[ty][tx];
        if (tx == 0) fx_lo += sm.EX[ty];
        if (ty == 0) fy_lo += sm.EY[tx];
        double Lu = minus_div3(sm.FX[ty][tx + 1] - fx_lo, sm.FY[ty + 1][tx] - fy_lo, fz - fz_prev, g.dx, g.rdx, g.dy,
                               g.rdy, g.dz, g.rdz);
        if (VISC) {
            const double Z = d4(sm.UR[R(0)][tid], sm.UR[R(1)][tid], u0, sm.UR[R(3)][tid], sm.UR[R(4)][tid]);
            Lu += XY + kc.kz * Z;
        }
        const double uo = stage == 1 ? u0 : unv;
        double unew;
        if (stage == 1)
            unew = uo + dt * Lu;
        else if (stage == 2)
            unew = 0.75 * uo + 0.25 * (u0 + dt * Lu);
        else
            unew = div_by(p2fma(2.0, u0 + dt * Lu, uo), 3.0, 1.0 / 3.0);  // (uo + 2(u + dt Lu)) / 3
        io(uout, k).store(scol, unew);
        const unsigned long long bb = active ? abs_bits(unew) : 0ull;
        vmax = bb > vmax ? bb : vmax;

        fz_prev = fz;
    };
    for (; kb < z1; kb += 7) {
        plane_step(std::integral_constant<int, 0>{});
        if (kb + 1 >= z1) break;
        plane_step(std::integral_constant<int, 1>{});
        if (kb + 2 >= z1) break;
        plane_step(std::integral_constant<int, 2>{});
        if (kb + 3 >= z1) break;
        plane_step(std::integral_constant<int, 3>{});
        if (kb + 4 >= z1) break;
        plane_step(std::integral_constant<int, 4>{});
        if (kb + 5 >= z1) break;
        plane_step(std::integral_constant<int, 5>{});
        if (kb + 6 >= z1) break;
        plane_step(std::integral_constant<int, 6>{});
    }
    return vmax;
}

// One stage over all tiles: the stage's max|u| bound (its input's slot and
// the ghost floor) picks the division sequence for every block alike; each
// block folds its stored |u_out| into the output slot, and the lead clears
// the slot the next-but-one stage fills.
template <int WENO, int P, bool VISC, int TX, int TY>
__global__ __launch_bounds__(TX * TY, 4) void k_burgers_ref_stage(const double *__restrict__ uin,
                                                                  const double *un, double *uout, RefArgs g,
                                                                  int stage, double dt, double eps,
                                                                  DiffCoef kc) {
    constexpr int NW = TX * TY / 64;
    __shared__ RefSmem<TX, TY> sm;
    const unsigned long long a_in = g.amax[stage - 1], a_gh = g.amax[3];
    const double amax = bits_double(a_in > a_gh ? a_in : a_gh);
    if (blockIdx.x == 0 && threadIdx.x == 0) g.amax[(stage + 1) % 3] = 0ull;
    unsigned long long vmax;
    if (fast_division_ok<WENO>(amax, eps))
        vmax = ref_stage_tile<WENO, P, VISC, TX, TY, true>(uin, un, uout, g, stage, dt, eps, kc, sm);
    else
        vmax = ref_stage_tile<WENO, P, VISC, TX, TY, false>(uin, un, uout, g, stage, dt, eps, kc, sm);
    vmax = wave_max_u64(vmax);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sm.red[wave] = vmax;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = sm.red[0];
#pragma unroll
        for (int w = 1; w < NW; w++) m = sm.red[w] > m ? sm.red[w] : m;
        atomicMax(&g.amax[stage % 3], m);
    }
}

// Slots for a call: [0] = [3] = max|u| over all nodes, [1] = [2] = 0.
__global__ void k_ref_amax_clear(unsigned long long *amax) {
    amax[0] = amax[1] = amax[2] = amax[3] = 0ull;
}

// What a call needs of u beside its steps, in one pass: max|u| over all nodes
// into slots 0 and 3, and the three ghost layers, which no stage writes, into
// the stage buffers w1 and w2.  A row is ceil(nx / 64) segments of a wave's
// width, and a wave takes eight consecutive segments at a time, of one row or of
// several: rows of the ghost planes and the first and last three of a plane are
// copied whole, of the others the first and last three nodes.  Bound by the
// read of u, 8 B a node, and on small grids by the atomics on one address, 13
// ns each: a block leaves them out where the slots already hold as much.
// us a call's set-up by two copies of u and a separate max|u| pass / by whole
// rows, one at a time / so: 26x26x300 35 / 52 / 16, 24x1024x1024 215 / 382 / 111,
// 7x7x4000 33 / 61 / 29, 100^3 74 / 58 / 19, 1601x986x35 439 / 103 / 97 (twice a
// call of one step less a call of two; the pass itself takes 120 us there).
constexpr int kPrepSegs = 8;  // segments, and so loads in flight, of a wave
__global__ __launch_bounds__(256) void k_ref_prepare(const double *__restrict__ u, double *__restrict__ w1,
                                                     double *__restrict__ w2, int nx, int ny, int nz,
                                                     unsigned long long *amax) {
    __shared__ unsigned long long red[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned segs = (static_cast<unsigned>(nx) + 63u) / 64u;
    const unsigned units = segs * static_cast<unsigned>(ny) * static_cast<unsigned>(nz);  // < 2^31
    const unsigned groups = (units + kPrepSegs - 1) / kPrepSegs;
    unsigned long long m = 0ull;
    for (unsigned g = 4u * blockIdx.x + static_cast<unsigned>(wave); g < groups; g += 4u * gridDim.x) {
        const unsigned first = g * kPrepSegs, left = units - first;
        const unsigned r0 = first / segs, s0 = first - r0 * segs, k0 = r0 / static_cast<unsigned>(ny);
        double v[kPrepSegs];
        unsigned r = r0, sg = s0;
#pragma unroll
        for (int q = 0; q < kPrepSegs; q++) {
            const unsigned i = min(sg * 64u + lane, static_cast<unsigned>(nx) - 1u);
            v[q] = u[static_cast<size_t>(r) * static_cast<unsigned>(nx) + i];
            if (q + 1u < left && ++sg == segs) {  // past the last segment: the last one again
                sg = 0;
                r++;
            }
        }
        r = r0;
        sg = s0;
        int j = static_cast<int>(r0 - k0 * static_cast<unsigned>(ny)), k = static_cast<int>(k0);
#pragma unroll
        for (int q = 0; q < kPrepSegs; q++) {
            const unsigned long long b = abs_bits(v[q]);
            m = b > m ? b : m;
            const int i = static_cast<int>(sg * 64u) + lane;
            const bool ghost = j < 3 || j >= ny - 3 || k < 3 || k >= nz - 3;
            if (i < nx && (ghost || i < 3 || i >= nx - 3)) {
                const size_t o = static_cast<size_t>(r) * static_cast<unsigned>(nx) + static_cast<unsigned>(i);
                w1[o] = v[q];
                w2[o] = v[q];
            }
            if (q + 1u < left && ++sg == segs) {
                sg = 0;
                r++;
                if (++j == ny) {
                    j = 0;
                    k++;
                }
            }
        }
    }
    m = wave_max_u64(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = red[0];
        for (int w = 1; w < 4; w++) m = red[w] > m ? red[w] : m;
        for (int s : {0, 3})
            if (m > __hip_atomic_load(&amax[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&amax[s], m);
    }
}

namespace {

using RefKernel = void (*)(const double *, const double *, double *, RefArgs, int, double, double, DiffCoef);

template <int WENO, int P, int TX, int TY>
RefKernel ref_kernel(bool visc) {
    return visc ? k_burgers_ref_stage<WENO, P, true, TX, TY> : k_burgers_ref_stage<WENO, P, false, TX, TY>;
}

template <int TX, int TY>
RefKernel ref_kernel_for(const mgad_scheme &sc, bool visc) {
    if (sc.weno == MGAD_WENO_JS) return ref_kernel<kWenoJS, 2, TX, TY>(visc);
    if (sc.p == 2) return ref_kernel<kWenoZ, 2, TX, TY>(visc);
    return ref_kernel<kWenoZ, 1, TX, TY>(visc);
}

struct RefLaunch {
    RefKernel fn;
    RefArgs g;
    unsigned blocks, threads;
};

// Tile width (TX x 16) and planes a block of a launch that is not one round of
// 32x32 tiles.  Grids with 2048 tiles of 32x16 or more take those, whole
// columns each.  Else the least of a CU's work, about 1.2 n (k + 1.5) us for n
// 16x16 blocks of k planes (32x16: 4 % less than two of them), and of the end
// of the launch, about 1.2 k.  us a stage before (32x16, 8 planes or more),
// then with this rule: 24^3 20.6, 7.6; 40^3 21.3, 11.2; 64^3 31.2, 15.1; 100^3
// 41.2, 31.6; 300x280x200 381, 360; 512x400x100 414, 390; 200x180x120 114, 115.
void ref_tiles(int ix, int iy, int iz, long cus, int &TX, int &kc) {
    const long ty = (iy + 15) / 16, wide = ((ix + 31) / 32) * ty, narrow = ((ix + 15) / 16) * ty;
    TX = 32;
    kc = iz;
    if (wide >= 2048) return;
    double least = 0.0;
    for (int q = 1; q <= std::min(iz, 64); q++) {
        const int bands = (iz + q - 1) / q, k = (iz + bands - 1) / bands;
        const double n = static_cast<double>((narrow * bands + cus - 1) / cus),
                     w = 1.92 * static_cast<double>((wide * bands + cus - 1) / cus);
        const double c16 = n * (k + 1.5) + k, c32 = w * (k + 1.5) + k;
        if (q == 1 || std::min(c16, c32) < least) {
            least = std::min(c16, c32);
            TX = c16 <= c32 ? 16 : 32;
            kc = k;
        }
    }
}

RefLaunch ref_launch(const mgad_scheme &sc, bool visc, unsigned nx, unsigned ny, unsigned nz, double dx, double dy,
                     double dz) {
    RefLaunch L{};
    const int ix = static_cast<int>(nx) - 6, iy = static_cast<int>(ny) - 6, iz = static_cast<int>(nz) - 6;
    // one round of 32x32 workgroups, one per CU, when the interior's tiles
    // fill the CUs (as for the periodic stage); else 32x16 or 16x16 tiles
    const int sq = ix > 0 && iy > 0 && iz > 0
                       ? square_bands(static_cast<long>((ix + 31) / 32) * ((iy + 31) / 32), static_cast<unsigned>(iz))
                       : 0;
    int TX = 32, TY = sq > 0 ? 32 : 16, kc = sq > 0 ? (iz + sq - 1) / sq : iz;
    if (sq == 0) ref_tiles(ix, iy, iz, resident_groups(1024), TX, kc);
    L.fn = sq > 0 ? ref_kernel_for<32, 32>(sc, visc)
                  : (TX == 32 ? ref_kernel_for<32, 16>(sc, visc) : ref_kernel_for<16, 16>(sc, visc));
    L.threads = TX * TY;
    RefArgs &g = L.g;
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    g.ntx = (ix + TX - 1) / TX;
    g.nty = (iy + TY - 1) / TY;
    g.kchunk = kc;
    g.dx = dx;
    g.dy = dy;
    g.dz = dz;
    g.rdx = 1.0 / dx;
    g.rdy = 1.0 / dy;
    g.rdz = 1.0 / dz;
    L.blocks = static_cast<unsigned>(g.ntx) * g.nty * ((iz + kc - 1) / kc);
    return L;
}

int enqueue_ref_step(hipStream_t s, const RefLaunch &L, double dt, double eps, DiffCoef kc, double *u, double *w1,
                     double *w2) {
    hipLaunchKernelGGL(L.fn, dim3(L.blocks), dim3(L.threads), 0, s, u, u, w1, L.g, 1, dt, eps, kc);
    hipLaunchKernelGGL(L.fn, dim3(L.blocks), dim3(L.threads), 0, s, w1, u, w2, L.g, 2, dt, eps, kc);
    hipLaunchKernelGGL(L.fn, dim3(L.blocks), dim3(L.threads), 0, s, w2, u, u, L.g, 3, dt, eps, kc);
    return check_launch();
}

// The max|u| slots of reference-step runs on a stream (4 per stream, kept
// for the process: graphs captured on the stream point at them).
unsigned long long *ref_amax_slots(hipStream_t s) {
    static std::map<hipStream_t, unsigned long long *> slots;
    auto it = slots.find(s);
    if (it != slots.end()) return it->second;
    unsigned long long *p = nullptr;
    if (check_hip(hipMalloc(&p, 4 * sizeof(unsigned long long)))) return nullptr;
    slots[s] = p;
    return p;
}

using RefGraphKey = std::tuple<hipStream_t, int, int, double, int, unsigned, unsigned, unsigned, double, double,
                               double, double, double, double, double, double *, double *, double *>;

std::map<RefGraphKey, KeptGraph> &ref_graphs() {
    static std::map<RefGraphKey, KeptGraph> m;
    return m;
}

}  // namespace

}  // namespace mgad

using namespace mgad;

extern "C" int mgad_burgers_ref_steps(hipStream_t stream, const mgad_scheme *scheme, int viscous, unsigned int nx,
                                      unsigned int ny, unsigned int nz, double dx, double dy, double dz, double dt,
                                      double *u, double *w1, double *w2, int nsteps, int use_graph) {
    if (!scheme || !u || !w1 || !w2 || u == w1 || u == w2 || w1 == w2 || nsteps < 0 || nx < 7 || ny < 7 ||
        nz < 7 || 1ull * nx * ny * nz >= (1ull << 31) || !(dx > 0) || !(dy > 0) || !(dz > 0) ||
        (scheme->weno != MGAD_WENO_Z && scheme->weno != MGAD_WENO_JS) || (scheme->p != 1 && scheme->p != 2)) {
        set_error(MGAD_ERR_INVALID_ARG);
        return MGAD_ERR_INVALID_ARG;
    }
    if (nsteps == 0) return MGAD_OK;
    std::lock_guard<std::recursive_mutex> lock(host_mutex());
    if (use_graph && stream != nullptr) {
        if (const int st = refuse_capture(stream)) return st;
    }
    RefLaunch L = ref_launch(*scheme, viscous != 0, nx, ny, nz, dx, dy, dz);
    L.g.amax = ref_amax_slots(stream);
    if (!L.g.amax) return MGAD_ERR_HIP;
    hipLaunchKernelGGL(k_ref_amax_clear, dim3(1), dim3(1), 0, stream, L.g.amax);
    // the stage buffers carry u's ghost layers (never written by any stage)
    const unsigned long long units = 1ull * ((nx + 63) / 64) * ny * nz;
    const unsigned blocks =
        static_cast<unsigned>(std::min<unsigned long long>((units + 4 * kPrepSegs - 1) / (4 * kPrepSegs), 2048));
    hipLaunchKernelGGL(k_ref_prepare, dim3(blocks), dim3(256), 0, stream, u, w1, w2, (int)nx, (int)ny, (int)nz,
                       L.g.amax);
    int st = check_launch();
    if (st) return st;
    const DiffCoef kc = viscous ? diff_coef() : DiffCoef{0.0, 0.0, 0.0};
    if (!use_graph || stream == nullptr) {
        for (int s = 0; s < nsteps && !st; s++) st = enqueue_ref_step(stream, L, dt, scheme->eps, kc, u, w1, w2);
        return st;
    }
    const RefGraphKey key{stream, scheme->weno, scheme->p, scheme->eps, viscous != 0, nx, ny, nz, dx, dy, dz, dt,
                          kc.kx, kc.ky, kc.kz, u, w1, w2};
    return replay_steps(ref_graphs(), 16, key, stream, nsteps, graph_steps(3),
                        [&] { return enqueue_ref_step(stream, L, dt, scheme->eps, kc, u, w1, w2); });
}
