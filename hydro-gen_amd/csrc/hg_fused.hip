// hg_fused.hip — the GRID step in two fused kernels.
//
//  hydro   : rain -> hydro_flux -> hydro_erosion -> sediment_transport
//            (glsl/rain.glsl, hydro_flux.glsl, hydro_erosion.glsl,
//            sediment_transport.glsl).  Reads the 9 state planes once and
//            writes them once (72 B/cell).
//  thermal : thermal_erosion + thermal_transport for layer 0 then layer 1,
//            then smoothing (glsl/thermal_erosion.glsl, thermal_transport.glsl,
//            smoothing.glsl).  Reads rock+dirt once, writes them once (16 B/cell).
//
// Both kernels work on a TX x TY output tile per workgroup.  The tile plus a
// halo of its dependency radius is staged in LDS, every intermediate stage is
// evaluated on a region that shrinks by one cell per stage, and only the tile
// is written back.  The per-cell arithmetic is the same inline code as the
// per-pass kernels (hg_cell.hpp), so the fused and per-pass paths agree bit
// for bit.
//
// The semi-Lagrangian gather of sediment_transport has no bounded radius
// (|v|*dt is unbounded).  The hydro kernel evaluates eroded sediment on the
// tile plus an HA-cell halo; a back-trace whose bilinear taps fall outside it
// recomputes the eroded sediment of those taps from the step's input planes
// (still intact: every pass is ping-pong), which is exact.
#include <algorithm>
#include <type_traits>

#include "hg_kernels.hpp"

namespace hgk {

namespace {

__device__ __forceinline__ size_t at(int x, int y, int nx) { return size_t(y) * size_t(nx) + size_t(x); }
// Output and tape planes are written once per launch and not read back by it.
// When the step's state outgrows the last-level cache (KParams::store_nt, a
// compile-time NTS in the kernels: a run-time choice between two stores of the
// same value is folded into one plain store) they are written with
// non-temporal stores: hydro kernel 270 -> 262 us at 4096^2, same results.
// Below that size ordinary stores are faster (the next launch reads the planes
// from the cache).  Non-temporal loads of the inputs read once per workgroup
// measured slower and are not used.
template <bool NTS>
__device__ __forceinline__ void st_out(float* p, float v) {
    if constexpr (NTS)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

template <bool NTS>
__device__ __forceinline__ void st_out2(float* p, float a, float b) {
    typedef float v2 __attribute__((ext_vector_type(2)));
    const v2 v = {a, b};
    if constexpr (NTS)
        __builtin_nontemporal_store(v, reinterpret_cast<v2*>(p));
    else
        *reinterpret_cast<v2*>(p) = v;
}

// ---------------------------------------------------------------------------
// Cells of the region of radius RAD around a TX x TY tile.  When the tile
// width is a multiple of 64, the region is split into its core columns (the
// tile's own: one wave per 64-wide row chunk, so lanes touch 64 consecutive
// LDS words, free of bank conflicts, and global rows start 256-B aligned) and
// the two side strips of RAD columns, spread over the threads.  Otherwise the
// region is walked linearly.
// ---------------------------------------------------------------------------
template <int TX, int TY, int NT, int RAD>
struct Region {
    static constexpr int W = TX + 2 * RAD, H = TY + 2 * RAD, N = W * H;
    static constexpr bool ROWS = TX % 64 == 0 && NT % 64 == 0;
    static constexpr int NW = NT / 64, CPR = TX / 64;       // waves; 64-wide chunks per row
    static constexpr int NCORE = H * CPR, NSIDE = 2 * RAD * H;
    static constexpr int ITC = ROWS ? (NCORE + NW - 1) / NW : 0;
    static constexpr int ITS = ROWS ? (NSIDE + NT - 1) / NT : 0;
    static constexpr int ITER = ROWS ? ITC + ITS : (N + NT - 1) / NT;
};

// Calls fn(it, rx, ry) for the cells of the region, in region coordinates
// rx in [0, W), ry in [0, H); `it` < Region::ITER numbers a thread's calls.
template <int TX, int TY, int NT, int RAD, class F>
__device__ __forceinline__ void tile_region_for(int tid, F&& fn) {
    using R = Region<TX, TY, NT, RAD>;
    if constexpr (R::ROWS) {
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
        for (int it = 0; it < R::ITC; ++it) {
            // The scalar guard stays even where every wave passes it: the
            // branch bounds how far the scheduler hoists LDS reads across
            // cells, which otherwise spills registers.
            const int q = wave + it * R::NW;              // wave-uniform
            if (q < R::NCORE) {
                const int row = q / R::CPR, c = q - row * R::CPR;
                fn(it, RAD + c * 64 + lane, row);
            }
        }
        if constexpr (RAD > 0) {
#pragma unroll
            for (int it = 0; it < R::ITS; ++it) {
                const int j = tid + it * NT;
                if (R::NSIDE % NT == 0 || j < R::NSIDE) {
                    const int row = j / (2 * RAD), c = j - row * (2 * RAD);
                    fn(R::ITC + it, c < RAD ? c : TX + c, row);
                }
            }
        }
    } else {
#pragma unroll
        for (int it = 0; it < R::ITER; ++it) {
            const int i = tid + it * NT;
            if (R::N % NT == 0 || i < R::N) {
                const int ry = i / R::W, rx = i - ry * R::W;
                fn(it, rx, ry);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// hydro kernel
// ---------------------------------------------------------------------------

template <int TX, int TY, int HA, int NT>
struct HydroTile {
    // input region: tile +- (HA+1) cells, loaded in aligned quads, so the LDS
    // region spans x in [x0 - QH*4, x0 + TX + QH*4)
    static constexpr int QH = (HA + 1 + 3) / 4;           // halo quads per side
    static constexpr int WI = TX + 8 * QH;                 // LDS row width (cells)
    static constexpr int OX = 4 * QH;                      // LDS x of tile column 0
    static constexpr int HI = TY + 2 * (HA + 1);           // LDS rows
    static constexpr int OY = HA + 1;                      // LDS y of tile row 0
    static constexpr int WE = TX + 2 * HA, HE = TY + 2 * HA;  // eroded-sediment region
    static constexpr int NE = WE * HE;
    static constexpr int NTILE = TX * TY;
    static constexpr int ITER_T = (NTILE + NT - 1) / NT;
    static constexpr int NLDS = WI * HI;
    // Where the list of cells with far taps lies after stage 1 (in the place of
    // the thermal stages' g in a STEP), and its length's distance from it.
    template <bool STEP>
    static constexpr int FAR = 2 * NE + 2 * NTILE + (STEP ? 2 * NE : 0);
    template <bool STEP>
    static constexpr int NFAR = STEP ? NE : NTILE;
    static_assert(NTILE <= NE, "the list fits g's place");
    static_assert(FAR<false> + NFAR<false> < 6 * NLDS, "aliased outputs must fit the input arrays");
    static_assert(TX % 4 == 0, "tile width must be a multiple of 4");
};

// One output tile (bx, by) of the hydro kernel; `lds` holds 6*NLDS floats.
// Ends with LDS still in use: callers looping over tiles must barrier first.
// EXTRA: also write the optional outputs (velocity, adjoint tape) that are
// not null; without it their pointers are never read, which keeps them out
// of the scalar registers of the common case.
// STEP (k_step_tile): rock and dirt after erosion are left in LDS on the whole
// region, as the thermal stages take them (see StepTile), and written to memory
// only as part of the tape.
template <int TX, int TY, int HA, int NT, bool EXTRA = false, bool NTS = false, bool STEP = false>
__device__ __forceinline__ void hydro_tile(float* lds, const HydroIO& io, int nx, int ny, int bx,
                                           int by, uint32_t step, uint32_t terrain, int rain,
                                           const KParams& k) {
    using T = HydroTile<TX, TY, HA, NT>;
    // LDS planes (pitch WI): rd = rock+dirt, b = water after rain, fl..fb = old flux.
    float* s_rd = lds;
    float* s_b = lds + T::NLDS;
    float* s_fl = lds + 2 * T::NLDS;
    float* s_fr = lds + 3 * T::NLDS;
    float* s_ft = lds + 4 * T::NLDS;
    float* s_fb = lds + 5 * T::NLDS;

    // Opaque to the optimiser: values derived from the thread index are then
    // recomputed per tile instead of being hoisted out of the batched tile
    // loop and held in registers across tiles.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int x0 = bx * TX, y0 = by * TY;
    const int lx0 = x0 - T::OX, ly0 = y0 - T::OY;   // grid coords of LDS (0,0)

    // ---- stage 0: stage inputs in aligned quads; rain is added here -------
    {
        constexpr int QW = T::WI / 4;
        constexpr int NQ = QW * T::HI;
        for (int q = tid; q < NQ; q += NT) {
            const int qy = q / QW, qxq = q - qy * QW;
            const int gx = lx0 + 4 * qxq, gy = ly0 + qy;
            const int li = qy * T::WI + 4 * qxq;
            float rd[4], b[4], fl[4], fr[4], ft[4], fb[4];
            if (gy >= 0 && gy < ny && gx >= 0 && gx + 3 < nx) {
                const size_t g = at(gx, gy, nx);
                const float4 r4 = *reinterpret_cast<const float4*>(io.r + g);
                const float4 d4 = *reinterpret_cast<const float4*>(io.d + g);
                const float4 b4 = *reinterpret_cast<const float4*>(io.b + g);
                const float4 l4 = *reinterpret_cast<const float4*>(io.fl + g);
                const float4 rr4 = *reinterpret_cast<const float4*>(io.fr + g);
                const float4 t4 = *reinterpret_cast<const float4*>(io.ft + g);
                const float4 bb4 = *reinterpret_cast<const float4*>(io.fb + g);
                rd[0] = r4.x + d4.x; rd[1] = r4.y + d4.y; rd[2] = r4.z + d4.z; rd[3] = r4.w + d4.w;
                b[0] = b4.x; b[1] = b4.y; b[2] = b4.z; b[3] = b4.w;
                fl[0] = l4.x; fl[1] = l4.y; fl[2] = l4.z; fl[3] = l4.w;
                fr[0] = rr4.x; fr[1] = rr4.y; fr[2] = rr4.z; fr[3] = rr4.w;
                ft[0] = t4.x; ft[1] = t4.y; ft[2] = t4.z; ft[3] = t4.w;
                fb[0] = bb4.x; fb[1] = bb4.y; fb[2] = bb4.z; fb[3] = bb4.w;
                if (rain) {
                    float inc[4];
                    if (k.rain_mode == HG_RAIN_UNIFORM) {
                        uint32_t o[4];
                        philox4x32_10(uint32_t(gx) >> 2, uint32_t(gy), step, terrain, k.seed_lo, k.seed_hi, o);
#pragma unroll
                        for (int j = 0; j < 4; ++j) inc[j] = k.rain_amount * u24(o[j]);
                    } else {
                        const float a = k.rain_mode == HG_RAIN_CONSTANT ? k.rain_amount : 0.0f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) inc[j] = a;
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) b[j] = b[j] + inc[j];
                }
            } else {
                // whole quad outside the grid (n is a multiple of 8, so quads
                // never straddle the border): flux reads a total of
                // HG_OOB_HEIGHT and zero flux, erosion reads rock+dirt 0.
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    rd[j] = 0.0f; b[j] = HG_OOB_HEIGHT;
                    fl[j] = 0.0f; fr[j] = 0.0f; ft[j] = 0.0f; fb[j] = 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s_rd[li + j] = rd[j]; s_b[li + j] = b[j];
                s_fl[li + j] = fl[j]; s_fr[li + j] = fr[j]; s_ft[li + j] = ft[j]; s_fb[li + j] = fb[j];
            }
        }
    }
    __syncthreads();

    // ---- stage 1: flux + erosion on the tile +- HA region -----------------
    // (region coordinates ex in [0, TX + 2HA), ey in [0, TY + 2HA))
    constexpr int IE = Region<TX, TY, NT, HA>::ITER;
    auto walk = [&](auto&& fn) { tile_region_for<TX, TY, NT, HA>(tid, fn); };
    float es0[IE], es1[IE], evx[IE], evy[IE];
#pragma unroll
    for (int it = 0; it < IE; ++it) { es0[it] = 0.0f; es1[it] = 0.0f; evx[it] = 0.0f; evy[it] = 0.0f; }
    // rock, dirt and sediment of the region, at clamped addresses, all
    // issued before the first cell is evaluated
    float gr[IE], gd[IE], g0[IE], g1[IE];
    float er[STEP ? IE : 1], ed[STEP ? IE : 1];
    if constexpr (STEP) {
#pragma unroll
        for (int it = 0; it < IE; ++it) er[it] = ed[it] = HG_OOB_HEIGHT;
    }
    walk([&](int it, int ex, int ey) {
        const int gx = min(max(x0 - HA + ex, 0), nx - 1), gy = min(max(y0 - HA + ey, 0), ny - 1);
        const size_t g = at(gx, gy, nx);
        gr[it] = io.r[g];
        gd[it] = io.d[g];
        g0[it] = io.s0[g];
        g1[it] = io.s1[g];
    });
    walk([&](int it, int ex, int ey) {
        const int gx = x0 - HA + ex, gy = y0 - HA + ey;
        if (gx < 0 || gy < 0 || gx >= nx || gy >= ny) return;
        const int li = (ey + 1) * T::WI + (ex + T::OX - HA);   // LDS index of this cell
        float f[4] = {s_fl[li], s_fr[li], s_ft[li], s_fb[li]};
        const float b = s_b[li];
        const float w = s_rd[li] + b;
        const float wn[4] = {s_rd[li - 1] + s_b[li - 1], s_rd[li + 1] + s_b[li + 1],
                             s_rd[li + T::WI] + s_b[li + T::WI], s_rd[li - T::WI] + s_b[li - T::WI]};
        const float fin[4] = {s_fr[li - 1], s_fl[li + 1], s_fb[li + T::WI], s_ft[li - T::WI]};
        const unsigned wall = (gx == 0 ? 1u : 0u) | (gx == nx - 1 ? 2u : 0u) | (gy == 0 ? 4u : 0u) |
                              (gy == ny - 1 ? 8u : 0u);
        float vx, vy, vz;
        const float d2 = flux_cell(f, b, w, wn, fin, wall, k, vx, vy, vz);
        const size_t g = at(gx, gy, nx);
        float r = gr[it], d = gd[it];
        float s0 = g0[it], s1 = g1[it];
        erosion_cell(r, d, s0, s1, vx, vy, vz, s_rd[li - 1], s_rd[li + 1], s_rd[li + T::WI],
                     s_rd[li - T::WI], k);
        es0[it] = s0; es1[it] = s1; evx[it] = vx; evy[it] = vy;
        if constexpr (STEP) { er[it] = r; ed[it] = d; }
        const bool tile = ex >= HA && ex < HA + TX && ey >= HA && ey < HA + TY;
        if (tile) {
            if (!STEP || EXTRA) {
                st_out<NTS>(&io.ro[g], r);
                st_out<NTS>(&io.dout[g], d);
            }
            st_out<NTS>(&io.bo[g], d2 * k.evap);     // sediment_transport.glsl:75
            st_out<NTS>(&io.flo[g], f[0]);
            st_out<NTS>(&io.fro[g], f[1]);
            st_out<NTS>(&io.fto[g], f[2]);
            st_out<NTS>(&io.fbo[g], f[3]);
            if (EXTRA && io.vx) {
                st_out<NTS>(&io.vx[g], vx);
                st_out<NTS>(&io.vy[g], vy);
                st_out<NTS>(&io.vz[g], vz);
            }
            if (EXTRA && io.tb1) {
                st_out<NTS>(&io.tb1[g], b);
                st_out<NTS>(&io.tb2[g], d2);
                st_out<NTS>(&io.ts0[g], s0);
                st_out<NTS>(&io.ts1[g], s1);
            }
        }
    });
    __syncthreads();   // all reads of the staged inputs are done

    // eroded sediment of the region and velocity of the tile, aliased over LDS
    float* s_s0 = lds;
    float* s_s1 = lds + T::NE;
    float* s_vx = lds + 2 * T::NE;
    float* s_vy = lds + 2 * T::NE + T::NTILE;
    if (tid == 0) reinterpret_cast<int*>(lds)[T::template FAR<STEP> + T::template NFAR<STEP>] = 0;
    walk([&](int it, int ex, int ey) {
        const int e = ey * T::WE + ex;
        s_s0[e] = es0[it];
        s_s1[e] = es1[it];
        if (ex >= HA && ex < HA + TX && ey >= HA && ey < HA + TY) {
            const int t = (ey - HA) * TX + (ex - HA);
            s_vx[t] = evx[it];
            s_vy[t] = evy[it];
        }
        if constexpr (STEP) {
            float* s_r = lds + 2 * T::NE + 2 * T::NTILE;
            s_r[e] = er[it];
            s_r[T::NE + e] = ed[it];
        }
    });
    __syncthreads();

    // ---- stage 2: back-trace + bilinear gather on the tile -----------------
    // Cells whose taps leave the halo are listed and done afterwards, four
    // lanes to a cell, one per tap: done where they are met, each wave with such
    // a lane recomputed its four taps one after the other.
    int* s_far = reinterpret_cast<int*>(lds) + T::template FAR<STEP>;
    int* s_nfar = s_far + T::template NFAR<STEP>;
    struct Taps {
        int ix, iy, ix1, iy1;
        float fx, fy;
    };
    auto taps_of = [&](int t) {
        const int ty = t / TX, tx = t - ty * TX;
        float bx, by;
        back_trace(x0 + tx, y0 + ty, s_vx[t], s_vy[t], k.dt, nx, ny, bx, by);
        Taps p;
        p.ix = int(bx);
        p.iy = int(by);
        p.fx = bx - float(p.ix);
        p.fy = by - float(p.iy);
        p.ix1 = min(p.ix + 1, nx - 1);
        p.iy1 = min(p.iy + 1, ny - 1);
        return p;
    };
    for (int t = tid; t < T::NTILE; t += NT) {
        const int ty = t / TX, tx = t - ty * TX;
        const int gx = x0 + tx, gy = y0 + ty;
        if (gx >= nx || gy >= ny) continue;
        const Taps p = taps_of(t);
        // region-local coordinates of the taps
        const int ex0 = p.ix - (x0 - HA), ey0 = p.iy - (y0 - HA);
        const int ex1 = p.ix1 - (x0 - HA), ey1 = p.iy1 - (y0 - HA);
        if (ex0 >= 0 && ey0 >= 0 && ex1 < T::WE && ey1 < T::HE) {
            const int e00 = ey0 * T::WE + ex0, e10 = ey0 * T::WE + ex1;
            const int e01 = ey1 * T::WE + ex0, e11 = ey1 * T::WE + ex1;
            const size_t g = at(gx, gy, nx);
            st_out<NTS>(&io.s0o[g], lerp1(lerp1(s_s0[e00], s_s0[e10], p.fx), lerp1(s_s0[e01], s_s0[e11], p.fx), p.fy));
            st_out<NTS>(&io.s1o[g], lerp1(lerp1(s_s1[e00], s_s1[e10], p.fx), lerp1(s_s1[e01], s_s1[e11], p.fx), p.fy));
        } else {
            s_far[atomicAdd(s_nfar, 1)] = t;
        }
    }
    __syncthreads();
    const int nfar = 4 * __builtin_amdgcn_readfirstlane(*s_nfar);
    if (nfar > 0) {
        for (int j = tid; j < nfar; j += NT) {
            const int t = s_far[j >> 2];
            const Taps p = taps_of(t);
            float v0, v1;
            eroded_sediment_global(io, (j & 1) ? p.ix1 : p.ix, (j & 2) ? p.iy1 : p.iy, nx, ny, step, terrain,
                                   rain != 0, k, v0, v1);
            // taps 00, 10, 01, 11 of lanes 0 .. 3 of the group
            auto tap = [](float v, auto c) {
                return __int_as_float(
                    __builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(c)::value * 0x55, 0xf, 0xf, true));
            };
            auto mix = [&](float v) {
                const float v00 = tap(v, std::integral_constant<int, 0>{}), v10 = tap(v, std::integral_constant<int, 1>{});
                const float v01 = tap(v, std::integral_constant<int, 2>{}), v11 = tap(v, std::integral_constant<int, 3>{});
                return lerp1(lerp1(v00, v10, p.fx), lerp1(v01, v11, p.fx), p.fy);
            };
            const float o0 = mix(v0), o1 = mix(v1);
            if ((j & 3) == 0) {
                const int ty = t / TX, tx = t - ty * TX;
                const size_t g = at(x0 + tx, y0 + ty, nx);
                st_out<NTS>(&io.s0o[g], o0);
                st_out<NTS>(&io.s1o[g], o1);
            }
        }
        if constexpr (STEP) __syncthreads();     // the list's place is the thermal stages' scale g
    }
}

// Tile of workgroup b in a 1-D grid of nb.  Workgroups are dealt to the 8 XCDs
// round robin (b -> XCD b mod 8); with `xcd` set, XCD x gets the contiguous run
// of tiles starting at x*q + min(x, r) (q = nb/8, r = nb mod 8), so a tile and
// its neighbours, whose halos overlap, are read through the same L2.
__device__ __forceinline__ void tile_of(int b, int nb, int gx, int xcd, int& bx, int& by) {
    if (xcd == 2 && (gx & 7) == 0 && (nb & 7) == 0) {
        // XCD x owns the column strip of tiles [x*sw, x*sw + sw) and walks it
        // row by row: its L2 sees both the horizontal and the vertical
        // neighbours of a tile, and all XCDs advance through the same rows
        const int sw = gx >> 3, x = b & 7, j = b >> 3;
        by = j / sw;
        bx = x * sw + (j - by * sw);
        return;
    }
    int t = b;
    if (xcd == 1) {
        const int q = nb >> 3, r = nb & 7, x = b & 7, j = b >> 3;
        t = x * q + min(x, r) + j;
    }
    by = t / gx;
    bx = t - by * gx;
}

// The order a launch's tiles are walked in for the caller's mode.  Column
// strips (2) need tile columns in multiples of 8.  Other shapes get
// contiguous runs (1) as long as two rows of tiles, at `bytes` read per cell,
// stay in 3 MB of an XCD's 4 MB L2, and row-major order beyond that.  Hydro, us
// per launch, runs against row-major: 640^2 9.7 / 12.7, 1088^2 20.2 / 29.5,
// 1408^2 28.7 / 45.5, 2240^2 86.9 / 99.4; 3000^2 173.3 / 170.6.
int tile_order(int mode, int nx, int tx, int ty, int bytes) {
    if (mode != 2) return mode;
    if (((nx + tx - 1) / tx) % 8 == 0) return 2;
    return size_t(2) * size_t(nx) * size_t(ty) * size_t(bytes) <= (size_t(3) << 20) ? 1 : 0;
}

template <int TX, int TY, int HA, int NT, bool EXTRA, bool NTS>
__global__ __launch_bounds__(NT) void k_fused_hydro(HydroIO io, int nx, int ny, uint32_t step,
                                                    uint32_t terrain, int rain, int xcd, KParams k) {
    __shared__ float lds[6 * HydroTile<TX, TY, HA, NT>::NLDS];
    int bx, by;
    tile_of(blockIdx.x, gridDim.x, (nx + TX - 1) / TX, xcd, bx, by);
    hydro_tile<TX, TY, HA, NT, EXTRA, NTS>(lds, io, nx, ny, bx, by, step, terrain, rain, k);
}

// ---------------------------------------------------------------------------
// thermal kernel: thermal layer 0, thermal layer 1, smoothing
//
// LDS holds rock, dirt and the outflow scale g on the tile +- 5 cells.  Stages
// (radius = cells around the tile they are evaluated on):
//   A r4: g of layer 0      B r3: rock += thermal change (written in place)
//   C r2: g of layer 1      D r1: dirt += thermal change (written in place)
//   E r0: smoothing, write back.
// In-place updates go through registers between two barriers.
// ---------------------------------------------------------------------------
constexpr int TH = 5;   // dependency radius of thermal L0 + L1 + smoothing

// Calls fn(it, lx, ly) for the cells of the region of radius RAD around the
// thermal tile, in LDS coordinates.
template <int TX, int TY, int NT, int RAD, class F>
__device__ __forceinline__ void region_for(int tid, F&& fn) {
    tile_region_for<TX, TY, NT, RAD>(tid, [&](int it, int rx, int ry) { fn(it, rx + (TH - RAD), ry + (TH - RAD)); });
}

template <int TX, int TY>
struct ThermalTile {
    static constexpr int W0 = TX + 2 * TH, N0 = W0 * (TY + 2 * TH);
};

// One output tile (bx, by) of the thermal kernel; `lds` holds 3*N0 floats.
// LOADED: its first two arrays already hold rock and dirt.
template <int TX, int TY, int NT, bool EXTRA = false, bool NTS = false, bool LOADED = false>
__device__ __forceinline__ void thermal_tile(float* lds, const ThermIO& io, int nx, int ny, int bx,
                                             int by, int do_thermal, int do_smooth, const KParams& k) {
    constexpr int W0 = ThermalTile<TX, TY>::W0, N0 = ThermalTile<TX, TY>::N0;
    float* s_r = lds;
    float* s_d = lds + N0;
    float* s_g = lds + 2 * N0;
    // Opaque to the optimiser: values derived from the thread index are then
    // recomputed per tile instead of being hoisted out of the batched tile
    // loop and held in registers across tiles.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int x0 = bx * TX - TH, y0 = by * TY - TH;   // grid coords of LDS (0,0)
    constexpr int DX[8] = {-1, 1, 0, 0, -1, 1, -1, 1};
    constexpr int DY[8] = {0, 0, 1, -1, 1, 1, -1, -1};
    constexpr int OFF[8] = {-1, 1, W0, -W0, W0 - 1, W0 + 1, -W0 - 1, -W0 + 1};
    (void)DX; (void)DY;
    auto in_grid = [&](int lx, int ly) {
        const int gx = x0 + lx, gy = y0 + ly;
        return gx >= 0 && gy >= 0 && gx < nx && gy < ny;
    };

    // load rock, dirt; out of grid reads HG_OOB_HEIGHT (thermal_erosion.glsl:20-26).
    // Loads use clamped addresses and are all issued before the first LDS write.
    if constexpr (!LOADED) {
        constexpr int IL = Region<TX, TY, NT, TH>::ITER;
        float lr[IL], ld[IL];
        region_for<TX, TY, NT, TH>(tid, [&](int it, int lx, int ly) {
            const int gx = x0 + lx, gy = y0 + ly;
            const size_t g = at(min(max(gx, 0), nx - 1), min(max(gy, 0), ny - 1), nx);
            const bool in = gx >= 0 && gy >= 0 && gx < nx && gy < ny;
            lr[it] = in ? io.r[g] : HG_OOB_HEIGHT;
            ld[it] = in ? io.d[g] : HG_OOB_HEIGHT;
        });
        region_for<TX, TY, NT, TH>(tid, [&](int it, int lx, int ly) {
            s_r[ly * W0 + lx] = lr[it];
            s_d[ly * W0 + lx] = ld[it];
        });
        __syncthreads();
    }

    if (do_thermal) {
        // ---- A: layer-0 outflow scale
        // (evaluated out of the grid too, on the out-of-grid height, and dropped)
        region_for<TX, TY, NT, 4>(tid, [&](int, int lx, int ly) {
            const int li = ly * W0 + lx;
            const float r = s_r[li];
            float D[8];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) D[kk] = r - s_r[li + OFF[kk]];
            const float g = thermal_g(D, r, 0, k);
            s_g[li] = in_grid(lx, ly) ? g : 0.0f;
        });
        __syncthreads();
        // ---- B: layer-0 transport, rock in place
        {
            float nr[Region<TX, TY, NT, 3>::ITER];
            region_for<TX, TY, NT, 3>(tid, [&](int it, int lx, int ly) {
                const int li = ly * W0 + lx;
                const float r = s_r[li], g = s_g[li];
                float acc = 0.0f;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    const float Dk = r - s_r[li + OFF[kk]];
                    acc = acc + thermal_term(Dk, g, s_g[li + OFF[kk]],
                                             kk < 4 ? k.tan_alpha[0] : k.thr_diag[0]);
                }
                nr[it] = r + acc;
            });
            __syncthreads();
            region_for<TX, TY, NT, 3>(tid, [&](int it, int lx, int ly) {
                if (in_grid(lx, ly)) s_r[ly * W0 + lx] = nr[it];
            });
            __syncthreads();
        }
        // ---- C: layer-1 outflow scale (rock after layer 0)
        region_for<TX, TY, NT, 2>(tid, [&](int, int lx, int ly) {
            const int li = ly * W0 + lx;
            const float r = s_r[li], d = s_d[li];
            float D[8];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) D[kk] = (r - s_r[li + OFF[kk]]) + (d - s_d[li + OFF[kk]]);
            const float g = thermal_g(D, d, 1, k);
            s_g[li] = in_grid(lx, ly) ? g : 0.0f;
        });
        __syncthreads();
        // ---- D: layer-1 transport, dirt in place
        {
            float nd[Region<TX, TY, NT, 1>::ITER];
            region_for<TX, TY, NT, 1>(tid, [&](int it, int lx, int ly) {
                const int li = ly * W0 + lx;
                const float r = s_r[li], d = s_d[li], g = s_g[li];
                float acc = 0.0f;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    const float Dk = (r - s_r[li + OFF[kk]]) + (d - s_d[li + OFF[kk]]);
                    acc = acc + thermal_term(Dk, g, s_g[li + OFF[kk]],
                                             kk < 4 ? k.tan_alpha[1] : k.thr_diag[1]);
                }
                nd[it] = d + acc;
            });
            __syncthreads();
            region_for<TX, TY, NT, 1>(tid, [&](int it, int lx, int ly) {
                if (in_grid(lx, ly)) s_d[ly * W0 + lx] = nd[it];
            });
            __syncthreads();
        }
    }

    // ---- E: smoothing on the tile, write back
    region_for<TX, TY, NT, 0>(tid, [&](int, int lx, int ly) {
        const int gx = x0 + lx, gy = y0 + ly;
        const int li = ly * W0 + lx;
        const float r0 = s_r[li], d0 = s_d[li];
        float r = r0, d = d0;
        if (do_smooth && gx > 0 && gy > 0 && gx < nx - 1 && gy < ny - 1)
            smooth_cell(r, d, s_r[li - 1], s_d[li - 1], s_r[li + 1], s_d[li + 1], s_r[li + W0],
                        s_d[li + W0], s_r[li - W0], s_d[li - W0], k.smooth_m);
        if (gx < nx && gy < ny) {
            const size_t g = at(gx, gy, nx);
            if (EXTRA && io.tr5) {
                st_out<NTS>(&io.tr5[g], r0);
                st_out<NTS>(&io.td6[g], d0);
            }
            st_out<NTS>(&io.ro[g], r);
            st_out<NTS>(&io.dout[g], d);
        }
    });
}

template <int TX, int TY, int NT, bool EXTRA, bool NTS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_fused_thermal(
    ThermIO io, int nx, int ny, int do_thermal, int do_smooth, int xcd, KParams k) {
    __shared__ float lds[3 * ThermalTile<TX, TY>::N0];
    int bx, by;
    tile_of(blockIdx.x, gridDim.x, (nx + TX - 1) / TX, xcd, bx, by);
    thermal_tile<TX, TY, NT, EXTRA, NTS>(lds, io, nx, ny, bx, by, do_thermal, do_smooth, k);
}

// ---------------------------------------------------------------------------
// The whole step on one tile, for small maps
//
// A small map's step is bound by its launches, not by their work: two kernels
// of about 6 us each with 4 us between them, and 3 us of host time per launch.
// One launch does both: the hydro stages run on the tile +- 5 cells the thermal
// stages need (2 cells otherwise), hand rock and dirt over in LDS, and the
// halo's repeated work is the price (2.1 times the cells of a 32 x 16 tile, 3
// times those of a 32 x 8 one).  us per step, alone / with three maps at once:
//         two kernels  32x8/768   32x16/512  64x16/1024
//    64^2  10.8/ 6.0    6.7/ 3.3   9.7/ 3.6  10.3/ 3.8
//   256^2  12.9/ 6.4    8.4/ 3.6  11.2/ 4.2  11.0/ 4.3
//   384^2  17.1/ 8.1   12.7/ 7.0  12.8/ 5.3  11.4/ 6.3
//   512^2  20.4/10.2   17.1/12.2  15.8/ 7.9  14.5/11.9
//   640^2  23.7/12.5   24.8/18.8  21.7/12.1  21.7/16.3
//   768^2  28.2/14.4   31.5/26.8  26.0/17.3  32.0/22.8
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct StepTile {
    using H = HydroTile<TX, TY, TH, 64>;
    static constexpr int THERMAL = 2 * H::NE + 2 * H::NTILE;     // rock, dirt, g of the thermal stages
    static constexpr int NLDS = 6 * H::NLDS;
    static_assert(THERMAL + 3 * H::NE < NLDS, "the thermal stages and the far list's length fit the input arrays");
    static_assert(H::NE == ThermalTile<TX, TY>::N0, "both stages number the tile +- 5 cells alike");
};

template <int TX, int TY, int NT, bool EXTRA>
__global__ __launch_bounds__(NT) void k_step_tile(HydroIO io, ThermIO tio, int nx, int ny, uint32_t step,
                                                  uint32_t terrain, int rain, int do_thermal, int do_smooth, int xcd,
                                                  KParams k) {
    __shared__ float lds[StepTile<TX, TY>::NLDS];
    int bx, by;
    tile_of(blockIdx.x, gridDim.x, (nx + TX - 1) / TX, xcd, bx, by);
    hydro_tile<TX, TY, TH, NT, EXTRA, false, true>(lds, io, nx, ny, bx, by, step, terrain, rain, k);
    thermal_tile<TX, TY, NT, EXTRA, false, true>(lds + StepTile<TX, TY>::THERMAL, tio, nx, ny, bx, by, do_thermal,
                                                 do_smooth, k);
}

// ---------------------------------------------------------------------------
// thermal kernel, marching form
//
// A wave owns a strip of 128 columns, two per lane, of which it writes the
// inner 116, and marches down its rows: each new row advances layer 0, layer 1
// and smoothing, each two to three rows behind the one before it.
// Vertical neighbours stay in registers and horizontal ones come from the
// adjacent lane (DPP wave shifts): no LDS, no barriers.
//
// Why: the tile form is bound by VALU issue (485 instructions per cell), and
// there every pair of neighbours is looked at four times, by both cells, once
// for the outflow scale and once for the transport.  Here a pair (an edge from
// cell p to cell q) is looked at once: its difference D = p - q gives
//   P = D > thr ? D : 0     what p sends towards q, over g_p
//   N = D < -thr ? D : 0    (-) what q sends towards p, over g_q
// both cells' sums over marked directions take P or -N, and when both g are
// known the transfer is T = P g_p + N g_q: one of the products is the tile
// form's G * D, the other is a zero.  p adds -T, q adds T, in the same
// order of directions as thermal_g and thermal_term, so the results are the
// same bit for bit, as long as the zeros meet no infinity or NaN, in a height or
// a g.  A wave that has seen one (its sums of products of them are not finite)
// runs its segment again in the ODD form, which takes thermal_term (a test per
// row instead, and the products or thermal_term after it: 5 % slower).
//
// About 265 VALU instructions per cell, times 1.10 for the columns and 1.12
// (at 49 rows) for the rows that are not its own, issued at one per 3.5 cycles
// per SIMD, near the rate of their mix (2.7 with two operands, 4.2 with three
// or a lane shift).  142 registers: three waves per SIMD; held to 128 for four
// it spills and slows down (150).  4096^2: 165 -> 126 us per launch, a step
// 430 -> 389 us, with three maps at once 402 -> 354; 2048^2 with three maps at
// once 104 -> 91 us per step.  (The check for infinities, 6 of the instructions,
// came later: 4 steps at 4096^2 1375 -> 1378 us.)
// ---------------------------------------------------------------------------
constexpr int MARCH_TX = 116;          // columns a wave writes
constexpr int MARCH_HX = 6;            // halo columns on each side (5 needed, even for the pairs)

// Value of the next (right) and the previous (left) lane.
__device__ __forceinline__ float lane_right(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));   // wave_shl:1
}
__device__ __forceinline__ float lane_left(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));   // wave_shr:1
}

// A row of the strip: the lane's two cells and the right lane's first cell.
// Layer 0 looks at rock alone, layer 1 at rock + dirt.
template <int LAYER>
struct MarchRow {
    float r[2], d[2], r_right, d_right;
};
template <int LAYER>
__device__ __forceinline__ float march_diff(float ra, float da, float rb, float db) {
    return LAYER == 0 ? ra - rb : (ra - rb) + (da - db);
}
struct MarchEdge {
    float D[2], P[2], N[2];
    __device__ __forceinline__ void mark(float thr) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            P[c] = D[c] > thr ? D[c] : 0.0f;
            N[c] = D[c] < -thr ? D[c] : 0.0f;
        }
    }
};
// What a layer carries from row to row.  a: the newest row; z: the row below it.
template <int LAYER>
struct MarchLayer {
    MarchRow<LAYER> a, z;
    MarchEdge h;                        // edges along row a: (x, x+1)
    float h_D_left, h_N_left;           // the left lane's second edge
    MarchEdge v, e, f;                  // edges z-a: (x,z)-(x,a), (x,z)-(x+1,a), (x+1,z)-(x,a); D unused
    float e_N_left;
    float mc[2], md[2];                 // largest difference of row a's cells towards row z
    float gz[2], gz_right;              // outflow scale of row z
    float finite;                       // so were all heights and g so far, if this is
    float th[2], th_left;               // transfers along row z
    float tv[2], te[2], te_left, tf[2]; // transfers between row z and the row below it
};

// Takes the next row b; returns in out[] the layer's new heights of row z
// (a.* are then b, z.* a).  in_a, in_z: whether this lane's cells of those rows
// are on the grid.
template <int LAYER, bool ODD>
__device__ __forceinline__ void march_advance(MarchLayer<LAYER>& s, const MarchRow<LAYER>& b, bool in_a, bool in_z,
                                              const KParams& k, float (&out)[2]) {
    const float ta = k.tan_alpha[LAYER], td = k.thr_diag[LAYER];
    const MarchRow<LAYER>& a = s.a;
    auto diff = [](float ra, float da, float rb, float db) { return march_diff<LAYER>(ra, da, rb, db); };
    MarchEdge v, e, f;
    v.D[0] = diff(a.r[0], a.d[0], b.r[0], b.d[0]);
    v.D[1] = diff(a.r[1], a.d[1], b.r[1], b.d[1]);
    e.D[0] = diff(a.r[0], a.d[0], b.r[1], b.d[1]);
    e.D[1] = diff(a.r[1], a.d[1], b.r_right, b.d_right);
    f.D[0] = diff(a.r[1], a.d[1], b.r[0], b.d[0]);
    f.D[1] = diff(a.r_right, a.d_right, b.r[1], b.d[1]);
    v.mark(ta);
    e.mark(td);
    f.mark(td);
    const float e_D_left = lane_left(e.D[1]), e_N_left = lane_left(e.N[1]);
    const float f_D_left = lane_left(f.D[1]), f_P_left = lane_left(f.P[1]);
    // outflow scale of row a (thermal_g)
    float g[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const float DL = c ? s.h.D[0] : s.h_D_left, NL = c ? s.h.N[0] : s.h_N_left;
        const float DLT = c ? f.D[0] : f_D_left, PLT = c ? f.P[0] : f_P_left;
        const float NLB = c ? s.e.N[0] : s.e_N_left;
        float bk = s.h.P[c] - NL;
        bk = bk + v.P[c];
        bk = bk - s.v.N[c];
        bk = bk + PLT;
        bk = bk + e.P[c];
        bk = bk - NLB;
        bk = bk - s.f.N[c];
        const float mc = fmaxf(fmaxf(-DL, s.h.D[c]), fmaxf(v.D[c], s.mc[c]));
        const float md = fmaxf(fmaxf(DLT, e.D[c]), s.md[c]);
        const float H = fminf(LAYER == 0 ? a.r[c] : a.d[c], fmaxf(fmaxf(mc, md), 0.0f));
        const float rmax = fmaxf(mc, md * 0.70710678118654752f);
        float sharp = fmaxf(1.0f + atanf(rmax) - k.Kalpha[LAYER], 1.0f);
        sharp = sharp * (sharp * sharp);
        const float S = (k.dt * k.Kspeed[LAYER] * 0.5f) * sharp * H;
        g[c] = (bk > 0.0f && in_a) ? S * rcp(bk) : 0.0f;
    }
    const float g_right = lane_right(g[0]);
    // transfers along row a and between rows z and a
    s.finite = fmaf(a.r[0], a.r[1], fmaf(g[0], g[1], s.finite));
    if constexpr (LAYER == 1) s.finite = fmaf(a.d[0], a.d[1], s.finite);
    float th[2], tv[2], te[2], tf[2];
    if constexpr (!ODD) {
        auto send = [](float P, float gp, float N, float gq) { return fmaf(N, gq, P * gp); };
        th[0] = send(s.h.P[0], g[0], s.h.N[0], g[1]);
        th[1] = send(s.h.P[1], g[1], s.h.N[1], g_right);
        tv[0] = send(s.v.P[0], s.gz[0], s.v.N[0], g[0]);
        tv[1] = send(s.v.P[1], s.gz[1], s.v.N[1], g[1]);
        te[0] = send(s.e.P[0], s.gz[0], s.e.N[0], g[1]);
        te[1] = send(s.e.P[1], s.gz[1], s.e.N[1], g_right);
        tf[0] = send(s.f.P[0], s.gz[1], s.f.N[0], g[0]);
        tf[1] = send(s.f.P[1], s.gz_right, s.f.N[1], g[1]);
    } else {
        const MarchRow<LAYER>& z = s.z;
        const float zr = lane_right(z.r[0]), zd = lane_right(z.d[0]);
        auto send = [](float D, float thr, float gp, float gq) { return -thermal_term(D, gp, gq, thr); };
        th[0] = send(s.h.D[0], ta, g[0], g[1]);
        th[1] = send(s.h.D[1], ta, g[1], g_right);
        tv[0] = send(diff(z.r[0], z.d[0], a.r[0], a.d[0]), ta, s.gz[0], g[0]);
        tv[1] = send(diff(z.r[1], z.d[1], a.r[1], a.d[1]), ta, s.gz[1], g[1]);
        te[0] = send(diff(z.r[0], z.d[0], a.r[1], a.d[1]), td, s.gz[0], g[1]);
        te[1] = send(diff(z.r[1], z.d[1], a.r_right, a.d_right), td, s.gz[1], g_right);
        tf[0] = send(diff(z.r[1], z.d[1], a.r[0], a.d[0]), td, s.gz[1], g[0]);
        tf[1] = send(diff(zr, zd, a.r[1], a.d[1]), td, s.gz_right, g[1]);
    }
    const float th_left = lane_left(th[1]), te_left = lane_left(te[1]), tf_left = lane_left(tf[1]);
    // new heights of row z: L, R, T, B, LT, RT, LB, RB
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float acc = (c ? s.th[0] : s.th_left) - s.th[c];
        acc = acc - tv[c];
        acc = acc + s.tv[c];
        acc = acc - (c ? tf[0] : tf_left);
        acc = acc - te[c];
        acc = acc + (c ? s.te[0] : s.te_left);
        acc = acc + s.tf[c];
        const float h = LAYER == 0 ? s.z.r[c] : s.z.d[c];
        out[c] = in_z ? h + acc : h;
    }
    // the next row
    s.h.D[0] = diff(b.r[0], b.d[0], b.r[1], b.d[1]);
    s.h.D[1] = diff(b.r[1], b.d[1], b.r_right, b.d_right);
    s.h.mark(ta);
    s.h_D_left = lane_left(s.h.D[1]);
    s.h_N_left = lane_left(s.h.N[1]);
    s.mc[0] = -v.D[0];
    s.mc[1] = -v.D[1];
    s.md[0] = fmaxf(-e_D_left, -f.D[0]);
    s.md[1] = fmaxf(-e.D[0], -f.D[1]);
    s.v = v;
    s.e = e;
    s.f = f;
    s.e_N_left = e_N_left;
    s.z = a;
    s.a = b;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        s.gz[c] = g[c];
        s.th[c] = th[c];
        s.tv[c] = tv[c];
        s.te[c] = te[c];
        s.tf[c] = tf[c];
    }
    s.gz_right = g_right;
    s.th_left = th_left;
    s.te_left = te_left;
}

// Rows per wave.  A wave also runs 4 to 10 rows of every stage above and below
// its own, and a workgroup (4 waves, one below the other) occupies a third of
// a CU: the most rows that still fill the 256 CUs three times over are the
// fastest, 49 at 4096^2 (us per launch: 16 rows 139, 37 rows 133, 49 rows 126,
// 56 rows 139, 64 rows 156).  Above 96 rows a second round costs less than the
// last one's idle CUs.
inline int march_rows(int nx, int ny) {
    const int strips = (nx + MARCH_TX - 1) / MARCH_TX;
    for (int rounds = 1;; ++rounds) {
        const int segs = std::max(1, rounds * 3 * 256 / strips);
        const int rows = (ny + 4 * segs - 1) / (4 * segs);
        if (rows <= 96) return std::max(rows, 8);
    }
}

// Rows [ys, ye) of the strip whose first written column is xs; false if the
// lane met a height or g that is not finite.
template <bool EXTRA, bool NTS, bool ODD>
__device__ __forceinline__ bool march_segment(const ThermIO& io, int nx, int ny, int xs, int ys, int ye, int do_thermal,
                                              int do_smooth, const KParams& k) {
    const int lane = int(threadIdx.x) & 63;
    const int x = xs - MARCH_HX + 2 * lane;                  // the lane's first column; even, like nx
    const bool inx = x >= 0 && x < nx;
    const bool mine = inx && lane >= MARCH_HX / 2 && lane < 64 - MARCH_HX / 2;
    const int xc = min(max(x, 0), nx - 2);
    auto iny = [&](int y) { return y >= 0 && y < ny; };
    auto load = [&](const float* p, int y) {
        return *reinterpret_cast<const float2*>(p + at(xc, min(max(y, 0), ny - 1), nx));
    };
    float r1[3][2], d1[3][2];                                // rows yo-1, yo, yo+1 after both layers
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c) r1[j][c] = d1[j][c] = 0.0f;
    auto push = [&](float ra, float rb, float da, float db) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            r1[0][c] = r1[1][c];
            r1[1][c] = r1[2][c];
            d1[0][c] = d1[1][c];
            d1[1][c] = d1[2][c];
        }
        r1[2][0] = ra;
        r1[2][1] = rb;
        d1[2][0] = da;
        d1[2][1] = db;
    };
    // smoothing of row yo, write it
    auto emit = [&](int yo) {
        const float r0 = r1[1][0], rr1 = r1[1][1], d0 = d1[1][0], dd1 = d1[1][1];
        float r[2] = {r0, rr1}, d[2] = {d0, dd1};
        const float rl = lane_left(rr1), rr = lane_right(r0), dl = lane_left(dd1), dr = lane_right(d0);
        const bool rows = do_smooth && yo > 0 && yo < ny - 1;
        if (rows && x > 0)
            smooth_cell(r[0], d[0], rl, dl, rr1, dd1, r1[2][0], d1[2][0], r1[0][0], d1[0][0], k.smooth_m);
        if (rows && x + 1 < nx - 1)
            smooth_cell(r[1], d[1], r0, d0, rr, dr, r1[2][1], d1[2][1], r1[0][1], d1[0][1], k.smooth_m);
        if (mine) {
            const size_t g = at(x, yo, nx);
            if (EXTRA && io.tr5) {
                st_out2<NTS>(&io.tr5[g], r0, rr1);
                st_out2<NTS>(&io.td6[g], d0, dd1);
            }
            st_out2<NTS>(&io.ro[g], r[0], r[1]);
            st_out2<NTS>(&io.dout[g], d[0], d[1]);
        }
    };
    if (!do_thermal) {                                       // smoothing alone
        for (int y = ys - 1; y <= ye; ++y) {
            const float2 r = load(io.r, y), d = load(io.d, y);
            push(r.x, r.y, d.x, d.y);
            if (y > ys) emit(y - 1);
        }
        return true;
    }
    MarchLayer<0> l0{};
    MarchLayer<1> l1{};
    float2 nr = load(io.r, ys - TH), nd = make_float2(0.0f, 0.0f);
    // y: the row layer 0 takes; layer 1 takes y - 2, smoothing gives y - 5
    auto row = [&](int y, bool upper) {
        const bool in = inx && iny(y);
        MarchRow<0> b;
        b.r[0] = in ? nr.x : HG_OOB_HEIGHT;
        b.r[1] = in ? nr.y : HG_OOB_HEIGHT;
        b.d[0] = b.d[1] = b.d_right = 0.0f;
        const float2 dd = nd;
        nr = load(io.r, y + 1);
        if (upper) nd = load(io.d, y - 1);
        b.r_right = lane_right(b.r[0]);
        float rz[2];
        march_advance<0, ODD>(l0, b, inx && iny(y - 1), inx && iny(y - 2), k, rz);
        if (!upper) return;
        const bool in2 = inx && iny(y - 2);
        MarchRow<1> q;
        q.r[0] = rz[0];
        q.r[1] = rz[1];
        q.d[0] = in2 ? dd.x : HG_OOB_HEIGHT;
        q.d[1] = in2 ? dd.y : HG_OOB_HEIGHT;
        q.r_right = lane_right(q.r[0]);
        q.d_right = lane_right(q.d[0]);
        const float rock[2] = {l1.z.r[0], l1.z.r[1]};        // rock of row y - 4
        float dz[2];
        march_advance<1, ODD>(l1, q, inx && iny(y - 3), inx && iny(y - 4), k, dz);
        push(rock[0], rock[1], dz[0], dz[1]);
        if (y - 5 >= ys && y - 5 < ye) emit(y - 5);
    };
    for (int y = ys - TH; y < ys - 1; ++y) row(y, false);
    nd = load(io.d, ys - 3);
    for (int y = ys - 1; y <= ye + 4; y += 2) {              // two at a time: the carried rows swap roles
        row(y, true);
        row(y + 1, true);
    }
    return fabsf(l0.finite) < INFINITY && fabsf(l1.finite) < INFINITY;
}

template <bool EXTRA, bool NTS>
__device__ __forceinline__ void thermal_march(const ThermIO& io, int nx, int ny, int xs, int ys, int ye, int do_thermal,
                                              int do_smooth, const KParams& k) {
    const bool finite = march_segment<EXTRA, NTS, false>(io, nx, ny, xs, ys, ye, do_thermal, do_smooth, k);
    if (__any(!finite)) (void)march_segment<EXTRA, NTS, true>(io, nx, ny, xs, ys, ye, do_thermal, do_smooth, k);
}

template <bool EXTRA, bool NTS>
__global__ __launch_bounds__(256) void k_march_thermal(ThermIO io, int nx, int ny, int rows, int do_thermal,
                                                       int do_smooth, int xcd, KParams k) {
    const int gx = (nx + MARCH_TX - 1) / MARCH_TX;
    int bx, by;
    tile_of(blockIdx.x, gridDim.x, gx, xcd, bx, by);
    const int ys = (by * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6)) * rows;
    if (ys >= ny) return;
    thermal_march<EXTRA, NTS>(io, nx, ny, bx * MARCH_TX, ys, min(ys + rows, ny), do_thermal, do_smooth, k);
}

// ---------------------------------------------------------------------------
// Batched persistent kernels: one launch per pass covers the tiles of every
// terrain of a batch.  Workgroup b processes work-list entries b, b+G, ...
// (G = grid size); an entry packs (terrain << 24) | (tile_y << 12) | tile_x.
// Each terrain's descriptor holds both buffers of its 9 state planes; bit p of
// `cur` selects which buffer of plane p is the current (input) one.
// ---------------------------------------------------------------------------
__device__ __forceinline__ HydroIO batch_hydro_io(const BatchTerrain& T, uint32_t cur) {
    HydroIO io;
    const float** in[9] = {&io.r, &io.d, &io.b, &io.fl, &io.fr, &io.ft, &io.fb, &io.s0, &io.s1};
    float** out[9] = {&io.ro, &io.dout, &io.bo, &io.flo, &io.fro, &io.fto, &io.fbo, &io.s0o, &io.s1o};
#pragma unroll
    for (int p = 0; p < 9; ++p) {
        const int c = (cur >> p) & 1;
        *in[p] = T.plane[p][c];
        *out[p] = T.plane[p][c ^ 1];
    }
    io.vx = io.vy = io.vz = nullptr;
    return io;
}

template <int TX, int TY, int HA, int NT, bool NTS>
__global__ __launch_bounds__(NT) void k_batch_hydro(const BatchTerrain* __restrict__ terr,
                                                    const uint32_t* __restrict__ tiles,
                                                    int ntiles, uint32_t cur, const uint32_t* step_ptr,
                                                    uint32_t step_off, int rain) {
    __shared__ float lds[6 * HydroTile<TX, TY, HA, NT>::NLDS];
    const uint32_t step = *step_ptr + step_off;
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const uint32_t e = tiles[t];
        if (e == 0xffffffffu) continue;
        const int ti = int(e >> 24), by = int((e >> 12) & 0xfffu), bx = int(e & 0xfffu);
        // copy the descriptor into registers: a reference into global memory
        // would be re-read after every global store of the tile
        const BatchTerrain& T = terr[ti];
        const HydroIO io = batch_hydro_io(T, cur);
        const KParams k = T.k;
        const int n = T.n;
        hydro_tile<TX, TY, HA, NT, false, NTS>(lds, io, n, n, bx, by, step, uint32_t(ti), rain, k);
        __syncthreads();
    }
}

// The marching form over a work-list of MARCH_TX x (4 rows) entries.
template <bool NTS>
__global__ __launch_bounds__(256) void k_batch_march(const BatchTerrain* __restrict__ terr,
                                                     const uint32_t* __restrict__ tiles, int ntiles, uint32_t cur,
                                                     int rows, int do_thermal, int do_smooth) {
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const uint32_t e = tiles[t];
        if (e == 0xffffffffu) continue;
        const int ti = int(e >> 24), by = int((e >> 12) & 0xfffu), bx = int(e & 0xfffu);
        const BatchTerrain& T = terr[ti];
        ThermIO io;
        const int cr = cur & 1, cd = (cur >> 1) & 1;
        io.r = T.plane[HG_P_ROCK][cr];
        io.ro = T.plane[HG_P_ROCK][cr ^ 1];
        io.d = T.plane[HG_P_DIRT][cd];
        io.dout = T.plane[HG_P_DIRT][cd ^ 1];
        const KParams k = T.k;
        const int n = T.n;
        const int ys = (by * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6)) * rows;
        if (ys < n) thermal_march<false, NTS>(io, n, n, bx * MARCH_TX, ys, min(ys + rows, n), do_thermal, do_smooth, k);
    }
}

template <int TX, int TY, int NT, bool NTS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_batch_thermal(
    const BatchTerrain* __restrict__ terr, const uint32_t* __restrict__ tiles, int ntiles,
    uint32_t cur, int do_thermal,
    int do_smooth) {
    __shared__ float lds[3 * ThermalTile<TX, TY>::N0];
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const uint32_t e = tiles[t];
        if (e == 0xffffffffu) continue;
        const int ti = int(e >> 24), by = int((e >> 12) & 0xfffu), bx = int(e & 0xfffu);
        const BatchTerrain& T = terr[ti];
        ThermIO io;
        const int cr = cur & 1, cd = (cur >> 1) & 1;
        io.r = T.plane[HG_P_ROCK][cr];
        io.ro = T.plane[HG_P_ROCK][cr ^ 1];
        io.d = T.plane[HG_P_DIRT][cd];
        io.dout = T.plane[HG_P_DIRT][cd ^ 1];
        const KParams k = T.k;
        const int n = T.n;
        thermal_tile<TX, TY, NT, false, NTS>(lds, io, n, n, bx, by, do_thermal, do_smooth, k);
        __syncthreads();
    }
}

// Compiled tile variants (the autotuner picks among them per grid size).
//                      TX   TY  HA   NT
#define HG_HYDRO_VARIANTS(X) \
    X(0,  64, 16, 2, 256)    \
    X(1,  64, 32, 2, 512)    \
    X(2, 128, 16, 2, 512)    \
    X(3,  64,  8, 2, 256)    \
    X(4,  64, 16, 3, 256)    \
    X(5, 128,  8, 2, 256)    \
    X(6,  64, 16, 2, 512)    \
    X(7, 128, 16, 2, 1024)   \
    X(8,  64,  8, 2, 512)
//                        TX   TY   NT
#define HG_THERMAL_VARIANTS(X) \
    X(0,  64, 16, 256)         \
    X(1,  64, 32, 256)         \
    X(2,  64, 32, 512)         \
    X(3,  64, 64, 512)         \
    X(4, 128, 32, 512)         \
    X(5,  32, 32, 256)         \
    X(6, 128, 16, 512)         \
    X(7,  64, 64, 1024)        \
    X(8, 128, 32, 1024)        \
    X(9,  64, 16, 512)         \
    X(10, 64,  8, 1024)
// the marching form follows them (in HG_THERMAL_VARIANTS' numbering)
constexpr int MARCH_VARIANT = 11;

}  // namespace

// The variants a map gets that was not tuned, by its number of 64 x 16 tiles
// (cells / 1024).  Few tiles leave CUs idle and each cell of a tile is on the
// critical path, so small maps get small tiles with more threads per cell;
// large ones get the tiles with less halo.  us per launch, alone / with three
// maps at once (hydro; thermal figures are of the whole step):
//          hydro 64x8/512  64x16/256  64x16/512  128x16/512
//   256^2     6.8/ 3.1     10.8/ 4.8
//   512^2     9.5/ 4.7     14.9/ 6.8      - / 4.8
//  1024^2                  22.4/15.5   18.3/13.7    - /14.6
//  2048^2                  72.6/61.8   69.7/62.9  70.4/62.7
//  4096^2                 265.7/253.0 265.2/258.1 261.8/249.6
//        thermal 64x8/1024 64x16/512  64x32/256  64x32/512
//   256^2    15.5/ 6.3       - / 6.6  28.7/10.1
//   512^2    20.2/ -         - / 8.8  31.8/11.3
//   768^2                  33.8/16.3  41.2/17.8    - /17.0
//  1024^2                  36.3/ -    41.4/23.4  36.7/22.0
//  2048^2                            126.3/99.9 118.0/97.8
int default_hydro_variant(size_t cells) {
    const size_t tiles = cells / 1024;
    return tiles < 512 ? 8 : tiles < 4096 ? 6 : 2;
}
int default_thermal_variant(size_t cells) {
    const size_t tiles = cells / 1024;
    return tiles < 128 ? 10 : tiles < 1024 ? 9 : tiles < 4096 ? 2 : MARCH_VARIANT;
}

// Rows of a thermal work-list entry for a batch of these sides.  The marching
// form has no fixed tile: a workgroup's rows cost about rows / 4 + 6 (see
// march_rows), times the rounds the entries take at 3 workgroups per CU.
int batch_thermal_rows(int variant, const int* sides, int count) {
    int tx = 0, ty = 0, h = 0, nt = 0;
    if (!thermal_variant_info(variant, &tx, &ty, &h, &nt) || variant != MARCH_VARIANT) return ty;
    long best_cost = 0;
    for (int rows = 8; rows <= 96; ++rows) {
        long entries = 0;
        for (int t = 0; t < count; ++t)
            entries += long((sides[t] + tx - 1) / tx) * ((sides[t] + 4 * rows - 1) / (4 * rows));
        const long cost = (entries + 3 * 256 - 1) / (3 * 256) * (rows + 6);
        if (rows == 8 || cost <= best_cost) {
            best_cost = cost;
            ty = 4 * rows;
        }
    }
    return ty;
}

int hydro_variant_count() {
#define X(i, tx, ty, ha, nt) +1
    return 0 HG_HYDRO_VARIANTS(X);
#undef X
}

int thermal_variant_count() {
#define X(i, tx, ty, nt) +1
    return 1 HG_THERMAL_VARIANTS(X);
#undef X
}

bool hydro_variant_info(int v, int* tx, int* ty, int* halo, int* nt) {
    switch (v) {
#define X(i, TX_, TY_, HA_, NT_) \
    case i: *tx = TX_; *ty = TY_; *halo = HA_; *nt = NT_; return true;
        HG_HYDRO_VARIANTS(X)
#undef X
        default: return false;
    }
}

bool thermal_variant_info(int v, int* tx, int* ty, int* halo, int* nt) {
    switch (v) {
        case MARCH_VARIANT: *tx = MARCH_TX; *ty = 4 * 48; *halo = TH; *nt = 256; return true;   // rows by size
#define X(i, TX_, TY_, NT_) \
    case i: *tx = TX_; *ty = TY_; *halo = TH; *nt = NT_; return true;
        HG_THERMAL_VARIANTS(X)
#undef X
        default: return false;
    }
}

hipError_t launch_fused_hydro(int variant, const HydroIO& io, int nx, int ny, uint32_t step,
                              uint32_t terrain, bool rain, int xcd_mode, const KParams& k, hipStream_t s) {
    switch (variant) {
#define X(i, TX_, TY_, HA_, NT_)                                                              \
    case i: {                                                                                 \
        const int xcd = tile_order(xcd_mode, nx, TX_, TY_, 36);                               \
        const unsigned grid = unsigned((nx + TX_ - 1) / TX_) * unsigned((ny + TY_ - 1) / TY_); \
        const bool ex = io.vx || io.tb1;                                                      \
        const int r = rain ? 1 : 0;                                                           \
        if (ex && k.store_nt)                                                                 \
            k_fused_hydro<TX_, TY_, HA_, NT_, true, true><<<grid, NT_, 0, s>>>(io, nx, ny, step, terrain, r, xcd, k); \
        else if (ex)                                                                          \
            k_fused_hydro<TX_, TY_, HA_, NT_, true, false><<<grid, NT_, 0, s>>>(io, nx, ny, step, terrain, r, xcd, k); \
        else if (k.store_nt)                                                                  \
            k_fused_hydro<TX_, TY_, HA_, NT_, false, true><<<grid, NT_, 0, s>>>(io, nx, ny, step, terrain, r, xcd, k); \
        else                                                                                  \
            k_fused_hydro<TX_, TY_, HA_, NT_, false, false><<<grid, NT_, 0, s>>>(io, nx, ny, step, terrain, r, xcd, k); \
        break;                                                                                \
    }
        HG_HYDRO_VARIANTS(X)
#undef X
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

//                        TX  TY   NT
#define HG_STEP_TILES(X)  \
    X(0, 32,  8, 768)     \
    X(1, 32, 16, 512)

// The k_step_tile variant of a map of `cells` cells that was not tuned; -1: the
// two kernels (figures at k_step_tile).
int default_step_tile(size_t cells) { return cells <= 288 * 288 ? 0 : cells <= 648 * 648 ? 1 : -1; }

int step_tile_count() {
#define X(i, tx, ty, nt) +1
    return 0 HG_STEP_TILES(X);
#undef X
}

bool step_tile_info(int v, int* tx, int* ty, int* nt) {
    switch (v) {
#define X(i, TX_, TY_, NT_) \
    case i: *tx = TX_; *ty = TY_; *nt = NT_; return true;
        HG_STEP_TILES(X)
#undef X
        default: return false;
    }
}

hipError_t launch_step_tile(int variant, const HydroIO& io, const ThermIO& tio, int nx, int ny, uint32_t step,
                            uint32_t terrain, bool rain, bool thermal, bool smooth, int xcd_mode, const KParams& k,
                            hipStream_t s) {
    switch (variant) {
#define X(i, TX_, TY_, NT_)                                                                       \
    case i: {                                                                                     \
        const unsigned grid = unsigned((nx + TX_ - 1) / TX_) * unsigned((ny + TY_ - 1) / TY_);    \
        const int xcd = tile_order(xcd_mode, nx, TX_, TY_, 36);                                   \
        const int r = rain ? 1 : 0, th = thermal ? 1 : 0, sm = smooth ? 1 : 0;                    \
        if (io.tb1)                                                                               \
            k_step_tile<TX_, TY_, NT_, true><<<grid, NT_, 0, s>>>(io, tio, nx, ny, step, terrain, r, th, sm, xcd, k);  \
        else                                                                                      \
            k_step_tile<TX_, TY_, NT_, false><<<grid, NT_, 0, s>>>(io, tio, nx, ny, step, terrain, r, th, sm, xcd, k); \
        break;                                                                                    \
    }
        HG_STEP_TILES(X)
#undef X
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_batch_hydro(int variant, const BatchTerrain* terr, const uint32_t* tiles, int ntiles,
                              int grid, uint32_t cur, const uint32_t* step_ptr, uint32_t step_off,
                              bool rain, bool nts, hipStream_t s) {
    switch (variant) {
#define X(i, TX_, TY_, HA_, NT_)                                                                   \
    case i:                                                                                        \
        if (nts)                                                                                   \
            k_batch_hydro<TX_, TY_, HA_, NT_, true><<<grid, NT_, 0, s>>>(terr, tiles, ntiles, cur, step_ptr, \
                                                                      step_off, rain ? 1 : 0);    \
        else                                                                                       \
            k_batch_hydro<TX_, TY_, HA_, NT_, false><<<grid, NT_, 0, s>>>(terr, tiles, ntiles, cur, step_ptr, \
                                                                       step_off, rain ? 1 : 0);   \
        break;
        HG_HYDRO_VARIANTS(X)
#undef X
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_batch_thermal(int variant, int tile_rows, const BatchTerrain* terr, const uint32_t* tiles,
                                int ntiles, int grid, uint32_t cur, bool thermal, bool smooth, bool nts,
                                hipStream_t s) {
    if (variant == MARCH_VARIANT) {
        const int th = thermal ? 1 : 0, sm = smooth ? 1 : 0;
        if (nts)
            k_batch_march<true><<<grid, 256, 0, s>>>(terr, tiles, ntiles, cur, tile_rows / 4, th, sm);
        else
            k_batch_march<false><<<grid, 256, 0, s>>>(terr, tiles, ntiles, cur, tile_rows / 4, th, sm);
        return hipGetLastError();
    }
    switch (variant) {
#define X(i, TX_, TY_, NT_)                                                                   \
    case i:                                                                                   \
        if (nts)                                                                              \
            k_batch_thermal<TX_, TY_, NT_, true><<<grid, NT_, 0, s>>>(terr, tiles, ntiles, cur, \
                                                                   thermal ? 1 : 0, smooth ? 1 : 0); \
        else                                                                                  \
            k_batch_thermal<TX_, TY_, NT_, false><<<grid, NT_, 0, s>>>(terr, tiles, ntiles, cur, \
                                                                    thermal ? 1 : 0, smooth ? 1 : 0); \
        break;
        HG_THERMAL_VARIANTS(X)
#undef X
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

__global__ void k_step_advance(uint32_t* step_ptr, uint32_t n) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *step_ptr += n;
}

hipError_t launch_step_advance(uint32_t* step_ptr, uint32_t n, hipStream_t s) {
    k_step_advance<<<1, 64, 0, s>>>(step_ptr, n);
    return hipGetLastError();
}

int batch_hydro_blocks_per_cu(int variant) {
    int nb = 0;
    switch (variant) {
#define X(i, TX_, TY_, HA_, NT_)                                                                  \
    case i:                                                                                       \
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_batch_hydro<TX_, TY_, HA_, NT_, true>, \
                                                         NT_, 0) != hipSuccess)                  \
            nb = 1;                                                                               \
        break;
        HG_HYDRO_VARIANTS(X)
#undef X
        default: nb = 1;
    }
    return nb > 0 ? nb : 1;
}

int batch_thermal_blocks_per_cu(int variant) {
    int nb = 0;
    switch (variant) {
        case MARCH_VARIANT: return 3;
#define X(i, TX_, TY_, NT_)                                                                   \
    case i:                                                                                   \
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_batch_thermal<TX_, TY_, NT_, true>, \
                                                         NT_, 0) != hipSuccess)              \
            nb = 1;                                                                           \
        break;
        HG_THERMAL_VARIANTS(X)
#undef X
        default: nb = 1;
    }
    return nb > 0 ? nb : 1;
}

hipError_t launch_fused_thermal(int variant, const ThermIO& io, int nx, int ny, bool thermal,
                                bool smooth, int xcd_mode, const KParams& k, hipStream_t s) {
    if (variant == MARCH_VARIANT) {
        const int rows = march_rows(nx, ny);
        const unsigned grid = unsigned((nx + MARCH_TX - 1) / MARCH_TX) * unsigned((ny + 4 * rows - 1) / (4 * rows));
        const int th = thermal ? 1 : 0, sm = smooth ? 1 : 0, xcd = tile_order(xcd_mode, nx, MARCH_TX, 4 * rows, 8);
        if (io.tr5 && k.store_nt)
            k_march_thermal<true, true><<<grid, 256, 0, s>>>(io, nx, ny, rows, th, sm, xcd, k);
        else if (io.tr5)
            k_march_thermal<true, false><<<grid, 256, 0, s>>>(io, nx, ny, rows, th, sm, xcd, k);
        else if (k.store_nt)
            k_march_thermal<false, true><<<grid, 256, 0, s>>>(io, nx, ny, rows, th, sm, xcd, k);
        else
            k_march_thermal<false, false><<<grid, 256, 0, s>>>(io, nx, ny, rows, th, sm, xcd, k);
        return hipGetLastError();
    }
    switch (variant) {
#define X(i, TX_, TY_, NT_)                                                                  \
    case i: {                                                                                \
        const int xcd = tile_order(xcd_mode, nx, TX_, TY_, 8);                               \
        const unsigned grid = unsigned((nx + TX_ - 1) / TX_) * unsigned((ny + TY_ - 1) / TY_); \
        const int th = thermal ? 1 : 0, sm = smooth ? 1 : 0;                                 \
        if (io.tr5 && k.store_nt)                                                            \
            k_fused_thermal<TX_, TY_, NT_, true, true><<<grid, NT_, 0, s>>>(io, nx, ny, th, sm, xcd, k); \
        else if (io.tr5)                                                                     \
            k_fused_thermal<TX_, TY_, NT_, true, false><<<grid, NT_, 0, s>>>(io, nx, ny, th, sm, xcd, k); \
        else if (k.store_nt)                                                                 \
            k_fused_thermal<TX_, TY_, NT_, false, true><<<grid, NT_, 0, s>>>(io, nx, ny, th, sm, xcd, k); \
        else                                                                                 \
            k_fused_thermal<TX_, TY_, NT_, false, false><<<grid, NT_, 0, s>>>(io, nx, ny, th, sm, xcd, k); \
        break;                                                                               \
    }
        HG_THERMAL_VARIANTS(X)
#undef X
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace hgk
