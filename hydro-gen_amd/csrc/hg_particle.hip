// hg_particle.hip — droplet (particle) erosion.
//
// A group of 16 lanes per droplet; the droplets of an iteration run concurrently
// and change the height planes with float atomic adds (global_atomic_add_f32),
// so a droplet sees the others' changes in whatever order the memory system
// applies them.  Height reads are relaxed atomic loads.  Erosion takes from a
// cell with a returning atomic add and gives back what was not there (take()),
// so concurrent droplets never drive a layer below 0.  Mass bookkeeping: every
// amount taken from the map is added to the droplet's load and every amount
// deposited is subtracted from it; sediment carried over the map edge is
// summed in `exported`, so sum(rock + dirt) + exported is conserved up to
// FP32 rounding.
//
// Model (Beyer-style droplets; the reference's particle mode,
// glsl/particle.glsl:64-136 and glsl/particle_erosion.glsl:22-128, is a
// different model): see hg_droplet_settings in include/hg.h.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "hg_kernels.hpp"
#include "hg_stencil.hpp"

namespace hgk {

namespace {

// The height planes are global memory, which the compiler no longer sees once a
// pointer has been through an array or a select.
using global_float = __attribute__((address_space(1))) float;
__device__ __forceinline__ float fetch_addf(float* p, float v) {
    return __builtin_amdgcn_global_atomic_fadd_f32((global_float*)p, v);
}
__device__ __forceinline__ void atomic_addf(float* p, float v) { (void)fetch_addf(p, v); }

// Height reads are relaxed device-scope atomic loads: they are served by L2,
// where the atomic adds land, and never by a stale line of the non-coherent
// per-CU vector cache (a droplet must see its own earlier erosion).
__device__ __forceinline__ float ld(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float height(const float* R, const float* D, size_t i) { return ld(R + i) + ld(D + i); }

// Cell of a position inside [0, n-1]^2; n-1 itself maps to cell n-2 (with
// fraction 1) so the 2x2 stencil stays in the grid.
__device__ __forceinline__ int cell_of(float p, int n) { return min(int(p), n - 2); }

// ---- a droplet is run by a group of kGroup consecutive lanes -----------------
//
// All lanes of a group hold the same droplet (the same registers, bit for
// bit, so they branch alike); what differs is which cell a lane touches: one
// of the 8 heights of a 2x2 stencil (4 corners x 2 layers), one of the 4
// corners of a deposit, one layer of one of 8 cells of a row of the erosion
// brush.  What neighbouring lanes touch in one cache line is one request.
//
// Requests are what bounds it: the L2s pass every atomic on to memory, which
// takes about 20 a ns (TCC_EA0_ATOMIC = TCC_ATOMIC = 474 million per iteration
// of 2^20 droplets at 2048^2 when 8 lanes ran a droplet on the two planes).
// So hg_step_particle runs on a map that holds rock and dirt of a cell next to
// each other (HeightMap, PAIRED): a brush row is one request for both layers,
// a stencil row too.  ms per iteration, 2^20 droplets of 64 steps at 2048^2 /
// 20000 of 30 steps at 512^2 (with the thermal pass):
//   a thread per droplet                            61.2 / 1.21
//   8 lanes, planes                                 23.7 / 0.37
//   16 lanes, paired                                20.5 / 0.25
// (hg_droplets_noalloc has no room for pairs: 16 lanes, planes, 26.8.)  367
// million atomic requests are left, a 40-byte row being 1.5 requests of 64
// bytes on average, and the arithmetic, at 4 droplets per wave, half the time.
// More in flight does not help: half the waves per CU run as fast, sending a
// step's dirt and rock atomics and the next step's loads together, or loading
// the brush beside the stencil, is slower (29 and 30 ms with planes).  Nor does
// running the droplets of one part of the map together (sorted by 0.5 to 4 MB
// regions, with or without each XCD keeping to its own): that halves the lines
// fetched, but the requests to a line then wait for each other, 31 to 73 ms.
constexpr int kGroup = 16;
constexpr int kRowCells = kGroup / 2;            // cells of a brush row in flight together
constexpr int kRows = 5;                         // brush rows in flight together (all of radius 3)
constexpr int kGotPitch = kRows * kRowCells + 4; // 16-byte rows; the groups of a wave start in different banks
constexpr int kSlots = 11 * 16;                  // brush rows padded to whole row chunks: radius 6 has 11 rows of 2
static_assert(kGroup == 16, "the lane exchanges are written for the 16 lanes of a DPP row");

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
struct GroupLanes {
    static __device__ __forceinline__ float other_layer(float v) { return dpp<0xb1>(v); }   // quad_perm 1, 0, 3, 2
    template <int L>
    static __device__ __forceinline__ float lane(float v) { return dpp<0x150 + L>(v); }     // row_newbcast:L
};
__device__ __forceinline__ float other_layer(float v) { return GroupLanes::other_layer(v); }

// The heights.  Planes: rock in a, dirt in b, row by row.  PAIRED: rows of
// (rock, dirt) pairs, those below `half` in a and the others in b, so that two
// separate planes of n x n floats hold them.
template <bool PAIRED>
struct HeightMap {
    float *a, *b;
    int n, half;
    __device__ __forceinline__ float* at(int layer, int x, int y) const {
        // 32-bit cell numbers: n <= 32768
        if constexpr (PAIRED) {
            const bool up = y >= half;
            const uint32_t i = uint32_t(up ? y - half : y) * uint32_t(2 * n) + uint32_t(2 * x + layer);
            return (up ? b : a) + size_t(i);
        } else {
            return (layer ? b : a) + size_t(uint32_t(y) * uint32_t(n) + uint32_t(x));
        }
    }
};

// Heights (rock + dirt) at the corners (0,0), (1,0), (0,1), (1,1) of cell (x,
// y): lane g of the group loads layer g & 1 of corner (g >> 1) & 1 of row
// (g >> 2) & 1, and every lane takes the four sums of lanes 0-7's loads.
template <class Map>
__device__ __forceinline__ void stencil_heights(const Map& m, int x, int y, int g, float& h00, float& h10, float& h01,
                                                float& h11) {
    const float v = ld(m.at(g & 1, x + ((g >> 1) & 1), y + ((g >> 2) & 1)));
    corner_heights<GroupLanes>(v, h00, h10, h01, h11);
}

// Bilinear deposit of `amount` into dirt around (px, py): the four dirt lanes
// of a stencil add a corner's share each.
template <class Map>
__device__ __forceinline__ void deposit(const Map& m, int g, float px, float py, float amount) {
    const int x = cell_of(px, m.n), y = cell_of(py, m.n);
    const float u = px - float(x), v = py - float(y);
    const bool right = (g & 2) != 0, top = (g & 4) != 0;
    const float share = amount * (right ? u : 1.0f - u) * (top ? v : 1.0f - v);
    if (g < 8 && (g & 1)) atomic_addf(m.at(1, x + (right ? 1 : 0), y + (top ? 1 : 0)), share);
}

// Taking material.  Up to `want` is removed from a cell, never more than it
// holds.  What a relaxed load says is there (`seen`) is subtracted with a
// returning atomic add; if other droplets took from the cell in between, the
// height it replaced is smaller, and the part that was not there is added
// back (taken).  Each take is then at most max(0, what the cell held at its
// atomic add, less the give-backs still outstanding), so the takes of all
// droplets from one cell never exceed what it held and it never ends below 0
// in exact arithmetic; in FP32 the subtraction and the give-back round, which
// can leave a residue of a few ulp of the amounts involved below 0.
__device__ __forceinline__ float estimate(float seen, float want) { return fminf(fmaxf(seen, 0.0f), want); }
__device__ __forceinline__ float taken(float* p, float old, float est) {
    // min(max(old, 0), est), spelt with two uses of `old`: with one, the compiler
    // moves the max behind the atomic, where it waits for the result
    const float got = est > 0.0f ? (!(old >= est) ? fmaxf(old, 0.0f) : est) : 0.0f;
    if (got < est) atomic_addf(p, est - got);
    return got;
}

// Start position of droplet `id` in an iteration: uniform over [0, n-1)^2.
__device__ __forceinline__ void droplet_start(uint32_t id, uint32_t iteration, const DropletParams& p, int n,
                                              float& px, float& py) {
    uint32_t o[4];
    philox4x32_10(id, iteration, 0x64726f70u, 0u, p.seed_lo, p.seed_hi, o);
    const float span = float(n - 1);
    px = u24(o[0]) * span;
    py = u24(o[1]) * span;
}

// Droplets of a workgroup: kDropletsPerBlock at a time, `rounds` times.  What
// a droplet still carries at the end of its life is dropped when the
// workgroup's other droplets have ended too: that deposit, up to a whole load
// in 4 cells, is the change a neighbour in another workgroup would feel most,
// and workgroups do not start at quite the same time.  With 256 threads and no
// wait, droplets that should hardly meet (one step each) left the map up to
// 2.0e-5 apart from run to run; so, up to 4e-6.
constexpr int kDropThreads = 1024;
constexpr int kDropletsPerBlock = kDropThreads / kGroup;
constexpr uint32_t kChunk = 64 / kGroup;         // droplets of a wave

// spread (coprime to the number of chunks): wave w runs chunk w * spread mod
// that number.  1 without an order; with one, neighbouring chunks of the order
// lie side by side on the map and are kept apart in time: run next to each
// other, their requests queue for the same lines (2048^2, 2^20 droplets sorted
// by tile, 8 lanes, planes: 48.8 ms per iteration, spread 19.2 ms).
//
// PARTIALS = false: the workgroup's exported mass and droplet steps are added
// atomically to *exported_out and *steps_out.  PARTIALS = true: they are
// written to partials[blockIdx.x], for k_droplet_totals to sum in a fixed
// order.
// ROWS: kRows, or 1 for the brush of radius 1, which is one cell: no loop over
// rows, and what it gave is passed on by a lane instead of through LDS.  us an
// iteration of 30 steps at 2048^2 on the planes, a thread per droplet / ROWS = 1:
// 1 droplet 55/52, 64 109/89, 65536 387/358, 2^20 6160/5345 (with kRows the last
// two take 421 and 6600).
template <bool PARTIALS, bool PAIRED, int ROWS>
__global__ __launch_bounds__(kDropThreads) void k_droplets(HeightMap<PAIRED> map, DropletParams p, Brush brush, uint32_t iteration,
                                                           uint32_t rounds, uint32_t spread,
                                                           const uint32_t* __restrict__ order,
                                                           double* exported_out, unsigned long long* steps_out,
                                                           DropletPartial* partials) {
    __shared__ double s_exp[kDropletsPerBlock];
    __shared__ unsigned s_steps[kDropletsPerBlock];
    __shared__ float s_w[kSlots];        // the brush's weights, its rows padded to whole chunks of kRowCells
    __shared__ __align__(16) float s_got[ROWS > 1 ? kDropletsPerBlock : 1][kGotPitch];   // what a group's brush cells gave
    const int g = int(threadIdx.x) & (kGroup - 1), group = int(threadIdx.x) / kGroup;
    const int n = map.n;
    const int reach = brush.r - 1, width = 2 * reach + 1;         // cells closer than r: rows and columns -reach .. reach
    const int twice = width > kRowCells ? 1 : 0;                  // a row is one chunk, or two (radius 5 and 6)
    const int row_slots = kRowCells << twice, chunks_of_rows = width << twice;
    static_assert(2 * kRowCells >= 11, "radius 6: rows of 11 cells");
    for (int t = int(threadIdx.x); t < kSlots; t += kDropThreads) s_w[t] = 0.0f;
    __syncthreads();
    if (int(threadIdx.x) < brush.count) {
        const int t = int(threadIdx.x);
        s_w[(brush.dy[t] + reach) * row_slots + brush.dx[t] + reach] = brush.w[t];
    }
    __syncthreads();
    double exported = 0.0;
    unsigned steps = 0;
    float end_px = 0.0f, end_py = 0.0f, end_sed = 0.0f;   // load left at the end of a life, and where
    for (uint32_t round = 0; round < rounds; ++round) {
        // a wave runs one chunk of consecutive slots
        const uint32_t w = (blockIdx.x * rounds + round) * (kDropThreads / 64) + threadIdx.x / 64;
        const uint32_t chunks = (p.count + kChunk - 1) / kChunk;
        if (w >= chunks) break;
        const uint32_t slot = uint32_t(uint64_t(w) * spread % chunks) * kChunk + uint32_t(group) % kChunk;
        if (slot >= p.count) continue;
        if (end_sed != 0.0f) deposit(map, g, end_px, end_py, end_sed);   // the round before
        const uint32_t id = order ? order[slot] : slot;
        const float span = float(n - 1);
        float px, py;
        droplet_start(id, iteration, p, n, px, py);
        float dx = 0.0f, dy = 0.0f, speed = p.init_speed, water = p.init_water, sed = 0.0f;
        bool alive = true;
        for (uint32_t life = 0; life < p.max_lifetime; ++life) {
            ++steps;
            const int cx = cell_of(px, n), cy = cell_of(py, n);
            const float u = px - float(cx), v = py - float(cy);
            float h00, h10, h01, h11;
            stencil_heights(map, cx, cy, g, h00, h10, h01, h11);
            const float gx = (h10 - h00) * (1.0f - v) + (h11 - h01) * v;
            const float gy = (h01 - h00) * (1.0f - u) + (h11 - h10) * u;
            const float h = h00 * (1.0f - u) * (1.0f - v) + h10 * u * (1.0f - v) + h01 * (1.0f - u) * v +
                            h11 * u * v;
            dx = dx * p.inertia - gx * (1.0f - p.inertia);
            dy = dy * p.inertia - gy * (1.0f - p.inertia);
            // correctly rounded sqrt and divide (as on the host): a droplet's
            // path is sensitive to the last bit of its direction.  Plain `/`
            // and sqrtf lower to the IEEE sequences; HIP's __fsqrt_rn lowers to
            // the native 3-ulp sqrt.
            const float len = sqrtf(dx * dx + dy * dy);
            if (len > 0.0f) {                     // one division: even lanes divide dx, odd lanes dy
                const float q = ((g & 1) ? dy : dx) / len, beside = other_layer(q);
                dx = (g & 1) ? beside : q;
                dy = (g & 1) ? q : beside;
            }
            const float ox = px, oy = py;
            if (dx == 0.0f && dy == 0.0f) {       // not moving: drop the load here
                deposit(map, g, px, py, sed);
                sed = 0.0f;
                alive = false;
                break;
            }
            px += dx;
            py += dy;
            if (!(px >= 0.0f && py >= 0.0f && px < span && py < span)) {   // over the edge (or NaN)
                exported += double(sed);
                sed = 0.0f;
                alive = false;
                break;
            }
            const int nx2 = cell_of(px, n), ny2 = cell_of(py, n);
            const float u2 = px - float(nx2), v2 = py - float(ny2);
            float k00, k10, k01, k11;
            stencil_heights(map, nx2, ny2, g, k00, k10, k01, k11);
            const float hn = k00 * (1.0f - u2) * (1.0f - v2) + k10 * u2 * (1.0f - v2) + k01 * (1.0f - u2) * v2 +
                             k11 * u2 * v2;
            const float dh = hn - h;
            const float cap = fmaxf(-dh, p.min_slope) * speed * water * p.capacity;
            if (sed > cap || dh > 0.0f) {
                const float amount = dh > 0.0f ? fminf(dh, sed) : (sed - cap) * p.deposition;
                sed -= amount;
                deposit(map, g, ox, oy, amount);
            } else {
                const float amount = fminf((cap - sed) * p.erosion, -dh);
                const bool interior = cx >= brush.r && cy >= brush.r && cx < n - brush.r && cy < n - brush.r;
                float wsum = 1.0f;
                if (!interior) {
                    wsum = 0.0f;
                    for (int t = 0; t < brush.count; ++t) {
                        const int x = cx + brush.dx[t], y = cy + brush.dy[t];
                        if (x >= 0 && y >= 0 && x < n && y < n) wsum += brush.w[t];
                    }
                }
                const float scale = interior ? amount : amount / wsum;
                for (int base = 0; base < (ROWS > 1 ? chunks_of_rows : 1); base += ROWS) {
                    // lane g: layer g & 1 of cell g >> 1 of each row chunk.  The
                    // dirt goes first, the rock gives the rest, both sent
                    // together as if all the dirt seen will be got.
                    float *at[ROWS], want[ROWS], seen[ROWS], est[ROWS], dirt[ROWS], old[ROWS];
#pragma unroll
                    for (int i = 0; i < ROWS; ++i) {
                        at[i] = map.a;
                        want[i] = seen[i] = 0.0f;
                        if (ROWS == 1 || base + i < chunks_of_rows) {
                            const int row = (base + i) >> twice, column = ((base + i) & twice) * kRowCells;
                            const int x = cx - reach + column + (g >> 1), y = cy - reach + row;
                            const float w = s_w[(base + i) * kRowCells + (g >> 1)];
                            if (w > 0.0f && (interior || (x >= 0 && y >= 0 && x < n && y < n))) {
                                at[i] = map.at(g & 1, x, y);
                                want[i] = scale * w;
                                seen[i] = ld(at[i]);
                            }
                        }
                    }
#pragma unroll
                    for (int i = 0; i < ROWS; ++i) {
                        const float beside = other_layer(seen[i]);
                        dirt[i] = estimate((g & 1) ? seen[i] : beside, want[i]);
                        est[i] = (g & 1) ? dirt[i] : estimate(seen[i], want[i] - dirt[i]);
                    }
#pragma unroll
                    for (int i = 0; i < ROWS; ++i) {
                        // any value where nothing is taken (taken() does not look
                        // at it): a 0 would have to be merged with the atomic's
                        // result, which waits for it before the next is sent
                        old[i] = __builtin_nondeterministic_value(old[i]);
                        if (est[i] > 0.0f) old[i] = fetch_addf(at[i], -est[i]);
                    }
                    if constexpr (ROWS == 1) {
                        float mine = taken(at[0], old[0], est[0]);
                        const float beside = other_layer(mine);
                        if (g == 0 && beside < dirt[0]) {    // as below
                            const float more = estimate(ld(at[0]), dirt[0] - beside);
                            if (more > 0.0f) mine += taken(at[0], fetch_addf(at[0], -more), more);
                        }
                        sed += GroupLanes::lane<0>(beside + mine);
                        continue;
                    }
                    // sed += dirt + rock, cell by cell in the brush's order
                    // (slots that gave nothing add 0): the group passes its
                    // cells' amounts round through LDS.  One wave reads and
                    // writes a group's row, and a wave's LDS accesses keep their
                    // order.
#pragma unroll
                    for (int i = 0; i < ROWS; ++i) {
                        const float mine = taken(at[i], old[i], est[i]);
                        const float beside = other_layer(mine);
                        if ((g & 1) == 0) {
                            float rock = mine;
                            if (beside < dirt[i]) {      // another droplet had the dirt: the rest from the rock after all
                                const float more = estimate(ld(at[i]), dirt[i] - beside);
                                if (more > 0.0f) rock += taken(at[i], fetch_addf(at[i], -more), more);
                            }
                            s_got[group][i * kRowCells + (g >> 1)] = beside + rock;
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    const int m = min(ROWS, chunks_of_rows - base) * (kRowCells / 4);
                    for (int q = 0; q < m; ++q) {
                        const float4 v4 = *reinterpret_cast<const float4*>(&s_got[group][4 * q]);
                        sed += v4.x;
                        sed += v4.y;
                        sed += v4.z;
                        sed += v4.w;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
            }
            speed = sqrtf(fmaxf(0.0f, speed * speed - dh * p.gravity));
            water = water * (1.0f - p.evaporation);
        }
        end_px = px;
        end_py = py;
        end_sed = alive ? sed : 0.0f;
    }
    __syncthreads();
    if (end_sed != 0.0f) deposit(map, g, end_px, end_py, end_sed);
    if (g == 0) {
        s_exp[group] = exported;
        s_steps[group] = steps;
    }
    __syncthreads();
    for (int s = kDropletsPerBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            s_exp[threadIdx.x] += s_exp[threadIdx.x + s];
            s_steps[threadIdx.x] += s_steps[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if constexpr (PARTIALS) {
            partials[blockIdx.x].exported = s_exp[0];
            partials[blockIdx.x].steps = s_steps[0];
        } else {
            if (s_exp[0] != 0.0) unsafeAtomicAdd(exported_out, s_exp[0]);
            atomicAdd(steps_out, (unsigned long long)s_steps[0]);
        }
    }
}

// Rock and dirt planes to rows of pairs and back: n * n cells, the first half
// of the rows in `low`, the other in `high`, 4 cells per thread, `quads` per
// half (n is a multiple of 8).
__global__ __launch_bounds__(256) void k_pair_heights(const float* __restrict__ rock, const float* __restrict__ dirt,
                                                      float* __restrict__ low, float* __restrict__ high,
                                                      size_t quads) {
    const size_t q = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (q >= 2 * quads) return;
    const float4 r = reinterpret_cast<const float4*>(rock)[q], d = reinterpret_cast<const float4*>(dirt)[q];
    float4* out = reinterpret_cast<float4*>(q < quads ? low : high) + 2 * (q < quads ? q : q - quads);
    out[0] = make_float4(r.x, d.x, r.y, d.y);
    out[1] = make_float4(r.z, d.z, r.w, d.w);
}
__global__ __launch_bounds__(256) void k_unpair_heights(const float* __restrict__ low, const float* __restrict__ high,
                                                        float* __restrict__ rock, float* __restrict__ dirt,
                                                        size_t quads) {
    const size_t q = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (q >= 2 * quads) return;
    const float4* in = reinterpret_cast<const float4*>(q < quads ? low : high) + 2 * (q < quads ? q : q - quads);
    const float4 a = in[0], b = in[1];
    reinterpret_cast<float4*>(rock)[q] = make_float4(a.x, a.z, b.x, b.z);
    reinterpret_cast<float4*>(dirt)[q] = make_float4(a.y, a.w, b.y, b.w);
}

// ---- droplet ordering (counting sort by start tile) --------------------------

__device__ __forceinline__ uint32_t start_tile(uint32_t id, uint32_t iteration, const DropletParams& p, int n,
                                               int side, int ntx) {
    float px, py;
    droplet_start(id, iteration, p, n, px, py);
    return uint32_t(int(py) / side) * uint32_t(ntx) + uint32_t(int(px) / side);
}

__global__ __launch_bounds__(256) void k_zero_u32(uint32_t* a, uint32_t count) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < count) a[i] = 0u;
}

__global__ __launch_bounds__(256) void k_drop_count(DropletParams p, int n, int side, int ntx, uint32_t iteration,
                                                    uint32_t* tiles) {
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id < p.count) atomicAdd(&tiles[start_tile(id, iteration, p, n, side, ntx)], 1u);
}

// Exclusive prefix sum of tiles[0, count) in place, one workgroup of 1024
// threads: each thread sums a contiguous run, the run totals are scanned in
// LDS, then each run is rewritten as offsets.
__global__ __launch_bounds__(1024) void k_drop_scan(uint32_t* tiles, uint32_t count) {
    __shared__ uint32_t s[1024];
    const uint32_t per = (count + 1023) / 1024;
    const uint32_t b = threadIdx.x * per, e = min(b + per, count);
    uint32_t sum = 0;
    for (uint32_t i = b; i < e; ++i) sum += tiles[i];
    s[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t off = 1; off < 1024; off <<= 1) {          // inclusive Hillis-Steele scan
        const uint32_t v = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = s[threadIdx.x] - sum;                      // exclusive
    for (uint32_t i = b; i < e; ++i) {
        const uint32_t c = tiles[i];
        tiles[i] = run;
        run += c;
    }
}

// Places droplet id at its sorted position (its tile's next free offset).
__global__ __launch_bounds__(256) void k_drop_scatter(DropletParams p, int n, int side, int ntx, uint32_t iteration,
                                                      uint32_t* tiles, uint32_t* order) {
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= p.count) return;
    order[atomicAdd(&tiles[start_tile(id, iteration, p, n, side, ntx)], 1u)] = id;
}

// Sums partials[0, nblocks) in a fixed order (thread t: blocks t, t + 256, ...;
// then a fixed tree) into *exported_out and *steps_out (either may be null),
// replacing them, or adding to them with `accumulate`.
__global__ __launch_bounds__(256) void k_droplet_totals(const DropletPartial* __restrict__ partials,
                                                        uint32_t nblocks, double* exported_out,
                                                        uint64_t* steps_out, int accumulate) {
    __shared__ double s_exp[256];
    __shared__ unsigned long long s_steps[256];
    double e = 0.0;
    unsigned long long st = 0;
    for (uint32_t b = threadIdx.x; b < nblocks; b += 256) {
        e += partials[b].exported;
        st += partials[b].steps;
    }
    s_exp[threadIdx.x] = e;
    s_steps[threadIdx.x] = st;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            s_exp[threadIdx.x] += s_exp[threadIdx.x + h];
            s_steps[threadIdx.x] += s_steps[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (exported_out) *exported_out = (accumulate ? *exported_out : 0.0) + s_exp[0];
        if (steps_out) *steps_out = (accumulate ? *steps_out : 0ull) + uint64_t(s_steps[0]);
    }
}

}  // namespace

Brush make_brush(int r) {
    // weights 1 - dist/r over cells with dist < r, normalised in double and
    // rounded to float once (the oracle builds the same table)
    Brush b{};
    b.r = r;
    double raw[HG_BRUSH_MAX];
    double sum = 0;
    for (int dy = -r; dy <= r; ++dy)
        for (int dx = -r; dx <= r; ++dx) {
            const double d = std::sqrt(double(dx * dx + dy * dy));
            if (d < r && b.count < HG_BRUSH_MAX) {
                b.dx[b.count] = int8_t(dx);
                b.dy[b.count] = int8_t(dy);
                raw[b.count] = 1.0 - d / r;
                sum += raw[b.count];
                ++b.count;
            }
        }
    for (int t = 0; t < b.count; ++t) b.w[t] = float(raw[t] / sum);
    return b;
}

// About 0.618 of the number of chunks, coprime to it.
static uint32_t chunk_spread(uint32_t count) {
    const uint32_t chunks = (count + kChunk - 1) / kChunk;
    uint32_t k = std::max(1u, uint32_t(uint64_t(chunks) * 618034u / 1000000u));
    while (std::gcd(k, chunks) != 1u) ++k;
    return k;
}

hipError_t launch_droplets(float* a, float* b, bool paired, int n, const DropletParams& p, const Brush& brush,
                           uint32_t iteration, const uint32_t* order, double* exported,
                           unsigned long long* steps, hipStream_t s) {
    if (p.count == 0) return hipSuccess;
    const uint32_t blocks = (p.count + kDropletsPerBlock - 1) / kDropletsPerBlock;
    const uint32_t spread = order ? chunk_spread(p.count) : 1u;
    auto launch = [&](auto kernel, auto map) {
        kernel<<<blocks, kDropThreads, 0, s>>>(map, p, brush, iteration, 1, spread, order, exported, steps, nullptr);
    };
    const HeightMap<true> pairs{a, b, n, n / 2};
    const HeightMap<false> planes{a, b, n, 0};
    if (brush.r == 1)
        paired ? launch(k_droplets<false, true, 1>, pairs) : launch(k_droplets<false, false, 1>, planes);
    else
        paired ? launch(k_droplets<false, true, kRows>, pairs) : launch(k_droplets<false, false, kRows>, planes);
    return hipGetLastError();
}

// Pairing and unpairing move 32 B a cell, 5.6 ps (once the planes are beyond the
// caches; 24 us at 2048^2, 380 at 8192^2).  Pairs shorten each step of a
// droplet's life by 1 to 1.5 us of the chain, and save 0.065 ns of atomics for
// each step of each droplet.  us an iteration, paired / on the planes:
//            64 x 20    4096 x 64   65536 x 64   262144 x 20
//   512^2    123/143     390/482    1988/2479     2429/3082
//  2048^2    119/131     380/447    1422/1699     1820/2234
//  8192^2    481/124     733/414    1762/1680     2147/2260
// A brush of one cell gains nothing on the chain, and by its atomics only where a
// cell is visited often (30 steps, on the planes / paired: 65536 at 512^2 504/481,
// 2^20 at 2048^2 5340/5380, 2^20 at 8192^2 5140/5510, 1 at 2048^2 53/72).
bool droplets_pair(int n, const DropletParams& p, int radius, uint32_t iterations) {
    const double lives = double(p.count > 0 ? p.max_lifetime : 0u) * iterations;
    if (radius == 1) return 8.0 * n * n <= lives * p.count;
    return double(n) * n < lives * (262144.0 + 12.0 * p.count);
}

hipError_t launch_pair_heights(const float* rock, const float* dirt, float* low, float* high, int n, hipStream_t s) {
    const size_t quads = size_t(n) * size_t(n) / 8;          // 4 cells each, per half
    k_pair_heights<<<unsigned((2 * quads + 255) / 256), 256, 0, s>>>(rock, dirt, low, high, quads);
    return hipGetLastError();
}

hipError_t launch_unpair_heights(const float* low, const float* high, float* rock, float* dirt, int n, hipStream_t s) {
    const size_t quads = size_t(n) * size_t(n) / 8;
    k_unpair_heights<<<unsigned((2 * quads + 255) / 256), 256, 0, s>>>(low, high, rock, dirt, quads);
    return hipGetLastError();
}

int droplet_tile_side(int n) { return std::max(16, (n + 127) / 128); }

int droplet_tile_count(int n) {
    const int side = droplet_tile_side(n), nt = (n + side - 1) / side;
    return nt * nt;
}

hipError_t launch_droplet_order(int n, const DropletParams& p, uint32_t iteration, uint32_t* tiles,
                                uint32_t* order, hipStream_t s) {
    if (p.count == 0) return hipSuccess;
    const int side = droplet_tile_side(n), ntx = (n + side - 1) / side;
    const uint32_t nt = uint32_t(ntx) * uint32_t(ntx), g = (p.count + 255) / 256;
    k_zero_u32<<<(nt + 255) / 256, 256, 0, s>>>(tiles, nt);
    k_drop_count<<<g, 256, 0, s>>>(p, n, side, ntx, iteration, tiles);
    k_drop_scan<<<1, 1024, 0, s>>>(tiles, nt);
    k_drop_scatter<<<g, 256, 0, s>>>(p, n, side, ntx, iteration, tiles, order);
    return hipGetLastError();
}

// Rounds per workgroup that keep the workgroups of a partials launch within
// HG_DROPLET_PARTIALS_MAX (1 up to 2^20 droplets, 4 at 2^22).
static_assert(kDropletsPerBlock * HG_DROPLET_PARTIALS_MAX == 1u << 20, "droplets of one round");
static uint32_t partial_rounds(uint32_t count) {
    const uint32_t per = uint32_t(kDropletsPerBlock) * HG_DROPLET_PARTIALS_MAX;
    return std::max(1u, (count + per - 1) / per);
}

uint32_t droplet_partial_blocks(uint32_t count) {
    const uint32_t per = uint32_t(kDropletsPerBlock) * partial_rounds(count);
    return (count + per - 1) / per;
}

hipError_t launch_droplets_partials(float* rock, float* dirt, int n, const DropletParams& p, const Brush& brush,
                                    uint32_t iteration, DropletPartial* partials, hipStream_t s) {
    if (p.count == 0) return hipSuccess;
    const HeightMap<false> map{rock, dirt, n, 0};
    auto launch = [&](auto kernel) {
        kernel<<<droplet_partial_blocks(p.count), kDropThreads, 0, s>>>(map, p, brush, iteration,
                                                                        partial_rounds(p.count), 1u, nullptr, nullptr,
                                                                        nullptr, partials);
    };
    brush.r == 1 ? launch(k_droplets<true, false, 1>) : launch(k_droplets<true, false, kRows>);
    return hipGetLastError();
}

hipError_t launch_droplet_totals(const DropletPartial* partials, uint32_t nblocks, double* exported,
                                 uint64_t* steps, bool accumulate, hipStream_t s) {
    k_droplet_totals<<<1, 256, 0, s>>>(partials, nblocks, exported, steps, accumulate ? 1 : 0);
    return hipGetLastError();
}

}  // namespace hgk
