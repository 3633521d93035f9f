// hg_particle.hip — droplet (particle) erosion.
//
// A group of 8 lanes per droplet; the droplets of an iteration run concurrently
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

namespace hgk {

namespace {

__device__ __forceinline__ void atomic_addf(float* p, float v) { unsafeAtomicAdd(p, v); }

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
// corners of a deposit, one cell in kGroup of the erosion brush.  A brush row
// or a stencil row is then one request of neighbouring lanes instead of one
// per cell, and a brush costs one round trip per layer instead of one per cell.
//
// With a thread per droplet a step was a chain of up to 2 x 25 dependent
// returning atomics (radius 3), each a request of its own.  2048^2 with 2^20
// droplets of 64 steps: 61.2 -> 23.6 ms per iteration; 512^2 with 20000 of 30
// steps: 1.20 -> 0.41 ms.  What bounds it now: the atomics, 474 million
// requests per iteration at 2048^2, all of which the L2s pass on to memory
// (TCC_EA0_ATOMIC = TCC_ATOMIC), 20 per ns.  Running the droplets of one part
// of the map together (sorted by 0.5 to 4 MB regions, with or without each XCD
// keeping to its own) halves the lines fetched and is slower, 31 to 73 ms:
// requests to the same lines then wait for each other.
constexpr int kGroup = 8;
constexpr int kBrushSlots = 32;                  // brush cells in flight together
constexpr int kPerLane = kBrushSlots / kGroup;
constexpr int kGotPitch = kBrushSlots + 4;       // 16-byte rows; the 8 groups of a wave start in different banks
static_assert(kGroup == 8, "the lane exchanges of stencil_heights are written for 8 lanes");

template <int CTRL, int BANKS>
__device__ __forceinline__ float dpp(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, 0xf, BANKS, false));
}

// Heights (rock + dirt) at the corners (0,0), (1,0), (0,1), (1,1) of cell c:
// lane g of the group loads corner g & 3 of layer g >> 2, adds the other
// layer's value from the lane 4 away and every lane takes the four sums.
__device__ __forceinline__ void stencil_heights(const float* R, const float* D, size_t c, int n, int g, float& h00,
                                                float& h10, float& h01, float& h11) {
    const float* layer = (g & 4) ? D : R;
    const float v = ld(layer + (c + size_t(g & 1) + ((g & 2) ? size_t(n) : size_t(0))));
    float o = dpp<0x104, 0x5>(v, v);             // row_shl:4 into lanes 0-3 and 8-11 of each 16
    o = dpp<0x114, 0xa>(o, v);                   // row_shr:4 into lanes 4-7 and 12-15
    const float h = v + o;
    h00 = dpp<0x00, 0xf>(h, h);                  // quad_perm broadcasts
    h10 = dpp<0x55, 0xf>(h, h);
    h01 = dpp<0xaa, 0xf>(h, h);
    h11 = dpp<0xff, 0xf>(h, h);
}

// Bilinear deposit of `amount` into dirt around (px, py): lane g < 4 of the
// group adds corner g's share.
__device__ __forceinline__ void deposit(float* D, int n, int g, float px, float py, float amount) {
    const int x = cell_of(px, n), y = cell_of(py, n);
    const float u = px - float(x), v = py - float(y);
    const float share = amount * ((g & 1) ? u : 1.0f - u) * ((g & 2) ? v : 1.0f - v);
    if (g < 4) atomic_addf(D + (size_t(y) * n + x + size_t(g & 1) + ((g & 2) ? size_t(n) : size_t(0))), share);
}

// Taking material.  Removes up to want[i] from p[idx[i]] for a lane's cells,
// never more than a cell holds, and returns in got[i] what was removed.  The
// amount `seen`, a relaxed load's value, says is there is subtracted with a
// returning atomic add; if other droplets took from the cell in between, the
// height it replaced is smaller, and the part that was not there is added
// back.  Each take is then at most max(0, what the cell held at its atomic
// add, less the give-backs still outstanding), so the takes of all droplets
// from one cell never exceed what it held and it never ends below 0 in exact
// arithmetic; in FP32 the subtraction and the give-back round, which can
// leave a residue of a few ulp of the amounts involved below 0.  All of a
// lane's atomics are issued before the first result is looked at.
__device__ __forceinline__ void take(float* p, const size_t (&idx)[kPerLane], const float (&seen)[kPerLane],
                                     const float (&want)[kPerLane], float (&got)[kPerLane]) {
    float est[kPerLane], old[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        est[i] = fminf(fmaxf(seen[i], 0.0f), want[i]);
        old[i] = 0.0f;
        if (est[i] > 0.0f) old[i] = atomicAdd(p + idx[i], -est[i]);
    }
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        got[i] = est[i] > 0.0f ? fminf(fmaxf(old[i], 0.0f), est[i]) : 0.0f;
        if (got[i] < est[i]) atomic_addf(p + idx[i], est[i] - got[i]);
    }
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
// by tile: 48.8 ms per iteration, spread 19.2 ms).
//
// PARTIALS = false: the workgroup's exported mass and droplet steps are added
// atomically to *exported_out and *steps_out.  PARTIALS = true: they are
// written to partials[blockIdx.x], for k_droplet_totals to sum in a fixed
// order.
template <bool PARTIALS>
__global__ __launch_bounds__(kDropThreads) void k_droplets(float* __restrict__ R, float* __restrict__ D, int n,
                                                           DropletParams p, Brush brush, uint32_t iteration,
                                                           uint32_t rounds, uint32_t spread,
                                                           const uint32_t* __restrict__ order,
                                                           double* exported_out, unsigned long long* steps_out,
                                                           DropletPartial* partials) {
    __shared__ double s_exp[kDropletsPerBlock];
    __shared__ unsigned s_steps[kDropletsPerBlock];
    __shared__ float s_w[HG_BRUSH_MAX];
    __shared__ int s_dxy[HG_BRUSH_MAX];                            // dx in the low half, dy in the high half
    __shared__ __align__(16) float s_got[kDropletsPerBlock][kGotPitch];   // what a group's brush cells gave
    const int g = int(threadIdx.x) & (kGroup - 1), group = int(threadIdx.x) / kGroup;
    if (threadIdx.x < HG_BRUSH_MAX) {
        const int t = int(threadIdx.x);
        s_w[t] = brush.w[t];
        s_dxy[t] = (int(brush.dx[t]) & 0xffff) | (int(brush.dy[t]) << 16);
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
        if (end_sed != 0.0f) deposit(D, n, g, end_px, end_py, end_sed);   // the round before
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
            stencil_heights(R, D, size_t(cy) * n + cx, n, g, h00, h10, h01, h11);
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
            if (len > 0.0f) {
                dx = dx / len;
                dy = dy / len;
            }
            const float ox = px, oy = py;
            if (dx == 0.0f && dy == 0.0f) {       // not moving: drop the load here
                deposit(D, n, g, px, py, sed);
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
            stencil_heights(R, D, size_t(ny2) * n + nx2, n, g, k00, k10, k01, k11);
            const float hn = k00 * (1.0f - u2) * (1.0f - v2) + k10 * u2 * (1.0f - v2) + k01 * (1.0f - u2) * v2 +
                             k11 * u2 * v2;
            const float dh = hn - h;
            const float cap = fmaxf(-dh, p.min_slope) * speed * water * p.capacity;
            if (sed > cap || dh > 0.0f) {
                const float amount = dh > 0.0f ? fminf(dh, sed) : (sed - cap) * p.deposition;
                sed -= amount;
                deposit(D, n, g, ox, oy, amount);
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
                for (int base = 0; base < brush.count; base += kBrushSlots) {
                    size_t idx[kPerLane];
                    float want[kPerLane], seen_d[kPerLane], seen_r[kPerLane], td[kPerLane], tr[kPerLane];
#pragma unroll
                    for (int i = 0; i < kPerLane; ++i) {
                        const int t = base + i * kGroup + g;
                        idx[i] = 0;
                        want[i] = seen_d[i] = seen_r[i] = 0.0f;
                        if (t < brush.count) {
                            const int dxy = s_dxy[t];
                            const int x = cx + int(int16_t(dxy & 0xffff)), y = cy + (dxy >> 16);
                            if (interior || (x >= 0 && y >= 0 && x < n && y < n)) {
                                idx[i] = size_t(y) * n + x;
                                want[i] = scale * s_w[t];
                                seen_d[i] = ld(D + idx[i]);
                                seen_r[i] = ld(R + idx[i]);
                            }
                        }
                    }
                    take(D, idx, seen_d, want, td);
#pragma unroll
                    for (int i = 0; i < kPerLane; ++i) want[i] = want[i] - td[i];
                    take(R, idx, seen_r, want, tr);
                    // sed += td + tr, cell by cell in the brush's order (cells
                    // that gave nothing add 0): the group passes its cells'
                    // amounts round through LDS.  One wave reads and writes a
                    // group's row, and a wave's LDS accesses keep their order.
#pragma unroll
                    for (int i = 0; i < kPerLane; ++i) s_got[group][i * kGroup + g] = td[i] + tr[i];
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    const int m = (min(kBrushSlots, brush.count - base) + 3) / 4;
                    for (int q = 0; q < m; ++q) {
                        const float4 a = *reinterpret_cast<const float4*>(&s_got[group][4 * q]);
                        sed += a.x;
                        sed += a.y;
                        sed += a.z;
                        sed += a.w;
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
    if (end_sed != 0.0f) deposit(D, n, g, end_px, end_py, end_sed);
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

hipError_t launch_droplets(float* rock, float* dirt, int n, const DropletParams& p, const Brush& brush,
                           uint32_t iteration, const uint32_t* order, double* exported,
                           unsigned long long* steps, hipStream_t s) {
    if (p.count == 0) return hipSuccess;
    const uint32_t blocks = (p.count + kDropletsPerBlock - 1) / kDropletsPerBlock;
    k_droplets<false><<<blocks, kDropThreads, 0, s>>>(rock, dirt, n, p, brush, iteration, 1,
                                                      order ? chunk_spread(p.count) : 1u, order, exported, steps, nullptr);
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
// HG_DROPLET_PARTIALS_MAX (1 up to 2^19 droplets, 8 at 2^22).
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
    k_droplets<true><<<droplet_partial_blocks(p.count), kDropThreads, 0, s>>>(
        rock, dirt, n, p, brush, iteration, partial_rounds(p.count), 1u, nullptr, nullptr, nullptr, partials);
    return hipGetLastError();
}

hipError_t launch_droplet_totals(const DropletPartial* partials, uint32_t nblocks, double* exported,
                                 uint64_t* steps, bool accumulate, hipStream_t s) {
    k_droplet_totals<<<1, 256, 0, s>>>(partials, nblocks, exported, steps, accumulate ? 1 : 0);
    return hipGetLastError();
}

}  // namespace hgk
