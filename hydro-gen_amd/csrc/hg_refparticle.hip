// hg_refparticle.hip — the reference's own particle mode.
//
// One Erosion::dispatch_particle (src/erosion.cpp:132-156) is four launches:
//  * k_refp_move: one thread per particle, glsl/particle.glsl:64-136 (spawn,
//    terrain normal and momentum sampled bilinearly, velocity and volume
//    update, capacity, kill tests).  The spawn range and the border test
//    use Map_settings_data.hmap_dims, which the reference leaves at
//    (1024, 1024) whatever the map size; here it is the grid's n unless
//    hg_set_ref_particle_dims sets it.  Particles outside the grid read 0
//    and their corner updates are dropped, like imageLoad/imageStore
//    outside an image;
//  * k_refp_erode: 4 lanes per particle, glsl/particle_erosion.glsl:22-128, one
//    for each corner of the particle's quad;
//  * the fused thermal kernel (both thermal layers and the grid smoothing of
//    rock and dirt), as for the grid step;
//  * k_refp_smooth_extra: the particle branch of glsl/smoothing.glsl:76-95
//    (momentum map and water display), per cell.
//
// The shader serialises the corner updates at a pixel with a per-pixel
// spinlock (glsl/particle_erosion.glsl:78-90).  Here every update of a pixel
// is an atomic operation of its own instead: the pure additions (deposits,
// the water display, the momentum accumulation) are float atomic adds, and a
// layer's dissolve, whose clamp at 0 reads the height, is one compare-and-swap
// loop on that layer.  The outcome is that of some serial order of the
// updates, as with the lock, except that a corner's dirt and rock updates are
// not one transaction: another particle can touch the pixel's rock between
// them.  A CAS loop that keeps failing gives up after a fixed number of tries
// and adds without the clamp (counted; the host reads the count).
//
// Arithmetic is FP32 in the shaders' order; division and square root are the
// correctly rounded ones and mix(a, b, t) is a + t (b - a), so that one
// particle on its own reproduces the FP32 oracle bit for bit.  The spawn
// hash's sin is hash_sinf below, whose operations a host compiles alike, so
// spawns reproduce it too.
#include <cmath>

#include "hg_kernels.hpp"

namespace hgk {

namespace {

constexpr int kCasTries = 4096;

__device__ __forceinline__ float fract_(float x) { return x - floorf(x); }

// sin of an FP32 argument for the spawn hash, evaluated in FP64 and rounded
// once: x = k pi/2 + r with pi/2 split into three parts (two of 24
// significant bits, so k * part is exact for |k| < 2^29, i.e. |x| < 8e8), the
// Taylor polynomials of sin r and cos r on |r| <= pi/4 to degree 15 and 16,
// and the quadrant of k.  The hash multiplies sin by 1e4 before taking the
// fraction, so any last-bit difference moves a spawn; GLSL leaves sin's
// precision to the implementation, and this one runs the same operations on
// the device and on a host (no contraction: -ffp-contract=off).
__device__ __forceinline__ float hash_sinf(float xf) {
    const double x = double(xf);
    const double k = rint(x * 0.6366197723675814);
    const double r = ((x - k * 1.570796251296997) - k * 7.549789415861596e-08) - k * 5.390302858158119e-15;
    const double z = r * r;
    const double sn = r * (1.0 + z * (-1.0 / 6.0 + z * (1.0 / 120.0 + z * (-1.0 / 5040.0 + z * (1.0 / 362880.0 +
                      z * (-1.0 / 39916800.0 + z * (1.0 / 6227020800.0 + z * (-1.0 / 1307674368000.0))))))));
    const double cs = 1.0 + z * (-0.5 + z * (1.0 / 24.0 + z * (-1.0 / 720.0 + z * (1.0 / 40320.0 +
                      z * (-1.0 / 3628800.0 + z * (1.0 / 479001600.0 + z * (-1.0 / 87178291200.0 +
                      z * (1.0 / 20922789888000.0))))))));
    const int q = int(static_cast<long long>(k) & 3);
    const double v = q == 0 ? sn : q == 1 ? cs : q == 2 ? -sn : -cs;
    return float(v);
}

// rand(vec2 p), glsl/particle.glsl:41-44
__device__ __forceinline__ float rp_rand(float x, float y) {
    return fract_(1e4f * hash_sinf(17.0f * x + y * 0.1f) * (0.1f + fabsf(hash_sinf(y * 13.0f + x))));
}

// img_bilinear (glsl/img_interpolation.glsl:3-22) of one plane; texels
// outside the image read 0.
__device__ __forceinline__ float rp_tex(const float* p, int n, int x, int y) {
    return (x >= 0 && y >= 0 && x < n && y < n) ? p[size_t(y) * n + x] : 0.0f;
}
__device__ __forceinline__ float rp_bilinear(const float* p, int n, float x, float y) {
    const int ix = int(x), iy = int(y);
    const float fx = fract_(x), fy = fract_(y);
    const float a = rp_tex(p, n, ix, iy), b = rp_tex(p, n, ix + 1, iy);
    const float c = rp_tex(p, n, ix, iy + 1), d = rp_tex(p, n, ix + 1, iy + 1);
    const float v1 = a + fx * (b - a);
    const float v2 = c + fx * (d - c);
    return v1 + fy * (v2 - v1);
}

// The four samples of get_terr_normal for a plane, at (x+1, y), (x-1, y), (x,
// y-1) and (x, y+1) around (px, py): their 16 texels are 12 cells of a 4 x 4
// patch, read row by row with 2- and 4-cell loads (cells are 4-byte aligned,
// which global loads of any width allow) instead of one by one.  2048^2 with
// 262144 particles at unrelated places: 93 -> 71 us per dispatch.
typedef float float2_u __attribute__((ext_vector_type(2), aligned(4)));
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));
struct RpPatch {
    float2_u below, above;     // rows y-1 and y+2, columns x, x+1
    float4_u at, next;         // rows y and y+1, columns x-1 .. x+2
};
__device__ __forceinline__ RpPatch rp_patch(const float* p, int n, int ix, int iy) {
    const float* q = p + size_t(iy) * n + ix;
    RpPatch a;
    a.below = *reinterpret_cast<const float2_u*>(q - n);
    a.at = *reinterpret_cast<const float4_u*>(q - 1);
    a.next = *reinterpret_cast<const float4_u*>(q + n - 1);
    a.above = *reinterpret_cast<const float2_u*>(q + 2 * size_t(n));
    return a;
}
__device__ __forceinline__ float rp_mix4(float a, float b, float c, float d, float x, float y) {
    const float fx = fract_(x), fy = fract_(y);
    const float v1 = a + fx * (b - a);
    const float v2 = c + fx * (d - c);
    return v1 + fy * (v2 - v1);
}
// Samples right, left, bottom, top of the patch.
__device__ __forceinline__ void rp_samples(const RpPatch& a, float px, float py, float& r, float& l, float& b, float& t) {
    r = rp_mix4(a.at[2], a.at[3], a.next[2], a.next[3], px + 1.0f, py);
    l = rp_mix4(a.at[0], a.at[1], a.next[0], a.next[1], px - 1.0f, py);
    b = rp_mix4(a.below[0], a.below[1], a.at[1], a.at[2], px, py - 1.0f);
    t = rp_mix4(a.next[1], a.next[2], a.above[0], a.above[1], px, py + 1.0f);
}
// Bilinear sample at (px, py) inside the image, two cells per load.
__device__ __forceinline__ float rp_inside(const float* p, int n, int ix, int iy, float px, float py) {
    const float2_u a = *reinterpret_cast<const float2_u*>(p + size_t(iy) * n + ix);
    const float2_u b = *reinterpret_cast<const float2_u*>(p + size_t(iy + 1) * n + ix);
    return rp_mix4(a[0], a[1], b[0], b[1], px, py);
}

// Correctly rounded division and square root: plain `/` and sqrtf lower to
// the IEEE sequences (HIP's __fsqrt_rn lowers to the native 3-ulp sqrt).
__device__ __forceinline__ float fdiv(float a, float b) { return a / b; }
__device__ __forceinline__ float fsqrt(float a) { return sqrtf(a); }

__global__ __launch_bounds__(256) void k_refp_move(hg_ref_particle* __restrict__ parts, uint32_t count,
                                                   const float* __restrict__ R, const float* __restrict__ D,
                                                   const float* __restrict__ B, const float* __restrict__ MX,
                                                   const float* __restrict__ MY, int n, RefParticleParams k,
                                                   float time, int should_rain) {
    const uint32_t id = blockIdx.x * 256u + threadIdx.x;
    if (id >= count) return;
    hg_ref_particle p = parts[id];
    if (p.iters == 0 && !should_rain) return;
    for (int i = 0; i < 2; ++i)
        if (p.sediment[i] < 0.0f || p.iters == 0) p.sediment[i] = 0.0f;
    if (p.iters == 0 || p.to_kill) {                                             // :71-86
        const float ax = fract_(time * 1.37f) * 1000.0f, ay = fract_(time * 7.21f) * 1000.0f;
        p.position[0] = fdiv(rp_rand(ax, float(id)) * float(k.dims_x - 4.0f), 1.0f) + 2.0f;
        p.position[1] = fdiv(rp_rand(ay, float(id) + 3.14f) * float(k.dims_y - 4.0f), 1.0f) + 2.0f;
        p.to_kill = 0u;
        p.velocity[0] = 0.0f;
        p.velocity[1] = 0.0f;
        p.volume = k.init_volume;
        if (!should_rain) return;          // p.iters = 0; return: nothing is written back
        p.iters = 1;
    }
    const float px = p.position[0], py = p.position[1];
    // get_terr_normal (:51-63)
    // Inside the image, and where px +- 1 round to the neighbouring cells (a
    // position just below a cell's end can round up to the next), the samples
    // are taken from the patch; elsewhere texel by texel.
    const int ix = int(px), iy = int(py);
    const bool inside = px >= 1.0f && py >= 1.0f && ix < n - 2 && iy < n - 2 && int(px + 1.0f) == ix + 1 &&
                        int(px - 1.0f) == ix - 1 && int(py + 1.0f) == iy + 1 && int(py - 1.0f) == iy - 1;
    float rr, rg, lr, lg, br, bg, tr, tg, mx, my, water;
    if (inside) {
        const RpPatch a = rp_patch(R, n, ix, iy), b = rp_patch(D, n, ix, iy);
        mx = rp_inside(MX, n, ix, iy, px, py);
        my = rp_inside(MY, n, ix, iy, px, py);
        water = rp_inside(B, n, ix, iy, px, py);
        rp_samples(a, px, py, rr, lr, br, tr);
        rp_samples(b, px, py, rg, lg, bg, tg);
    } else {
        rr = rp_bilinear(R, n, px + 1.0f, py); rg = rp_bilinear(D, n, px + 1.0f, py);
        lr = rp_bilinear(R, n, px - 1.0f, py); lg = rp_bilinear(D, n, px - 1.0f, py);
        br = rp_bilinear(R, n, px, py - 1.0f); bg = rp_bilinear(D, n, px, py - 1.0f);
        tr = rp_bilinear(R, n, px, py + 1.0f); tg = rp_bilinear(D, n, px, py + 1.0f);
        mx = rp_bilinear(MX, n, px, py);
        my = rp_bilinear(MY, n, px, py);
        water = rp_bilinear(B, n, px, py);
    }
    const float dx = rr + rg - lr - lg;
    const float dz = tr + tg - br - bg;
    const float cx = dx * 2.0f - 0.0f * dz, cy = 0.0f * 0.0f - 2.0f * 2.0f, cz = 2.0f * dz - dx * 0.0f;
    const float cl = fsqrt(cx * cx + cy * cy + cz * cz);
    const float nx = fdiv(cx, cl), ny = fdiv(cy, cl), nz = fdiv(cz, cl);
    float vx = p.velocity[0], vy = p.velocity[1];
    vx = vx - fdiv(k.dt * nx, p.volume) * k.G;                                   // :101
    vy = vy - fdiv(k.dt * nz, p.volume) * k.G;
    const float mlen = fsqrt(mx * mx + my * my);
    float vlen = fsqrt(vx * vx + vy * vy);
    if (mlen > 0.0f && vlen > 0.0f) {                                            // :103-105
        const float d = fdiv(mx, mlen) * fdiv(vx, vlen) + fdiv(my, mlen) * fdiv(vy, vlen);
        const float t = fdiv(k.inertia * d, p.volume + 1e5f * water);
        vx = vx + t * mx;
        vy = vy + t * my;
    }
    vlen = fsqrt(vx * vx + vy * vy);
    if (vlen > 1.0f) {                                                           // :108-110
        vx = fdiv(vx, vlen);
        vy = fdiv(vy, vlen);
    }
    float qx = px + k.dt * vx, qy = py + k.dt * vy;                              // :113
    if (qx <= 1.0f || qy <= 1.0f || qx * 1.0f >= float(k.dims_x - 2) || qy * 1.0f >= float(k.dims_y - 2)) {   // :114-124
        qx = px;
        qy = py;
        vx = 0.0f;
        vy = 0.0f;
        p.to_kill = 1u;
    }
    const float fr = 1.0f - k.dt * k.friction * ny;                              // :125
    vx = vx * fr;
    vy = vy * fr;
    p.volume = p.volume - k.dt * k.Ke;                                           // :126
    const float sin_a = fsqrt(1.0f - ny * ny);                                   // :129
    vlen = fsqrt(vx * vx + vy * vy);
    const float m02 = 0.02f < sin_a ? sin_a : 0.02f;                             // GLSL max(0.02, sin_a)
    const float sc = k.Kc * p.volume * vlen * m02;
    p.sc = 0.0f < sc ? sc : 0.0f;                                                // :131
    p.iters += 1;
    if (p.volume <= k.min_volume || vlen < k.min_velocity || uint32_t(p.iters) >= k.ttl) p.to_kill = 1u;
    p.position[0] = qx;
    p.position[1] = qy;
    p.velocity[0] = vx;
    p.velocity[1] = vy;
    parts[id] = p;
}

__device__ __forceinline__ void atomic_addf(float* p, float v) { unsafeAtomicAdd(p, v); }

// h' = max-with-clamp of h - eroded (h' = 0 when h - eroded < 0) as one atomic
// update of *p.  Returns the height it replaced; `t` = that height - eroded.
__device__ float dissolve(float* p, float eroded, float& t, unsigned long long* giveups) {
    unsigned int* u = reinterpret_cast<unsigned int*>(p);
    unsigned int old = __hip_atomic_load(u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int tries = 0; tries < kCasTries; ++tries) {
        const float h = __uint_as_float(old);
        const float tt = h - eroded;
        const float nv = tt < 0.0f ? 0.0f : tt;
        unsigned int expected = old;
        if (__hip_atomic_compare_exchange_strong(u, &expected, __float_as_uint(nv), __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            t = tt;
            return h;
        }
        old = expected;
    }
    const float h = atomicAdd(p, -eroded);
    t = h - eroded;
    atomicAdd(giveups, 1ull);
    return h;
}

// Value of lane c of the caller's group of 4 lanes.
template <int C>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), C * 0x55, 0xf, 0xf, true));
}

// A group of 4 lanes per particle, one per corner of its quad.  The kernel is
// paced by the atomics, which the L2s pass on to memory one request at a time
// (see hg_particle.hip): two corners of a row are now one request per plane,
// and the corners' read-modify-write chains overlap instead of following each
// other.  2048^2 with 262144 particles: 200 -> 134 us per dispatch.
// The corners' cells are distinct, and the shader's corner loop hands only the
// particle's sediment from one corner to the next; every lane replays that
// chain, in the shader's order, from what the four corners did.
__global__ __launch_bounds__(256) void k_refp_erode(hg_ref_particle* __restrict__ parts, uint32_t count,
                                                    float* R, float* D, float* B, float* MZ, float* MW, int n,
                                                    RefParticleParams k, unsigned long long* giveups) {
    const uint32_t id = blockIdx.x * 64u + threadIdx.x / 4u;
    const int c = int(threadIdx.x & 3u);
    if (id >= count) return;
    const hg_ref_particle part = parts[id];
    if (part.iters == 0) return;
    const float px = part.position[0] * 1.0f, py = part.position[1] * 1.0f;
    // corners (0,0), (1,0), (1,1), (0,1)
    const bool right = c == 1 || c == 2, top = c >= 2;
    const int qx = int(px) + (right ? 1 : 0), qy = int(py) + (top ? 1 : 0);
    const float fx = fract_(px), fy = fract_(py);
    const float multipl = (right ? fx : 1.0f - fx) * (top ? fy : 1.0f - fy);
    const bool on_grid = qx >= 0 && qy >= 0 && qx < n && qy < n;         // imageStore outside: dropped
    // what this corner does to the particle's sediment of layer l: set[l] its
    // new value (to_kill: the amount taken off), done[l] whether it is reached
    float set[2] = {0.0f, 0.0f};
    bool done[2] = {false, false};
    if (on_grid) {
        const size_t i = size_t(qy) * n + qx;
        float* layer[2] = {R, D};
        float cap = 0.0f;
#pragma unroll
        for (int l = 1; l >= 0; --l) {
            float* h = layer[l] + i;
            done[l] = true;
            if (part.to_kill) {                                                  // :36-42
                const float sed = part.sediment[l] * multipl;
                atomic_addf(h, sed);
                set[l] = sed;
                continue;
            }
            const float Kls = k.dt * k.Ks[l], Kld = k.dt * k.Kd[l];
            const float cs = part.sc - cap;
            const float cc = 0.0f < cs ? cs : 0.0f;
            float s1 = part.sediment[l];
            if (cc > s1) {                                                       // :52-63
                const float eroded = multipl * Kls * (cc - s1);
                s1 = s1 + eroded;
                float t;
                const float old_terr = dissolve(h, eroded, t, giveups);
                if (t < 0.0f) {
                    s1 = s1 + t;
                    cap = cap + old_terr;
                } else {
                    set[l] = s1;
                    break;
                }
            } else {                                                             // :65-69
                const float deposit = multipl * Kld * (s1 - cc);
                s1 = s1 - deposit;
                atomic_addf(h, deposit);
            }
            set[l] = s1;
        }
        atomic_addf(B + i, 1e-5f * part.volume * multipl);                       // :79
        atomic_addf(MZ + i, part.volume * part.velocity[0] * multipl);          // :81
        atomic_addf(MW + i, part.volume * part.velocity[1] * multipl);
    }
    float sed0 = part.sediment[0], sed1 = part.sediment[1];
    const float flags = (on_grid ? 1.0f : 0.0f) + (done[0] ? 2.0f : 0.0f);
    auto corner = [&](float v1, float v0, float f) {
        if (f < 1.0f) return;                                                    // off the grid
        sed1 = part.to_kill ? sed1 - v1 : v1;
        if (f > 2.0f) sed0 = part.to_kill ? sed0 - v0 : v0;
        const float conv = sed0 * k.Kconv * k.dt;                               // :71-75
        sed1 = sed1 + conv;
        sed0 = sed0 - conv;
    };
    corner(quad_lane<0>(set[1]), quad_lane<0>(set[0]), quad_lane<0>(flags));
    corner(quad_lane<1>(set[1]), quad_lane<1>(set[0]), quad_lane<1>(flags));
    corner(quad_lane<2>(set[1]), quad_lane<2>(set[0]), quad_lane<2>(flags));
    corner(quad_lane<3>(set[1]), quad_lane<3>(set[0]), quad_lane<3>(flags));
    if (c == 0) {
        parts[id].sediment[0] = sed0;
        parts[id].sediment[1] = sed1;
    }
}

// glsl/smoothing.glsl:76-95 on the interior cells (border cells return before it).
__global__ __launch_bounds__(256) void k_refp_smooth_extra(float* B, float* MX, float* MY, float* MZ, float* MW,
                                                           int n, float cnt) {
    const size_t cells = size_t(n) * n;
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= cells) return;
    const int y = int(i / size_t(n)), x = int(i - size_t(y) * n);
    if (x == 0 || y == 0 || x == n - 1 || y == n - 1) return;
    const float fm0 = 1.0f - (1e-12f * cnt), fb0 = 1.0f - (8e-8f * cnt);
    const float fm = fminf(fmaxf(fm0, 0.0f), 1.0f), fb = fminf(fmaxf(fb0, 0.0f), 1.0f);
    float mx = MX[i] * fm, my = MY[i] * fm;
    mx = mx + (1e-12f * cnt) * MZ[i];
    my = my + (1e-12f * cnt) * MW[i];
    MZ[i] = 0.0f;
    MW[i] = 0.0f;
    float b = B[i] * fb;
    if (b < 1e-6f) b = 0.0f;
    if (fsqrt(mx * mx + my * my) < 1e-12f) {
        mx = 0.0f;
        my = 0.0f;
    }
    MX[i] = mx;
    MY[i] = my;
    B[i] = b;
}

}  // namespace

static_assert(sizeof(hg_ref_particle) == 48, "Particle is 48 bytes in std430");

hipError_t launch_ref_particle_move(hg_ref_particle* parts, uint32_t count, const float* rock, const float* dirt,
                                    const float* water, const float* mx, const float* my, int n,
                                    const RefParticleParams& k, float time, int should_rain, hipStream_t s) {
    if (count == 0) return hipSuccess;
    k_refp_move<<<(count + 255) / 256, 256, 0, s>>>(parts, count, rock, dirt, water, mx, my, n, k, time, should_rain);
    return hipGetLastError();
}

hipError_t launch_ref_particle_erode(hg_ref_particle* parts, uint32_t count, float* rock, float* dirt, float* water,
                                     float* mz, float* mw, int n, const RefParticleParams& k,
                                     unsigned long long* giveups, hipStream_t s) {
    if (count == 0) return hipSuccess;
    k_refp_erode<<<(count + 63) / 64, 256, 0, s>>>(parts, count, rock, dirt, water, mz, mw, n, k, giveups);
    return hipGetLastError();
}

hipError_t launch_ref_particle_smooth_extra(float* water, float* mx, float* my, float* mz, float* mw, int n,
                                            uint32_t particle_count, hipStream_t s) {
    const size_t cells = size_t(n) * n;
    k_refp_smooth_extra<<<unsigned((cells + 255) / 256), 256, 0, s>>>(water, mx, my, mz, mw, n,
                                                                        float(particle_count));
    return hipGetLastError();
}

}  // namespace hgk
