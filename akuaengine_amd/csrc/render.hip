// render.hip -- headless point-sprite rendering of the particles (akua_render, include/akua_io.h).
//
// The reference draws its particle VBO with GL point sprites (Renderer.cpp:28-56;
// fluidParticle.vert: gl_PointSize = size / |world - camera|; fluidParticle.frag: discard where
// |gl_PointCoord - 0.5| > 0.5, colour * exp(-3 d^2)) over a floor mesh (floor.frag: checker of
// floor(x) + floor(z)), depth test GL_LESS, particles in buffer order.  Here:
//   k_render_clear   every pixel key to the maximum (no sprite), and the draw order's inverse;
//   k_render_splat   one lane per particle: the clip-volume test of a GL point, the sprite
//                    square, and by one or more lanes for each fragment centre inside the disc an
//                    atomic minimum of (window depth bits << 32 | draw index) -- the smallest depth
//                    wins and, at equal depth, the earlier particle in buffer order, which is what
//                    GL_LESS keeps when the sprites are drawn in that order;
//   k_render_huge    the same for the sprites that k_render_splat lists as too large for a wave;
//   k_render_resolve one thread per pixel: the winning sprite's colour at this fragment, or the
//                    floor where a ray through the pixel centre meets it nearer, or the clear
//                    colour; written as RGB8 rows from the top.
#include "render.h"

#include <algorithm>
#include <cmath>

namespace akua {

namespace {

constexpr float kMaxPointSize = 256.0f;  // GL clamps sprites to an implementation range
constexpr float kFloorY = -0.02f;        // FLOOR_LEVEL (Application.cpp:16)
constexpr float kFloorExtent = 100.0f;   // floor quad x, z in [0, 100] (Application.cpp:130-135)

// Empties the pixels' keys and the list of huge sprites and inverts the draw order: phys[k], the slot drawn k-th.
__global__ void k_render_clear(unsigned long long* __restrict__ z, uint32_t pixels, const uint32_t* __restrict__ lid,
                               uint32_t* __restrict__ phys, uint32_t n, uint32_t* __restrict__ huge) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0u) huge[0] = 0u;
    if (i < pixels) z[i] = ~0ull;
    if (i < n) {
        const uint32_t k = lid[i];
        if (k < n) phys[k] = i;
    }
}

struct Sprite {
    float xw, yw, zw, s;  // window centre (pixels, origin bottom-left), depth in [0, 1], size
};

// The sprite of the particle at world position p, or false when GL would clip the point.
__device__ __forceinline__ bool sprite_of(const RenderParams& R, float px, float py, float pz,
                                          float size, Sprite& out) {
    const float* m = R.vp;
    const float cx = ((m[0] * px + m[1] * py) + m[2] * pz) + m[3];
    const float cy = ((m[4] * px + m[5] * py) + m[6] * pz) + m[7];
    const float cz = ((m[8] * px + m[9] * py) + m[10] * pz) + m[11];
    const float cw = ((m[12] * px + m[13] * py) + m[14] * pz) + m[15];
    if (!(cw > 0.0f) || !(fabsf(cx) <= cw) || !(fabsf(cy) <= cw) || !(fabsf(cz) <= cw)) return false;
    const float nx = cx / cw, ny = cy / cw, nz = cz / cw;
    out.xw = (nx * 0.5f + 0.5f) * (float)R.width;
    out.yw = (ny * 0.5f + 0.5f) * (float)R.height;
    out.zw = nz * 0.5f + 0.5f;
    const float dx = px - R.eye[0], dy = py - R.eye[1], dz = pz - R.eye[2];
    const float dist = sqrtf((dx * dx + dy * dy) + dz * dz);
    float s = size / dist;
    s = fminf(fmaxf(s, 1.0f), kMaxPointSize);
    if (!(s == s)) return false;
    out.s = s;
    return true;
}

// Squared distance of fragment (fx, fy) from the sprite centre in sprite coordinates (0.25 is the
// disc's edge).
__device__ __forceinline__ float sprite_d2(const Sprite& sp, int fx, int fy) {
    const float x0 = sp.xw - 0.5f * sp.s, y0 = sp.yw - 0.5f * sp.s;
    const float ox = ((float)fx + 0.5f - x0) / sp.s - 0.5f;
    const float oy = ((float)fy + 0.5f - y0) / sp.s - 0.5f;
    return ox * ox + oy * oy;
}

// A sprite's fragments on the screen: the rectangle's first column and row, its width and size, and the key
// (depth, then draw order) that its pixels take the smallest of.
struct Splat {
    Sprite sp;
    int fx0, fy0;
    uint32_t w, count;  // count 0: nothing to draw
    unsigned long long key;
};

__device__ __forceinline__ Splat splat_of(const RenderParams& R, float4 x, float size, uint32_t draw) {
    Splat s;
    s.count = 0u;
    if (!sprite_of(R, x.x, x.y, x.z, size, s.sp)) return s;
    const float x0 = s.sp.xw - 0.5f * s.sp.s, y0 = s.sp.yw - 0.5f * s.sp.s;
    // fragments whose centres f + 0.5 lie in [x0, x0 + s)
    int fx0 = (int)ceilf(x0 - 0.5f), fx1 = (int)ceilf(x0 + s.sp.s - 0.5f) - 1;
    int fy0 = (int)ceilf(y0 - 0.5f), fy1 = (int)ceilf(y0 + s.sp.s - 0.5f) - 1;
    fx0 = max(fx0, 0);
    fy0 = max(fy0, 0);
    fx1 = min(fx1, R.width - 1);
    fy1 = min(fy1, R.height - 1);
    if (fx1 < fx0 || fy1 < fy0) return s;
    s.fx0 = fx0;
    s.fy0 = fy0;
    s.w = (uint32_t)(fx1 - fx0 + 1);
    s.count = s.w * (uint32_t)(fy1 - fy0 + 1);  // at most 257 x 257
    s.key = ((unsigned long long)__float_as_uint(s.sp.zw) << 32) | (unsigned long long)draw;
    return s;
}

// Fragments first, first + kStride, ... of the rectangle row by row, kSplatBatch at a time: their pixels' keys are
// read together.  A key that the pixel already undercuts needs no atomic (keys only fall, so an old value
// read decides the same): sprites overlap many deep.
constexpr uint32_t kSplatBatch = 4;
template <uint32_t kStride>
__device__ __forceinline__ void splat_draw(const RenderParams& R, const Splat& s, uint32_t first, unsigned long long* zbuf) {
    uint32_t row = first / s.w, column = first - row * s.w;
    for (uint32_t f = first; f < s.count; f += kStride * kSplatBatch) {
        unsigned long long* at[kSplatBatch];
        unsigned long long old[kSplatBatch];
#pragma unroll
        for (uint32_t u = 0; u < kSplatBatch; ++u) {
            const int fx = s.fx0 + (int)column, fy = s.fy0 + (int)row;
            const bool in = f + u * kStride < s.count && !(sprite_d2(s.sp, fx, fy) > 0.25f);
            at[u] = in ? &zbuf[(size_t)(R.height - 1 - fy) * (size_t)R.width + (size_t)fx] : nullptr;
            old[u] = in ? __hip_atomic_load(at[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0ull;
            for (column += kStride; column >= s.w; column -= s.w) ++row;
        }
#pragma unroll
        for (uint32_t u = 0; u < kSplatBatch; ++u)
            if (old[u] > s.key) atomicMin(at[u], s.key);
    }
}

// A wave projects kPer particles, one per lane.  A sprite of a few fragments is drawn by its lane, a
// larger one by sixteen, four sprites at a time: at the reference's point size a near sprite has some 80
// fragments, a serial chain for one lane, and a distant one a few, for which sixteen lanes are idle.  Sprites of
// more than kSplatHuge fragments, close to the camera, are listed for a launch of their own (kList): those of one
// wave would keep it busy long after the others.  Measured at 1280 x 720, us with one lane per sprite / with
// sixteen / so: 27,000 particles in the default view 267 / 53 / 53, in sprites of about one pixel 3 / 7 / 4; 1M from
// (5, 4, 16) 459 / 249 / 176, in sprites of 1-5 pixels 34 / 148 / 58, from within 6,602 / 1,658 / 286; 8M 526 / 1,166
// / 517 and 300 / 1,182 / 307.
constexpr uint32_t kSplatLanes = 16, kSplatHuge = 1024;

template <uint32_t kPer, bool kList>
__global__ __launch_bounds__(256) void k_render_splat(const float4* __restrict__ X, const float* __restrict__ size,
                                                      const uint32_t* __restrict__ id,
                                                      const uint32_t* __restrict__ lid, uint32_t n, RenderParams R,
                                                      unsigned long long* zbuf, uint32_t* __restrict__ huge) {
    constexpr uint32_t kOwn = kPer == 4u ? 4u : 8u;  // with four particles all of them have their lanes at once
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t i = (blockIdx.x * (256u / 64u) + (threadIdx.x >> 6)) * kPer + lane;
    Splat mine;
    mine.count = 0u;
    if (lane < kPer && i < n) mine = splat_of(R, X[i], R.pointSize > 0.0f ? R.pointSize : size[id[i]], lid[i]);
    if (mine.count != 0u && mine.count <= kOwn) splat_draw<1u>(R, mine, 0u, zbuf);
    if (kList) {
        const bool listed = mine.count > kSplatHuge;
        const unsigned long long all = __ballot(listed);
        if (all != 0ull) {
            uint32_t at = 0;
            if (lane == 0u) at = atomicAdd(huge, (uint32_t)__builtin_popcountll(all));
            at = (uint32_t)__shfl((int)at, 0, 64) + (uint32_t)__builtin_popcountll(all & ~(~0ull << lane));
            if (listed) {
                huge[1u + at] = i;
                mine.count = 0u;
            }
        }
    }
    for (unsigned long long large = __ballot(mine.count > kOwn); large != 0ull;) {
        // the next four: this lane's sixteen take the (lane / 16)th
        uint32_t from = 64u;
#pragma unroll
        for (uint32_t g = 0; g < 64u / kSplatLanes; ++g) {
            if (g == lane / kSplatLanes && large != 0ull) from = (uint32_t)__builtin_ctzll(large);
            large &= large - 1ull;
        }
        const int of = (int)(from & 63u);
        Splat s;
        s.sp.xw = __shfl(mine.sp.xw, of, 64);
        s.sp.yw = __shfl(mine.sp.yw, of, 64);
        s.sp.s = __shfl(mine.sp.s, of, 64);
        s.fx0 = __shfl(mine.fx0, of, 64);
        s.fy0 = __shfl(mine.fy0, of, 64);
        s.w = (uint32_t)__shfl((int)mine.w, of, 64);
        s.count = (uint32_t)__shfl((int)mine.count, of, 64);
        s.key = (unsigned long long)__shfl((long long)mine.key, of, 64);
        if (from < 64u) splat_draw<kSplatLanes>(R, s, lane % kSplatLanes, zbuf);
    }
}

// The listed sprites, a workgroup each.
constexpr uint32_t kHugeBlock = 256, kHugeBlocks = 2048;
__global__ __launch_bounds__(kHugeBlock) void k_render_huge(const float4* __restrict__ X, const float* __restrict__ size,
                                                            const uint32_t* __restrict__ id,
                                                            const uint32_t* __restrict__ lid, uint32_t n, RenderParams R,
                                                            unsigned long long* zbuf, const uint32_t* __restrict__ huge) {
    const uint32_t count = min(huge[0], n);
    for (uint32_t q = blockIdx.x; q < count; q += gridDim.x) {
        const uint32_t i = min(huge[1u + q], n - 1u);
        const Splat s = splat_of(R, X[i], R.pointSize > 0.0f ? R.pointSize : size[id[i]], lid[i]);
        if (s.count != 0u) splat_draw<kHugeBlock>(R, s, threadIdx.x, zbuf);
    }
}

__device__ __forceinline__ unsigned char to_u8(float c) {
    c = fminf(fmaxf(c, 0.0f), 1.0f);
    return (unsigned char)__float2int_rn(c * 255.0f);
}

__global__ void k_render_resolve(const float4* __restrict__ X, const float4* __restrict__ color,
                                 const float* __restrict__ size, const uint32_t* __restrict__ id,
                                 const uint32_t* __restrict__ phys, RenderParams R,
                                 const unsigned long long* __restrict__ zbuf,
                                 unsigned char* __restrict__ rgb) {
    const uint32_t pix = blockIdx.x * blockDim.x + threadIdx.x;
    if (pix >= (uint32_t)(R.width * R.height)) return;
    const int row = (int)(pix / (uint32_t)R.width), fx = (int)(pix % (uint32_t)R.width);
    const int fy = R.height - 1 - row;
    float r = 0.15f, g = 0.15f, b = 0.18f;  // glClearColor (Application.cpp:72)
    bool floorHit = false;
    float zf = 1.0f;
    if (R.drawFloor) {
        // the ray through the pixel centre against the floor plane
        const float nx = ((float)fx + 0.5f) / (float)R.width * 2.0f - 1.0f;
        const float ny = ((float)fy + 0.5f) / (float)R.height * 2.0f - 1.0f;
        const float a = nx * R.tanHalf * R.aspect, c = ny * R.tanHalf;
        const float dx = (R.front[0] + a * R.right[0]) + c * R.up[0];
        const float dy = (R.front[1] + a * R.right[1]) + c * R.up[1];
        const float dz = (R.front[2] + a * R.right[2]) + c * R.up[2];
        if (dy != 0.0f) {
            const float t = (kFloorY - R.eye[1]) / dy;
            const float hx = R.eye[0] + t * dx, hz = R.eye[2] + t * dz;
            if (t > 0.0f && hx >= 0.0f && hx <= kFloorExtent && hz >= 0.0f && hz <= kFloorExtent) {
                const float* m = R.vp;
                const float cz = ((m[8] * hx + m[9] * kFloorY) + m[10] * hz) + m[11];
                const float cw = ((m[12] * hx + m[13] * kFloorY) + m[14] * hz) + m[15];
                if (cw > 0.0f && fabsf(cz) <= cw) {
                    floorHit = true;
                    zf = (cz / cw) * 0.5f + 0.5f;
                    const int check = ((int)floorf(hx) + (int)floorf(hz)) & 1;
                    r = g = b = check ? 0.5f : 0.8f;  // mix(color1, color2, check)
                }
            }
        }
    }
    const unsigned long long key = zbuf[pix];
    if (key != ~0ull) {
        const float zp = __uint_as_float((uint32_t)(key >> 32));
        if (!floorHit || zp < zf) {
            const uint32_t slot = phys[(uint32_t)(key & 0xFFFFFFFFull)];  // draw index -> slot
            const float4 x = X[slot];
            const float sz = R.pointSize > 0.0f ? R.pointSize : size[id[slot]];
            Sprite sp;
            if (sprite_of(R, x.x, x.y, x.z, sz, sp)) {
                const float d2 = sprite_d2(sp, fx, fy);
                const float alpha = expf(-3.0f * d2);
                const float4 col = color[id[slot]];
                r = col.x * alpha;
                g = col.y * alpha;
                b = col.z * alpha;
            }
        }
    }
    rgb[3 * (size_t)pix + 0] = to_u8(r);
    rgb[3 * (size_t)pix + 1] = to_u8(g);
    rgb[3 * (size_t)pix + 2] = to_u8(b);
}

}  // namespace

void camera_setup(const float position[3], float yawDeg, float pitchDeg, float fovYDeg, float nearZ,
                  float farZ, int width, int height, RenderParams& R) {
    const double d2r = 3.14159265358979323846 / 180.0;
    const double yaw = yawDeg * d2r, pitch = pitchDeg * d2r;
    // Camera::updateVectors (Camera.cpp:76-87), then glm::lookAt's basis
    double f[3] = {std::cos(yaw) * std::cos(pitch), std::sin(pitch), std::sin(yaw) * std::cos(pitch)};
    auto norm = [](double* v) {
        const double l = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        for (int k = 0; k < 3; ++k) v[k] /= l;
    };
    auto cross = [](const double* a, const double* b, double* o) {
        o[0] = a[1] * b[2] - a[2] * b[1];
        o[1] = a[2] * b[0] - a[0] * b[2];
        o[2] = a[0] * b[1] - a[1] * b[0];
    };
    norm(f);
    const double worldUp[3] = {0.0, 1.0, 0.0};
    double rt[3], up[3];
    cross(f, worldUp, rt);
    norm(rt);
    cross(rt, f, up);
    norm(up);
    const double eye[3] = {position[0], position[1], position[2]};
    // glm::lookAt(eye, eye + f, up): rows s, u, -f with translations
    double s[3], u[3];
    cross(f, up, s);
    norm(s);
    cross(s, f, u);
    double V[16] = {s[0], s[1], s[2], -(s[0] * eye[0] + s[1] * eye[1] + s[2] * eye[2]),
                    u[0], u[1], u[2], -(u[0] * eye[0] + u[1] * eye[1] + u[2] * eye[2]),
                    -f[0], -f[1], -f[2], (f[0] * eye[0] + f[1] * eye[1] + f[2] * eye[2]),
                    0.0, 0.0, 0.0, 1.0};
    // glm::perspective (right-handed, depth in [-1, 1])
    const double aspect = (double)width / (double)height;
    const double th = std::tan(fovYDeg * d2r / 2.0);
    const double n = nearZ, fz = farZ;
    double P[16] = {1.0 / (aspect * th), 0, 0, 0,
                    0, 1.0 / th, 0, 0,
                    0, 0, -(fz + n) / (fz - n), -(2.0 * fz * n) / (fz - n),
                    0, 0, -1.0, 0};
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
            double acc = 0.0;
            for (int k = 0; k < 4; ++k) acc += P[4 * r + k] * V[4 * k + c];
            R.vp[4 * r + c] = (float)acc;
        }
    for (int k = 0; k < 3; ++k) {
        R.eye[k] = (float)eye[k];
        R.front[k] = (float)f[k];
        R.right[k] = (float)s[k];
        R.up[k] = (float)u[k];
    }
    R.tanHalf = (float)th;
    R.aspect = (float)aspect;
    R.width = width;
    R.height = height;
}

void launch_render(hipStream_t st, const float4* X, const float4* color, const float* size,
                   const uint32_t* id, const uint32_t* lid, uint32_t* phys, uint32_t n,
                   const RenderParams& R, unsigned long long* zbuf, unsigned char* rgb, uint32_t* huge) {
    const uint32_t pixels = (uint32_t)(R.width * R.height);
    k_render_clear<<<(std::max(pixels, n) + 255) / 256, 256, 0, st>>>(zbuf, pixels, lid, phys, n, huge);
    // Particles per wave: fewer where few waves would draw them all, and up to 2^21 no more than sixteen, as the
    // sprites of a wave lie side by side and one near the camera is at work for longest (1M from (3, 2, 6) after 30
    // steps, us with one lane per sprite / sixteen / so with 64 / so with 16: 896 / 191 / 485 / 205).
    const auto splat = [&](auto kernel, uint32_t per) {
        const uint32_t waves = (n + per - 1u) / per;
        kernel<<<(waves + 3u) / 4u, 256, 0, st>>>(X, size, id, lid, n, R, zbuf, huge);
    };
    if (n > (1u << 21))
        splat(k_render_splat<64, true>, 64u);
    else if (n > (1u << 15))
        splat(k_render_splat<16, true>, 16u);
    else if (n)
        splat(k_render_splat<4, false>, 4u);
    if (n > (1u << 15)) k_render_huge<<<kHugeBlocks, kHugeBlock, 0, st>>>(X, size, id, lid, n, R, zbuf, huge);
    k_render_resolve<<<(pixels + 255) / 256, 256, 0, st>>>(X, color, size, id, phys, R, zbuf, rgb);
}

}  // namespace akua
