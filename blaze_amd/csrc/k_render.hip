// k_render.hip — the solver's consumer: volume ray marching of the
// temperature grid.
//
// Reference: RenderEngine::render (asiroisvigneux/Blaze
// src/RenderEngine.cu:312-365): write_scatter_to_3d_tex_kernel :76-101 (4x
// downsample of T above the ramp's low end), gaussian_blur_texture_kernel
// :51-74 (3x3x3 [1 2 1]-type filter, clamped), render_kernel :149-225
// (camera ray, box clip, primary march with emission, multi-scatter and one
// shadow march per directional light), bbox_intersect_kernel :112-147,
// Camera (src/Camera.h:31-60), Light (src/Light.h:31-55), Shader
// (src/Shader.h:33-75), ColorRamp (src/ColorRamp.h:32-80).
//
// Every expression keeps the reference's evaluation order. Three things are
// defined here instead of by the hardware or CUDA's library: the texture
// lookup is an explicit FP32 trilinear filter with clamped texel indices
// (the reference's clamp-addressed linear-filtered textures, whose weights
// the hardware stores in 8-bit fixed point), normalize divides by sqrtf
// (the reference multiplies by an approximate rsqrtf), and exp is the
// Cody-Waite reduction with a degree-7 Taylor polynomial below (the CPU
// oracle restates the same steps, so the image is reproducible bit for
// bit). A shadow ray that misses the box (only possible for degenerate
// directions; the reference would march it forever) leaves full
// transmittance, and both marches stop after 65536 samples.
#include <mutex>
#include <string>
#include <type_traits>

#include "solver.h"

namespace blz {

namespace {

constexpr int RES_STEP = 8; // frames are multiples of the reference's 8x8 launch tiles
constexpr int MAX_MARCH = 1 << 16;

struct V3 {
    float x, y, z;
};
__device__ __forceinline__ V3 mkv(float x, float y, float z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return mkv(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return mkv(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ V3 operator*(V3 a, V3 b) { return mkv(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ V3 operator*(V3 a, float s) { return mkv(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ V3 operator*(float s, V3 a) { return mkv(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ float sqlen(V3 v) { return v.x * v.x + v.y * v.y + v.z * v.z; }

// exp(x): x = k ln2 + r with ln2 split so that k*ln2_hi is exact (|k| <=
// 128), exp(r) by Taylor to degree 7 (|r| <= ln2/2, truncation < 1e-8
// relative), times 2^k. Below -87.34 (results under FLT_MIN) it returns 0,
// above 88.72 infinity.
// 2^k as one v_ldexp_f32: the product is exact down to FLT_MIN either way.
__device__ __forceinline__ float bexp(float x) {
    const float k = floorf(x * 1.44269502f + 0.5f);
    float r = x - k * 0.693145751953125f;
    r = r - k * 1.42860677e-06f;
    float p = 1.98412701e-04f;
    p = p * r + 1.38888892e-03f;
    p = p * r + 8.33333377e-03f;
    p = p * r + 4.16666679e-02f;
    p = p * r + 1.66666672e-01f;
    p = p * r + 0.5f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    float e = __builtin_amdgcn_ldexpf(p, (int)k);
    e = x > 88.7228394f ? __int_as_float(0x7f800000) : e;
    e = x < -87.3365479f ? 0.0f : e;
    return x != x ? x : e;
}
__device__ __forceinline__ V3 bexp3(V3 a) { return mkv(bexp(a.x), bexp(a.y), bexp(a.z)); }

// linear-filtered, clamp-addressed lookup at unnormalised coordinates
// (texel centres at integer + 0.5): the lower texel of each axis (-1 .. n)
// and the weights of the upper ones
struct Texel {
    int i, j, k;
    float a, b, c;
};
__device__ __forceinline__ Texel texel_at(int nx, int ny, int nz, V3 g) {
    const float xb = g.x - 0.5f, yb = g.y - 0.5f, zb = g.z - 0.5f;
    const float fx = floorf(xb), fy = floorf(yb), fz = floorf(zb);
    return Texel{(int)fminf(fmaxf(fx, -1.0f), (float)nx), (int)fminf(fmaxf(fy, -1.0f), (float)ny),
                 (int)fminf(fmaxf(fz, -1.0f), (float)nz), xb - fx, yb - fy, zb - fz};
}

typedef float f2a4 __attribute__((ext_vector_type(2), aligned(4)));

// PAIR: the two texels of a row as one 8-byte load (the pair moved inside the
// row at its ends), where a wave's lanes are spread along rays. Lanes beside
// each other in the image read beside each other, and there the eight 4-byte
// loads take half the time: 1920x1080 through a full 256^3, one light, 8.6 ms
// against 11.3. WIDE: volumes of 4 GiB and more, whose byte offsets do not fit
// 32 bits.
template <bool WIDE, bool PAIR>
__device__ __forceinline__ float tex_lin(const float* __restrict__ v, int nx, int ny, int nz, const Texel& q) {
    const int ya = min(max(q.j, 0), ny - 1), yc = min(max(q.j + 1, 0), ny - 1);
    const int za = min(max(q.k, 0), nz - 1), zc = min(max(q.k + 1, 0), nz - 1);
    const int x = min(max(q.i, 0), max(nx - 2, 0)), xa = min(max(q.i, 0), nx - 1), xc = min(max(q.i + 1, 0), nx - 1);
    const bool low = q.i < 0, high = q.i >= nx - 1;
    auto at = [&](int i, int j, int k) {
        if (WIDE) return v + ((size_t)k * ny + j) * nx + i;
        return (const float*)((const char*)v + (unsigned)((k * ny + j) * nx + i) * 4u);
    };
    auto row = [&](int j, int k) {
        if (!PAIR) return (1.0f - q.a) * *at(xa, j, k) + q.a * *at(xc, j, k);
        const float* p = at(x, j, k);
        if (nx < 2) return (1.0f - q.a) * p[0] + q.a * p[0]; // uniform
        const f2a4 t = *(const f2a4*)p;
        return (1.0f - q.a) * (high ? t[1] : t[0]) + q.a * (low ? t[0] : t[1]);
    };
    const float c00 = row(ya, za), c10 = row(yc, za), c01 = row(ya, zc), c11 = row(yc, zc);
    return (1.0f - q.c) * ((1.0f - q.b) * c00 + q.b * c10) + q.c * ((1.0f - q.b) * c01 + q.b * c11);
}

// Bricks of 2^sh cells per axis (4 or more, at most OCC_WORDS * 32 bricks):
// a brick's bit is clear where every texel that a lookup starting in it
// reads gives a density below the cutoff, which adds nothing to either march.
constexpr int OCC_WORDS = 1024;
struct Occ {
    int sh, nx, ny, nz, words;
    int box;      // the box of the bricks that are not clear follows the words
    float lim;    // |T| below which a sample is under the cutoff; negative: no brick is clear
    float margin; // of positions and box, per unit of a ray origin's coordinates, and at the domain's own
    float margin_dom;
};

// scene constants computed on the host in the reference's order
struct RScene {
    V3 origin, top_left, horizontal, vertical;
    float res_x, res_y;
    V3 dom_min, dom_max, dom_size;
    float dx;
    int W, H, D, Ws, Hs, Ds;
    float p_step, s_step, cutoff;
    float density_scale, shadow_density_scale, gain, emission_scale;
    V3 albedo, extinction;
    int ramp_size;
    float ramp_in, ramp_out;
    float ramp_keys[BLZ_MAX_RAMP];
    V3 ramp_colors[BLZ_MAX_RAMP];
    V3 ms_color;
    float ms_scale, ms_mask_a, ms_mask_b;
    int light_count;
    V3 light_dir[BLZ_MAX_LIGHTS], light_illum[BLZ_MAX_LIGHTS];
};

__device__ __forceinline__ V3 ramp_color(const RScene& s, float temp) {
    const float remap = fminf(fmaxf((temp - s.ramp_in) / (s.ramp_out - s.ramp_in), 0.0f), 1.0f);
    if (s.ramp_size == 1) return s.ramp_colors[0];
    int prev = 0, next = 0;
    for (int i = 0; i < s.ramp_size; ++i) {
        if (s.ramp_keys[i] <= remap) {
            prev = i;
        } else {
            next = i;
            break;
        }
    }
    const float range = s.ramp_keys[next] - s.ramp_keys[prev];
    const float blend = (remap - s.ramp_keys[prev]) / range;
    return s.ramp_colors[prev] + blend * (s.ramp_colors[next] - s.ramp_colors[prev]);
}

__device__ __forceinline__ float smoothstep_f(float a, float b, float x) {
    const float y = fmaxf(0.0f, fminf((x - a) / (b - a), 1.0f));
    return y * y * (3.0f - (2.0f * y));
}

struct Ray {
    V3 o, d, inv;
    int sx, sy, sz;
    float t0, t1;
};
__device__ __forceinline__ Ray make_ray(V3 o, V3 d) {
    Ray r;
    r.o = o;
    r.d = d;
    r.inv = mkv(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    r.sx = r.inv.x < 0.0f;
    r.sy = r.inv.y < 0.0f;
    r.sz = r.inv.z < 0.0f;
    r.t0 = 0.0f;
    r.t1 = __int_as_float(0x7f800000);
    return r;
}

// slab test of src/RenderEngine.cu:112-147 (sets t0 = max(tmin, 0), t1)
__device__ __forceinline__ bool box_hit(Ray& r, V3 lo, V3 hi) {
    const V3 b[2] = {lo, hi};
    float tmin = (b[r.sx].x - r.o.x) * r.inv.x;
    float tmax = (b[1 - r.sx].x - r.o.x) * r.inv.x;
    const float tymin = (b[r.sy].y - r.o.y) * r.inv.y;
    const float tymax = (b[1 - r.sy].y - r.o.y) * r.inv.y;
    if ((tmin > tymax) || (tymin > tmax)) return false;
    if (tymin > tmin) tmin = tymin;
    if (tymax < tmax) tmax = tymax;
    const float tzmin = (b[r.sz].z - r.o.z) * r.inv.z;
    const float tzmax = (b[1 - r.sz].z - r.o.z) * r.inv.z;
    if ((tmin > tzmax) || (tzmin > tmax)) return false;
    if (tzmin > tmin) tmin = tzmin;
    if (tzmax < tmax) tmax = tzmax;
    r.t0 = fmaxf(tmin, 0.0f);
    r.t1 = tmax;
    if (r.t1 < 0.0f) return false;
    return true;
}

// Grid::worldToGridNoOffset (src/Grid.h:292-296): y flipped
template <class S>
__device__ __forceinline__ V3 w2g(const RScene& s, const S& sc, V3 p) {
    return mkv(sc(p.x - s.dom_min.x), sc(s.dom_size.y - (p.y - s.dom_min.y)), sc(p.z - s.dom_min.z));
}

// write_scatter_to_3d_tex_kernel: mean over the 4x4x4 block of T above tmin
__global__ void __launch_bounds__(256) k_rnd_scatter(const float* __restrict__ T, int W, int H, int Ws, int Hs,
                                                     int Ds, float tmin, float* __restrict__ out) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= Ws * Hs * Ds) return;
    const int i = t % Ws, j = (t / Ws) % Hs, k = t / (Ws * Hs);
    float acc = 0.0f;
    for (int io = 0; io < 4; ++io)
        for (int jo = 0; jo < 4; ++jo)
            for (int ko = 0; ko < 4; ++ko) {
                const float v = T[(size_t)(i * 4 + io) + (size_t)(j * 4 + jo) * W + (size_t)(k * 4 + ko) * W * H];
                acc += v > tmin ? v : 0.0f;
            }
    out[t] = acc / 64.0f;
}

// gaussian_blur_texture_kernel: 27 taps (k outer, then j, then i), samples
// at texel centres of the clamped volume, weights w[tap] (sum 1)
struct BlurW {
    float w[27];
};
__global__ void __launch_bounds__(256) k_rnd_blur(const float* __restrict__ in, float* __restrict__ out, int Ws,
                                                  int Hs, int Ds, BlurW w) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= Ws * Hs * Ds) return;
    const int i = t % Ws, j = (t / Ws) % Hs, k = t / (Ws * Hs);
    float acc = 0.0f;
    int q = 0;
    for (int dk = -1; dk <= 1; ++dk)
        for (int dj = -1; dj <= 1; ++dj)
            for (int di = -1; di <= 1; ++di, ++q) {
                const int x = min(max(i + di, 0), Ws - 1), y = min(max(j + dj, 0), Hs - 1),
                          z = min(max(k + dk, 0), Ds - 1);
                acc += in[(size_t)x + (size_t)y * Ws + (size_t)z * Ws * Hs] * w.w[q];
            }
    out[t] = acc;
}

// one bit per brick; a workgroup per word, eight lanes along x per brick
__global__ void __launch_bounds__(256) k_rnd_occ(const float* __restrict__ T, int W, int H, int D, int nbricks, Occ o,
                                                 unsigned* __restrict__ bits) {
    const int b = blockIdx.x * 32 + (threadIdx.x >> 3), lane = threadIdx.x & 7, E = 1 << o.sh;
    bool any = false;
    if (b < nbricks) {
        const int bx = b % o.nx, by = (b / o.nx) % o.ny, bz = b / (o.nx * o.ny);
        const int x1 = min(bx * E + E, W - 1), y1 = min(by * E + E, H - 1), z1 = min(bz * E + E, D - 1);
        for (int x = bx * E + lane; x <= x1; x += 8)
            for (int z = bz * E; z <= z1; ++z)
#pragma unroll 4
                for (int y = by * E; y <= y1; ++y)
                    any |= !(fabsf(T[((size_t)z * H + y) * W + x]) < o.lim); // NaN is kept
    }
    const unsigned long long m = __ballot(any);
    __shared__ unsigned sm[4];
    if ((threadIdx.x & 63) == 0) {
        unsigned w = 0;
        for (int q = 0; q < 8; ++q)
            if ((m >> (8 * q)) & 255) w |= 1u << q;
        sm[threadIdx.x >> 6] = w;
    }
    __syncthreads();
    if (threadIdx.x == 0) bits[blockIdx.x] = sm[0] | sm[1] << 8 | sm[2] << 16 | sm[3] << 24;
}

// The box around the bricks that are not clear, in world space, six floats
// (lower, upper): one workgroup
__global__ void __launch_bounds__(1024) k_rnd_box(unsigned* __restrict__ bits, Occ o, V3 dom_min, V3 dom_size,
                                                  float dx) {
    __shared__ int lo[3], hi[3];
    if (threadIdx.x < 3) {
        lo[threadIdx.x] = 1 << 30;
        hi[threadIdx.x] = -1;
    }
    __syncthreads();
    // a thread per row of bricks, 32 of its bits at a time
    for (int row = threadIdx.x; row < o.ny * o.nz; row += 1024) {
        int first = 1 << 30, last = -1;
        for (int x = 0; x < o.nx; x += 32) {
            const int b = row * o.nx + x, w = b >> 5;
            const unsigned long long two = bits[w] | (unsigned long long)(w + 1 < o.words ? bits[w + 1] : 0u) << 32;
            unsigned m = (unsigned)(two >> (b & 31));
            if (o.nx - x < 32) m &= (1u << (o.nx - x)) - 1u;
            if (!m) continue;
            first = min(first, x + __ffs(m) - 1);
            last = x + 31 - __clz(m);
        }
        if (last < 0) continue;
        const int l[3] = {first, row % o.ny, row / o.ny}, h[3] = {last, l[1], l[2]};
        for (int a = 0; a < 3; ++a) {
            if (l[a] < lo[a]) atomicMin(&lo[a], l[a]);
            if (h[a] > hi[a]) atomicMax(&hi[a], h[a]);
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    // a lookup starts in brick b from b E + 0.5 to (b + 1) E + 0.5, at the
    // grid's sides from anywhere beyond; y runs downwards
    const float inf = __int_as_float(0x7f800000), E = (float)(1 << o.sh);
    float l[3], h[3];
    const int n[3] = {o.nx, o.ny, o.nz};
    for (int a = 0; a < 3; ++a) {
        l[a] = lo[a] == 0 ? -inf : ((float)lo[a] * E + 0.5f) * dx;
        h[a] = hi[a] == n[a] - 1 ? inf : ((float)(hi[a] + 1) * E + 0.5f) * dx;
    }
    float* out = (float*)(bits + o.words);
    const bool none = hi[0] < 0;
    out[0] = none ? inf : dom_min.x + l[0];
    out[1] = none ? inf : dom_min.y + (dom_size.y - h[1]);
    out[2] = none ? inf : dom_min.z + l[2];
    out[3] = none ? -inf : dom_min.x + h[0];
    out[4] = none ? -inf : dom_min.y + (dom_size.y - l[1]);
    out[5] = none ? -inf : dom_min.z + h[2];
}

// The part of a ray in the box of the bricks that are not clear, widened by
// `margin` (two cells and many times the rounding of positions): samples
// outside [t0, t1] are in clear bricks. A NaN bounds nothing.
struct Span {
    float t0, t1;
};
__device__ __forceinline__ Span box_span(const Ray& r, V3 lo, V3 hi, float margin) {
    Span s{-__int_as_float(0x7f800000), __int_as_float(0x7f800000)};
    auto axis = [&](float o, float d, float inv, float l, float h) {
        l = l - margin - o;
        h = h + margin - o;
        float n = (inv < 0.0f ? h : l) * inv, f = (inv < 0.0f ? l : h) * inv;
        if (d == 0.0f) { // in the slab all along, or nowhere
            n = (l <= 0.0f && h >= 0.0f) ? -__int_as_float(0x7f800000) : __int_as_float(0x7f800000);
            f = -n;
        }
        s.t0 = n > s.t0 ? n : s.t0;
        s.t1 = f < s.t1 ? f : s.t1;
    };
    axis(r.o.x, r.d.x, r.inv.x, lo.x, hi.x);
    axis(r.o.y, r.d.y, r.inv.y, lo.y, hi.y);
    axis(r.o.z, r.d.z, r.inv.z, lo.z, hi.z);
    return s;
}

// Could the sample at q reach the cutoff? (A coordinate that is not finite
// gives NaN weights, and NaN samples are taken.)
__device__ __forceinline__ bool occupied(const unsigned* bits, const Occ& o, const RScene& s, const Texel& q) {
    const int x = min(max(q.i, 0), s.W - 1) >> o.sh, y = min(max(q.j, 0), s.H - 1) >> o.sh,
              z = min(max(q.k, 0), s.D - 1) >> o.sh;
    const int b = (z * o.ny + y) * o.nx + x;
    const float w = q.a + q.b + q.c;
    return ((bits[b >> 5] >> (b & 31)) & 1u) || w != w;
}

// transmittance from `pos` to a light: SU samples at a time, so that their
// loads overlap (the exponentials still follow each other); BITS: samples in
// clear bricks are passed over
template <int SU, bool BITS, bool PAIR, class S, bool WIDE>
__device__ __forceinline__ V3 shadow_march(const float* __restrict__ T, const unsigned* bits, const RScene& s,
                                           const S& sc, const Occ& o, V3 lo, V3 hi, V3 pos, V3 dir) {
    V3 strans = mkv(1.0f, 1.0f, 1.0f);
    Ray sr = make_ray(pos, dir);
    if (!box_hit(sr, s.dom_min, s.dom_max)) return strans;
    float st = sr.t0 + s.dx * 0.5f;
    const bool gain = s.gain != 0.0f || !(st < 1e30f); // else the divisor is 1
    const Span span = box_span(sr, lo, hi, o.margin_dom);
    const float end = span.t1 < sr.t1 ? span.t1 : sr.t1;
    int m = 0;
    for (; st < span.t0 && st <= end && m < MAX_MARCH; ++m) st += s.s_step;
    for (; st <= end && m < MAX_MARCH; m += SU) {
        Texel q[SU];
        float at[SU];
        bool take[SU], any = false;
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            q[u] = texel_at(s.W, s.H, s.D, w2g(s, sc, sr.o + st * sr.d));
            take[u] = st <= end && m + u < MAX_MARCH && (!BITS || occupied(bits, o, s, q[u]));
            any |= take[u];
            at[u] = st;
            st += s.s_step;
        }
        if (!any) continue;
        float sd[SU];
#pragma unroll
        for (int u = 0; u < SU; ++u)
            sd[u] = tex_lin<WIDE, PAIR>(T, s.W, s.H, s.D, q[u]) * s.density_scale * s.shadow_density_scale;
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            if (!take[u] || sd[u] < s.cutoff) continue;
            V3 e = s.extinction * sd[u] * s.s_step;
            if (gain) {
                const float den = 1.0f + at[u] * s.gain;
                e = mkv(e.x / den, e.y / den, e.z / den);
            }
            strans = strans * bexp3(e);
            if (sqlen(strans) < s.cutoff) return strans;
        }
    }
    return strans;
}

// a sample's emission (render_kernel :190-203)
template <bool PAIR, bool WIDE>
__device__ __forceinline__ V3 emission_at(const float* __restrict__ scat, const RScene& s, V3 g, float temp) {
    if (!(s.emission_scale > 0.0f)) return mkv(0.0f, 0.0f, 0.0f);
    const float scatter = tex_lin<WIDE, PAIR>(
        scat, s.Ws, s.Hs, s.Ds, texel_at(s.Ws, s.Hs, s.Ds, mkv(g.x / 4.0f, g.y / 4.0f, g.z / 4.0f)));
    return ramp_color(s, temp) * s.emission_scale +
           s.ms_color * scatter * s.ms_scale * smoothstep_f(s.ms_mask_a, s.ms_mask_b, temp);
}

// the camera ray of pixel (i, j): Camera::getRay, normalize(top_left +
// u*horizontal + v*vertical - origin)
__device__ __forceinline__ Ray camera_ray(const RScene& s, int i, int j) {
    const V3 q = s.top_left + (((float)i + 0.5f) / s.res_x) * s.horizontal +
                 (((float)j + 0.5f) / s.res_y) * s.vertical - s.origin;
    const float inv_len = 1.0f / sqrtf(q.x * q.x + q.y * q.y + q.z * q.z);
    return make_ray(s.origin, q * inv_len);
}

// the box of the bricks that are not clear, and a camera ray's part in it
struct Box {
    V3 lo, hi;
};
__device__ __forceinline__ Box brick_box(const unsigned* __restrict__ occ, const Occ& o) {
    const float inf = __int_as_float(0x7f800000);
    const float* b = (const float*)(occ + o.words);
    if (!o.box) return Box{mkv(-inf, -inf, -inf), mkv(inf, inf, inf)};
    return Box{mkv(b[0], b[1], b[2]), mkv(b[3], b[4], b[5])};
}
__device__ __forceinline__ Span camera_span(const Ray& r, const Box& box, const RScene& s, const Occ& o) {
    return box_span(r, box.lo, box.hi,
                    o.margin_dom + o.margin * (fabsf(s.origin.x) + fabsf(s.origin.y) + fabsf(s.origin.z)));
}

// render_kernel: a workgroup of RW waves per RT x RT pixels. Along a ray only
// the transmittance is a chain, and it needs the densities alone; so the tile
// takes up to SPW RW samples of its rays at a time, a thread per sample (a
// wave: SPW samples of every ray, neighbours in space). Each thread has its
// sample's density, emission and exp; each wave runs the chain; the waves draw
// (light, SPW samples) shadow marches from a counter; each thread weights its
// sample's light; and wave 0 adds it up in the reference's order while the
// other starts on the next samples. Rays are cut to the box of the bricks that
// are not clear, and samples in clear bricks read nothing. Bound by the vector
// instructions of the shadow marches. Small tiles spread the few heavy rays of
// a small frame over the chip; each lane walks its ray's chain of SPW RW
// samples, so large tiles do less of it. Which frame gets which:
// render_with.
//
// The kernel over 256^3 at 640x360, three lights, gas in 4% of the pixels: one
// wave per 8x8 tile that marches alone took 9.9 ms, the heaviest tiles last;
// 2x2 tiles 0.70 (one wave: 0.80, four with 64 samples at a time: 1.1; SU = 1:
// 0.75).
constexpr int RW = 2, RTASKS = 10;
template <int RT, bool PAIR, class S, bool WIDE>
__global__ void __launch_bounds__(RW * 64) k_render(const float* __restrict__ T, const float* __restrict__ scat,
                                                    const unsigned* __restrict__ occ, float* __restrict__ fb,
                                                    RScene s, S sc, Occ o, int groups) {
    constexpr int PX = RT * RT;  // pixels of a tile
    constexpr int SPW = 64 / PX; // samples of each ray that a wave takes
    static_assert(3 * PX <= 64, "wave 0 has a lane per channel and pixel");
    __shared__ unsigned bits[OCC_WORDS];
    __shared__ unsigned long long act[2][RW];
    // [group of SPW samples of each ray][lane]
    __shared__ float s_pt[RW][64], s_dT[3][RW][64], s_em[3][RW][64], s_str[RTASKS][3][64];
    __shared__ int next;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int px = lane % PX;
    const int i = blockIdx.x * RT + px % RT, j = blockIdx.y * RT + px / RT;
    for (int t = threadIdx.x; t < o.words; t += RW * 64) bits[t] = occ[t];
    Ray pr = camera_ray(s, i, j);
    bool alive = box_hit(pr, s.dom_min, s.dom_max);
    V3 trans = mkv(1.0f, 1.0f, 1.0f);
    const V3 one = mkv(1.0f, 1.0f, 1.0f);
    const Box box = brick_box(occ, o);
    const Span span = camera_span(pr, box, s, o);
    const float end = span.t1 < pr.t1 ? span.t1 : pr.t1;
    float lumi = 0.0f; // of wave 0's lane (channel, pixel)
    const int rn = SPW * groups, ntask = groups * s.light_count;
    const int k = SPW * wv + lane / PX; // this thread's sample of each round
    float pt0 = pr.t0 + s.dx * 0.5f, pt = pt0;
    for (int t = 0; t < k; ++t) pt += s.p_step;
    __syncthreads();
    // every wave holds the same pt0, trans and alive of a pixel, so all go the same way
    for (int n = 0, par = 0; n < MAX_MARCH && __any(alive && pt0 <= end); n += rn) {
        const float from = pt;
        for (int t = 0; t < rn; ++t) {
            pt += s.p_step;
            pt0 += s.p_step;
        }
        if (!__any(alive && pt0 >= span.t0)) continue; // all in clear bricks
        if (threadIdx.x == 0) next = 0;
        par ^= 1;
        V3 dT = one, emission = mkv(0.0f, 0.0f, 0.0f);
        if (wv < groups) {
            bool on = alive && from <= end && n + k < MAX_MARCH;
            const V3 g = w2g(s, sc, pr.o + from * pr.d);
            const Texel tq = texel_at(s.W, s.H, s.D, g);
            on = on && occupied(bits, o, s, tq);
            if (on) {
                const float temp = tex_lin<WIDE, PAIR>(T, s.W, s.H, s.D, tq);
                const float dens = temp * s.density_scale;
                on = !(dens < s.cutoff);
                if (on) {
                    emission = emission_at<PAIR, WIDE>(scat, s, g, temp);
                    dT = bexp3(s.extinction * dens * s.p_step);
                    s_pt[wv][lane] = from;
                    s_dT[0][wv][lane] = dT.x;
                    s_dT[1][wv][lane] = dT.y;
                    s_dT[2][wv][lane] = dT.z;
                }
            }
            const unsigned long long m = __ballot(on);
            if (lane == 0) act[par][wv] = m;
        }
        __syncthreads();
        unsigned long long any = 0;
        for (int w = 0; w < groups; ++w) any |= act[par][w];
        if (!any) continue;
        // the chain: which samples count, and the transmittance before this thread's
        V3 before = trans;
        unsigned long long use = 0;
        for (int w = 0; w < groups; ++w) {
            const unsigned long long m = act[par][w] >> px;
            if (!m) continue;
#pragma unroll
            for (int u = 0; u < SPW; ++u) {
                if (SPW * w + u == k) before = trans;
                if (!alive || !((m >> (PX * u)) & 1)) continue;
                use |= 1ull << (SPW * w + u);
                const int e = PX * u + px;
                trans = trans * mkv(s_dT[0][w][e], s_dT[1][w][e], s_dT[2][w][e]);
                if (sqlen(trans) < s.cutoff) alive = false;
            }
        }
        for (;;) {
            int t = 0;
            if (lane == 0) t = atomicAdd(&next, 1);
            t = __builtin_amdgcn_readfirstlane(t);
            if (t >= ntask) break;
            const int l = t / groups, w = t - l * groups;
            if (!((use >> (SPW * w + lane / PX)) & 1)) continue;
            const V3 str = shadow_march<2, true, PAIR, S, WIDE>(T, bits, s, sc, o, box.lo, box.hi,
                                                                pr.o + s_pt[w][lane] * pr.d, -1.0f * s.light_dir[l]);
            s_str[t][0][lane] = str.x;
            s_str[t][1][lane] = str.y;
            s_str[t][2][lane] = str.z;
        }
        __syncthreads();
        // this sample's light, weighted; zero (which adds nothing) if it does not count
        if (wv < groups) {
            const bool on = (use >> k) & 1;
            const V3 left = one - dT;
            for (int l = 0; l < s.light_count; ++l) {
                float(*st)[64] = s_str[l * groups + wv];
                const V3 c = s.albedo * mkv(st[0][lane], st[1][lane], st[2][lane]) * before * s.light_illum[l] * left;
                st[0][lane] = on ? c.x : 0.0f;
                st[1][lane] = on ? c.y : 0.0f;
                st[2][lane] = on ? c.z : 0.0f;
            }
            const V3 c = before * emission * left;
            s_em[0][wv][lane] = on ? c.x : 0.0f;
            s_em[1][wv][lane] = on ? c.y : 0.0f;
            s_em[2][wv][lane] = on ? c.z : 0.0f;
        }
        __syncthreads();
        if (wv == 0 && lane < 3 * PX) {
            const int ch = lane / PX;
            for (int w = 0; w < groups; ++w)
#pragma unroll
                for (int u = 0; u < SPW; ++u) {
                    for (int l = 0; l < s.light_count; ++l) lumi = lumi + s_str[l * groups + w][ch][PX * u + px];
                    lumi = lumi + s_em[ch][w][PX * u + px];
                }
        }
    }
    if (wv == 0 && lane < 3 * PX) fb[3 * ((size_t)i + (size_t)(int)s.res_x * j) + lane / PX] = lumi;
}

// A thread per pixel, 8x8 pixels per wave, each marching its ray and its
// samples' shadow rays alone: the least work of all, and with enough waves on
// every CU their unlike lengths even out. The bricks' bits cost more than they
// save here; the box does not.
//
// 1920x1080 over 256^3 (steps of two cells), 2x2 and 4x4 tiles against this:
// full of gas, one light 22 and 9.5 against 8.7 ms; one cell in a thousand,
// three lights 14 and 4.4 against 3.0; gas in 4% of the pixels, one light 3.4
// and 2.1 against 2.1.
constexpr int PT = 8;
template <class S, bool WIDE>
__global__ void __launch_bounds__(PT * PT) k_render_px(const float* __restrict__ T, const float* __restrict__ scat,
                                                       const unsigned* __restrict__ occ, float* __restrict__ fb,
                                                       RScene s, S sc, Occ o) {
    const int i = blockIdx.x * PT + threadIdx.x % PT, j = blockIdx.y * PT + threadIdx.x / PT;
    const Ray pr = camera_ray(s, i, j);
    V3 lumi = mkv(0.0f, 0.0f, 0.0f), trans = mkv(1.0f, 1.0f, 1.0f);
    const V3 one = mkv(1.0f, 1.0f, 1.0f);
    if (Ray r = pr; box_hit(r, s.dom_min, s.dom_max)) {
        const Box box = brick_box(occ, o);
        const Span span = camera_span(r, box, s, o);
        const float end = span.t1 < r.t1 ? span.t1 : r.t1;
        float pt = r.t0 + s.dx * 0.5f;
        int n = 0;
        for (; pt < span.t0 && pt <= end && n < MAX_MARCH; ++n) pt += s.p_step;
        for (; pt <= end && n < MAX_MARCH; pt += s.p_step, ++n) {
            const V3 pos = r.o + pt * r.d;
            const V3 g = w2g(s, sc, pos);
            const float temp = tex_lin<WIDE, false>(T, s.W, s.H, s.D, texel_at(s.W, s.H, s.D, g));
            const float dens = temp * s.density_scale;
            if (dens < s.cutoff) continue;
            const V3 emission = emission_at<false, WIDE>(scat, s, g, temp);
            const V3 dT = bexp3(s.extinction * dens * s.p_step);
            for (int l = 0; l < s.light_count; ++l) {
                const V3 str = shadow_march<1, false, false, S, WIDE>(T, nullptr, s, sc, o, box.lo, box.hi, pos,
                                                                      -1.0f * s.light_dir[l]);
                lumi = lumi + s.albedo * str * trans * s.light_illum[l] * (one - dT);
            }
            lumi = lumi + trans * emission * (one - dT);
            trans = trans * dT;
            if (sqlen(trans) < s.cutoff) break;
        }
    }
    float* p = fb + 3 * ((size_t)i + (size_t)(int)s.res_x * j);
    p[0] = lumi.x;
    p[1] = lumi.y;
    p[2] = lumi.z;
}

inline unsigned nblk(size_t n) { return (unsigned)((n + 255) / 256); }

// zero fill (a kernel, not a memset node, so a captured render replays it)
__global__ void __launch_bounds__(256) k_rnd_zero(float* __restrict__ d, size_t n) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t < n) d[t] = 0.0f;
}

// Scratch of blz_render_noalloc: the two multi-scatter volumes and the
// device frame buffer, in place of the handle's grow-only allocation.
// 32 MiB per device (held until the process ends): a 256^3 grid's volumes
// (2 x 64^3 floats) plus a 1920x1080 frame (6.2M floats) fit. Every call
// on a device shares its copy; calls that overlap on one device race.
constexpr size_t RND_SCRATCH_FLOATS = (size_t)8 << 20;
static __device__ __align__(256) float scratch[RND_SCRATCH_FLOATS];

V3 h3(const float* a) { return V3{a[0], a[1], a[2]}; }
V3 hadd(V3 a, V3 b) { return V3{a.x + b.x, a.y + b.y, a.z + b.z}; }
V3 hsub(V3 a, V3 b) { return V3{a.x - b.x, a.y - b.y, a.z - b.z}; }
V3 hmul(V3 a, float s) { return V3{a.x * s, a.y * s, a.z * s}; }
V3 hmulf(float s, V3 a) { return V3{s * a.x, s * a.y, s * a.z}; }

} // namespace

// get_buf(n, &p): n floats of device scratch for the scatter volumes and the
// frame, or an error
template <class GetBuf>
static int render_with(Solver& s, const blz_render_settings& r, float* host_rgb, GetBuf get_buf) {
    if (r.width <= 0 || r.height <= 0 || r.width % RES_STEP || r.height % RES_STEP || r.width > 16384 || r.height > 16384) {
        set_error("render size must be positive multiples of 8 (at most 16384)");
        return BLZ_E_INVALID;
    }
    if (!(r.p_step > 0.0f) || !(r.s_step > 0.0f) || r.light_count < 0 || r.light_count > BLZ_MAX_LIGHTS ||
        r.ramp_size < 1 || r.ramp_size > BLZ_MAX_RAMP || r.ms_blur_iter < 0) {
        set_error("invalid render settings (steps > 0, 0..10 lights, 1..10 ramp keys, blur iterations >= 0)");
        return BLZ_E_INVALID;
    }
    RScene sc{};
    // Camera (src/Camera.h:42-53), host FP32 in the same order
    {
        const V3 o = h3(r.cam_trans), u = h3(r.cam_u), v = h3(r.cam_v), w = h3(r.cam_w);
        const float aspect = (float)r.width / (float)r.height;
        const float half_w = 0.5f * r.cam_aperture;
        const float half_h = half_w / aspect;
        sc.origin = o;
        sc.top_left = hadd(hsub(hsub(o, hmulf(r.cam_focal, w)), hmulf(half_w, u)), hmulf(half_h, v));
        sc.horizontal = hmulf(2.0f * half_w, u);
        sc.vertical = hmulf(-2.0f * half_h, v);
        sc.res_x = (float)(unsigned)r.width;
        sc.res_y = (float)(unsigned)r.height;
    }
    sc.dom_min = V3{s.s.domain_min[0], s.s.domain_min[1], s.s.domain_min[2]};
    sc.dom_max = V3{s.s.domain_max[0], s.s.domain_max[1], s.s.domain_max[2]};
    sc.dom_size = hsub(sc.dom_max, sc.dom_min);
    sc.dx = s.dx;
    sc.W = s.W;
    sc.H = s.H;
    sc.D = s.D;
    sc.Ws = s.W / 4;
    sc.Hs = s.H / 4;
    sc.Ds = s.D / 4;
    sc.p_step = r.p_step;
    sc.s_step = r.s_step;
    sc.cutoff = r.cutoff;
    sc.density_scale = r.density_scale;
    sc.shadow_density_scale = r.shadow_density_scale;
    sc.gain = r.gain;
    sc.emission_scale = r.emission_scale;
    // Shader (src/Shader.h:52-63)
    {
        const V3 col = h3(r.volume_color), sca = h3(r.scattering);
        const V3 den = V3{sca.x + r.absorption, sca.y + r.absorption, sca.z + r.absorption};
        const V3 num = V3{col.x * sca.x, col.y * sca.y, col.z * sca.z};
        sc.albedo = V3{num.x / den.x, num.y / den.y, num.z / den.z};
        sc.extinction = hmul(V3{sca.x + r.absorption, sca.y + r.absorption, sca.z + r.absorption}, -1.0f);
    }
    sc.ramp_size = r.ramp_size;
    sc.ramp_in = r.temp_range[0];
    sc.ramp_out = r.temp_range[1];
    for (int q = 0; q < r.ramp_size; ++q) {
        sc.ramp_keys[q] = r.ramp_keys[q];
        sc.ramp_colors[q] = h3(r.ramp_colors[q]);
    }
    sc.ms_color = h3(r.ms_color);
    sc.ms_scale = r.ms_scale;
    sc.ms_mask_a = r.ms_mask[0];
    sc.ms_mask_b = r.ms_mask[1];
    // Light (src/Light.h:43-50): colour * intensity * 2^exposure
    sc.light_count = r.light_count;
    for (int l = 0; l < r.light_count; ++l) {
        sc.light_dir[l] = h3(r.light_dir[l]);
        sc.light_illum[l] = hmul(hmul(h3(r.light_color[l]), r.light_intensity[l]), std::pow(2.0f, r.light_exposure[l]));
    }
    // buffers: two scatter volumes (at least one cell each) and the frame
    const size_t ns = (size_t)std::max(1, sc.Ws) * std::max(1, sc.Hs) * std::max(1, sc.Ds);
    const size_t nf = (size_t)r.width * r.height * 3;
    float* buf = nullptr;
    if (int e = get_buf(2 * ns + nf, &buf)) return e;
    float* scat[2] = {buf, buf + ns};
    float* fb = buf + 2 * ns;
    const float* T = s.f[F_T].front();
    const bool have_scatter = sc.Ws > 0 && sc.Hs > 0 && sc.Ds > 0;
    if (!have_scatter) {
        sc.Ws = sc.Hs = sc.Ds = 1;
    }
    if (r.ms_scale > 0.0f && have_scatter) {
        hipLaunchKernelGGL(k_rnd_scatter, dim3(nblk(ns)), dim3(256), 0, s.stream, T, s.W, s.H, sc.Ws, sc.Hs, sc.Ds,
                           r.temp_range[0], scat[0]);
        // blur weights: filter / its sum (src/RenderEngine.cu:33-47, :262-276)
        static const float filt[27] = {0, 1, 0, 1, 2, 1, 0, 1, 0, 1, 2, 1, 2, 4, 2, 1, 2, 1, 0, 1, 0, 1, 2, 1, 0, 1, 0};
        float sum = 0.0f;
        for (int q = 0; q < 27; ++q) sum += filt[q];
        BlurW bw;
        for (int q = 0; q < 27; ++q) bw.w[q] = filt[q] / sum;
        for (int it = 0; it < r.ms_blur_iter; ++it) {
            hipLaunchKernelGGL(k_rnd_blur, dim3(nblk(ns)), dim3(256), 0, s.stream, scat[0], scat[1], sc.Ws, sc.Hs,
                               sc.Ds, bw);
            std::swap(scat[0], scat[1]);
        }
    } else {
        hipLaunchKernelGGL(k_rnd_zero, dim3(nblk(ns)), dim3(256), 0, s.stream, scat[0], ns);
    }
    // bricks of empty space, kept in the scatter volume that is free now: it
    // has a float per 4x4x4 cells, the bricks a bit, up to 8 times as many
    Occ o{};
    int nbricks = 0;
    for (o.sh = 2;; ++o.sh) {
        const int E = 1 << o.sh;
        o.nx = (s.W + E - 1) / E;
        o.ny = (s.H + E - 1) / E;
        o.nz = (s.D + E - 1) / E;
        const long long nb = (long long)o.nx * o.ny * o.nz;
        if (nb <= OCC_WORDS * 32) {
            nbricks = (int)nb;
            break;
        }
    }
    o.words = (nbricks + 31) / 32;
    // the filter, density and product roundings stay within 1e-5
    o.lim = r.cutoff / (std::fabs(r.density_scale) * std::max(1.0f, std::fabs(r.shadow_density_scale))) * 0.99999f;
    if (!(o.lim > 1e-30f)) o.lim = -1.0f;
    unsigned* occ = (unsigned*)scat[1];
    hipLaunchKernelGGL(k_rnd_occ, dim3((unsigned)o.words), dim3(256), 0, s.stream, T, s.W, s.H, s.D, nbricks, o, occ);
    // their box, where the volume has room for it (grids down to 12^3 have)
    o.box = ns >= (size_t)o.words + 6;
    float reach = 0.0f;
    for (int a = 0; a < 3; ++a)
        reach = std::max(reach, std::max(std::fabs(s.s.domain_min[a]), std::fabs(s.s.domain_max[a])));
    o.margin = 1e-5f;
    o.margin_dom = 2.0f * s.dx + 1e-5f * reach;
    if (o.box)
        hipLaunchKernelGGL(k_rnd_box, dim3(1), dim3(1024), 0, s.stream, occ, o, sc.dom_min, sc.dom_size, s.dx);
    // groups of SPW samples per round: one per wave, fewer where the shadow
    // marches of more than RTASKS / RW lights need the room
    const int groups = std::min(RW, RTASKS / std::max(1, r.light_count));
    // The tile by the frame's pixels and lights. ms of a call with 2x2 tiles /
    // 4x4 tiles / a thread per pixel over 256^3, with gas in 4% of the pixels,
    // full of gas, and with one cell in a thousand:
    //   64x64, 3 lights      0.51 / 0.76 / 5.0   1.8 / 3.0 / 25    1.3 / 1.7 / 11
    //   320x184, 3 lights    0.55 / 0.82 / 4.3   6.9 / 10 / 24     2.5 / 1.8 / 12
    //   320x184, none        0.27 / 0.25 / 0.33  0.47 / 0.38 / 0.46  0.39 / 0.32 / 0.46
    //   640x360, 3 lights    1.03 / 0.94 / 3.8   21 / 12 / 24      4.5 / 2.2 / 6.1
    //   640x360, none        0.48 / 0.40 / 0.44  1.2 / 0.71 / 0.64 0.84 / 0.57 / 0.55
    //   1280x720, 3 lights   3.0 / 2.1 / 5.3     72 / 41 / 58      13 / 4.2 / 4.8
    //   1280x720, 1 light    1.6 / 1.1 / 1.3     10 / 4.4 / 4.7    4.1 / 1.7 / 1.4
    //   1920x1080, 3 lights  4.1 / 2.5 / 3.0     54 / 26 / 28      14 / 4.4 / 3.0
    // Against the first build (a wave per 8x8 pixels alone) this rule took 0.04
    // to 1.04 of the time on eleven volumes of 32^3 to 256^3 at 17 frame sizes;
    // 2x2 tiles for all took up to 4.5 times as long (1920x1080 of the last).
    const long long pixels = (long long)r.width * r.height;
    const int tile = pixels >= 200000 + 500000ll * r.light_count ? PT
                     : pixels >= (r.light_count ? 200000 : 30000) ? 4 : 2;
    const dim3 grid((unsigned)(r.width / tile), (unsigned)(r.height / tile));
    const bool wide = (size_t)s.W * s.H * s.D >= ((size_t)1 << 30);
    auto launch = [&](auto scale, auto w) {
        using S = decltype(scale);
        constexpr bool WIDE = decltype(w)::value;
        if (tile == PT)
            hipLaunchKernelGGL((k_render_px<S, WIDE>), grid, dim3(PT * PT), 0, s.stream, T, scat[0], occ, fb, sc,
                               scale, o);
        else if (tile == 4)
            hipLaunchKernelGGL((k_render<4, false, S, WIDE>), grid, dim3(RW * 64), 0, s.stream, T, scat[0], occ, fb,
                               sc, scale, o, groups);
        else
            hipLaunchKernelGGL((k_render<2, true, S, WIDE>), grid, dim3(RW * 64), 0, s.stream, T, scat[0], occ, fb,
                               sc, scale, o, groups);
    };
    float inv = 0.0f;
    if (dx_pow2(s.dx, &inv)) {
        if (wide) launch(MulDx{inv}, std::true_type{});
        else launch(MulDx{inv}, std::false_type{});
    } else {
        if (wide) launch(DivDx{s.dx}, std::true_type{});
        else launch(DivDx{s.dx}, std::false_type{});
    }
    BLZ_HIP(hipGetLastError());
    BLZ_HIP(hipMemcpyAsync(host_rgb, fb, nf * sizeof(float), hipMemcpyDeviceToHost, s.stream));
    BLZ_HIP(hipStreamSynchronize(s.stream));
    return BLZ_OK;
}

int render_frame(Solver& s, const blz_render_settings& r, float* host_rgb) {
    return render_with(s, r, host_rgb, [&s](size_t n, float** out) -> int {
        const size_t bytes = n * sizeof(float);
        if (bytes > s.rnd_bytes) {
            if (s.rnd_buf) BLZ_HIP(hipFree(s.rnd_buf));
            s.rnd_buf = nullptr;
            s.rnd_bytes = 0;
            if (hipMalloc(&s.rnd_buf, bytes) != hipSuccess) {
                set_error("hipMalloc failed for render buffers");
                return BLZ_E_NOMEM;
            }
            s.rnd_bytes = bytes;
        }
        *out = s.rnd_buf;
        return BLZ_OK;
    });
}

// Device address of `scratch` on each device, looked up once per device
// (with that device current) by hipGetSymbolAddress; host code uses these
// addresses, never the array's name (a host-side stand-in).
static std::mutex g_scratch_mu;
static float* g_scratch_dev[64] = {};

static int scratch_on(int device, float** out) {
    if (device < 0 || device >= 64) {
        set_error("blz_render_noalloc: device index out of range");
        return BLZ_E_INVALID;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[device]) {
        int cur = -1;
        BLZ_HIP(hipGetDevice(&cur));
        if (cur != device) {
            set_error("blz_render_noalloc: the solver's device must be current");
            return BLZ_E_INVALID;
        }
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
            return BLZ_E_HIP;
        }
        g_scratch_dev[device] = (float*)p;
    }
    *out = g_scratch_dev[device];
    return BLZ_OK;
}

int render_frame_noalloc(Solver& s, const blz_render_settings& r, float* host_rgb) {
    float* base = nullptr;
    if (int e = scratch_on(s.device, &base)) return e;
    return render_with(s, r, host_rgb, [base](size_t n, float** out) -> int {
        if (n > RND_SCRATCH_FLOATS) {
            set_error("blz_render_noalloc: scatter volumes plus frame need " + std::to_string(n) +
                      " floats, above the scratch limit of " + std::to_string(RND_SCRATCH_FLOATS));
            return BLZ_E_INVALID;
        }
        *out = base;
        return BLZ_OK;
    });
}

} // namespace blz
