// Device-side core of the MI355X path tracer (gfx950, wave64).
//
// Estimator semantics follow the reference kernel (src/tfg-pathtracer/):
//   camera ray          kernel.cu:260-337      hit attributes   Tri.hpp:38-160
//   material fetch      kernel.cu:54-119       Disney           Disney.hpp:41-253
//   sampling            Sampling.hpp:10-54     point light NEE  kernel.cu:175-205
//   HDRI NEE            kernel.cu:210-258, HDRI.hpp:130-162, Texture.hpp:95-207
//   MIS combine         kernel.cu:339-358      path loop        kernel.cu:369-481
// Defined behaviour where the reference is undefined or replaced:
//   * RNG: Philox4x32-10 (Salmon et al., SC'11) keyed by (seed, scene) with
//     counter (pixel, sample, block, 0); uniforms in [0,1) from the top 24 bits.
//   * The HDRI NEE pdf is computed whether or not the shadow ray is blocked
//     (the reference leaves it uninitialised when blocked, kernel.cu:248/254).
//   * Point-light visibility: blocked iff some triangle is hit at
//     t < dist - 0.001 from the offset origin (the reference compares the
//     closest hit's smooth-shading position, kernel.cu:193-197; the two differ
//     only for an occluder within the shading offset of the light).
//   * The HDRI pixel is binarySearch(cdf, r1) bit for bit, found through a
//     guide table (hdri_table.hpp); the point light uses the same r1.
//   * acos arguments are clamped to [-1, 1] for the environment lookup.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "child_order.hpp"
#include "hdri_table.hpp"
#include "work_turns.hpp"

namespace eleven {
namespace dev {

#define EL_PI 3.14159265358979323846f

// Traversal variants (compile-time).
#ifndef EL_LEAF_PIPE   // leaf triangles: next record loaded before the current one is tested
#define EL_LEAF_PIPE 1
#endif

// ---------------------------------------------------------------- vectors --
struct v3 {
    float x, y, z;
};
__device__ __forceinline__ v3 mk(float x, float y, float z) { return v3{x, y, z}; }
__device__ __forceinline__ v3 operator+(v3 a, v3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ v3 operator-(v3 a, v3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ v3 operator*(v3 a, v3 b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ v3 operator*(v3 a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ v3 operator*(float s, v3 a) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ v3 operator/(v3 a, float s) { return mk(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ v3 operator/(v3 a, v3 b) { return mk(a.x / b.x, a.y / b.y, a.z / b.z); }
__device__ __forceinline__ float dot(v3 a, v3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
// Vector.hpp:229-231 form (y component negated difference).
__device__ __forceinline__ v3 cross(v3 a, v3 b) {
    return mk(a.y * b.z - a.z * b.y, -(a.x * b.z - a.z * b.x), a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ float length(v3 a) { return sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }
// Vector.hpp:173-176: zero vectors pass through unchanged.
__device__ __forceinline__ v3 normalized(v3 a) {
    float l = length(a);
    if (l == 0.f) return a;
    return a / l;
}
// Hardware reciprocal and square roots (v_rcp_f32, v_sqrt_f32, v_rsq_f32:
// 1 ulp) for value arithmetic only -- BRDF and pdf values, MIS weights,
// throughput.  Every quantity that decides a direction, an index or a branch
// of the path (sampling, bases, ray and shadow directions, texel and HDRI
// index math, intersection) keeps IEEE division and square root.
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
// normalized() for value arithmetic: zero vectors pass through unchanged.
__device__ __forceinline__ v3 fnormalized(v3 a) {
    float l2 = dot(a, a);
    return l2 == 0.f ? a : a * __builtin_amdgcn_rsqf(l2);
}
__device__ __forceinline__ float lerpf(float a, float b, float c) { return a + c * (b - a); }  // FAST_LERP
__device__ __forceinline__ v3 lerp3(v3 a, v3 b, float c) {
    return mk(lerpf(a.x, b.x, c), lerpf(a.y, b.y, c), lerpf(a.z, b.z, c));
}
__device__ __forceinline__ float clampf(float a, float b, float c) { return a < b ? b : (a > c ? c : a); }
__device__ __forceinline__ float minf(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float maxf(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ v3 ld3(const float* p) { return mk(p[0], p[1], p[2]); }

// ------------------------------------------------------------------- RNG --
// Philox4x32-10, Salmon, Moraes, Dror, Shaw: "Parallel random numbers: as
// easy as 1, 2, 3", SC'11.  Multipliers and Weyl key increments as published.
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        // one 32 x 32 -> 64-bit multiply per product (v_mad_u64_u32) instead
        // of separate high and low multiplies
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x, p1 = (uint64_t)0xCD9E8D57u * c.z;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        c = make_uint4(hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0);
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c;
}
__device__ __forceinline__ float u01(uint32_t u) { return (float)(u >> 8) * (1.0f / 16777216.0f); }

// Random numbers of one path, one Philox block per use:
//   block 0      camera r1..r4          block 1 .x   camera r5
//   block 2 + b  bounce b: DisneySample r1, r2, r3 (.x .y .z), shade r1 (.w)
// (shade's r2 and r3 are never read on the reference's HDRI-IS path,
// kernel.cu:234-257, so they are not drawn).
struct PathRng {
    uint32_t k0, k1, pixel, sample, scene;
    __device__ __forceinline__ uint4 block(uint32_t b) const {
        return philox4x32_10(make_uint4(pixel, sample, b, scene), k0, k1);
    }
};

// ----------------------------------------------------------- scene layout --
// Texel storage: kTexF32 = RGB FP32 in the float pool (offset = first
// float); kTexLdr + k = one 32-bit word per texel in the 8-bit pool (offset =
// first texel), bytes R, G, B indexing the loader's byte -> value table k
// (0 sRGB, 1 linear): the same FP32 values in a third of the bytes.
constexpr int32_t kTexF32 = 0, kTexLdr = 1;
struct DevTex {
    int32_t w, h;
    float xTile, yTile, xOffset, yOffset;
    int32_t filter;
    int32_t format;
    uint64_t offset;
};

struct DevMaterial {
    int32_t albedoTex, emissionTex, roughnessTex, metallicTex, normalTex, pad0;
    float albedo[3], emission[3];
    float roughness, metallic, clearcoatGloss, clearcoat, anisotropic, eta, transmission, specular,
        specularTint, sheenTint, subsurface, sheen;
    float roughnessEff, metallicEff;   // powf(roughness, 2.2f), powf(metallic, 2.2f) (kernel.cu:113-114)
    float pad1[2];
};

struct DevCamera {
    uint32_t xRes, yRes;
    float focalLength, sensorWidth, sensorHeight, aperture, focusDistance;
    float cosRot[3], sinRot[3];   // cos/sin of the Euler angles in radians, per camera
    float pos[3];
    int32_t bokeh;
};

// Shading record per original triangle: 8 float4 = 128 B, one cache line
// per hit: [0..8] v0 v1 v2 | [9..17] n0 n1 n2 | [18..23] uv0 uv1 uv2 (x,y) |
// [24] material id (int bits) | [25] tangentsSign | [26..31] unused.
// The corner tangents, needed only for normal maps and the tangent AOVs,
// are a separate stream of 3 float4 per triangle: t0 t1 t2 | unused.
constexpr int kShadeWords = 8, kShadeFloats = 4 * kShadeWords;
constexpr int kTanWords = 3, kTanFloats = 4 * kTanWords;

struct DevScene {
    const void* nodes;             // WideNode<W>[]
    const float4* tris;            // 3 float4 per leaf-order triangle
    const float4* shade;           // kShadeWords per original triangle
    const float4* tangents;        // kTanWords per original triangle
    const DevMaterial* mats;
    const DevTex* texs;
    const float* texels;           // pool of all textures (RGB FP32)
    const uint32_t* texels8;       // 8-bit copies of the LDR textures (DevTex::format)
    const float* texLut;           // 2 x 256 byte -> value tables (sRGB, linear)
    const float* lights;           // 6 floats per light: position, radiance
    const float* envCdf;           // HDRI CDF (L + 1)
    const int32_t* envGuide;       // guide table (2^envLog2G + 1 pairs)
    const int32_t* envMap;         // per interval: open-interval and tie results
    const uint32_t* envBad;        // 2^16-bit map: random-number buckets whose HDRI pdf may be 0 or inf
    const float4* envTab;          // 2 per HDRI pixel k: envSampleAt(k) (direction + pdf, value)
    DevTex env;                    // env texture (texels in the pool)
    float envRadianceSum;
    int32_t envLog2G;
    int32_t nLights;
    int32_t nTris;
    int32_t width;                 // BVH width (4 or 8)
    int32_t gcap;                  // global stack entries per thread (a stack per lane)
    int32_t quads;                 // BVH4 within kQuadStack: short queues give a ray to a quad of lanes
    float slabUnit;                // factor of the slab distances' scale (slabUnitOf)
    DevCamera cam;
    // batches only: the scene's RNG key and accumulation buffers
    uint32_t seedLo, seedHi;
    float4* accum;
    uint32_t* counts;
};

// --------------------------------------------------------------- textures --
struct TexPools {
    const float* f32;
    const uint32_t* u8;
    const float* lut;   // the byte -> value tables (global or an LDS copy)
};
__device__ __forceinline__ TexPools texPools(const DevScene& s, const float* lut = nullptr) {
    return TexPools{s.texels, s.texels8, lut ? lut : s.texLut};
}
// Texture::getValueFromCoordinates (Texture.hpp:95-106).
__device__ __forceinline__ v3 texel(const TexPools& P, const DevTex& t, int x, int y) {
    x = (int)(t.xTile * (x + t.xOffset * t.w)) % t.w;
    y = (int)(t.yTile * (y + t.yOffset * t.h)) % t.h;
    // Out-of-range coordinates (negative uv) are undefined in the reference;
    // wrap them into the texture instead of reading out of bounds.
    if (x < 0) x += t.w;
    if (y < 0) y += t.h;
    const uint64_t i = (uint64_t)y * t.w + x;
    if (t.format == kTexF32) return ld3(P.f32 + t.offset + 3 * i);
    const uint32_t v = P.u8[t.offset + i];
    const float* L = P.lut + 256 * (t.format - kTexLdr);
    return mk(L[v & 255u], L[(v >> 8) & 255u], L[(v >> 16) & 255u]);
}
// Index (texel units, within the texture) that texel() reads for (x, y).
__device__ __forceinline__ uint32_t texelIndex(const DevTex& t, int x, int y) {
    x = (int)(t.xTile * (x + t.xOffset * t.w)) % t.w;
    y = (int)(t.yTile * (y + t.yOffset * t.h)) % t.h;
    if (x < 0) x += t.w;
    if (y < 0) y += t.h;
    return (uint32_t)y * (uint32_t)t.w + (uint32_t)x;
}
__device__ __forceinline__ v3 texUV(const TexPools& pool, const DevTex& t, float u, float v) {
    return texel(pool, t, (int)(u * t.w), (int)(v * t.h));
}
// Texture.hpp:114-135
__device__ __forceinline__ v3 texBilinear(const TexPools& pool, const DevTex& t, float u, float v) {
    float x = u * t.w, y = v * t.h;
    float t1x = floorf(x), t1y = floorf(y);
    float t2x = t1x + 1, t2y = t1y + 1;
    float a = (x - t1x) / (t2x - t1x), b = (y - t1y) / (t2y - t1y);
    v3 v1 = texel(pool, t, (int)t1x, (int)t1y), v2 = texel(pool, t, (int)t2x, (int)t1y);
    v3 v3_ = texel(pool, t, (int)t1x, (int)t2y), v4 = texel(pool, t, (int)t2x, (int)t2y);
    return lerp3(lerp3(v1, v2, a), lerp3(v3_, v4, a), b);
}
__device__ __forceinline__ v3 texFiltered(const TexPools& pool, const DevTex& t, float u, float v) {
    return t.filter == 1 ? texBilinear(pool, t, u, v) : texUV(pool, t, u, v);
}

// Texture::sphericalMapping (Texture.hpp:144-156) for a unit sphere at origin.
__device__ __forceinline__ void sphericalMapping(v3 p, float& u, float& v) {
    float theta = acosf(clampf(-p.y, -1.f, 1.f));
    float phi = atan2f(-p.z, p.x) + EL_PI;
    u = phi / (2 * EL_PI);
    v = theta / EL_PI;
    // limitUV (Math.hpp:38-41)
    u += -(float)(u > 1) + -(float)(u < 0);
    v += -(float)(v > 1) + -(float)(v < 0);
}

// -------------------------------------------------------------- sampling --
__device__ __forceinline__ v3 cosineSampleHemisphere(float u1, float u2) {   // Sampling.hpp:31-41
    float r = sqrtf(u1);
    float phi = 2.0f * EL_PI * u2;
    v3 d;
    d.x = r * cosf(phi);
    d.y = r * sinf(phi);
    d.z = sqrtf(maxf(0.0f, 1.0f - d.x * d.x - d.y * d.y));
    return d;
}
__device__ __forceinline__ v3 importanceSampleGGX(float rgh, float r1, float r2) {   // Sampling.hpp:43-54
    float a = maxf(0.001f, rgh);
    float phi = r1 * EL_PI * 2;
    float cosTheta = sqrtf((1.0f - r2) / (1.0f + (a * a - 1.0f) * r2));
    float sinTheta = clampf(sqrtf(1.0f - (cosTheta * cosTheta)), 0.0f, 1.0f);
    return mk(sinTheta * cosf(phi), sinTheta * sinf(phi), cosTheta);
}
__device__ __forceinline__ void uniformCircleSampling(float u1, float u2, float u3, float& x, float& y) {
    float t = 2 * EL_PI * u1;
    float u = u2 + u3;
    float r = u > 1 ? 2 - u : u;
    x = r * cosf(t);
    y = r * sinf(t);
}

// ---------------------------------------------------------------- Disney --
struct HitData {
    float metallic, roughness, clearcoatGloss, clearcoat, anisotropic, eta, transmission, specular,
        specularTint, sheenTint, subsurface, sheen;
    v3 emission, albedo, normal;
};

__device__ __forceinline__ void createBasis(v3 n, v3& t, v3& b) {   // Disney.hpp:41-45
    t = normalized(cross(mk(0, 1, 0), n));
    b = normalized(cross(n, t));
}
__device__ __forceinline__ float schlickFresnel(float u) {
    float m = clampf(1.0f - u, 0.0f, 1.0f);
    float m2 = m * m;
    return m2 * m2 * m;
}
// The microfacet terms below are value arithmetic (frcp, fsqrt).
__device__ __forceinline__ float GTR1(float NDotH, float a) {
    if (a >= 1.0f) return 1.0f / EL_PI;
    float a2 = a * a;
    float t = 1.0f + (a2 - 1.0f) * NDotH * NDotH;
    return (a2 - 1.0f) * frcp(EL_PI * logf(a2) * t);
}
// 1 / (pi ax ay c^2) with rax = 1 / ax, ray = 1 / ay, piAxAy = pi * ax * ay.
__device__ __forceinline__ float GTR2_aniso(float NDotH, float HDotX, float HDotY, float rax, float ray,
                                            float piAxAy) {
    float a = HDotX * rax, b = HDotY * ray;
    float c = a * a + b * b + NDotH * NDotH;
    return frcp(piAxAy * c * c);
}
__device__ __forceinline__ float smithG_GGX(float NDotV, float alphaG) {
    float a = alphaG * alphaG, b = NDotV * NDotV;
    return frcp(NDotV + fsqrt(a + b - a * b));
}
__device__ __forceinline__ float smithG_GGX_aniso(float NDotV, float VDotX, float VDotY, float ax, float ay) {
    float a = VDotX * ax, b = VDotY * ay, c = NDotV;
    return frcp(NDotV + fsqrt(a * a + b * b + c * c));
}

// Anisotropic GGX widths of Disney.hpp:128-130 / 213-215.
struct GgxWidths {
    float ax, ay, rax, ray, piAxAy;
};
__device__ __forceinline__ GgxWidths ggxWidths(const HitData& h) {
    GgxWidths g;
    float aspect = fsqrt(1.0f - h.anisotropic * 0.9f);
    float ra = frcp(aspect);
    g.ax = maxf(0.001f, h.roughness * ra);
    g.ay = maxf(0.001f, h.roughness * aspect);
    g.rax = frcp(g.ax);
    g.ray = frcp(g.ay);
    g.piAxAy = EL_PI * g.ax * g.ay;
    return g;
}

// Disney.hpp:108-147 given the half vector H = normalize(L + V) and
// Ds = GTR2_aniso(N.H, H.T, H.B).  `dir` is the incoming ray direction
// (V = -dir).  With clearcoat == 0 the GTR1/GTR2 mix weight is exactly 1.
__device__ __forceinline__ float disneyPdfH(const HitData& h, v3 L, v3 H, float NDotH, float Ds) {
    v3 N = h.normal;
    if (dot(N, L) <= 0.0f) return 1.0f;
    float diffuseRatio = 0.5f * (1.0f - h.metallic);
    float specularRatio = 1.0f - diffuseRatio;
    float pdfGTR2 = Ds * NDotH;
    float mix = pdfGTR2;
    if (h.clearcoat != 0.0f) {
        float clearcoatAlpha = lerpf(0.1f, 0.001f, h.clearcoatGloss);
        float pdfGTR1 = GTR1(NDotH, clearcoatAlpha) * NDotH;
        mix = lerpf(pdfGTR1, pdfGTR2, frcp(1.0f + h.clearcoat));
    }
    float pdfSpec = mix * frcp(4.0f * fabsf(dot(L, H)));
    float pdfDiff = fabsf(dot(L, N)) * (1.0f / EL_PI);
    return diffuseRatio * pdfDiff + specularRatio * pdfSpec;
}
__device__ __forceinline__ float disneyPdf(v3 dir, const HitData& h, v3 L) {
    v3 V = dir * -1.0f;
    v3 H = fnormalized(L + V);
    v3 T, B;
    createBasis(h.normal, T, B);
    float NDotH = fabsf(dot(h.normal, H));
    GgxWidths g = ggxWidths(h);
    return disneyPdfH(h, L, H, NDotH, GTR2_aniso(NDotH, dot(H, T), dot(H, B), g.rax, g.ray, g.piAxAy));
}

// Disney.hpp:150-177
__device__ __forceinline__ v3 disneySample(v3 dir, const HitData& h, float r1, float r2, float r3) {
    v3 N = h.normal;
    v3 V = dir * -1.0f;
    v3 T, B;
    createBasis(h.normal, T, B);
    float diffuseRatio = 0.5f * (1.0f - h.metallic);
    if (r3 < diffuseRatio) {
        v3 H = cosineSampleHemisphere(r1, r2);
        return T * H.x + B * H.y + N * H.z;
    }
    v3 H = importanceSampleGGX(h.roughness, r1, r2);
    H = T * H.x + B * H.y + N * H.z;
    v3 v1 = V * -1.0f;
    return v1 - 2 * dot(v1, H) * H;   // reflect (Vector.hpp:218-220)
}

// Disney.hpp:179-253; with PDF also disneyPdf(dir, h, L) into `pdf`, which
// shares the half vector and the GTR2 term.  The clearcoat lobe is skipped
// when its weight is 0 (it is finite, so it adds exactly 0).
template <bool PDF>
__device__ __forceinline__ v3 disneyEvalT(v3 dir, const HitData& h, v3 L, float& pdf) {
    v3 V = dir * -1.0f;
    v3 T, B;
    createBasis(h.normal, T, B);
    v3 H = fnormalized(L + V);
    float NDotL = fabsf(dot(h.normal, L));
    float NDotV = fabsf(dot(h.normal, V));
    float NDotH = fabsf(dot(h.normal, H));
    float LDotH = fabsf(dot(L, H));
    GgxWidths g = ggxWidths(h);
    float Ds = GTR2_aniso(NDotH, dot(H, T), dot(H, B), g.rax, g.ray, g.piAxAy);
    if (PDF) pdf = disneyPdfH(h, L, H, NDotH, Ds);
    v3 brdf = mk(0, 0, 0);
    if (h.transmission < 1.0f && dot(h.normal, L) > 0.0f && dot(h.normal, V) > 0.0f) {
        v3 Cdlin = h.albedo;
        float Cdlum = 0.3f * Cdlin.x + 0.6f * Cdlin.y + 0.1f * Cdlin.z;
        v3 Ctint = Cdlum > 0.0f ? Cdlin * frcp(Cdlum) : mk(1, 1, 1);
        v3 Cspec0 = lerp3(h.specular * 0.08f * lerp3(mk(1, 1, 1), Ctint, h.specularTint), Cdlin, h.metallic);
        v3 Csheen = lerp3(mk(1, 1, 1), Ctint, h.sheenTint);
        float FL = schlickFresnel(NDotL), FV = schlickFresnel(NDotV);
        float Fd90 = 0.5f + 2.0f * LDotH * LDotH * h.roughness;
        float Fd = lerpf(1.0f, Fd90, FL) * lerpf(1.0f, Fd90, FV);
        float Fss90 = LDotH * LDotH * h.roughness;
        float Fss = lerpf(1.0f, Fss90, FL) * lerpf(1.0f, Fss90, FV);
        float ss = 1.25f * (Fss * (frcp(NDotL + NDotV) - 0.5f) + 0.5f);
        float FH = schlickFresnel(LDotH);
        v3 Fs = lerp3(Cspec0, mk(1, 1, 1), FH);
        float Gs = smithG_GGX_aniso(NDotL, dot(L, T), dot(L, B), g.ax, g.ay);
        Gs *= smithG_GGX_aniso(NDotV, dot(V, T), dot(V, B), g.ax, g.ay);
        v3 Fsheen = FH * h.sheen * Csheen;
        brdf = ((1.0f / EL_PI) * lerpf(Fd, ss, h.subsurface) * Cdlin + Fsheen) * (1.0f - h.metallic) + Gs * Fs * Ds;
        if (h.clearcoat != 0.0f) {
            float Dr = GTR1(NDotH, lerpf(0.1f, 0.001f, h.clearcoatGloss));
            float Fr = lerpf(0.04f, 1.0f, FH);
            float Gr = smithG_GGX(NDotL, 0.25f) * smithG_GGX(NDotV, 0.25f);
            brdf = brdf + mk(1, 1, 1) * (0.25f * h.clearcoat * Gr * Fr * Dr);
        }
    }
    return brdf;
}
__device__ __forceinline__ v3 disneyEval(v3 dir, const HitData& h, v3 L) {
    float unused;
    return disneyEvalT<false>(dir, h, L, unused);
}
__device__ __forceinline__ v3 disneyEvalPdf(v3 dir, const HitData& h, v3 L, float& pdf) {
    return disneyEvalT<true>(dir, h, L, pdf);
}

// d disneyEval / d (albedo.x, albedo.y, albedo.z, roughness, metallic,
// specular) of HitData (effective values, after generateHitData's pow 2.2),
// written out analytically from the expression above; used by the adjoint.
__device__ __forceinline__ void disneyEvalGrad(v3 dir, const HitData& h, v3 L, v3 (&df)[6]) {
#pragma unroll
    for (int k = 0; k < 6; k++) df[k] = mk(0, 0, 0);
    v3 V = dir * -1.0f;
    v3 T, B;
    createBasis(h.normal, T, B);
    v3 H = normalized(L + V);
    float NDotL = fabsf(dot(h.normal, L));
    float NDotV = fabsf(dot(h.normal, V));
    float NDotH = fabsf(dot(h.normal, H));
    float LDotH = fabsf(dot(L, H));
    if (!(h.transmission < 1.0f && dot(h.normal, L) > 0.0f && dot(h.normal, V) > 0.0f)) return;
    const v3 C = h.albedo;
    const float wl[3] = {0.3f, 0.6f, 0.1f};
    const float lum = wl[0] * C.x + wl[1] * C.y + wl[2] * C.z;
    const v3 Ctint = lum > 0.0f ? C / lum : mk(1, 1, 1);
    const float mu = h.metallic, rho = h.roughness;
    const v3 tintMix = mk(1, 1, 1) + (Ctint - mk(1, 1, 1)) * h.specularTint;
    const float S0 = h.specular * 0.08f;
    const v3 Cspec0 = S0 * tintMix + (C - S0 * tintMix) * mu;
    const v3 Csheen = mk(1, 1, 1) + (Ctint - mk(1, 1, 1)) * h.sheenTint;
    const float FL = schlickFresnel(NDotL), FV = schlickFresnel(NDotV), FH = schlickFresnel(LDotH);
    const float Fd90 = 0.5f + 2.0f * LDotH * LDotH * rho;
    const float A = 1 + FL * (Fd90 - 1), Bd = 1 + FV * (Fd90 - 1);
    const float Fd = A * Bd, dFd = 2 * LDotH * LDotH * (FL * Bd + FV * A);
    const float Fss90 = LDotH * LDotH * rho;
    const float A2 = 1 + FL * (Fss90 - 1), B2 = 1 + FV * (Fss90 - 1);
    const float Fss = A2 * B2, dFss = LDotH * LDotH * (FL * B2 + FV * A2);
    const float k1 = 1.0f / (NDotL + NDotV) - 0.5f;
    const float ss = 1.25f * (Fss * k1 + 0.5f), dss = 1.25f * k1 * dFss;
    const float D0 = Fd + h.subsurface * (ss - Fd), dD0 = dFd + h.subsurface * (dss - dFd);
    const float aspect = sqrtf(1.0f - h.anisotropic * 0.9f);
    const float ax = maxf(0.001f, rho / aspect), ay = maxf(0.001f, rho * aspect);
    const float dax = rho / aspect > 0.001f ? 1.0f / aspect : 0.0f, day = rho * aspect > 0.001f ? aspect : 0.0f;
    const float HX = dot(H, T), HY = dot(H, B);
    const float a = HX / ax, b = HY / ay, c = a * a + b * b + NDotH * NDotH;
    const float Ds = 1.0f / (EL_PI * ax * ay * c * c);
    const float dDs = Ds * (-1.0f / ax + 4.0f * a * a / (c * ax)) * dax + Ds * (-1.0f / ay + 4.0f * b * b / (c * ay)) * day;
    float GL, dGL, GV, dGV;
    {
        float X = dot(L, T), Y = dot(L, B);
        float q = sqrtf((X * ax) * (X * ax) + (Y * ay) * (Y * ay) + NDotL * NDotL);
        GL = 1.0f / (NDotL + q);
        dGL = -GL * GL * ((X * X * ax) * dax + (Y * Y * ay) * day) / q;
    }
    {
        float X = dot(V, T), Y = dot(V, B);
        float q = sqrtf((X * ax) * (X * ax) + (Y * ay) * (Y * ay) + NDotV * NDotV);
        GV = 1.0f / (NDotV + q);
        dGV = -GV * GV * ((X * X * ax) * dax + (Y * Y * ay) * day) / q;
    }
    const float Gs = GL * GV, dGs = dGL * GV + GL * dGV;
    const v3 Fs = Cspec0 + (mk(1, 1, 1) - Cspec0) * FH;
    const v3 Fsheen = Csheen * (FH * h.sheen);
    const v3 diffusePart = C * ((1.0f / EL_PI) * D0) + Fsheen;
    const float spec = Gs * Ds * (1.0f - FH);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const v3 e = mk(k == 0 ? 1.f : 0.f, k == 1 ? 1.f : 0.f, k == 2 ? 1.f : 0.f);
        const v3 dCtint = lum > 0.0f ? e / lum - C * (wl[k] / (lum * lum)) : mk(0, 0, 0);
        const v3 dCspec0 = (S0 * h.specularTint * (1.0f - mu)) * dCtint + e * mu;
        const v3 dFsheen = dCtint * (FH * h.sheen * h.sheenTint);
        df[k] = (e * ((1.0f / EL_PI) * D0) + dFsheen) * (1.0f - mu) + dCspec0 * spec;
    }
    df[3] = C * ((1.0f / EL_PI) * dD0 * (1.0f - mu)) + Fs * (dGs * Ds + Gs * dDs);
    df[4] = diffusePart * -1.0f + (C - S0 * tintMix) * spec;
    df[5] = tintMix * (0.08f * (1.0f - mu) * spec);
}

// ----------------------------------------------------------------- camera --
// kernel.cu:260-337 (double-promoted terms kept as in the reference).
__device__ __forceinline__ void cameraRay(const DevCamera& c, int x, int y, float r1, float r2, float r3, float r4,
                                          float r5, v3& o, v3& d) {
    float dx = c.pos[0] + ((float)x) / ((float)c.xRes) * c.sensorWidth;
    float dy = c.pos[1] + ((float)y) / ((float)c.yRes) * c.sensorHeight;
    float odx = (float)((-c.sensorWidth / 2.0) + dx);
    float ody = (float)((-c.sensorHeight / 2.0) + dy);
    float rx = (float)((1.0 / (float)c.xRes) * (r1 - 0.5) * c.sensorWidth);
    float ry = (float)((1.0 / (float)c.yRes) * (r2 - 0.5) * c.sensorHeight);
    float SPx = odx + rx, SPy = ody + ry;
    float SPz = c.pos[2] + c.focalLength;
    // XYZ Euler rotation; the per-camera cos/sin are evaluated once on the host
    // (the reference evaluates the same six values for every ray)
    const float cx = c.cosRot[0], sx = c.sinRot[0], cy = c.cosRot[1], sy = c.sinRot[1];
    const float cz = c.cosRot[2], sz = c.sinRot[2];
    v3 dir = mk(SPx, SPy, SPz) - mk(c.pos[0], c.pos[1], c.pos[2]);
    v3 dX = mk(dir.x, dir.y * cx - dir.z * sx, dir.y * sx + dir.z * cx);
    v3 dY = mk(dX.x * cy + dX.z * sy, dX.y, dX.z * cy - dX.x * sy);
    v3 dZ = mk(dY.x * cz - dY.y * sz, dY.x * sz + dY.y * cz, dY.z);
    o = mk(c.pos[0], c.pos[1], c.pos[2]);
    d = normalized(dZ);
    if (c.bokeh) {
        float diameter = c.focalLength / c.aperture;
        float l = c.focusDistance + c.focalLength;
        v3 focus = o + d * l;
        float px, py;
        uniformCircleSampling(r3, r4, r5, px, py);
        px *= diameter * 0.5f;
        py *= diameter * 0.5f;
        v3 orig = o + mk(px, py, 0);
        o = orig;
        d = normalized(focus - orig);
    }
}

// --------------------------------------------------------------- hit data --
struct SurfaceHit {
    v3 position, normal;
    float tu, tv;
    int32_t material, tri;
    float u, v, sign;   // barycentrics and tangentsSign, for surfaceTangents
};

// Tri::hit's attribute part (Tri.hpp:70-157) from the traversal's (t, u, v).
__device__ __forceinline__ SurfaceHit surfaceAt(const DevScene& s, int tri, float t, float u, float v, v3 o, v3 d) {
    const float4* R = s.shade + (uint64_t)tri * kShadeWords;
    const float4 A = R[0], B = R[1], C = R[2], D = R[3], E = R[4], F = R[5], G = R[6];
    SurfaceHit h;
    v3 v0 = mk(A.x, A.y, A.z), v1 = mk(A.w, B.x, B.y), v2 = mk(B.z, B.w, C.x);
    v3 n0 = mk(C.y, C.z, C.w), n1 = mk(D.x, D.y, D.z), n2 = mk(D.w, E.x, E.y);
    float uv0x = E.z, uv0y = E.w, uv1x = F.x, uv1y = F.y, uv2x = F.z, uv2y = F.w;
    h.material = __float_as_int(G.x);
    h.sign = G.y;
    h.tri = tri;
    h.u = u;
    h.v = v;
    h.tu = uv0x + (uv1x - uv0x) * u + (uv2x - uv0x) * v;
    h.tv = uv0y + (uv1y - uv0y) * u + (uv2y - uv0y) * v;
    v3 geom = o + d * t;
    v3 Ns = n0 + (n1 - n0) * u + (n2 - n0) * v;
    v3 p0 = geom - dot(geom - v0, n0) * n0;
    v3 p1 = geom - dot(geom - v1, n1) * n1;
    v3 p2 = geom - dot(geom - v2, n2) * n2;
    v3 sp = p0 + (p1 - p0) * u + (p2 - p0) * v;
    bool convex = dot(sp - geom, Ns) > 0.0f;
    h.position = convex ? sp : geom;
    h.normal = Ns;
    return h;
}

// Tangent frame at a hit (Tri.hpp:78-79, 153): the interpolated corner
// tangents (not renormalised) and bitangent = tangentsSign * N x T.
__device__ __forceinline__ void surfaceTangents(const DevScene& s, const SurfaceHit& h, v3& T, v3& B) {
    const float4* R = s.tangents + (uint64_t)h.tri * kTanWords;
    const float4 a = R[0], b = R[1], c = R[2];
    const v3 t0 = mk(a.x, a.y, a.z), t1 = mk(a.w, b.x, b.y), t2 = mk(b.z, b.w, c.x);
    T = t0 + (t1 - t0) * h.u + (t2 - t0) * h.v;
    B = h.sign * cross(h.normal, T);
}

// generateHitData (kernel.cu:54-119)
// `lut`: an LDS copy of s.texLut, or null for the global one.
__device__ __forceinline__ HitData hitData(const DevScene& s, const SurfaceHit& h, const float* lut = nullptr) {
    const DevMaterial& m = s.mats[h.material];
    const TexPools P = texPools(s, lut);
    HitData d;
    d.albedo = m.albedoTex < 0 ? ld3(m.albedo) : texFiltered(P, s.texs[m.albedoTex], h.tu, h.tv);
    d.emission = m.emissionTex < 0 ? ld3(m.emission) : texFiltered(P, s.texs[m.emissionTex], h.tu, h.tv);
    // powf(x, 2.2f) of kernel.cu:113-114: for untextured parameters computed
    // once per material at upload
    d.roughness = m.roughnessTex < 0 ? m.roughnessEff
                                     : powf(texFiltered(P, s.texs[m.roughnessTex], h.tu, h.tv).x, 2.2f);
    d.metallic = m.metallicTex < 0 ? m.metallicEff
                                   : powf(texFiltered(P, s.texs[m.metallicTex], h.tu, h.tv).x, 2.2f);
    if (m.normalTex < 0) {
        d.normal = h.normal;
    } else {
        v3 c = texUV(P, s.texs[m.normalTex], h.tu, h.tv);
        v3 ln = c * 2.0f - mk(1, 1, 1);
        v3 T, B;
        surfaceTangents(s, h, T, B);
        d.normal = normalized(ln.x * T - ln.y * B + ln.z * h.normal);
    }
    d.clearcoatGloss = m.clearcoatGloss;
    d.clearcoat = m.clearcoat;
    d.anisotropic = m.anisotropic;
    d.eta = m.eta;
    d.transmission = m.transmission;
    d.specular = m.specular;
    d.specularTint = m.specularTint;
    d.sheenTint = m.sheenTint;
    d.subsurface = m.subsurface;
    d.sheen = m.sheen;
    return d;
}

// Escaped ray: env(-dir), nearest/filtered lookup (kernel.cu:414-419).
__device__ __forceinline__ v3 envLookup(const DevScene& s, v3 d) {
    float u, v;
    sphericalMapping(d * -1.0f, u, v);
    return texFiltered(texPools(s), s.env, u, v);
}

// HDRI NEE sample (kernel.cu:236-254 with HDRI.hpp:145-162, Texture.hpp:177-207).
struct EnvSample {
    v3 dir, value;
    float pdf;
    v3 shadowDir;   // normalized(dir), the shadow ray's direction
};
// Everything the NEE sample derives from the environment pixel k alone;
// tabulated per pixel at upload (envTab) by this same code.
__device__ __forceinline__ EnvSample envSampleAt(const DevScene& s, int k) {
    const DevTex& t = s.env;
    int x = k % t.w, y = k / t.w;
    float nu = x / (float)t.w, nv = y / (float)t.h;
    // inverseTransformUV
    int ix = (int)(nu * t.w), iy = (int)(nv * t.h);
    ix = (int)(t.xTile * (ix - t.xOffset * t.w)) % t.w;
    iy = (int)(t.yTile * (iy - t.yOffset * t.h)) % t.h;
    float iu = (float)ix / (float)t.w, iv = (float)iy / (float)t.h;
    iu += -(float)(iu > 1) + -(float)(iu < 0);
    iv += -(float)(iv > 1) + -(float)(iv < 0);
    // reverseSphericalMapping, negated and normalised
    float phi = iu * 2 * EL_PI, theta = iv * EL_PI;
    float px = cosf(phi - EL_PI), py = -cosf(theta), pz = -sinf(phi - EL_PI);
    float a = sqrtf(1 - py * py);
    EnvSample e;
    e.dir = normalized(mk(a * px, py, a * pz)) * -1.0f;
    e.value = texUV(texPools(s), t, iu, iv);
    // HDRI::pdf((int)(iu*W), (int)(iv*H))
    int qx = (int)(iu * t.w), qy = (int)(iv * t.h);
    v3 dv = texel(texPools(s), t, qx, qy);
    float th = (((float)qy / (float)t.h)) * EL_PI;
    e.pdf = ((dv.x + dv.y + dv.z) / s.envRadianceSum) * (float)(t.w * t.h) / (2.0f * EL_PI * sinf(th));
    e.shadowDir = normalized(e.dir);
    return e;
}
__device__ __forceinline__ EnvSample envSample(const DevScene& s, float r1) {
    // HDRI::sample(r1): exactly binarySearch(cdf, r1, W*H)
    const int k = hdriLookup(s.envCdf, s.envGuide, s.envMap, s.envLog2G, r1);
    const float4 a = s.envTab[2 * k], b = s.envTab[2 * k + 1];
    EnvSample e;
    e.dir = mk(a.x, a.y, a.z);
    e.pdf = a.w;
    e.value = mk(b.x, b.y, b.z);
    e.shadowDir = normalized(e.dir);   // as envSampleAt
    return e;
}

// ------------------------------------------------------------- traversal --
// Moller-Trumbore exactly as Tri::hit (Tri.hpp:38-68): FP32, no contraction,
// IEEE division for 1/det, inclusive barycentric bounds, t >= 0.
__device__ __forceinline__ bool mtHit(float4 A, float4 B, float4 C, float ox, float oy, float oz, float dx, float dy,
                                      float dz, float& t, float& u, float& v) {
#pragma clang fp contract(off)
    const float EPS = 0.0000001f;
    float e1x = A.w, e1y = B.x, e1z = B.y;
    float e2x = B.z, e2y = B.w, e2z = C.x;
    float px = dy * e2z - dz * e2y;
    float py = -(dx * e2z - dz * e2x);
    float pz = dx * e2y - dy * e2x;
    float det = e1x * px + e1y * py + e1z * pz;
    if (det > -EPS && det < EPS) return false;
    float inv = 1.0f / det;
    float tx = ox - A.x, ty = oy - A.y, tz = oz - A.z;
    u = (tx * px + ty * py + tz * pz) * inv;
    if (u < 0.0f || u > 1.0f) return false;
    float qx = ty * e1z - tz * e1y;
    float qy = -(tx * e1z - tz * e1x);
    float qz = tx * e1y - ty * e1x;
    v = (dx * qx + dy * qy + dz * qz) * inv;
    if (v < 0.0f || (u + v) > 1.0f) return false;
    t = (e2x * qx + e2y * qy + e2z * qz) * inv;
    if (t < 0.0f) return false;
    return true;
}

constexpr int kShortStack = 16;   // LDS entries per lane (power of two)

// Per-lane traversal stack.  Its newest entries live in LDS, in a ring of
// kShortStack rows of one int per lane (4 KB per wave); older ones spill to a
// global per-thread area (g[row * gstride + lane]).  Row 0 holds -1, the code that ends
// a traversal, so that a pop needs no test for an empty stack.  sp and lo are
// byte offsets of the ring, kStackRow per entry, not yet wrapped: an entry's
// address is one AND and one addition (both issue in half the time of a multiply
// or a shift with addition).  A BVH4 visit writes all four rows above sp, whatever it
// hit, after room() has made them free.  The host sizes the global part from the
// tree's worst-case depth (spillRows) so it never overflows; if it would, the
// entry is dropped and counted (no out-of-bounds access).
constexpr uint32_t kStackRow = 256, kStackWrap = (kShortStack - 1) * kStackRow;
constexpr int kVisitRows = 4;   // rows a visit may write above the stack's top
static_assert((kShortStack & (kShortStack - 1)) == 0 && kVisitRows < kShortStack, "the ring wraps by a mask");
// Global entries per thread for a tree whose traversals hold up to `bound` codes (the row of -1 comes on top).
inline int spillRows(int bound) {
    const int rows = bound + 1 + kVisitRows - kShortStack;
    return rows > 1 ? rows : 1;
}
struct TravStack {
    int* lds;   // the lane's column of its wave's ring
    int* g;     // its wave's part of the global area (wave-uniform)
    int gstride;
    int gcap;
    unsigned long long* dropped;   // counts entries that did not fit
    uint32_t sp, lo;
    __device__ __forceinline__ int& at(uint32_t off) { return *(int*)((char*)lds + (off & kStackWrap)); }
    __device__ __forceinline__ void reset() {
        sp = kStackRow;
        lo = 0;
        at(0) = -1;
    }
    // Makes the kVisitRows rows above sp free: the oldest entries go to the global area.
    __device__ __forceinline__ void room() {
        while (sp - lo > (kShortStack - kVisitRows) * kStackRow) {
            const int old = at(lo), row = (int)(lo / kStackRow);
            if (row < gcap)
                g[(uint64_t)row * gstride + __lane_id()] = old;
            else
                atomicAdd(dropped, 1ull);
            lo += kStackRow;
        }
    }
    // After room(), at most kVisitRows times.
    __device__ __forceinline__ void push(int e) {
        at(sp) = e;
        sp += kStackRow;
    }
    __device__ __forceinline__ int pop() {
        sp -= kStackRow;
        int e = at(sp);
        if (sp < lo) {   // spilled
            lo = sp;
            const int row = (int)(sp / kStackRow);
            e = row < gcap ? g[(uint64_t)row * gstride + __lane_id()] : -1;
        }
        return e;
    }
};

// Quantized wide node as uploaded, in 16-byte words.
//   W = 8: eleven::QNode<8> as it is, 6 words (header, q0-11 in three words,
//          child0-7 in two).
//   W = 4: 4 words, one per child (packLaneNode, bvh.hpp): word j holds child
//          j's code, its six plane bytes, and the grid origin and step of
//          axis j (j < 3), so that the four lanes of a quad that share a ray
//          read a node with one load, 16 bytes each, and each lane has its
//          own child and its own axis:
//            x  child code; of an inner node its first word, 4 * node
//            y  lo x | lo y << 8 | exponent of axis j << 23 (the step's FP32 bits) | 1 << 31 in an empty slot
//            z  lo z | hi x << 8 | hi y << 16 | hi z << 24
//            w  grid origin of axis j (FP32 bits)
template <int W>
struct QNodeWords {
    static constexpr int kWords = W == 4 ? 4 : 6;
};

struct TraceResult {
    int32_t tri;   // original index, -1 if none
    float t, u, v;
};

struct TraceCounters {
    uint32_t nodes, tris;
};

// Byte selectors (v_perm_b32 over z : y of a BVH4 node word) that gather a
// child's near and far plane bytes (x, y, z) for a ray direction's signs.
struct PlaneSel {
    uint32_t nearXY, farXY, z;   // (near x, near y), (far x, far y), (near z, far z)
};
__device__ __forceinline__ PlaneSel planeSel(float ix, float iy, float iz) {
    PlaneSel s;
    // y bytes 0, 1: lo x, lo y (selectors 0, 1); z bytes 0..3: lo z, hi x, hi y, hi z (4..7); 0x0c: zero
    s.nearXY = 0x0c000c00u | (ix < 0 ? 5u : 0u) | (iy < 0 ? 6u << 16 : 1u << 16);
    s.farXY = 0x0c000c00u | (ix < 0 ? 0u : 5u) | (iy < 0 ? 1u << 16 : 6u << 16);
    s.z = iz < 0 ? 0x0c040c07u : 0x0c070c04u;
    return s;
}
// Two plane bytes as the halves of a word, each the FP16 number q 2^-24 (a
// denormal, exact): v_fma_mix_f32 takes them as they are, so a plane needs no
// conversion of its own.
using HalfPair = _Float16 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ HalfPair planePair(const uint4& w, uint32_t sel) {
    return __builtin_bit_cast(HalfPair, __builtin_amdgcn_perm(w.z, w.y, sel));
}
// Slab distances are in units of 1 / scale: kSlabScale keeps q 2^-24 * (2^24
// step / direction) finite down to components of 1e-30, and near planes below 1,
// where they may be clamped for nothing (fma's clamp modifier), for distances up to
// 2^24.  A direction longer than 2^20 takes scale 1 instead, as its distances would
// become denormal otherwise, and components of 2^24 * 1e-30 count as zero.  Either
// is multiplied by the scene's slabUnit: 1, or less where the grid steps of its
// nodes are so large (2^28 and more) that 2^24 step / direction overflows all the same.
// A plane distance may overflow by its node's origin, which misses nothing (an
// infinity less its widening is no number, and the axis is left out), but
// not by the step alone: a near plane behind the ray would be infinitely far ahead.
constexpr float kSlabScale = 1.0f / 16777216.0f, kSlabScaleInv = 16777216.0f;
struct SlabScale {
    float scale, tiny;   // tiny: the smallest direction component told from zero
};
__device__ __forceinline__ SlabScale slabScale(float dx, float dy, float dz, float unit) {
    const bool longer = fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz)) > 1048576.0f;
    return SlabScale{longer ? unit : kSlabScale * unit, longer ? 1e-30f * kSlabScaleInv : 1e-30f};
}
// Scaled reciprocal of a direction component for the slab tests (at most 2^-24 * 1e30).
__device__ __forceinline__ float slabInv(float d, const SlabScale& c) {
    return 1.0f / (fabsf(d) > c.tiny ? d : copysignf(c.tiny, d)) * c.scale;
}
// The slabUnit of a scene whose largest grid step is 2^exponent: 2^24 step * kSlabScale / 1e-30 is then below
// 2^127.  No less than 2^-82, which keeps the reciprocals of components up to 2^20 normal numbers: with steps
// of 2^109 a triangle's determinant has long overflown.
inline float slabUnitOf(int exponent) { return std::ldexp(1.0f, std::max(-82, std::min(0, 27 - exponent))); }
// Widening of a slab distance A + q B: near planes use A - |A| kSlabEps, far planes A + |A| kSlabEps (see visitWords).
constexpr float kSlabEps = 1.0f / 524288.0f, kFarEps = 1.0f / 1048576.0f;

// A ray prepared for slab tests: origin, direction, the slab distances' scale and the scaled reciprocal.
struct TRay {
    float ox, oy, oz, dx, dy, dz, ix, iy, iz, scale;
};

__device__ __forceinline__ TRay makeTRay(float ox, float oy, float oz, float dx, float dy, float dz, float unit) {
    const SlabScale c = slabScale(dx, dy, dz, unit);
    return TRay{ox, oy, oz, dx, dy, dz, slabInv(dx, c), slabInv(dy, c), slabInv(dz, c), c.scale};
}

// Visits an inner node: slab-tests its W children against [0, tcull] and
// returns the nearest one hit, the others being pushed far to near; with none hit
// the stack's top.  With UNSORTED (any-hit queries, whose result does not depend
// on the visiting order) the hit children are taken in slot order instead.
// Child encoding: >= 0 inner node, <= -2 leaf, -1 empty slot or stack.
//
// Planes decode exactly (p + q * step is an FP32 value by construction).
// visitWords tests a node whose words are already loaded; visitNode loads them.
//
// Plane b = p + q s, so (b - o) / d = A + q B per axis with A = (p - o) inv
// and B = s inv (exact: s is a power of two), and fma(q, B, A) rounds once; A
// carries two roundings, so a distance is off by at most 2^-23 |A| + 2^-24
// |t|.  Near planes use A - E and far planes A + E with E = 2^-19 |A| of their
// own axis (an axis whose direction is near zero has a huge A, but also huge
// distances of its own), and the 2^-20 tf widening covers the |t| term (a far
// distance below zero is a miss either way): the
// test stays conservative.  An empty slot (child -1) has an inverted box, 255
// grid steps from near to far plane; where 255 steps are below the rounding
// of A (a node smaller than ~4e-6 of its distance from the origin on every
// axis) the box passes the widened test, so the slot is checked as
// well: entering it would end the traversal (-1 is the empty stack's code).
//
// What bounds a long launch is the instructions it issues, and not all cost the
// same: measured, an FP32 add, multiply or fma and a 32-bit add, and, or and shift
// take 2.0-2.7 cycles of a SIMD per wave; a minimum, maximum, comparison, select,
// conversion, byte permute or anything with a scalar operand besides takes 4.1-4.6.
// So W = 4 is written in the cheap ones where there is a choice: planes
// come as FP16 pairs (3 permutes and 6 mixed fmas instead of 2, 6 conversions and 6
// fmas), misses are sign masks, and the children are not sorted (10 minima and
// maxima, then 3 comparisons and 3 selects for each child pushed): the sign of
// a difference of keys counts for each child the hit ones behind it, which is its row
// above the stack's top, every child is written to its row (a miss counts as
// nearest of all, so its row is above the last hit), and the nearest comes
// back with the pop.  A 1920 x 1080 frame of 64 samples over 1,048,576 triangles renders in
// 84.5 instead of 91.6 ms, 2 M closest hits take 213 instead of 263 us.
template <int W, bool UNSORTED = false>
__device__ __forceinline__ int visitWords(const uint4* np, const TRay& ray, float tcull, TravStack& st) {
    float px, py, pz, sx, sy, sz;
    if constexpr (W == 4) {
        px = __uint_as_float(np[0].w), py = __uint_as_float(np[1].w), pz = __uint_as_float(np[2].w);
        sx = __uint_as_float(np[0].y & 0x7f800000u), sy = __uint_as_float(np[1].y & 0x7f800000u);
        sz = __uint_as_float(np[2].y & 0x7f800000u);
    } else {
        const uint4 h = np[0];
        px = __uint_as_float(h.x), py = __uint_as_float(h.y), pz = __uint_as_float(h.z);
        sx = __uint_as_float((h.w & 0xffu) << 23);
        sy = __uint_as_float(((h.w >> 8) & 0xffu) << 23);
        sz = __uint_as_float(((h.w >> 16) & 0xffu) << 23);
    }
    const float Ax = (px - ray.ox) * ray.ix, Ay = (py - ray.oy) * ray.iy, Az = (pz - ray.oz) * ray.iz;
    const float Ex = fabsf(Ax * kSlabEps), Ey = fabsf(Ay * kSlabEps), Ez = fabsf(Az * kSlabEps);
    const float Anx = Ax - Ex, Afx = Ax + Ex, Any = Ay - Ey, Afy = Ay + Ey, Anz = Az - Ez, Afz = Az + Ez;
    tcull = (UNSORTED ? tcull : fabsf(tcull)) * ray.scale;
    if constexpr (W == 4) {
        const float Bx = sx * (ray.ix * kSlabScaleInv), By = sy * (ray.iy * kSlabScaleInv), Bz = sz * (ray.iz * kSlabScaleInv);
        const PlaneSel sel = planeSel(ray.ix, ray.iy, ray.iz);
        uint32_t miss[4], key[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const HalfPair n = planePair(np[i], sel.nearXY), f = planePair(np[i], sel.farXY), z = planePair(np[i], sel.z);
            const float tz = __builtin_amdgcn_fmed3f(fmaf((float)z.x, Bz, Anz), 0.0f, 1.0f);
            const float tn = entryDistance(fmaf((float)n.x, Bx, Anx), fmaf((float)n.y, By, Any), tz);
            float tf = fminf(fmaf((float)z.y, Bz, Afz), tcull);
            tf = fminf(fminf(fmaf((float)f.x, Bx, Afx), fmaf((float)f.y, By, Afy)), tf) * (1.0f + kFarEps);
            miss[i] = (uint32_t)((__float_as_int(tf - tn) | (int)np[i].y) >> 31);
            key[i] = childKey(__float_as_uint(tn), miss[i]);
        }
        st.room();
        if constexpr (UNSORTED) {
#pragma unroll
            for (int i = 3; i >= 0; i--)
                if (!miss[i]) st.push((int)np[i].x);
            return st.pop();
        } else {
            uint32_t above[4];
            childRows(key, above);
#pragma unroll
            for (int i = 0; i < 4; i++) st.at(st.sp + above[i] * kStackRow) = (int)np[i].x;
            st.sp += (4u + miss[0] + miss[1] + miss[2] + miss[3]) * kStackRow;
            return st.pop();
        }
    } else {
        uint32_t keys[W];
        int32_t child[W];
        const float Bx = sx * ray.ix, By = sy * ray.iy, Bz = sz * ray.iz;
        auto key = [&](int i, uint32_t qnx, uint32_t qny, uint32_t qnz, uint32_t qfx, uint32_t qfy, uint32_t qfz) {
            const float tx0 = fmaf((float)qnx, Bx, Anx), tx1 = fmaf((float)qfx, Bx, Afx);
            const float ty0 = fmaf((float)qny, By, Any), ty1 = fmaf((float)qfy, By, Afy);
            const float tz0 = fmaf((float)qnz, Bz, Anz), tz1 = fmaf((float)qfz, Bz, Afz);
            const float tn = fmaxf(fmaxf(tx0, ty0), fmaxf(tz0, 0.0f));
            float tf = fminf(fminf(tx1, ty1), fminf(tz1, tcull));
            tf = fmaf(fabsf(tf), kFarEps, tf);
            keys[i] = (tn <= tf && child[i] != -1) ? ((__float_as_uint(tn) & ~7u) | (uint32_t)i) : 0xFFFFFFFFu;
        };
        const uint4 a = np[1], b = np[2], c = np[3], d = np[4], e = np[5];
        const uint32_t q[12] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w};
        child[0] = (int32_t)d.x, child[1] = (int32_t)d.y, child[2] = (int32_t)d.z, child[3] = (int32_t)d.w;
        child[W - 4] = (int32_t)e.x, child[W - 3] = (int32_t)e.y, child[W - 2] = (int32_t)e.z, child[W - 1] = (int32_t)e.w;
        // near / far plane bytes per axis by the direction's sign (q index: axis * 4 + side * 2 + dword)
        const bool nx = ray.ix < 0, ny = ray.iy < 0, nz = ray.iz < 0;
        uint32_t nf[6][2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            nf[0][k] = nx ? q[2 + k] : q[k], nf[3][k] = nx ? q[k] : q[2 + k];
            nf[1][k] = ny ? q[6 + k] : q[4 + k], nf[4][k] = ny ? q[4 + k] : q[6 + k];
            nf[2][k] = nz ? q[10 + k] : q[8 + k], nf[5][k] = nz ? q[8 + k] : q[10 + k];
        }
#pragma unroll
        for (int i = 0; i < W; i++) {
            const int k = i >> 2, sh = 8 * (i & 3);
            key(i, (nf[0][k] >> sh) & 0xffu, (nf[1][k] >> sh) & 0xffu, (nf[2][k] >> sh) & 0xffu,
                (nf[3][k] >> sh) & 0xffu, (nf[4][k] >> sh) & 0xffu, (nf[5][k] >> sh) & 0xffu);
        }
        if constexpr (UNSORTED) {
            int next = -2;   // the lowest hit slot is visited next, the others are pushed
            st.room();
#pragma unroll
            for (int i = W - 1; i >= 0; i--) {
                if (i == 3) st.room();
                if (keys[i] == 0xFFFFFFFFu) continue;
                if (next != -2) st.push(child[next]);
                next = i;
            }
            return next == -2 ? st.pop() : child[next];
        }
        // ascending sort (tn >= 0, so float bits order as unsigned)
        int nh = 0;
#pragma unroll
        for (int i = 1; i < W; i++)
#pragma unroll
            for (int j = i; j > 0; j--) {
                const uint32_t lo = min(keys[j - 1], keys[j]), hi = max(keys[j - 1], keys[j]);
                keys[j - 1] = lo;
                keys[j] = hi;
            }
#pragma unroll
        for (int i = 0; i < W; i++) nh += keys[i] != 0xFFFFFFFFu;
        if (nh == 0) return st.pop();
        if (nh > 1) st.room();
#pragma unroll
        for (int i = W - 1; i >= 1; i--) {
            if (i == 3 && nh > 4) st.room();
            if (i < nh) st.push(child[keys[i] & 7u]);
        }
        return child[keys[0] & 7u];
    }
}

template <int W, bool UNSORTED = false>
__device__ __forceinline__ int visitNode(const uint4* __restrict__ nodes, int cur, const TRay& ray, float tcull,
                                         TravStack& st) {
    constexpr int K = QNodeWords<W>::kWords;
    const uint4* np = nodes + (W == 4 ? (uint64_t)(uint32_t)cur : (uint64_t)cur * K);
    uint4 w[K];
#pragma unroll
    for (int k = 0; k < K; k++) w[k] = np[k];
    return visitWords<W, UNSORTED>(w, ray, tcull, st);
}

// Tests one triangle record and updates the closest hit: smaller t wins,
// equal t goes to the lower original index.  For ANY the first hit below
// r.t is taken and true is returned (the query ends).
template <bool ANY, class Ray>
__device__ __forceinline__ bool hitTriangle(const float4& A, const float4& B, const float4& C, const Ray& ray,
                                            TraceResult& r) {
    float t, u, v;
    if (mtHit(A, B, C, ray.ox, ray.oy, ray.oz, ray.dx, ray.dy, ray.dz, t, u, v)) {
        const int id = __float_as_int(C.y);
        if (ANY) {
            if (t < r.t) {
                r.tri = id;
                r.t = t;
                r.u = u;
                r.v = v;
                return true;
            }
        } else if (t < r.t || (t == r.t && (unsigned)id < (unsigned)r.tri)) {
            r.tri = id;
            r.t = t;
            r.u = u;
            r.v = v;
        }
    }
    return false;
}

// Tests the triangles of leaf `code` (<= -2), as hitTriangle.  The leaf's
// triangles are contiguous records; the three words of the next
// triangle are loaded before the current one is tested, and all three
// words of a triangle together (the vertex word is otherwise fetched only
// after the determinant test), so a leaf costs about one memory round trip
// instead of two per triangle.
template <bool ANY, bool COUNT>
__device__ __forceinline__ bool testLeaf(const float4* __restrict__ tris, int code, const TRay& ray, TraceResult& r,
                                         TraceCounters& cnt) {
    const uint32_t k = (uint32_t)(-code - 2), first = k >> 4;
    const int count = (int)(k & 15u) + 1;
    const float4* p = tris + first * 3u;
#if EL_LEAF_PIPE
    float4 nA = p[0], nB = p[1], nC = p[2];
#endif
    for (int i = 0; i < count; i++) {
#if EL_LEAF_PIPE
        const float4 A = nA, B = nB, C = nC;
        if (i + 1 < count) {
            nA = p[3 * (i + 1)];
            nB = p[3 * (i + 1) + 1];
            nC = p[3 * (i + 1) + 2];
        }
#else
        float4 A = p[3 * i], B = p[3 * i + 1], C = p[3 * i + 2];
#endif
        if (COUNT) cnt.tris++;
        if (hitTriangle<ANY>(A, B, C, ray, r)) return true;
    }
    return false;
}

// Culling bound for child boxes: closest-hit keeps boxes slightly beyond the
// current hit so an equal-t hit with a lower index is still found.
template <bool ANY>
__device__ __forceinline__ float cullT(float t) {
    return ANY ? t : t * (1.0f + 1.0f / 1048576.0f);
}

// One ray, one thread: depth-first traversal with nearest-child-first order.
template <int W, bool ANY, bool COUNT>
__device__ __forceinline__ TraceResult traceRay(const DevScene& s, float ox, float oy, float oz, float dx, float dy,
                                                float dz, float tmax, TravStack& st, TraceCounters& cnt) {
    const uint4* __restrict__ nodes = (const uint4*)s.nodes;
    const TRay ray = makeTRay(ox, oy, oz, dx, dy, dz, s.slabUnit);
    TraceResult r;
    r.tri = -1;
    r.t = tmax;
    r.u = r.v = 0.f;
    st.reset();
    int cur = 0;
    while (cur != -1) {
        if (cur >= 0) {
            if (COUNT) cnt.nodes++;
            cur = visitNode<W, ANY>(nodes, cur, ray, cullT<ANY>(r.t), st);
        } else {
            bool done = testLeaf<ANY, COUNT>(s.tris, cur, ray, r, cnt);
            cur = done ? -1 : st.pop();
        }
    }
    return r;
}

// The lanes of the wave for which p holds.
__device__ __forceinline__ unsigned long long waveMask(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// How many of them have a lower index than the caller's lane.
__device__ __forceinline__ uint32_t lanesBelow(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Persistent traversal of the items [begin, end) owned by one wave, with
// in-wave refill: a lane whose ray is finished takes the wave's next item, so
// the wave keeps its lanes busy instead of waiting for its slowest ray (the
// refill happens once at least `refill` lanes are idle, or all are).  Inner
// nodes and leaves are separated (Aila & Laine, "Understanding the Efficiency
// of Ray Traversal on GPUs", HPG 2009, speculative while-while): a lane that
// reaches a leaf postpones it and keeps descending until every live lane of
// the wave holds a leaf, then the wave tests leaves together.  With one BVH
// per wave a lane may postpone a second leaf and go on descending instead
// of idling while the other lanes look for their first (measured: a third
// does not pay, nor does a second with per-ray BVHs, whose lanes hold more
// registers).  A new ray starts at the root like any other visit: a visit of
// its own at the refill would run with only the lanes refilled (a 1080p frame of 64
// samples over 1,048,576 triangles 86.3 instead of 84.6 ms, 2 M closest hits 220 instead of 213 us).  The
// lane's state should fit 64 registers, what is the same for a wave is kept
// once (the count of rays, the spill area's address, the count of dropped
// entries in memory) and a queue's entry is looked up once a ray: with 0 to 5
// registers spilled in launches over one BVH and 6 to 19 in batches, 10 to 27
// before, a batch of 12 scenes takes 10.65 instead of 11.1 ms, 2 M closest hits
// 205 instead of 210 us.  The
// closest hit is order-independent (t, then lower index), so results are
// identical to traceRay.
//
//   load(i, ox, oy, oz, dx, dy, dz, tmax, bvh, item) -> false if item i has no
//                                   ray; with PER_RAY_BVH it also sets the BVH
//                                   (nodes, triangles) the ray traverses; item:
//                                   what store is to know it by.  The lanes that
//                                   call together have consecutive i
//   store(item, result, traced)     once per item
//
// Every lane of the wave must call with the same begin/end.
struct BvhPtr {
    const uint4* nodes;
    const float4* tris;
};

// The items a wave traces: chunks of `chunk` items, either in turn (each turn
// every wave takes one, without counters) or, with waves == 0, handed out at
// run time.  From turn to turn a wave moves on by 5/8 of the waves: a queue
// starts as a whole number of frames, and a wave that kept its place would
// often get the same part of the image every time (the first launch of a 256 x
// 256 frame of 16 samples: all 8 chunks of a wave from one tile, so its waves
// worked 19 % of its 325 us on average; moving on, the frame renders in 0.88
// instead of 0.95 ms, a 512 x 512 one in 2.32 instead of 2.53).  Everything that
// is the same for a wave is kept in scalar registers (readfirstlane): with 64
// vector registers a lane every one that is not spilled counts (a 128 x 128
// gradient's render 770 -> 730 us).  Then chunk c belongs to share c % parts;
// share x is counted by ctr[x * stride].  A wave draws from its home share
// first, then from the others, so waves that meet cheap rays take more chunks
// and a launch ends when the work does, not when its slowest wave's share
// does.  One scene uses 8 shares (one per XCD: the waves of an XCD draw
// neighbouring chunks, which keeps their rays coherent in its L2), a batch 64
// (measured faster there).  Every counter starts the launch at 0.  A share is
// skipped without an atomic once a coherent read shows it drawn out (a read
// never runs ahead of the counter, so no chunk is lost).
constexpr uint32_t kWorkShares = 64;   // shares of a wide WorkSource (one per lane of a wave)
struct WorkSource {
    uint32_t* ctr;
    uint32_t n, chunk, stride, parts, home;
    uint32_t chunks;   // ceil(n / chunk)
    uint32_t first;    // this wave's first chunk (waves != 0)
    uint32_t waves;    // 0: drawn from the counters
};

// A wave's place in its items (wave-uniform).
struct WorkCursor {
    uint32_t cursor = 0, end = 0;
    WorkTurns turns;
    uint32_t tried = 0;      // narrow source: shares found drawn out
    __device__ __forceinline__ WorkCursor(const WorkSource& ws) : turns(ws.first) {}
    // The next chunk after [cursor, end) is used up; false: no items left,
    // and none will come.  One-scene launches do not ask again then; batches
    // do, with a load a time, since the test costs their kernels more in
    // registers (a batch of 12 scenes 8.67 and 8.75 ms of GPU).
    // The whole wave must call.
    template <bool WIDE>
    __device__ __forceinline__ bool draw(const WorkSource& ws) {
        if (ws.waves) return take(ws, turns.next(ws.waves, ws.chunks, ws.first));
        const uint32_t lane = __lane_id();
        // Wide sources (batches, parts == 64): lane l looks at share
        // (home + l) % 64 at once (one load per lane instead of 64
        // dependent loads), and the wave draws from the first share with
        // chunks left.  Share x holds the chunks x, x + 64, ...:
        // (chunks - x + 63) / 64 of them.
        while (WIDE) {
            const uint32_t x = (ws.home + lane) & (kWorkShares - 1);
            const uint32_t seen =
                __hip_atomic_load(ws.ctr + x * ws.stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool left = x < ws.chunks && seen < ((ws.chunks - x + kWorkShares - 1) >> 6);
            const unsigned long long have = __ballot(left);
            if (!have) return false;
            const uint32_t pick = (ws.home + (uint32_t)(__ffsll((long long)have) - 1)) & (kWorkShares - 1);
            uint32_t k = 0;
            if (lane == 0) k = atomicAdd(ws.ctr + pick * ws.stride, 1u);
            k = __builtin_amdgcn_readfirstlane(k);
            if (take(ws, (uint64_t)pick + (uint64_t)kWorkShares * k)) return true;
        }
        // Narrow sources (one scene, parts == 8): one share at a time, from
        // the wave's home share on; a share found drawn out is not looked at
        // again.
        while (!WIDE && tried < ws.parts) {
            const uint32_t x = (ws.home + tried) % ws.parts;
            uint32_t* const c = ws.ctr + x * ws.stride;
            const uint32_t seen = __builtin_amdgcn_readfirstlane(
                __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (((uint64_t)x + (uint64_t)ws.parts * seen) * ws.chunk < ws.n) {
                uint32_t k = 0;
                if (lane == (uint32_t)(__ffsll((long long)__ballot(true)) - 1)) k = atomicAdd(c, 1u);
                k = __builtin_amdgcn_readfirstlane(k);
                if (take(ws, (uint64_t)x + (uint64_t)ws.parts * k)) return true;
            }
            tried++;
        }
        return false;
    }
    __device__ __forceinline__ bool take(const WorkSource& ws, uint64_t chunk) {
        const uint64_t first = chunk * ws.chunk;
        if (first >= ws.n) return false;
        cursor = __builtin_amdgcn_readfirstlane((uint32_t)first);
        end = __builtin_amdgcn_readfirstlane((uint32_t)(first + ws.chunk < ws.n ? first + ws.chunk : ws.n));
        return true;
    }
};

template <int W, bool ANY, bool COUNT, bool PER_RAY_BVH = false, class Load, class Store>
__device__ __forceinline__ void traceWaveRange(const DevScene& s, TravStack& st, const WorkSource& ws,
                                               uint32_t refill, Load&& load, Store&& store, TraceCounters& cnt,
                                               uint32_t& traced) {
    if (ws.waves && ws.first >= ws.chunks) return;   // no chunk for this wave
    BvhPtr bvh{(const uint4*)s.nodes, s.tris};
    WorkCursor wc(ws);
    bool more = true;   // wave-uniform: items may remain
    bool live = false;
    uint32_t item = 0;
    TRay ray{};
    TraceResult r{};
    int cur = -1, leaf = -1, leaf2 = -1;
    while (true) {
        // ---- refill idle lanes from the wave's range or the next chunk
        const unsigned long long idle = waveMask(!live);
        const uint32_t nIdle = (uint32_t)__popcll(idle);
        const bool want = nIdle >= refill || nIdle == 64;
        if ((PER_RAY_BVH || more) && want && wc.cursor >= wc.end) more = wc.draw<PER_RAY_BVH>(ws);
        if (want && more) {
            if (!live) {
                uint32_t i = wc.cursor + lanesBelow(idle);
                if (i < wc.end) {
                    float ox, oy, oz, dx, dy, dz, tmax;
                    BvhPtr rb = bvh;
                    if (load(i, ox, oy, oz, dx, dy, dz, tmax, rb, item)) {
                        if (PER_RAY_BVH) bvh = rb;
                        ray = makeTRay(ox, oy, oz, dx, dy, dz, s.slabUnit);
                        r.tri = -1;
                        r.t = tmax;
                        r.u = r.v = 0.f;
                        st.reset();
                        leaf = leaf2 = -1;
                        cur = 0;
                        live = true;
                    } else {
                        TraceResult dead;
                        dead.tri = -2;
                        dead.t = dead.u = dead.v = 0.f;
                        store(item, dead, false);
                    }
                }
            }
            wc.cursor += nIdle;
            traced += nIdle - (uint32_t)__popcll(waveMask(!live));
        } else if (nIdle == 64 && !more) {
            break;   // no items left and every lane finished
        }
        // ---- inner nodes: descend until every live lane holds a leaf
        while (true) {
            const bool act = live && cur >= 0;
            if ((waveMask(cur >= 0) & waveMask(leaf == -1)) == 0) break;   // also when no lane can descend
            // closest hit, one BVH per wave: with enough lanes finished and
            // items left, test the leaves held so far and refill instead of
            // idling until the descent ends (any-hit queries and per-ray
            // BVHs measured slower with it)
            if (!ANY && !PER_RAY_BVH && more &&
                (uint32_t)__popcll(waveMask((cur & leaf) == -1)) >= refill)
                break;
            if (act) {
                if (COUNT) cnt.nodes++;
                cur = visitNode<W, ANY>(PER_RAY_BVH ? bvh.nodes : (const uint4*)s.nodes, cur, ray, cullT<ANY>(r.t),
                                        st);
                if (cur <= -2 && (PER_RAY_BVH ? leaf : leaf2) == -1) {   // a leaf: postponed
                    leaf2 = PER_RAY_BVH ? -1 : leaf;
                    leaf = cur;
                    cur = st.pop();
                }
            }
        }
        // ---- leaves: the postponed one, then any leaves that follow on the stack
        while (true) {
            const bool has = live && (leaf != -1 || cur <= -2);
            if ((waveMask(leaf != -1) | waveMask(cur <= -2)) == 0) break;
            if (has) {
                int code;
                if (!PER_RAY_BVH && leaf2 != -1) {
                    code = leaf2;
                    leaf2 = -1;
                } else if (leaf != -1) {
                    code = leaf;
                    leaf = -1;
                } else {
                    code = cur;
                    cur = st.pop();
                }
                if (testLeaf<ANY, COUNT>(PER_RAY_BVH ? bvh.tris : s.tris, code, ray, r, cnt)) {
                    cur = -1;   // any-hit: done
                    leaf = leaf2 = -1;
                }
            }
        }
        // ---- finished rays
        if (live && cur == -1 && leaf == -1) {
            store(item, r, true);
            live = false;
        }
    }
}

// --------------------------------------------------------- quad traversal --
// Short BVH4 launches give a ray to a quad (4 neighbouring lanes of a wave, 16
// rays per wave): lane j tests child j of the ray's node and triangle j of its
// leaf.  What such a launch waits for is one ray's chain of visits, each a
// load and then the instructions that lead to the next node's address; with
// a child per lane a visit is one coalesced 64-byte load and ~70 instructions,
// and the quad's exchanges are DPP moves, which cost no LDS round trip.  A
// launch over 3,072 rays takes 12-27 us instead of 35-53.
constexpr int kQuadStack = 64;        // LDS entries per ray: 4 KB per wave, as kShortStack per lane
constexpr uint32_t kQuadEntry = 64;   // bytes from a ray's stack entry to its next (16 rays interleaved)

// Value of lane J (0..3) of the caller's quad, and of the lane whose index in
// the quad differs by the bits of X.  The lanes of a quad always run together.
template <int J>
__device__ __forceinline__ uint32_t quadLane(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, J * 0x55, 0xf, 0xf, true);
}
template <int J>
__device__ __forceinline__ float quadLane(float v) {
    return __uint_as_float(quadLane<J>(__float_as_uint(v)));
}
template <int X>
__device__ __forceinline__ uint32_t quadXor(uint32_t v) {
    constexpr int ctrl = (0 ^ X) | (1 ^ X) << 2 | (2 ^ X) << 4 | (3 ^ X) << 6;
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, ctrl, 0xf, 0xf, true);
}
template <int X>
__device__ __forceinline__ float quadXor(float v) {
    return __uint_as_float(quadXor<X>(__float_as_uint(v)));
}
__device__ __forceinline__ float quadMin(float v) {
    v = fminf(v, quadXor<1>(v));
    return fminf(v, quadXor<2>(v));
}
__device__ __forceinline__ uint32_t quadOr(uint32_t v) {
    v |= quadXor<1>(v);
    return v | quadXor<2>(v);
}

// A quad's stack: entry i at lds[16 i], the code -1 of an empty stack at entry
// 0 (popped at most once per ray).  Trees whose worst case is deeper than
// kQuadStack - 2 are traversed with a stack per lane, which can spill.
// Entries written by one lane are read by all four: the wave barrier keeps
// the compiler from moving reads over writes.
struct QuadStack {
    int* lds;
    uint32_t sp;   // kQuadEntry x entries
    __device__ __forceinline__ int& at(uint32_t off) { return *(int*)((char*)lds + off); }
    __device__ __forceinline__ void reset() {
        at(0) = -1;
        sp = kQuadEntry;
    }
    __device__ __forceinline__ int pop() {
        sp -= kQuadEntry;
        return at(sp);
    }
};

struct QuadRay {
    float ox, oy, oz, dx, dy, dz;
    float oa, ia, scale;   // origin and slabInv of this lane's axis (lanes 0..2), slabScale
    PlaneSel sel;
};
__device__ __forceinline__ QuadRay makeQuadRay(float ox, float oy, float oz, float dx, float dy, float dz,
                                               float unit, uint32_t j) {
    QuadRay r{ox, oy, oz, dx, dy, dz};
    r.oa = j == 0 ? ox : j == 1 ? oy : oz;
    const SlabScale c = slabScale(dx, dy, dz, unit);
    r.scale = c.scale;
    r.ia = slabInv(j == 0 ? dx : j == 1 ? dy : dz, c);
    r.sel = planeSel(quadLane<0>(r.ia), quadLane<1>(r.ia), quadLane<2>(r.ia));
    return r;
}

// visitWords of a BVH4 node by the four lanes of a quad: pushes the hit
// children far to near (ANY: in slot order).
template <bool ANY>
__device__ __forceinline__ void visitQuad(const uint4* __restrict__ nodes, int cur, const QuadRay& ray, float tcull,
                                          uint32_t j, QuadStack& st) {
    const uint4 w = nodes[(uint32_t)cur + j];
    const float A = (__uint_as_float(w.w) - ray.oa) * ray.ia;
    const float B = __uint_as_float(w.y & 0x7f800000u) * (ray.ia * kSlabScaleInv);
    const float An = fmaf(-fabsf(A), kSlabEps, A), Af = fmaf(fabsf(A), kSlabEps, A);
    const HalfPair n = planePair(w, ray.sel.nearXY), f = planePair(w, ray.sel.farXY), z = planePair(w, ray.sel.z);
    const float Bx = quadLane<0>(B), By = quadLane<1>(B), Bz = quadLane<2>(B);
    const float tx0 = fmaf((float)n.x, Bx, quadLane<0>(An)), tx1 = fmaf((float)f.x, Bx, quadLane<0>(Af));
    const float ty0 = fmaf((float)n.y, By, quadLane<1>(An)), ty1 = fmaf((float)f.y, By, quadLane<1>(Af));
    const float tz0 = fmaf((float)z.x, Bz, quadLane<2>(An)), tz1 = fmaf((float)z.y, Bz, quadLane<2>(Af));
    const float tn = fmaxf(fmaxf(tx0, ty0), fmaxf(tz0, 0.0f));
    float tf = fminf(fminf(tx1, ty1), fminf(tz1, tcull * ray.scale));
    tf = fmaf(fabsf(tf), kFarEps, tf);
    const bool hit = tn <= tf && (int)w.x != -1;
    uint32_t at = st.sp, top;
    if constexpr (ANY) {
        const uint32_t nib = quadOr(hit ? 1u << j : 0u);
        top = (uint32_t)__popc(nib) * kQuadEntry;
        at += (uint32_t)__popc(nib >> (j + 1)) * kQuadEntry;   // below the children taken after it
    } else {
        // distances as non-negative integers, so that a difference's sign bit is the comparison
        const int key = childKeyOfLane(__float_as_uint(tn), j, hit);
        const uint32_t nearer = nearerKey((int)quadXor<1>((uint32_t)key), key) +
                                nearerKey((int)quadXor<2>((uint32_t)key), key) +
                                nearerKey((int)quadXor<3>((uint32_t)key), key);
        uint32_t c = hit ? kQuadEntry : 0u;
        c += quadXor<1>(c);
        top = c + quadXor<2>(c);
        at += top - kQuadEntry - nearer * kQuadEntry;
    }
    if (hit) st.at(at) = (int)w.x;
    st.sp += top;
    __builtin_amdgcn_wave_barrier();
}

// Tests the triangles of leaf `code`, lane j every fourth from the j-th on, as
// hitTriangle into the lane's own best r.  ANY: true in every lane of the
// quad if one of them hit.
template <bool ANY, bool COUNT>
__device__ __forceinline__ bool testLeafQuad(const float4* __restrict__ tris, int code, const QuadRay& ray, uint32_t j,
                                             TraceResult& r, TraceCounters& cnt) {
    const uint32_t k = (uint32_t)(-code - 2), first = k >> 4, count = (k & 15u) + 1;
    bool found = false;
    for (uint32_t i = j; i < count; i += 4) {
        const float4* p = tris + 3 * (uint64_t)(first + i);
        const float4 A = p[0], B = p[1], C = p[2];
        if (COUNT) cnt.tris++;
        found |= hitTriangle<ANY>(A, B, C, ray, r);
    }
    return ANY && quadOr(found ? 1u : 0u) != 0u;
}

// The ray's closest hit from the best hits of its four lanes: smaller t, then
// lower index (a lane without a hit has t = tmax, tri -1).
__device__ __forceinline__ void quadClosest(TraceResult& r) {
    auto take = [&](float t, uint32_t id, float u, float v) {
        if (t < r.t || (t == r.t && id < (uint32_t)r.tri)) {
            r.t = t;
            r.tri = (int32_t)id;
            r.u = u;
            r.v = v;
        }
    };
    {
        const float t = quadXor<1>(r.t), u = quadXor<1>(r.u), v = quadXor<1>(r.v);
        const uint32_t id = quadXor<1>((uint32_t)r.tri);
        take(t, id, u, v);
    }
    const float t = quadXor<2>(r.t), u = quadXor<2>(r.u), v = quadXor<2>(r.v);
    const uint32_t id = quadXor<2>((uint32_t)r.tri);
    take(t, id, u, v);
}

// traceWaveRange for BVH4 with a quad per ray.  A quad without a ray has cur,
// leaf and leaf2 -1.
template <bool ANY, bool COUNT, bool PER_RAY_BVH = false, class Load, class Store>
__device__ __forceinline__ void traceQuadRange(const DevScene& s, QuadStack& st, const WorkSource& ws,
                                               uint32_t refill, Load&& load, Store&& store, TraceCounters& cnt,
                                               uint32_t& traced) {
    if (ws.waves && ws.first >= ws.chunks) return;   // no chunk for this wave
    BvhPtr bvh{(const uint4*)s.nodes, s.tris};
    const uint32_t lane = __lane_id(), j = lane & 3u;
    WorkCursor wc(ws);
    bool more = true;   // wave-uniform: items may remain
    bool live = false;
    uint32_t item = 0;
    QuadRay ray{};
    TraceResult r{};
    float tq = 0.f;   // the quad's culling distance
    int cur = -1, leaf = -1, leaf2 = -1;
    while (true) {
        // ---- refill idle quads from the wave's range or the next chunk
        const unsigned long long idle = waveMask(!live);
        const uint32_t nIdle = (uint32_t)__popcll(idle);
        const bool want = nIdle >= refill || nIdle == 64;
        if ((PER_RAY_BVH || more) && want && wc.cursor >= wc.end) more = wc.draw<PER_RAY_BVH>(ws);
        if (want && more) {
            if (!live) {
                const uint32_t i = wc.cursor + (lanesBelow(idle) >> 2);   // quads are idle as a whole
                if (i < wc.end) {
                    float ox, oy, oz, dx, dy, dz, tmax;
                    BvhPtr rb = bvh;
                    if (load(i, ox, oy, oz, dx, dy, dz, tmax, rb, item)) {
                        if (PER_RAY_BVH) bvh = rb;
                        ray = makeQuadRay(ox, oy, oz, dx, dy, dz, s.slabUnit, j);
                        r.tri = -1;
                        r.t = tmax;
                        r.u = r.v = 0.f;
                        tq = cullT<ANY>(tmax);
                        st.reset();
                        cur = 0;
                        live = true;
                    } else if (j == 0) {
                        TraceResult dead;
                        dead.tri = -2;
                        dead.t = dead.u = dead.v = 0.f;
                        store(item, dead, false);
                    }
                }
            }
            wc.cursor += nIdle >> 2;
            traced += (nIdle - (uint32_t)__popcll(waveMask(!live))) >> 2;
        } else if (nIdle == 64 && !more) {
            break;   // no items left and every quad finished
        }
        // ---- inner nodes: descend until every live quad holds a leaf
        while (waveMask(cur >= 0 && leaf == -1)) {
            if (cur >= 0) {
                if (COUNT) cnt.nodes += j == 0;
                visitQuad<ANY>(PER_RAY_BVH ? bvh.nodes : (const uint4*)s.nodes, cur, ray, tq, j, st);
                cur = st.pop();
                if (cur <= -2 && (PER_RAY_BVH ? leaf : leaf2) == -1) {   // postponed: leaf2 is the older one
                    leaf2 = leaf;
                    leaf = cur;
                    cur = st.pop();
                }
            }
        }
        // ---- leaves: the postponed ones, then any that follow on the stack
        while (true) {
            const bool has = leaf != -1 || cur <= -2;
            if (!waveMask(has)) break;
            if (has) {
                int code;
                if (leaf2 != -1) {
                    code = leaf2;
                    leaf2 = -1;
                } else if (leaf != -1) {
                    code = leaf;
                    leaf = -1;
                } else {
                    code = cur;
                    cur = st.pop();
                }
                if (testLeafQuad<ANY, COUNT>(PER_RAY_BVH ? bvh.tris : s.tris, code, ray, j, r, cnt)) {
                    cur = -1;   // any-hit: done
                    leaf = leaf2 = -1;
                }
                if (!ANY) tq = quadMin(cullT<ANY>(r.t));
            }
        }
        // ---- finished rays
        if (live && cur == -1) {
            quadClosest(r);
            if (j == 0) store(item, r, true);
            live = false;
        }
    }
}

}  // namespace dev
}  // namespace eleven
