// C-ABI device context: scene upload (renderSetup), rendering (renderCuda),
// readback (getBuffers / getSamples) and the ray-query hooks.
//
// Reference host side (src/tfg-pathtracer/kernel.cu:485-724) deep-copies the
// AoS scene with one cudaMemcpy per array plus "pointer binding", keeps the
// accumulation in fixed 1920x1080 device globals and reads it back on a
// fresh, unsynchronised stream.  Here one context owns one stream; the scene
// becomes a handful of SoA buffers; accumulation is sized to the camera; and
// every readback is ordered after the last render on the same stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/eleven.h"
#include "adjoint_plan.hpp"
#include "bvh.hpp"
#include "dev_buf.hpp"
#include "hdri_table.hpp"
#include "host_parallel.hpp"
#include "kernels.hpp"
#include "pt_device.hpp"
#include "scene.hpp"
#include "stage.hpp"
#include "wf_buffers.hpp"

using namespace eleven;
using eleven::dev::DevScene;

namespace {

constexpr int kCounterWords = kXcds * kStatSlots;   // per-XCD copies of the tallies (kernels.hpp)

static_assert(kCounterWords <= (int)Stage::kTallyWords, "the stage holds the tallies");

// Sum of the per-XCD copies of tally `slot`.
inline unsigned long long tally(const unsigned long long* h, int slot) {
    unsigned long long s = 0;
    for (int x = 0; x < kXcds; x++) s += h[x * kStatSlots + slot];
    return s;
}

}  // namespace

// ---------------------------------------------------- static device scratch --
// The scratch of el_trace_closest_noalloc: the tallies (kCounterWords 64-bit
// words) and the traversal stack's per-thread spill area, one array per GPU
// that lives until the process ends.  Host code never passes `scratch`
// itself to a kernel (on the host it is only a stand-in for the symbol): each
// device's address comes from hipGetSymbolAddress, looked up once per device
// by el_create with that device current.
constexpr size_t kScratchCounterBytes = 512;                  // >= kCounterWords * 8
constexpr size_t kScratchSpillInts = (size_t(4) << 20) + 1024;   // 16 MiB of spill slots and a block's visit rows
constexpr size_t kScratchBytes = kScratchCounterBytes + kScratchSpillInts * sizeof(int);
static_assert(kScratchCounterBytes >= sizeof(unsigned long long) * kXcds * kStatSlots, "tallies fit");
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static std::mutex g_scratchMu;
static std::vector<void*> g_scratchPtr;   // per device, null until looked up

// Device address of `scratch` on the current device `device`.
static hipError_t scratchAddress(int device, void** out) {
    std::lock_guard<std::mutex> lock(g_scratchMu);
    if ((size_t)device >= g_scratchPtr.size()) g_scratchPtr.resize(device + 1, nullptr);
    if (!g_scratchPtr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratchPtr[device] = p;
    }
    *out = g_scratchPtr[device];
    return hipSuccess;
}

struct el_ctx {
    int device = 0;
    void* scratch = nullptr;       // this device's static scratch (scratchAddress)
    hipStream_t stream = nullptr;
    std::string err;
    int cus = 0;
    uint32_t maxThreads = 0;
    uint32_t block = kDefaultBlock;
    uint32_t refill = kDefaultRefill;

    bool hasScene = false;
    uint32_t ntri = 0;
    std::vector<float> verts;
    Bvh2 bvh2;
    WideBvh wide;
    int width = 4;
    int gcap = 1;

    DevScene ds{};
    el_camera cam{};
    std::vector<dev::DevMaterial> mats;
    std::vector<dev::DevTex> texs;
    std::vector<uint64_t> texF32;   // FP32-pool offset of each texture (el_set_texture)

    DevBuf dNodes, dTris, dShade, dMats, dTexs, dTexels, dLights, dEnvCdf, dEnvGuide, dEnvMap, dEnvBad, dEnvTab, dTexels8, dTexLut, dTangents;
    DevBuf dGstack, dAccum, dCounts, dAov, dCounters;
    WfBuffers wf;

    DevBuf tRays, tTmax, tTri, tT, tUV, tOcc;   // scratch for host-pointer ray queries

    uint32_t sampleBase = 0;
    uint64_t accSeed = 0;          // seed / depth / RNG scene word of the renders in the accumulation
    uint32_t accDepth = 0, accScene = 0;
    bool accPending = false;       // the accumulation is empty, but its buffers are not cleared
    bool accMixed = false;         // renders since el_clear used different seeds or depths
    DevBuf dRec;                   // per (sample, pixel) path radiance of a recorded render
    DevBuf dRecHits, dRecVis, wVis;  // its vertices (RenderArgs::recHits / recVis)
    bool adjSumValid = false;      // aMat / aTex hold the sums of the el_adjoint calls so far
    int32_t adjSumTex = -1;        // their grad_texture
    bool recValid = false;         // the record covers the whole accumulation
    uint64_t totalRays = 0, totalVerts = 0, totalPaths = 0;
    DevBuf aImage, aMat, aTex;     // adjoint image, FP64 material and FP32 texel gradients
    DevBuf aHits, aVis, aQueue;    // el_adjoint: a generation's hits and shadow answers, the replay's queue counts
    DevBuf aTarget, aLoss;         // el_residual_l2: target image, FP64 loss
    size_t residualPx = 0;         // aImage holds el_residual_l2's residual for this many pixels (0: none)
    el_stats stats{};
    bool aovOn = false;

    std::vector<hipEvent_t> evPool;
};

static int fail(el_ctx* c, int code, const std::string& what) {
    if (c) c->err = what;
    return code;
}
static int failHip(el_ctx* c, const char* what, hipError_t e) {
    return fail(c, EL_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

#define EL_HIP(ctx, x)                                   \
    do {                                                 \
        hipError_t e_ = (x);                             \
        if (e_ != hipSuccess) return failHip(ctx, #x, e_); \
    } while (0)

static hipError_t upload(DevBuf& b, const void* src, size_t bytes, hipStream_t st) {
    hipError_t e = b.ensure(bytes);
    if (e != hipSuccess) return e;
    if (bytes) e = hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, st);
    return e;
}

// The tallies to the stage; waits for the stream.
static hipError_t readTallies(StageLease& stage, const unsigned long long* ctr) {
    stage.inFlight(true);
    hipError_t e = hipMemcpyAsync(stage->tallies, ctr, sizeof(unsigned long long) * kCounterWords, hipMemcpyDeviceToHost,
                                  stage.stream());
    if (e == hipSuccess) e = hipStreamSynchronize(stage.stream());
    if (e == hipSuccess) stage.inFlight(false);
    return e;
}

static LaunchCfg cfgOf(el_ctx* c) {
    LaunchCfg l;
    l.stream = c->stream;
    l.block = c->block;
    l.shadeBlock = 256;
    l.refill = c->refill;
    l.maxThreads = l.quadThreads = c->maxThreads;
    l.gstack = c->dGstack.as<int>();
    return l;
}

extern "C" {

int el_device_count(int* out) {
    if (!out) return EL_ERR_ARG;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) n = 0;
    *out = n;
    return EL_OK;
}

int el_create(el_ctx** out, int device) {
    if (!out) return EL_ERR_ARG;
    *out = nullptr;
    std::unique_ptr<el_ctx> c(new el_ctx());
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return EL_ERR_HIP;
    if (device < 0 || device >= n) return EL_ERR_ARG;
    c->device = device;
    if (hipSetDevice(device) != hipSuccess) return EL_ERR_HIP;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return EL_ERR_HIP;
    c->cus = prop.multiProcessorCount;
    // resident-thread capacity: 32 waves of 64 lanes per CU
    c->maxThreads = (uint32_t)c->cus * 2048u;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) return EL_ERR_HIP;
    if (c->dCounters.ensure(sizeof(unsigned long long) * kCounterWords) != hipSuccess) return EL_ERR_HIP;
    if (scratchAddress(device, &c->scratch) != hipSuccess) return EL_ERR_HIP;
    stagePool().contexts(device, 1);
    *out = c.release();
    return EL_OK;
}

void el_destroy(el_ctx* c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (auto e : c->evPool) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    stagePool().contexts(c->device, -1);
    delete c;
}

const char* el_last_error(const el_ctx* c) { return c ? c->err.c_str() : "null context"; }

}  // extern "C"

// Pack and upload the wide BVH of the current width.
// 8-bit copy of an RGB FP32 texture: R | G << 8 | B << 16 per texel, each
// byte the index of the value in `table` (bit-exact); false if some value is
// not in the table.  The table is non-decreasing (the loader's fastPow of
// i / 255), so each value is found by binary search.
static bool packLdr(const float* rgb, size_t n, const float (&table)[256], uint32_t* out) {
    std::atomic<bool> ok{true};
    parallelFor(n, [&](size_t i0, size_t i1) {
        for (size_t i = i0; i < i1 && ok.load(std::memory_order_relaxed); i++) {
            uint32_t w = 0;
            for (int ch = 0; ch < 3; ch++) {
                const float v = rgb[3 * i + ch];
                const float* p = std::lower_bound(table, table + 256, v);
                if (p == table + 256 || std::memcmp(p, &v, 4) != 0) {
                    ok = false;
                    return;
                }
                w |= (uint32_t)(p - table) << (8 * ch);
            }
            out[i] = w;
        }
    });
    return ok;
}

// The device camera: the host fields plus the six trig values the reference
// evaluates per ray (kernel.cu:304-306) after rotation *= (PI / 180.0) as
// Vector3 *= float (kernel.cu:301).
static dev::DevCamera devCamera(const el_camera& cam) {
    dev::DevCamera dc{};
    dc.xRes = cam.x_res;
    dc.yRes = cam.y_res;
    dc.focalLength = cam.focal_length;
    dc.sensorWidth = cam.sensor_width;
    dc.sensorHeight = cam.sensor_height;
    dc.aperture = cam.aperture;
    dc.focusDistance = cam.focus_distance;
    const float toRad = (float)(3.14159265358979323846f / 180.0);
    const float rx = cam.rotation.x * toRad, ry = cam.rotation.y * toRad, rz = cam.rotation.z * toRad;
    dc.cosRot[0] = std::cos(rx);
    dc.sinRot[0] = std::sin(rx);
    dc.cosRot[1] = std::cos(ry);
    dc.sinRot[1] = std::sin(ry);
    dc.cosRot[2] = std::cos(rz);
    dc.sinRot[2] = std::sin(rz);
    dc.pos[0] = cam.position.x;
    dc.pos[1] = cam.position.y;
    dc.pos[2] = cam.position.z;
    dc.bokeh = cam.bokeh;
    return dc;
}

// Material values as the kernels read them (texture ids are set by the
// caller); for untextured roughness and metallic also generateHitData's
// powf(x, 2.2f) (kernel.cu:113-114), once per material.
static void setMaterialValues(dev::DevMaterial& d, const el_material& m) {
    d.albedo[0] = m.albedo.x;
    d.albedo[1] = m.albedo.y;
    d.albedo[2] = m.albedo.z;
    d.emission[0] = m.emission.x;
    d.emission[1] = m.emission.y;
    d.emission[2] = m.emission.z;
    d.roughness = m.roughness;
    d.metallic = m.metallic;
    d.roughnessEff = powf(m.roughness, 2.2f);
    d.metallicEff = powf(m.metallic, 2.2f);
    d.clearcoatGloss = m.clearcoat_gloss;
    d.clearcoat = m.clearcoat;
    d.anisotropic = m.anisotropic;
    d.eta = m.eta;
    d.transmission = m.transmission;
    d.specular = m.specular;
    d.specularTint = m.specular_tint;
    d.sheenTint = m.sheen_tint;
    d.subsurface = m.subsurface;
    d.sheen = m.sheen;
}

static int uploadBvh(el_ctx* c, int width) {
    try {
        c->wide = collapseWide(c->bvh2, c->verts.data(), (int)c->ntri, width);
        if (width == 4)   // the nodes as the device reads them, in the place of the others
            parallelFor(c->wide.nodeCount, [&](size_t i0, size_t i1) {
                for (size_t i = i0; i < i1; i++) {
                    unsigned char* const at = c->wide.nodes.data() + i * sizeof(QNode<4>);
                    QNode<4> n;
                    uint32_t words[16];
                    static_assert(sizeof words == sizeof n, "a node keeps its size");
                    std::memcpy(&n, at, sizeof n);
                    packLaneNode(n, words);
                    std::memcpy(at, words, sizeof words);
                }
            });
    } catch (const std::exception& ex) {
        return fail(c, EL_ERR_RANGE, ex.what());
    }
    c->width = width;
    EL_HIP(c, upload(c->dNodes, c->wide.nodes.data(), c->wide.nodes.size(), c->stream));
    EL_HIP(c, upload(c->dTris, c->wide.triStream.data(), c->wide.triStream.size() * sizeof(float), c->stream));
    c->gcap = dev::spillRows(c->wide.stackBound);
    EL_HIP(c, c->dGstack.ensure((size_t)c->gcap * c->maxThreads * sizeof(int)));
    c->ds.nodes = c->dNodes.p;
    c->ds.tris = c->dTris.as<float4>();
    c->ds.width = width;
    c->ds.gcap = c->gcap;
    c->ds.quads = width == 4 && c->wide.stackBound + 2 <= dev::kQuadStack;
    c->ds.slabUnit = dev::slabUnitOf(c->wide.maxStepExponent);
    c->stats.bvh_width = (uint32_t)width;
    c->stats.stack_bound = (uint32_t)c->wide.stackBound;
    c->stats.node_bytes = c->wide.nodes.size();
    c->stats.tri_bytes = c->wide.triStream.size() * sizeof(float);
    c->stats.node_stride = (uint32_t)c->wide.nodeStride;
    c->stats.tri_stride = 12 * sizeof(float);
    EL_HIP(c, hipStreamSynchronize(c->stream));
    return EL_OK;
}

// Gives back the buffers of a recording render (EL_FLAG_RECORD_PATHS), which
// cover only the accumulation they were recorded into: at the next render that
// does not record, with the scene, and with the accumulation if they
// are larger than kKeptRecord (recording steps in a row keep smaller ones, whose
// allocation takes as long as the step's rays).
constexpr size_t kKeptRecord = size_t(2) << 30;
static void releaseRecord(el_ctx* c) {
    c->dRec.release();
    c->dRecHits.release();
    c->dRecVis.release();
    c->wVis.release();
}

// Empties the accumulation.  Its sums and counts are not written here: the next
// wavefront render starts them from zero (RenderArgs::fresh), and whatever
// else reads them first clears them (clearPending).
static int clearAccum(el_ctx* c) {
    if (c->dAov.p) EL_HIP(c, hipMemsetAsync(c->dAov.p, 0, c->dAov.n, c->stream));
    c->accPending = true;
    c->sampleBase = 0;
    c->accMixed = false;
    c->recValid = false;
    if (c->dRec.n + c->dRecHits.n + c->dRecVis.n + c->wVis.n > kKeptRecord) releaseRecord(c);
    c->totalRays = c->totalVerts = c->totalPaths = 0;
    return EL_OK;
}
static hipError_t clearPending(el_ctx* c) {
    if (!c->accPending) return hipSuccess;
    const size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    hipError_t e = hipMemsetAsync(c->dAccum.p, 0, npx * sizeof(float4), c->stream);
    if (e == hipSuccess) e = hipMemsetAsync(c->dCounts.p, 0, npx * sizeof(uint32_t), c->stream);
    if (e == hipSuccess) c->accPending = false;
    return e;
}

extern "C" {

int el_upload_scene(el_ctx* c, const el_scene_view* v) {
    if (!c || !v) return fail(c, EL_ERR_ARG, "null argument");
    if (v->tri_count && (!v->vertices || !v->object_id)) return fail(c, EL_ERR_ARG, "missing triangle arrays");
    if (v->camera.x_res == 0 || v->camera.y_res == 0) return fail(c, EL_ERR_ARG, "camera resolution is zero");
    if ((uint64_t)v->camera.x_res * v->camera.y_res > (1ull << 28))
        return fail(c, EL_ERR_RANGE, "resolution above 2^28 pixels");
    if (v->tri_count >= (uint32_t)kLeafFirstLimit) return fail(c, EL_ERR_RANGE, "more than 2^27 triangles");
    if (v->material_count == 0 || !v->materials) return fail(c, EL_ERR_ARG, "at least one material is required");
    if (v->mesh_count == 0 || !v->mesh_material) return fail(c, EL_ERR_ARG, "mesh table missing");
    if (!v->hdri.data || v->hdri.width <= 0 || v->hdri.height <= 0) return fail(c, EL_ERR_ARG, "hdri missing");
    if (v->light_count && !v->lights) return fail(c, EL_ERR_ARG, "lights missing");
    for (uint32_t i = 0; i < v->texture_count; i++)
        if (!v->textures[i].data || v->textures[i].width <= 0 || v->textures[i].height <= 0)
            return fail(c, EL_ERR_ARG, "texture " + std::to_string(i) + " is empty");
    EL_HIP(c, hipSetDevice(c->device));
    c->hasScene = false;
    c->adjSumValid = false;
    c->residualPx = 0;
    releaseRecord(c);
    c->ntri = v->tri_count;
    c->cam = v->camera;

    // geometry + BVH
    c->verts.assign(v->vertices, v->vertices + (size_t)v->tri_count * 9);
    c->bvh2 = buildBvh2(c->verts.data(), (int)c->ntri);
    int rc = uploadBvh(c, c->width);
    if (rc) return rc;

    // shading records and corner tangents, indexed by original triangle
    std::vector<float> shade((size_t)v->tri_count * dev::kShadeFloats, 0.f);
    std::vector<float> tans((size_t)v->tri_count * dev::kTanFloats, 0.f);
    parallelFor(v->tri_count, [&](size_t i0, size_t i1) {
        for (uint32_t i = (uint32_t)i0; i < (uint32_t)i1; i++) {
            float* S = &shade[(size_t)i * dev::kShadeFloats];
            std::memcpy(S, v->vertices + (size_t)i * 9, 9 * sizeof(float));
            if (v->normals) std::memcpy(S + 9, v->normals + (size_t)i * 9, 9 * sizeof(float));
            if (v->uvs) std::memcpy(S + 18, v->uvs + (size_t)i * 6, 6 * sizeof(float));
            int32_t obj = v->object_id[i];
            int32_t mat = (obj >= 0 && (uint32_t)obj < v->mesh_count) ? v->mesh_material[obj] : 0;
            if (mat < 0 || (uint32_t)mat >= v->material_count) mat = 0;
            std::memcpy(&S[24], &mat, 4);
            S[25] = v->tangent_sign ? v->tangent_sign[i] : 0.f;
            if (v->tangents) std::memcpy(&tans[(size_t)i * dev::kTanFloats], v->tangents + (size_t)i * 9, 9 * sizeof(float));
        }
    });
    EL_HIP(c, upload(c->dShade, shade.data(), shade.size() * sizeof(float), c->stream));
    EL_HIP(c, upload(c->dTangents, tans.data(), tans.size() * sizeof(float), c->stream));

    // textures: one FP32 pool, the environment map last.  A texture whose
    // every value is an entry of one of the loader's byte -> value tables
    // (an 8-bit file) also gets an 8-bit copy, which the kernels read.
    std::vector<float> pool;
    std::vector<uint32_t> pool8;
    float tables[2][256];
    ldrTable(sRGB, tables[0]);
    ldrTable(LINEAR, tables[1]);
    c->texs.clear();
    c->texF32.clear();
    auto addTex = [&](const el_texture& t, bool mayPack) {
        dev::DevTex d{};
        d.w = t.width;
        d.h = t.height;
        d.xTile = t.x_tile;
        d.yTile = t.y_tile;
        d.xOffset = t.x_offset;
        d.yOffset = t.y_offset;
        d.filter = t.filter;
        d.format = dev::kTexF32;
        d.offset = pool.size();
        const size_t n = (size_t)t.width * t.height;
        pool.insert(pool.end(), t.data, t.data + n * 3);
        for (int k = 0; mayPack && k < 2; k++) {
            std::vector<uint32_t> words(n);
            if (!packLdr(t.data, n, tables[k], words.data())) continue;
            d.format = dev::kTexLdr + k;
            d.offset = pool8.size();
            pool8.insert(pool8.end(), words.begin(), words.end());
            break;
        }
        return d;
    };
    for (uint32_t i = 0; i < v->texture_count; i++) {
        c->texF32.push_back(pool.size());
        c->texs.push_back(addTex(v->textures[i], true));
    }
    dev::DevTex env = addTex(v->hdri, false);
    EL_HIP(c, upload(c->dTexels, pool.data(), pool.size() * sizeof(float), c->stream));
    EL_HIP(c, upload(c->dTexels8, pool8.data(), pool8.size() * sizeof(uint32_t), c->stream));
    EL_HIP(c, upload(c->dTexLut, tables, sizeof tables, c->stream));
    c->stats.texels_8bit = pool8.size();
    EL_HIP(c, upload(c->dTexs, c->texs.data(), c->texs.size() * sizeof(dev::DevTex), c->stream));

    // materials
    c->mats.assign(v->material_count, dev::DevMaterial{});
    for (uint32_t i = 0; i < v->material_count; i++) {
        const el_material& m = v->materials[i];
        dev::DevMaterial& d = c->mats[i];
        auto texOk = [&](int32_t id) { return (id >= 0 && (uint32_t)id < v->texture_count) ? id : -1; };
        d.albedoTex = texOk(m.albedo_tex);
        d.emissionTex = texOk(m.emission_tex);
        d.roughnessTex = texOk(m.roughness_tex);
        d.metallicTex = texOk(m.metallic_tex);
        d.normalTex = texOk(m.normal_tex);
        setMaterialValues(d, m);
    }
    EL_HIP(c, upload(c->dMats, c->mats.data(), c->mats.size() * sizeof(dev::DevMaterial), c->stream));

    // lights
    std::vector<float> lights((size_t)v->light_count * 6);
    for (uint32_t i = 0; i < v->light_count; i++) {
        const el_point_light& l = v->lights[i];
        float* L = &lights[(size_t)i * 6];
        L[0] = l.position.x;
        L[1] = l.position.y;
        L[2] = l.position.z;
        L[3] = l.radiance.x;
        L[4] = l.radiance.y;
        L[5] = l.radiance.z;
    }
    EL_HIP(c, upload(c->dLights, lights.data(), lights.size() * sizeof(float), c->stream));

    // HDRI CDF exactly as HDRI::generateCDF at construction (offsets still 0),
    // then the alias table of the search's effective distribution.
    const el_texture& h = v->hdri;
    HdriSampler hs = buildHdriSampler(h.data, h.width, h.height);
    EL_HIP(c, upload(c->dEnvCdf, hs.cdf.data(), hs.cdf.size() * sizeof(float), c->stream));
    EL_HIP(c, upload(c->dEnvGuide, hs.guide.data(), hs.guide.size() * sizeof(int32_t), c->stream));
    EL_HIP(c, upload(c->dEnvMap, hs.map2.data(), hs.map2.size() * sizeof(int32_t), c->stream));
    const std::vector<uint32_t> badBits =
        hdriBadBuckets(hs, h.data, h.width, h.height, h.x_tile, h.y_tile, h.x_offset, h.y_offset);
    EL_HIP(c, upload(c->dEnvBad, badBits.data(), badBits.size() * sizeof(uint32_t), c->stream));

    // accumulation
    size_t npx = (size_t)v->camera.x_res * v->camera.y_res;
    EL_HIP(c, c->dAccum.ensure(npx * sizeof(float4)));
    EL_HIP(c, c->dCounts.ensure(npx * sizeof(uint32_t)));
    c->dAov.release();

    DevScene& s = c->ds;
    s.shade = c->dShade.as<float4>();
    s.tangents = c->dTangents.as<float4>();
    s.mats = c->dMats.as<dev::DevMaterial>();
    s.texs = c->dTexs.as<dev::DevTex>();
    s.texels = c->dTexels.as<float>();
    s.texels8 = c->dTexels8.as<uint32_t>();
    s.texLut = c->dTexLut.as<float>();
    s.lights = c->dLights.as<float>();
    s.envCdf = c->dEnvCdf.as<float>();
    s.envGuide = c->dEnvGuide.as<int32_t>();
    s.envMap = c->dEnvMap.as<int32_t>();
    s.envBad = c->dEnvBad.as<uint32_t>();
    s.env = env;
    s.envRadianceSum = hs.radianceSum;
    EL_HIP(c, c->dEnvTab.ensure((size_t)h.width * h.height * 2 * sizeof(float4)));
    s.envTab = c->dEnvTab.as<float4>();
    s.envLog2G = hs.log2G;
    s.nLights = (int32_t)v->light_count;
    s.nTris = (int32_t)v->tri_count;
    s.cam = devCamera(v->camera);
    EL_HIP(c, launchEnvTable(c->stream, s, c->dEnvTab.as<float4>()));
    rc = clearAccum(c);
    if (rc) return rc;
    EL_HIP(c, hipStreamSynchronize(c->stream));   // the uploads: a batch uses the scene on another stream
    c->hasScene = true;
    return EL_OK;
}

int el_set_camera(el_ctx* c, const el_camera* cam) {
    if (!c || !cam) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (cam->x_res == 0 || cam->y_res == 0) return fail(c, EL_ERR_ARG, "camera resolution is zero");
    if ((uint64_t)cam->x_res * cam->y_res > (1ull << 28)) return fail(c, EL_ERR_RANGE, "resolution above 2^28 pixels");
    EL_HIP(c, hipSetDevice(c->device));
    const size_t npx = (size_t)cam->x_res * cam->y_res;
    EL_HIP(c, c->dAccum.ensure(npx * sizeof(float4)));
    EL_HIP(c, c->dCounts.ensure(npx * sizeof(uint32_t)));
    if (cam->x_res != c->cam.x_res || cam->y_res != c->cam.y_res) c->dAov.release();
    c->cam = *cam;
    c->ds.cam = devCamera(*cam);
    c->residualPx = 0;   // the residual of el_residual_l2 belongs to the previous view
    return clearAccum(c);
}

int el_clear(el_ctx* c) {
    if (!c) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    EL_HIP(c, hipSetDevice(c->device));
    return clearAccum(c);
}

}  // extern "C"

// Generations with fewer paths trace every bounce's shadows in one launch with
// the next extension; larger ones from the third bounce on (bounceTogether).
constexpr uint32_t kTogetherPaths = 16u << 20;

// Large launches keep the GPU busy on their own, and rays of different queues
// side by side cost cache hits (the extension's L2 hit rate fell from 0.70 to
// 0.62 next to the first bounce's shadows); small ones last one ray's chain
// of dependent fetches, which the three queues then spend at once.
static bool bounceTogether(uint32_t paths, uint32_t bounce) { return paths < kTogetherPaths || bounce >= 2; }

static hipEvent_t poolEvent(el_ctx* c, size_t i) {
    while (c->evPool.size() <= i) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        c->evPool.push_back(e);
    }
    return c->evPool[i];
}

// Generation size and wavefront state for `total` work items of a frame
// with `npad` padded pixels: Q paths per generation (queueCap, or by default
// as many as a quarter of the free device memory holds), rounded to whole
// sample passes or 64-path groups; q points at the context's buffers.
static int wfPlan(el_ctx* c, const LaunchCfg& lc, uint64_t total, uint64_t npad, uint64_t queueCap, bool aov,
                  WfState& q, uint64_t& Q) {
    // Default: as many paths in flight as a quarter of the free device
    // memory holds (~216 B of queue and path state per path), so a
    // 1080p x 64 spp frame runs as a single generation.
    Q = queueCap;
    if (!Q && total <= c->wf.cap && (!aov || c->wf.aov.n >= total * 48)) Q = total;   // held already
    if (!Q) {
        size_t freeB = 0, totalB = 0;
        EL_HIP(c, hipMemGetInfo(&freeB, &totalB));
        const uint64_t perPath = 6 * 32 + 60 + (aov ? 48 : 0);
        Q = std::max<uint64_t>(1u << 20, freeB / 4 / perPath);
    }
    if (Q >= npad)
        Q = (Q / npad) * npad;
    else
        Q = std::max<uint64_t>(64, (Q / 64) * 64);
    if (Q > total) Q = total;
    if (Q > 0x7fffffffull) return fail(c, EL_ERR_RANGE, "queue capacity above 2^31");
    // Entries one XCD's blocks can append in one launch: at most
    // ceil(Q/8) + maxThreads/8 + block (grid-stride over <= maxThreads,
    // block <= kMaxBlock).
    const uint64_t segSize = (Q + kXcds - 1) / kXcds + lc.maxThreads / kXcds + kMaxBlock;
    const uint64_t qcap = std::max<uint64_t>(Q, kXcds * segSize);
    EL_HIP(c, c->wf.ensure(Q, qcap, aov, kQCounters * sizeof(uint32_t)));
    if (!c->wf.holds(Q, qcap, aov))
        return fail(c, EL_ERR_STATE, "wavefront buffers smaller than the generation (internal error)");
    q.ray[0] = c->wf.ray0.as<float4>();
    q.ray[1] = c->wf.ray1.as<float4>();
    q.hits = c->wf.hits.as<float4>();
    q.shadowH = c->wf.shadowH.as<float4>();
    q.shadowP = c->wf.shadowP.as<float4>();
    q.pathT = c->wf.pathT.as<float4>();
    q.pathL = c->wf.pathL.as<float4>();
    q.pathPix = c->wf.pix.as<uint32_t>();
    q.pathSample = c->wf.sample.as<uint32_t>();
    q.pathQuiet = c->wf.quiet.as<uint64_t>();
    q.pathAov = aov ? c->wf.aov.as<float4>() : nullptr;
    q.pendP = c->wf.pend.as<float4>();
    q.counters = c->wf.counters.as<uint32_t>();
    q.segSize = (uint32_t)segSize;
    q.cap = qcap;
    q.gstack = lc.gstack;
    q.gthreads = lc.maxThreads;
    return EL_OK;
}

// Camera rays and every bounce of the generation a.genCount: extend -> shade ->
// both shadow queues.  Where the launches are small, the shadows of bounce b
// and the extension of bounce b + 1 are one launch (launchWfTrace).  With
// EL_FLAG_KERNEL_TIMES in `flags` the launches are timed by evPool's events
// from `ev` on (`timed`: event index, kind 0 extend, 1 shade, 2 shadow).
static int wfWalk(el_ctx* c, const LaunchCfg& lc, RenderArgs a, WfState q, uint32_t flags,
                  std::vector<std::pair<size_t, int>>& timed, size_t& ev, unsigned long long* ctr) {
    const bool apart = (flags & (EL_FLAG_SERIAL_SHADOWS | EL_FLAG_KERNEL_TIMES | EL_FLAG_COUNT_TRAVERSAL)) != 0;
    const bool kernelTimes = (flags & EL_FLAG_KERNEL_TIMES) != 0;
    auto launch = [&](int kind, auto&& f) -> hipError_t {   // one launch, timed if asked
        if (!kernelTimes) return f();
        hipEvent_t x0 = poolEvent(c, ev), x1 = poolEvent(c, ev + 1);
        if (!x0 || !x1) return hipErrorOutOfMemory;
        hipError_t e = hipEventRecord(x0, c->stream);
        if (e == hipSuccess) e = f();
        if (e == hipSuccess) e = hipEventRecord(x1, c->stream);
        timed.push_back({ev, kind});
        ev += 2;
        return e;
    };
    EL_HIP(c, launchWfCamera(lc, c->ds, a, q, ctr));
    bool extended = false;   // bounce b's closest hits were traced with the previous bounce's shadows
    for (uint32_t b = 0; b < a.maxDepth; b++) {
        const bool together = !apart && bounceTogether(a.genCount, b), more = b + 1 < a.maxDepth;
        a.bounce = b;
        q.parity = b & 1u;
        q.deferP = together ? 1u : 0u;
        q.visBit = q.pathVis ? 1u << (2 * b) : 0u;
        const int cur = b & 1, nxt = cur ^ 1;
        uint32_t* cntCur = q.counters + (cur ? kQRay1 : kQRay0);
        uint32_t* cntNxt = q.counters + (nxt ? kQRay1 : kQRay0);
        if (!extended)
            EL_HIP(c, launch(0, [&] {
                return launchWfExtend(lc, c->ds, q, q.ray[cur], cntCur, cntNxt, a.genCount,
                                      (flags & EL_FLAG_COUNT_TRAVERSAL) != 0, ctr);
            }));
        EL_HIP(c, launch(1, [&] {
            return launchWfShade(lc, c->ds, a, q, q.ray[cur], cntCur, q.ray[nxt], cntNxt, a.genCount, ctr);
        }));
        if (together) {
            EL_HIP(c, launchWfTrace(lc, c->ds, q, more ? q.ray[nxt] : nullptr, cntNxt, cntCur, a.genCount, ctr));
        } else {
            for (int light = 0; light < 2; light++)
                EL_HIP(c, launch(2, [&] { return launchWfShadow(lc, c->ds, q, light, a.genCount, ctr); }));
        }
        extended = together && more;
    }
    return EL_OK;
}

extern "C" int el_render(el_ctx* c, const el_render_params* p) {
    if (!c || !p) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (p->mode != EL_MODE_PLAIN && p->mode != EL_MODE_WAVEFRONT) return fail(c, EL_ERR_ARG, "unknown mode");
    if (p->bvh_width != 0 && p->bvh_width != 4 && p->bvh_width != 8) return fail(c, EL_ERR_ARG, "bvh_width must be 4 or 8");
    if (p->block != 0 && (p->block % 64 != 0 || p->block > (uint32_t)kMaxBlock))
        return fail(c, EL_ERR_ARG, "block must be a multiple of 64, at most 256");
    uint32_t depth = p->max_depth ? p->max_depth : 5;
    if (depth > 64) return fail(c, EL_ERR_RANGE, "max_depth above 64");
    EL_HIP(c, hipSetDevice(c->device));
    if (p->spp == 0) return EL_OK;
    StageLease stage(c->device, c->stream);
    EL_HIP(c, stage.take());
    if (p->bvh_width && (int)p->bvh_width != c->width) {
        int rc = uploadBvh(c, (int)p->bvh_width);
        if (rc) return rc;
    }
    if (p->refill > 64) return fail(c, EL_ERR_ARG, "refill must be 0..64");
    c->block = p->block ? p->block : kDefaultBlock;
    c->refill = p->refill ? p->refill : kDefaultRefill;
    bool aov = (p->flags & EL_FLAG_AOV) != 0;
    size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    if (aov && !c->dAov.p) {
        EL_HIP(c, c->dAov.ensure(npx * 3 * sizeof(float4)));
        EL_HIP(c, hipMemsetAsync(c->dAov.p, 0, c->dAov.n, c->stream));
    }
    c->aovOn = c->aovOn || aov;
    float4* aovBuf = aov ? c->dAov.as<float4>() : nullptr;
    unsigned long long* ctr = c->dCounters.as<unsigned long long>();
    if (p->mode == EL_MODE_PLAIN) {
        EL_HIP(c, hipMemsetAsync(ctr, 0, sizeof(unsigned long long) * kCounterWords, c->stream));
        EL_HIP(c, clearPending(c));
    }
    LaunchCfg lc = cfgOf(c);
    RenderArgs a{};
    a.k0 = (uint32_t)p->seed;
    a.k1 = (uint32_t)(p->seed >> 32);
    a.scene = p->rng_scene;
    a.maxDepth = depth;
    a.sample = c->sampleBase;
    a.cull = (p->flags & EL_FLAG_NO_CULL) ? 0u : 1u;
    bool record = (p->flags & EL_FLAG_RECORD_PATHS) != 0;
    if (record && c->sampleBase != 0) return fail(c, EL_ERR_STATE, "EL_FLAG_RECORD_PATHS needs a cleared accumulation");
    // Wavefront renders record every vertex's hit and shadow answers (16 B per
    // vertex + 4 B per path) and the paths' radiance (16 B), from which el_adjoint
    // replays without tracing, when the radiance fits half of the free device
    // memory and the vertices a quarter of the rest.  Without the vertices the
    // adjoint walks the paths again, and has no use for their radiance.
    record = record && p->mode != EL_MODE_PLAIN && depth <= (uint32_t)dev::kAdjMaxDepthHost;
    if (record) {
        const size_t recBytes = (size_t)p->spp * npx * sizeof(float4), hitBytes = recBytes * depth;
        auto holds = [](const DevBuf& b, size_t n) { return b.p && n <= b.n && n >= b.n / 4; };
        // buffers of another size go back first: the rules are about the memory without them
        if (!holds(c->dRec, recBytes) || !holds(c->dRecHits, hitBytes)) {
            releaseRecord(c);
            size_t freeB = 0, totalB = 0;
            EL_HIP(c, hipMemGetInfo(&freeB, &totalB));
            record = recBytes <= freeB / 2 && hitBytes <= (freeB - recBytes) / 4;
        }
    }
    if (record) {
        const size_t paths = (size_t)p->spp * npx;
        EL_HIP(c, c->dRec.ensure(paths * sizeof(float4)));
        EL_HIP(c, c->dRecHits.ensure(paths * depth * sizeof(float4)));
        EL_HIP(c, c->dRecVis.ensure(paths * sizeof(uint32_t)));
        a.rec = c->dRec.as<float4>();
        a.recHits = c->dRecHits.as<float4>();
        a.recVis = c->dRecVis.as<uint32_t>();
        a.recStride = paths;
    } else if (c->dRec.p) {
        releaseRecord(c);
    }
    c->recValid = false;

    hipEvent_t e0 = poolEvent(c, 0), e1 = poolEvent(c, 1);
    if (!e0 || !e1) return fail(c, EL_ERR_HIP, "event creation failed");
    double extendMs = 0, shadeMs = 0, shadowMs = 0;
    uint64_t extendLaunches = 0;
    EL_HIP(c, hipEventRecord(e0, c->stream));
    const unsigned long long* const h = stage->tallies;   // the launches' tallies, read back with the last sync

    if (p->mode == EL_MODE_PLAIN) {
        for (uint32_t s = 0; s < p->spp; s++) {
            a.sample = c->sampleBase + s;
            EL_HIP(c, launchPlain(lc, c->ds, a, c->dAccum.as<float4>(), c->dCounts.as<uint32_t>(), aovBuf, ctr));
        }
    } else {
        const uint32_t tilesX = (c->cam.x_res + 7) / 8, tilesY = (c->cam.y_res + 7) / 8;
        const uint64_t npad = (uint64_t)tilesX * tilesY * 64;
        uint64_t total = (uint64_t)p->spp * npad;
        if (npad >= (1ull << 31)) return fail(c, EL_ERR_RANGE, "frame too large for the wavefront renderer");
        uint64_t Q = 0;
        WfState q{};
        int rc = wfPlan(c, lc, total, npad, p->queue_cap, aov, q, Q);
        if (rc) return rc;
        if (record) {
            EL_HIP(c, c->wVis.ensure(Q * sizeof(uint32_t)));
            q.pathVis = c->wVis.as<uint32_t>();
        }
        a.npad = (uint32_t)npad;
        size_t ev = 2;
        std::vector<std::pair<size_t, int>> timed;   // (event index, kind) kind 0 extend 1 shade 2 shadow
        for (uint64_t start = 0; start < total; start += Q) {
            a.genPixel = (uint32_t)(start % npad);
            a.genSample = (uint32_t)(start / npad);
            a.genCount = (uint32_t)std::min<uint64_t>(Q, total - start);
            a.run = a.genPixel == 0 && a.genCount % npad == 0 ? (uint32_t)(a.genCount / npad) : 0u;
            a.fresh = c->accPending ? 1u : 0u;
            a.zeroTallies = start == 0 ? 1u : 0u;
            rc = wfWalk(c, lc, a, q, p->flags, timed, ev, ctr);
            if (rc) return rc;
            extendLaunches += depth;
            EL_HIP(c, launchWfFinalize(lc, c->ds, a, q, c->dAccum.as<float4>(), c->dCounts.as<uint32_t>(), aovBuf,
                                       ctr));
        }
        c->accPending = false;
        EL_HIP(c, hipEventRecord(e1, c->stream));
        EL_HIP(c, readTallies(stage, ctr));   // the tallies and every event
        for (auto& t : timed) {
            float ms = 0;
            EL_HIP(c, hipEventElapsedTime(&ms, c->evPool[t.first], c->evPool[t.first + 1]));
            (t.second == 0 ? extendMs : t.second == 1 ? shadeMs : shadowMs) += ms;
        }
    }
    if (p->mode == EL_MODE_PLAIN) {
        EL_HIP(c, hipEventRecord(e1, c->stream));
        EL_HIP(c, readTallies(stage, ctr));
    }
    float totalMs = 0;
    EL_HIP(c, hipEventElapsedTime(&totalMs, e0, e1));
    if (c->sampleBase == 0) {
        c->accSeed = p->seed;
        c->accDepth = depth;
        c->accScene = p->rng_scene;
    } else if (c->accSeed != p->seed || c->accDepth != depth || c->accScene != p->rng_scene) {
        c->accMixed = true;
    }
    c->sampleBase += p->spp;
    c->recValid = record;
    c->stats.record_bytes = record ? c->dRec.n + c->dRecHits.n + c->dRecVis.n + c->wVis.n : 0;
    c->totalRays += tally(h, kStatRays);
    c->totalVerts += tally(h, kStatVerts);
    c->totalPaths += tally(h, kStatPaths);
    c->stats.rays = tally(h, kStatRays);
    c->stats.vertices = tally(h, kStatVerts);
    c->stats.paths = tally(h, kStatPaths);
    c->stats.render_ms = totalMs;
    c->stats.extend_ms = extendMs;
    c->stats.shade_ms = shadeMs;
    c->stats.shadow_ms = shadowMs;
    c->stats.extend_launches = extendLaunches;
    c->stats.extend_rays = tally(h, kStatExtRays);
    c->stats.node_fetches = tally(h, kStatNodes);
    c->stats.tri_tests = tally(h, kStatTris);
    if (tally(h, kStatOverflow)) return fail(c, EL_ERR_RANGE, "traversal stack or queue overflow (results incomplete)");
    return EL_OK;
}

extern "C" int el_residual_l2(el_ctx* c, const float* target, double* loss) {
    if (!c || !target) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (c->sampleBase == 0) return fail(c, EL_ERR_STATE, "nothing rendered since el_clear");
    EL_HIP(c, hipSetDevice(c->device));
    const size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    EL_HIP(c, c->aImage.ensure(npx * 3 * sizeof(float)));
    EL_HIP(c, c->aTarget.ensure(npx * 3 * sizeof(float)));
    EL_HIP(c, c->aLoss.ensure(sizeof(double)));
    EL_HIP(c, hipMemcpyAsync(c->aTarget.p, target, npx * 3 * sizeof(float), hipMemcpyHostToDevice, c->stream));
    EL_HIP(c, hipMemsetAsync(c->aLoss.p, 0, sizeof(double), c->stream));
    EL_HIP(c, launchResidualL2(c->stream, c->dAccum.as<float4>(), c->dCounts.as<uint32_t>(), c->aTarget.as<float>(),
                               (uint32_t)npx, c->aImage.as<float>(), c->aLoss.as<double>()));
    double h = 0.0;
    EL_HIP(c, hipMemcpyAsync(&h, c->aLoss.p, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    EL_HIP(c, hipStreamSynchronize(c->stream));
    if (loss) *loss = h;
    c->residualPx = npx;
    return EL_OK;
}

// Bytes of an output of el_adjoint up to which it is copied with the tallies.
constexpr size_t kOneWait = 1u << 20;

extern "C" int el_adjoint(el_ctx* c, const el_adjoint_params* p, const float* dimage, float* dmat, float* dtex,
                          int devp) {
    const bool accumulate = (p && (p->flags & EL_ADJ_ACCUMULATE) != 0);
    const bool devResidual = (p && (p->flags & EL_ADJ_DEVICE_RESIDUAL) != 0);
    if (!c || !p || (!dimage && !devResidual)) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (c->sampleBase == 0) return fail(c, EL_ERR_STATE, "nothing rendered since el_clear: no image to differentiate");
    if (c->accMixed) return fail(c, EL_ERR_STATE, "the accumulation mixes renders of different seeds or depths");
    if (c->accDepth > (uint32_t)dev::kAdjMaxDepthHost) return fail(c, EL_ERR_RANGE, "adjoint supports max_depth <= 16");
    if (p->block != 0 && (p->block % 64 != 0 || p->block > (uint32_t)kMaxBlock))
        return fail(c, EL_ERR_ARG, "block must be a multiple of 64, at most 256");
    const int gtex = p->grad_texture;
    if (gtex >= (int)c->texs.size()) return fail(c, EL_ERR_ARG, "grad_texture out of range");
    if (accumulate && (!c->adjSumValid || c->adjSumTex != gtex))
        return fail(c, EL_ERR_STATE, "EL_ADJ_ACCUMULATE without a previous el_adjoint with the same grad_texture");
    EL_HIP(c, hipSetDevice(c->device));
    StageLease stage(c->device, c->stream);
    EL_HIP(c, stage.take());
    const size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    const size_t M = c->mats.size();
    const size_t ntex = gtex >= 0 ? (size_t)c->texs[gtex].w * c->texs[gtex].h * 3 : 0;
    const hipMemcpyKind h2d = devp ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    if (devResidual) {
        if (c->residualPx != npx)
            return fail(c, EL_ERR_STATE, "EL_ADJ_DEVICE_RESIDUAL without an el_residual_l2 at this resolution");
    } else {
        EL_HIP(c, c->aImage.ensure(npx * 3 * sizeof(float)));
        EL_HIP(c, hipMemcpyAsync(c->aImage.p, dimage, npx * 3 * sizeof(float), h2d, c->stream));
        c->residualPx = 0;
    }
    if (!accumulate) {
        EL_HIP(c, c->aMat.ensure(std::max<size_t>(1, M) * 6 * sizeof(double)));
        EL_HIP(c, hipMemsetAsync(c->aMat.p, 0, M * 6 * sizeof(double), c->stream));
        if (ntex) {
            EL_HIP(c, c->aTex.ensure(ntex * sizeof(float)));
            EL_HIP(c, hipMemsetAsync(c->aTex.p, 0, ntex * sizeof(float), c->stream));
        }
        c->adjSumValid = false;
    }
    unsigned long long* ctr = c->dCounters.as<unsigned long long>();
    EL_HIP(c, hipMemsetAsync(ctr, 0, sizeof(unsigned long long) * kCounterWords, c->stream));
    LaunchCfg lc = cfgOf(c);
    if (p->block) lc.block = p->block;
    const uint32_t depth = c->accDepth;
    RenderArgs a{};
    a.k0 = (uint32_t)c->accSeed;
    a.k1 = (uint32_t)(c->accSeed >> 32);
    a.scene = c->accScene;
    a.maxDepth = depth;
    a.sample = 0;
    a.cull = 1;   // exact: a zero-throughput path adds neither radiance nor gradient
    AdjArgs g{};
    g.dimage = c->aImage.as<float>();
    g.counts = c->dCounts.as<uint32_t>();
    g.gradTex = gtex;
    g.dmat = c->aMat.as<double>();
    g.dtex = ntex ? c->aTex.as<float>() : nullptr;
    g.ldsMats = M <= kAdjLdsMats ? (uint32_t)M : 0u;
    // The paths are replayed a generation at a time.  Recorded ones (a
    // wavefront EL_FLAG_RECORD_PATHS render) are traced no more: the
    // recording stopped no earlier than the replay does.  Others are walked
    // again here, recording the generation's hits and shadow answers.
    const bool recorded = c->recValid;
    const uint64_t npad = (uint64_t)((c->cam.x_res + 7) / 8) * ((c->cam.y_res + 7) / 8) * 64;
    const uint64_t total = (uint64_t)c->sampleBase * npad;
    if (npad >= (1ull << 31)) return fail(c, EL_ERR_RANGE, "frame too large for the adjoint");
    uint64_t Q = 0;
    WfState q{};
    const AdjointMemory memory{WfBuffers::kEntryBytes, WfBuffers::kSlotBytes,
                               lc.maxThreads + (uint64_t)kXcds * (kMaxBlock + 1), recorded ? 0 : 16ull * depth + 4,
                               c->wf.cap, c->wf.qcap, c->aHits.n + c->aVis.n};
    hipError_t asked = hipSuccess;
    const uint64_t cap = adjointPaths(memory, total, [&]() -> uint64_t {
        size_t freeB = 0, totalB = 0;
        asked = hipMemGetInfo(&freeB, &totalB);
        return freeB;
    });
    EL_HIP(c, asked);
    int rc = wfPlan(c, lc, total, npad, cap, false, q, Q);
    if (rc) return rc;
    if (recorded) {
        a.recHits = c->dRecHits.as<float4>();
        a.recVis = c->dRecVis.as<uint32_t>();
        a.recStride = (uint64_t)c->sampleBase * npx;
        g.rec = c->dRec.as<float4>();
    } else {
        EL_HIP(c, c->aHits.ensure(Q * depth * sizeof(float4)));
        EL_HIP(c, c->aVis.ensure(Q * sizeof(uint32_t)));
        a.recHits = c->aHits.as<float4>();
        a.recStride = Q;
        a.recBySlot = 1;
        q.pathVis = c->aVis.as<uint32_t>();
    }
    const size_t countBytes = (depth + 1) * kXcds * sizeof(uint32_t);
    EL_HIP(c, c->aQueue.ensure(countBytes));
    g.queueCount = c->aQueue.as<uint32_t>();
    a.npad = (uint32_t)npad;
    hipEvent_t e0 = poolEvent(c, 0), e1 = poolEvent(c, 1);
    if (!e0 || !e1) return fail(c, EL_ERR_HIP, "event creation failed");
    EL_HIP(c, hipEventRecord(e0, c->stream));
    for (uint64_t start = 0; start < total; start += Q) {
        a.genPixel = (uint32_t)(start % npad);
        a.genSample = (uint32_t)(start / npad);
        a.genCount = (uint32_t)std::min<uint64_t>(Q, total - start);
        a.run = a.genPixel == 0 && a.genCount % npad == 0 ? (uint32_t)(a.genCount / npad) : 0u;
        if (!recorded) {
            std::vector<std::pair<size_t, int>> timed;
            size_t ev = 2;
            rc = wfWalk(c, lc, a, q, 0, timed, ev, ctr);
            if (rc) return rc;
        }
        EL_HIP(c, hipMemsetAsync(c->aQueue.p, 0, countBytes, c->stream));
        // the walk's ray and shadow queues are free: the replay's go there
        float4* const state[2] = {q.shadowH, q.shadowP};
        for (uint32_t b = 0; b < depth; b++) {
            a.bounce = b;
            const int cur = b & 1, nxt = cur ^ 1;
            EL_HIP(c, launchAdjBounce(lc, c->ds, a, q, g, q.ray[cur], state[cur], q.ray[nxt], state[nxt], ctr));
        }
    }
    EL_HIP(c, hipEventRecord(e1, c->stream));
    const unsigned long long* const h = stage->tallies;
    // The material sums and the texels come with the tallies, in one wait, up to
    // kOneWait each: a copy to pageable memory is a wait of its own, and so is a
    // chunk of stageOut, which takes larger textures once the GPU is done.
    const size_t matBytes = dmat ? M * 6 * sizeof(double) : 0, texBytes = ntex && dtex && !devp ? ntex * sizeof(float) : 0;
    const size_t matStaged = matBytes <= kOneWait ? matBytes : 0, texStaged = texBytes <= kOneWait ? texBytes : 0;
    if (ntex && dtex && devp)
        EL_HIP(c, hipMemcpyAsync(dtex, c->aTex.p, ntex * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
    std::vector<double> large(matBytes > matStaged ? M * 6 : 0);
    if (!large.empty()) EL_HIP(c, hipMemcpyAsync(large.data(), c->aMat.p, matBytes, hipMemcpyDeviceToHost, c->stream));
    if (matStaged + texStaged) {
        EL_HIP(c, stage->ensure(matStaged + texStaged));
        stage.inFlight(true);
    }
    if (matStaged) EL_HIP(c, launchCopyOut(c->stream, c->aMat.p, stage->p, matStaged / 4));
    if (texStaged) EL_HIP(c, launchCopyOut(c->stream, c->aTex.p, stage->p + matStaged, texStaged / 4));
    EL_HIP(c, readTallies(stage, ctr));
    float ms = 0;
    EL_HIP(c, hipEventElapsedTime(&ms, e0, e1));
    if (dmat) {
        const double* const hm = matStaged ? (const double*)stage->p : large.data();
        std::vector<float> fm(M * 6);
        for (size_t i = 0; i < M * 6; i++) fm[i] = (float)hm[i];
        if (devp)
            EL_HIP(c, hipMemcpy(dmat, fm.data(), fm.size() * sizeof(float), hipMemcpyHostToDevice));
        else
            std::memcpy(dmat, fm.data(), fm.size() * sizeof(float));
    }
    if (texStaged) std::memcpy(dtex, stage->p + matStaged, texStaged);
    if (texBytes > texStaged)
        EL_HIP(c, stageOut(
                      stage, ntex, sizeof(float),
                      [&](size_t first, size_t n, unsigned char* chunk) {
                          return launchCopyOut(c->stream, c->aTex.as<float>() + first, chunk, n);
                      },
                      [&](size_t first, size_t, const unsigned char* chunk, size_t i0, size_t i1) {
                          std::memcpy(dtex + first + i0, (const float*)chunk + i0, (i1 - i0) * sizeof(float));
                      }));
    c->adjSumValid = true;
    c->adjSumTex = gtex;
    c->stats.adjoint_ms = ms;
    c->stats.adjoint_rays = tally(h, kStatRays);
    c->stats.adjoint_bytes = (recorded ? 0 : c->aHits.n + c->aVis.n) + c->aQueue.n + c->aImage.n + c->aMat.n + c->aTex.n;
    if (tally(h, kStatOverflow)) return fail(c, EL_ERR_RANGE, "traversal stack overflow (gradients incomplete)");
    return EL_OK;
}

// The mean image of sums[i * stride] over the accepted samples, and their
// counts, to host arrays (either may be null): divided on the GPU, which writes
// it to the stage.  A 1920 x 1080 frame takes 1.9 ms, of which a caller's fresh
// arrays cost 1.6; sums and counts copied to pageable memory and divided by the
// host took 12.9.
static hipError_t readMean(el_ctx* c, const float4* sums, uint32_t stride, size_t npx, float* rgba,
                           uint32_t* samples) {
    if (hipError_t e = clearPending(c); e != hipSuccess) return e;
    StageLease stage(c->device, c->stream);
    if (hipError_t e = stage.take(); e != hipSuccess) return e;
    const size_t nR = rgba ? sizeof(float4) : 0, nS = samples ? sizeof(uint32_t) : 0;
    // a chunk of n pixels: n float4, then n counts
    return stageOut(
        stage, npx, nR + nS,
        [&](size_t first, size_t n, unsigned char* chunk) {
            return launchResolve(c->stream, sums, stride, c->dCounts.as<uint32_t>(), (uint32_t)first, (uint32_t)n,
                                 nR ? (float4*)chunk : nullptr, nS ? (uint32_t*)(chunk + n * nR) : nullptr);
        },
        [&](size_t first, size_t n, const unsigned char* chunk, size_t i0, size_t i1) {
            if (nR) std::memcpy(rgba + 4 * (first + i0), chunk + i0 * nR, (i1 - i0) * nR);
            if (nS) std::memcpy(samples + first + i0, chunk + n * nR + i0 * nS, (i1 - i0) * nS);
        });
}

extern "C" {

int el_read_passes(el_ctx* c, float* rgba, uint32_t* samples, uint64_t* rays, uint64_t* vertices) {
    if (!c) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    EL_HIP(c, hipSetDevice(c->device));
    size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    if (rgba || samples) EL_HIP(c, readMean(c, c->dAccum.as<float4>(), 1, npx, rgba, samples));
    if (rays) *rays = c->totalRays;
    if (vertices) *vertices = c->totalVerts;
    return EL_OK;
}

int el_read_aov(el_ctx* c, int pass, float* rgba) {
    if (!c || !rgba) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (pass != EL_PASS_NORMAL && pass != EL_PASS_TANGENT && pass != EL_PASS_BITANGENT)
        return fail(c, EL_ERR_ARG, "pass must be NORMAL, TANGENT or BITANGENT");
    if (!c->dAov.p) return fail(c, EL_ERR_STATE, "no AOV rendered (EL_FLAG_AOV)");
    EL_HIP(c, hipSetDevice(c->device));
    size_t npx = (size_t)c->cam.x_res * c->cam.y_res;
    EL_HIP(c, readMean(c, c->dAov.as<float4>() + (pass - EL_PASS_NORMAL), 3, npx, rgba, nullptr));
    return EL_OK;
}

int el_get_stats(el_ctx* c, el_stats* out) {
    if (!c || !out) return EL_ERR_ARG;
    *out = c->stats;
    return EL_OK;
}

int el_set_materials(el_ctx* c, const el_material* m, uint32_t count) {
    if (!c || !m) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (count != c->mats.size()) return fail(c, EL_ERR_ARG, "material count differs from the uploaded scene");
    for (uint32_t i = 0; i < count; i++) {
        setMaterialValues(c->mats[i], m[i]);
    }
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipMemcpyAsync(c->dMats.p, c->mats.data(), count * sizeof(dev::DevMaterial), hipMemcpyHostToDevice,
                             c->stream));
    EL_HIP(c, hipStreamSynchronize(c->stream));
    return EL_OK;
}

int el_set_texture(el_ctx* c, int32_t id, const float* rgb) {
    if (!c || !rgb) return EL_ERR_ARG;
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (id < 0 || (size_t)id >= c->texs.size()) return fail(c, EL_ERR_ARG, "texture id out of range");
    // new values go to the FP32 copy, which the texture reads from then on
    dev::DevTex& t = c->texs[id];
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipMemcpyAsync(c->dTexels.as<float>() + c->texF32[id], rgb, (size_t)t.w * t.h * 3 * sizeof(float),
                             hipMemcpyHostToDevice, c->stream));
    if (t.format != dev::kTexF32) {
        c->stats.texels_8bit -= (uint64_t)t.w * t.h;
        t.format = dev::kTexF32;
        t.offset = c->texF32[id];
        EL_HIP(c, hipMemcpyAsync(c->dTexs.as<dev::DevTex>() + id, &t, sizeof t, hipMemcpyHostToDevice, c->stream));
    }
    EL_HIP(c, hipStreamSynchronize(c->stream));
    return EL_OK;
}

}  // extern "C"

// ---------------------------------------------------------------- queries --
// Host queries of up to this many rays (160 KB of rays and answers) leave the
// copies out: 1000 rays take 47 instead of 95 us.
constexpr uint32_t kDirectRays = 4096;

static int traceCommon(el_ctx* c, const el_ray* rays, const float* tmax, uint32_t n, int32_t* tri, float* t,
                       float* uv, uint8_t* occ, int devp, bool any, bool count, uint64_t* nodes, uint64_t* tris) {
    if (!c || !rays) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (any && (!tmax || !occ)) return fail(c, EL_ERR_ARG, "null argument");
    if (!any && !count && (!tri || !t)) return fail(c, EL_ERR_ARG, "null argument");
    if (n == 0) return EL_OK;
    EL_HIP(c, hipSetDevice(c->device));
    const float* dR = (const float*)rays;
    const float* dTm = tmax;
    int32_t* dTri = tri;
    float* dT = t;
    float* dUV = uv;
    uint8_t* dOcc = occ;
    StageLease stage(c->device, c->stream);
    EL_HIP(c, stage.take());
    Stage& st = *stage;
    // A short host query (a pick) goes through the stage: the kernel reads the
    // rays from it and writes the answers to it, without a copy each way.
    const bool direct = !devp && !count && n <= kDirectRays;
    const size_t rayBytes = (size_t)n * sizeof(el_ray);
    if (direct) {
        EL_HIP(c, st.ensure(kDirectRays * (sizeof(el_ray) + 16)));
        std::memcpy(st.p, rays, rayBytes);
        dR = (const float*)st.p;
        unsigned char* out = st.p + rayBytes;
        if (any) {
            std::memcpy(out, tmax, (size_t)n * 4);
            dTm = (const float*)out;
            dOcc = out + (size_t)n * 4;
        } else {
            dTri = (int32_t*)out;
            dT = (float*)(out + (size_t)n * 4);
            if (uv) dUV = (float*)(out + (size_t)n * 8);
        }
    } else if (!devp) {
        EL_HIP(c, upload(c->tRays, rays, rayBytes, c->stream));
        dR = c->tRays.as<float>();
        if (any) {
            EL_HIP(c, upload(c->tTmax, tmax, (size_t)n * 4, c->stream));
            dTm = c->tTmax.as<float>();
            EL_HIP(c, c->tOcc.ensure(n));
            dOcc = c->tOcc.as<uint8_t>();
        } else if (uv) {
            EL_HIP(c, c->tUV.ensure((size_t)n * 8));
            dUV = c->tUV.as<float>();
        }
    }
    if (!any && !direct && (!devp || count)) {
        EL_HIP(c, c->tTri.ensure((size_t)n * 4));
        EL_HIP(c, c->tT.ensure((size_t)n * 4));
        if (!devp || !dTri) dTri = c->tTri.as<int32_t>();
        if (!devp || !dT) dT = c->tT.as<float>();
    }
    unsigned long long* ctr = c->dCounters.as<unsigned long long>();
    EL_HIP(c, hipMemsetAsync(ctr, 0, sizeof(unsigned long long) * kCounterWords, c->stream));
    stage.inFlight(direct);
    EL_HIP(c, launchTrace(cfgOf(c), c->ds, dR, dTm, n, dTri, dT, dUV, dOcc, any, count, ctr));
    if (!devp && !direct && !count) {
        // a chunk of n rays: each answer's n values after the other's
        const std::vector<std::pair<void*, size_t>> host =
            any ? std::vector<std::pair<void*, size_t>>{{occ, 1}}
                : std::vector<std::pair<void*, size_t>>{{tri, 4}, {t, 4}, {uv, uv ? 8 : 0}};
        const unsigned char* const dev[3] = {any ? (unsigned char*)dOcc : (unsigned char*)dTri, (unsigned char*)dT,
                                             (unsigned char*)dUV};
        size_t bytes = 0;
        for (auto& o : host) bytes += o.second;
        EL_HIP(c, stageOut(
                      stage, n, bytes,
                      [&](size_t first, size_t m, unsigned char* chunk) {
                          hipError_t e = hipSuccess;
                          for (size_t k = 0; k < host.size() && e == hipSuccess; k++) {
                              const size_t w = host[k].second;
                              if (w) e = hipMemcpyAsync(chunk, dev[k] + first * w, m * w, hipMemcpyDeviceToHost, c->stream);
                              chunk += m * w;
                          }
                          return e;
                      },
                      [&](size_t first, size_t m, const unsigned char* chunk, size_t i0, size_t i1) {
                          for (auto& o : host) {
                              const size_t w = o.second;
                              if (w) std::memcpy((unsigned char*)o.first + (first + i0) * w, chunk + i0 * w, (i1 - i0) * w);
                              chunk += m * w;
                          }
                      }));
    }
    EL_HIP(c, readTallies(stage, ctr));
    const unsigned long long* const h = st.tallies;
    if (direct && any) std::memcpy(occ, dOcc, n);
    if (direct && !any) {
        std::memcpy(tri, dTri, (size_t)n * 4);
        std::memcpy(t, dT, (size_t)n * 4);
        if (uv) std::memcpy(uv, dUV, (size_t)n * 8);
    }
    if (nodes) *nodes = tally(h, kStatNodes);
    if (tris) *tris = tally(h, kStatTris);
    if (tally(h, kStatOverflow)) return fail(c, EL_ERR_RANGE, "traversal stack overflow (results incomplete)");
    return EL_OK;
}

extern "C" {

int el_trace_closest(el_ctx* c, const el_ray* rays, uint32_t n, int32_t* tri, float* t, float* uv, int devp) {
    return traceCommon(c, rays, nullptr, n, tri, t, uv, nullptr, devp, false, false, nullptr, nullptr);
}

int el_trace_any(el_ctx* c, const el_ray* rays, const float* tmax, uint32_t n, uint8_t* occ, int devp) {
    return traceCommon(c, rays, tmax, n, nullptr, nullptr, nullptr, occ, devp, true, false, nullptr, nullptr);
}

int el_trace_count(el_ctx* c, const el_ray* rays, uint32_t n, uint64_t* nodes, uint64_t* tris, int devp) {
    if (!nodes || !tris) return fail(c, EL_ERR_ARG, "null argument");
    return traceCommon(c, rays, nullptr, n, nullptr, nullptr, nullptr, nullptr, devp, false, true, nodes, tris);
}

int el_trace_closest_noalloc(el_ctx* c, const el_ray* d_rays, uint32_t n, int32_t* d_tri, float* d_t,
                             float* d_uv) {
    if (!c || !d_rays || !d_tri || !d_t) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    if (!c->scratch) return fail(c, EL_ERR_STATE, "no device scratch");
    if (n == 0) return EL_OK;
    EL_HIP(c, hipSetDevice(c->device));
    // as many resident threads as the spill area holds at the scene's depth (by quads, which spill nothing, all)
    LaunchCfg lc = cfgOf(c);
    const uint64_t fit = kScratchSpillInts / (uint64_t)c->gcap;
    uint32_t threads = (uint32_t)std::min<uint64_t>(c->maxThreads, fit);
    threads -= threads % lc.block;
    if (threads < lc.block)
        return fail(c, EL_ERR_RANGE, "the scene's traversal stack (" + std::to_string(c->gcap) +
                                         " spill slots per thread) exceeds the static scratch for one block");
    lc.maxThreads = threads;
    lc.gstack = (int*)((unsigned char*)c->scratch + kScratchCounterBytes);
    unsigned long long* ctr = (unsigned long long*)c->scratch;
    EL_HIP(c, hipMemsetAsync(ctr, 0, sizeof(unsigned long long) * kCounterWords, c->stream));
    EL_HIP(c, launchTrace(lc, c->ds, (const float*)d_rays, nullptr, n, d_tri, d_t, d_uv, nullptr, false, false, ctr));
    unsigned long long h[kCounterWords];
    EL_HIP(c, hipMemcpyAsync(h, ctr, sizeof h, hipMemcpyDeviceToHost, c->stream));
    EL_HIP(c, hipStreamSynchronize(c->stream));
    if (tally(h, kStatOverflow)) return fail(c, EL_ERR_RANGE, "traversal stack overflow (results incomplete)");
    return EL_OK;
}

int el_trace_bench(el_ctx* c, const el_ray* d_rays, uint32_t n, int32_t* d_tri, float* d_t, int iters,
                   double* mean_ms) {
    if (!c || !d_rays || !d_tri || !d_t || !mean_ms || iters <= 0) return fail(c, EL_ERR_ARG, "null argument");
    if (!c->hasScene) return fail(c, EL_ERR_STATE, "no scene uploaded");
    EL_HIP(c, hipSetDevice(c->device));
    unsigned long long* ctr = c->dCounters.as<unsigned long long>();
    hipEvent_t e0 = poolEvent(c, 0), e1 = poolEvent(c, 1);
    double total = 0;
    for (int i = 0; i < iters; i++) {
        EL_HIP(c, hipEventRecord(e0, c->stream));
        EL_HIP(c, launchTrace(cfgOf(c), c->ds, (const float*)d_rays, nullptr, n, d_tri, d_t, nullptr, nullptr, false,
                              false, ctr));
        EL_HIP(c, hipEventRecord(e1, c->stream));
        EL_HIP(c, hipEventSynchronize(e1));
        float ms = 0;
        EL_HIP(c, hipEventElapsedTime(&ms, e0, e1));
        total += ms;
    }
    *mean_ms = total / iters;
    return EL_OK;
}

int el_device_alloc(el_ctx* c, size_t bytes, void** out) {
    if (!c || !out) return EL_ERR_ARG;
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipMalloc(out, bytes ? bytes : 16));
    return EL_OK;
}

int el_device_free(el_ctx* c, void* p) {
    if (!c) return EL_ERR_ARG;
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipFree(p));
    return EL_OK;
}

int el_memcpy_htod(el_ctx* c, void* dst, const void* src, size_t bytes) {
    if (!c || !dst || !src) return EL_ERR_ARG;
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    EL_HIP(c, hipStreamSynchronize(c->stream));
    return EL_OK;
}

int el_memcpy_dtoh(el_ctx* c, void* dst, const void* src, size_t bytes) {
    if (!c || !dst || !src) return EL_ERR_ARG;
    EL_HIP(c, hipSetDevice(c->device));
    EL_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    EL_HIP(c, hipStreamSynchronize(c->stream));
    return EL_OK;
}

}  // extern "C"

// ---------------------------------------------------------------- batches --
// Many scenes rendered by one wavefront loop.  Each scene is uploaded into
// its own context (geometry, textures, HDRI tables and its accumulation stay
// in that context's buffers); the batch owns the queues, the traversal
// stack, a device array of the scenes' DevScene records and the generation
// plan.  Work items are enumerated scene after scene, sample-major inside a
// scene; a generation takes the next queue_cap of them, whatever scenes they
// belong to, and a segment table tells the camera and finalize kernels which
// scene each path slot belongs to.  With EL_BATCH_GRAPH the whole launch
// sequence is captured once into a hipGraph and replayed.
struct el_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err, log;
    uint32_t maxThreads = 0;
    std::vector<el_ctx*> scenes;
    std::vector<uint32_t> spp;
    std::vector<uint64_t> seed;
    int width = 4;
    DevBuf dScenes, dSegs, dGstack, dCounters;
    WfBuffers wf;
    hipGraphExec_t graph = nullptr;
    std::string graphKey;
    el_stats stats{};
    hipEvent_t e0 = nullptr, e1 = nullptr;
};

static int bfail(el_batch* b, int code, const std::string& what) {
    if (b) b->err = what;
    return code;
}

#define EL_BHIP(b, x)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (x);                                                                   \
        if (e_ != hipSuccess) return bfail(b, EL_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct BatchGen {
    size_t segOffset;
    uint32_t nseg, count, finTotal;
};

extern "C" {

int el_batch_create(el_batch** out, int device) {
    if (!out) return EL_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return EL_ERR_HIP;
    if (device < 0 || device >= n) return EL_ERR_ARG;
    std::unique_ptr<el_batch> b(new el_batch());
    b->device = device;
    if (hipSetDevice(device) != hipSuccess) return EL_ERR_HIP;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return EL_ERR_HIP;
    b->maxThreads = (uint32_t)prop.multiProcessorCount * 2048u;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return EL_ERR_HIP;
    if (hipEventCreate(&b->e0) != hipSuccess || hipEventCreate(&b->e1) != hipSuccess) return EL_ERR_HIP;
    if (b->dCounters.ensure(sizeof(unsigned long long) * kCounterWords) != hipSuccess) return EL_ERR_HIP;
    *out = b.release();
    return EL_OK;
}

void el_batch_destroy(el_batch* b) {
    if (!b) return;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    if (b->graph) (void)hipGraphExecDestroy(b->graph);
    for (auto* c : b->scenes) el_destroy(c);
    if (b->e0) (void)hipEventDestroy(b->e0);
    if (b->e1) (void)hipEventDestroy(b->e1);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

const char* el_batch_last_error(const el_batch* b) { return b ? b->err.c_str() : "null batch"; }
const char* el_batch_log(const el_batch* b) { return b ? b->log.c_str() : ""; }

int el_batch_add(el_batch* b, const el_scene_view* view, uint32_t spp, uint64_t seed, int32_t* index) {
    if (!b || !view) return bfail(b, EL_ERR_ARG, "null argument");
    if (spp == 0) return bfail(b, EL_ERR_ARG, "spp must be positive");
    if (b->scenes.size() >= 65536) return bfail(b, EL_ERR_RANGE, "at most 65536 scenes per batch");
    el_ctx* c = nullptr;
    int rc = el_create(&c, b->device);
    if (rc) return bfail(b, rc, "context creation failed");
    rc = el_upload_scene(c, view);
    if (rc) {
        std::string m = el_last_error(c);
        el_destroy(c);
        return bfail(b, rc, m);
    }
    if (c->width != b->width) {
        rc = uploadBvh(c, b->width);
        if (rc) {
            std::string m = el_last_error(c);
            el_destroy(c);
            return bfail(b, rc, m);
        }
    }
    b->scenes.push_back(c);
    b->spp.push_back(spp);
    b->seed.push_back(seed);
    if (b->graph) {
        (void)hipGraphExecDestroy(b->graph);
        b->graph = nullptr;
    }
    if (index) *index = (int32_t)b->scenes.size() - 1;
    return EL_OK;
}

int el_batch_read(el_batch* b, int32_t scene, float* rgba, uint32_t* samples) {
    if (!b) return EL_ERR_ARG;
    if (scene < 0 || (size_t)scene >= b->scenes.size()) return bfail(b, EL_ERR_ARG, "scene index out of range");
    int rc = el_read_passes(b->scenes[scene], rgba, samples, nullptr, nullptr);
    if (rc) return bfail(b, rc, el_last_error(b->scenes[scene]));
    return EL_OK;
}

int el_batch_stats(el_batch* b, el_stats* out) {
    if (!b || !out) return EL_ERR_ARG;
    *out = b->stats;
    return EL_OK;
}

}  // extern "C"

// Renders every scene of the batch from a cleared accumulation with spp[i]
// (capped at sppCap if nonzero).  Returns the device time in *ms.
static int batchRender(el_batch* b, const el_batch_params* p, uint32_t sppCap, double* ms) {
    const size_t S = b->scenes.size();
    if (S == 0) return bfail(b, EL_ERR_STATE, "empty batch");
    const uint32_t depth = p->max_depth ? p->max_depth : 5;
    if (depth > 64) return bfail(b, EL_ERR_RANGE, "max_depth above 64");
    if (p->bvh_width != 0 && p->bvh_width != 4 && p->bvh_width != 8) return bfail(b, EL_ERR_ARG, "bvh_width must be 4 or 8");
    if (p->block != 0 && (p->block % 64 != 0 || p->block > (uint32_t)kMaxBlock))
        return bfail(b, EL_ERR_ARG, "block must be a multiple of 64, at most 256");
    if (p->refill > 64) return bfail(b, EL_ERR_ARG, "refill must be 0..64");
    EL_BHIP(b, hipSetDevice(b->device));
    StageLease stage(b->device, b->stream);
    EL_BHIP(b, stage.take());
    const int width = p->bvh_width ? (int)p->bvh_width : b->width;
    if (width != b->width) {
        for (auto* c : b->scenes) {
            int rc = uploadBvh(c, width);
            if (rc) return bfail(b, rc, el_last_error(c));
        }
        b->width = width;
    }
    // scene records: shared spill capacity and slab unit, per-scene key and accumulation
    int gcap = 1, quads = 1;
    float slabUnit = 1.0f;
    for (auto* c : b->scenes) {
        gcap = std::max(gcap, c->gcap);
        quads &= c->ds.quads;
        slabUnit = std::min(slabUnit, c->ds.slabUnit);
    }
    std::vector<DevScene> recs(S);
    std::vector<uint64_t> work(S), npadv(S);
    uint64_t total = 0;
    for (size_t i = 0; i < S; i++) {
        el_ctx* c = b->scenes[i];
        recs[i] = c->ds;
        recs[i].gcap = gcap;
        recs[i].quads = quads;
        recs[i].slabUnit = slabUnit;
        recs[i].seedLo = (uint32_t)b->seed[i];
        recs[i].seedHi = (uint32_t)(b->seed[i] >> 32);
        recs[i].accum = c->dAccum.as<float4>();
        recs[i].counts = c->dCounts.as<uint32_t>();
        const uint64_t tx = (c->cam.x_res + 7) / 8, ty = (c->cam.y_res + 7) / 8;
        npadv[i] = tx * ty * 64;
        const uint32_t spp = sppCap ? std::min(sppCap, b->spp[i]) : b->spp[i];
        work[i] = (uint64_t)spp * npadv[i];
        total += work[i];
    }
    EL_BHIP(b, upload(b->dScenes, recs.data(), S * sizeof(DevScene), b->stream));
    EL_BHIP(b, b->dGstack.ensure((size_t)gcap * b->maxThreads * sizeof(int)));
    // generation plan
    uint64_t Q = p->queue_cap;
    if (!Q) {
        size_t freeB = 0, totalB = 0;
        EL_BHIP(b, hipMemGetInfo(&freeB, &totalB));
        Q = std::max<uint64_t>(1u << 20, freeB / 4 / (6 * 32 + 60));
    }
    Q = std::max<uint64_t>(64, (Q / 64) * 64);
    if (Q > total) Q = total;
    if (Q > 0x7fffffffull) return bfail(b, EL_ERR_RANGE, "queue capacity above 2^31");
    std::vector<BatchSeg> segs;
    std::vector<BatchGen> gens;
    {
        size_t sc = 0;
        uint64_t sceneBase = 0;
        for (uint64_t gs = 0; gs < total; gs += Q) {
            const uint64_t ge = std::min(total, gs + Q);
            BatchGen g{segs.size(), 0, (uint32_t)(ge - gs), 0};
            uint64_t w = gs;
            while (w < ge) {
                while (w >= sceneBase + work[sc]) {
                    sceneBase += work[sc];
                    sc++;
                }
                const uint64_t segEnd = std::min(ge, sceneBase + work[sc]);
                BatchSeg s{};
                s.slotStart = (uint32_t)(w - gs);
                s.count = (uint32_t)(segEnd - w);
                s.scene = (uint32_t)sc;
                s.npad = (uint32_t)npadv[sc];
                s.wStart = w - sceneBase;
                s.finStart = g.finTotal;
                s.run = s.wStart % s.npad == 0 && s.count % s.npad == 0 ? s.count / s.npad : 0u;
                g.finTotal += std::min<uint32_t>(s.count, s.npad);
                segs.push_back(s);
                g.nseg++;
                w = segEnd;
            }
            gens.push_back(g);
        }
    }
    EL_BHIP(b, upload(b->dSegs, segs.data(), segs.size() * sizeof(BatchSeg), b->stream));
    LaunchCfg lc;
    lc.stream = b->stream;
    lc.block = p->block ? p->block : kDefaultBlock;
    lc.shadeBlock = 256;
    lc.maxThreads = lc.quadThreads = b->maxThreads;
    lc.refill = p->refill ? p->refill : kDefaultRefill;
    lc.gstack = b->dGstack.as<int>();
    const uint64_t segSize = (Q + kXcds - 1) / kXcds + lc.maxThreads / kXcds + kMaxBlock;
    const uint64_t qcap = std::max<uint64_t>(Q, kXcds * segSize);
    EL_BHIP(b, b->wf.ensure(Q, qcap, false, kQCounters * sizeof(uint32_t)));
    if (!b->wf.holds(Q, qcap, false))
        return bfail(b, EL_ERR_STATE, "wavefront buffers smaller than the generation (internal error)");
    WfState q{};
    q.ray[0] = b->wf.ray0.as<float4>();
    q.ray[1] = b->wf.ray1.as<float4>();
    q.hits = b->wf.hits.as<float4>();
    q.shadowH = b->wf.shadowH.as<float4>();
    q.shadowP = b->wf.shadowP.as<float4>();
    q.pathT = b->wf.pathT.as<float4>();
    q.pathL = b->wf.pathL.as<float4>();
    q.pathPix = b->wf.pix.as<uint32_t>();
    q.pathSample = b->wf.sample.as<uint32_t>();
    q.pathQuiet = b->wf.quiet.as<uint64_t>();
    q.pathAov = nullptr;
    q.pendP = b->wf.pend.as<float4>();
    q.counters = b->wf.counters.as<uint32_t>();
    q.segSize = (uint32_t)segSize;
    q.cap = qcap;
    q.gstack = lc.gstack;
    q.gthreads = lc.maxThreads;
    unsigned long long* ctr = b->dCounters.as<unsigned long long>();
    const DevScene* dsc = b->dScenes.as<DevScene>();
    const bool apart = (p->flags & EL_BATCH_SERIAL_SHADOWS) != 0;
    auto launchAll = [&]() -> hipError_t {   // the launches of el_render's loop
        hipError_t e;
        for (const BatchGen& g : gens) {
            const BatchSeg* gseg = b->dSegs.as<BatchSeg>() + g.segOffset;
            if ((e = launchBtCamera(lc, dsc, gseg, g.nseg, g.count, depth, !(p->flags & EL_BATCH_NO_CULL), q,
                                    &g == &gens[0], ctr)) != hipSuccess)
                return e;
            bool extended = false;
            for (uint32_t bo = 0; bo < depth; bo++) {
                const bool together = !apart && bounceTogether(g.count, bo), more = bo + 1 < depth;
                RenderArgs a{};
                a.maxDepth = depth;
                a.bounce = bo;
                a.cull = (p->flags & EL_BATCH_NO_CULL) ? 0u : 1u;
                const int cur = bo & 1, nxt = cur ^ 1;
                uint32_t* cntCur = q.counters + (cur ? kQRay1 : kQRay0);
                uint32_t* cntNxt = q.counters + (nxt ? kQRay1 : kQRay0);
                WfState qb = q;
                qb.parity = bo & 1u;
                qb.deferP = together ? 1u : 0u;
                if (!extended &&
                    (e = launchBtExtend(lc, dsc, width, qb, q.ray[cur], cntCur, cntNxt, g.count, ctr)) != hipSuccess)
                    return e;
                if ((e = launchBtShade(lc, dsc, a, qb, q.ray[cur], cntCur, q.ray[nxt], cntNxt, g.count, ctr)) !=
                    hipSuccess)
                    return e;
                if (together) {
                    e = launchBtTrace(lc, dsc, width, qb, more ? q.ray[nxt] : nullptr, cntNxt, cntCur, g.count, ctr);
                    if (e != hipSuccess) return e;
                } else {
                    for (int light = 0; light < 2; light++)
                        if ((e = launchBtShadow(lc, dsc, width, qb, light, g.count, ctr)) != hipSuccess) return e;
                }
                extended = together && more;
            }
            if ((e = launchBtFinalize(lc, dsc, gseg, g.nseg, g.finTotal, q, ctr)) != hipSuccess) return e;
        }
        return hipSuccess;
    };
    const bool useGraph = (p->flags & EL_BATCH_GRAPH) != 0;
    if (useGraph) {
        // the captured sequence depends on the plan and the launch shape
        // FNV-1a of the segment table and the generations: kernel arguments
        // (segment counts, slot totals) are baked into the graph
        uint64_t plan = 1469598103934665603ull;
        auto mix = [&](const void* p, size_t n) {
            for (size_t i = 0; i < n; i++) plan = (plan ^ ((const unsigned char*)p)[i]) * 1099511628211ull;
        };
        mix(segs.data(), segs.size() * sizeof(BatchSeg));
        for (const BatchGen& g : gens) {
            const uint64_t f[4] = {g.segOffset, g.nseg, g.count, g.finTotal};
            mix(f, sizeof f);
        }
        std::string key = std::to_string(S) + "/" + std::to_string(depth) + "/" + std::to_string(width) + "/" +
                          std::to_string(p->flags & ~EL_BATCH_GRAPH) + "/" + std::to_string(plan) + "/" +
                          std::to_string(lc.block) + "/" + std::to_string(lc.refill) + "/" + std::to_string(Q) +
                          "/" + std::to_string(sppCap) + "/" + std::to_string(total) + "/" +
                          std::to_string(allocationsOf(b->dScenes, b->dSegs, b->dGstack, b->dCounters) + b->wf.allocations());
        if (!b->graph || key != b->graphKey) {
            if (b->graph) {
                EL_BHIP(b, hipGraphExecDestroy(b->graph));
                b->graph = nullptr;
            }
            EL_BHIP(b, hipStreamSynchronize(b->stream));
            hipGraph_t gph = nullptr;
            EL_BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
            hipError_t le = launchAll();
            hipError_t ce = hipStreamEndCapture(b->stream, &gph);
            if (le != hipSuccess) return bfail(b, EL_ERR_HIP, std::string("capture: ") + hipGetErrorString(le));
            if (ce != hipSuccess) return bfail(b, EL_ERR_HIP, std::string("end capture: ") + hipGetErrorString(ce));
            hipError_t ie = hipGraphInstantiate(&b->graph, gph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(gph);
            if (ie != hipSuccess) {
                b->graph = nullptr;
                return bfail(b, EL_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(ie));
            }
            b->graphKey = key;
        }
        EL_BHIP(b, hipEventRecord(b->e0, b->stream));
        EL_BHIP(b, hipGraphLaunch(b->graph, b->stream));
        EL_BHIP(b, hipEventRecord(b->e1, b->stream));
    } else {
        EL_BHIP(b, hipEventRecord(b->e0, b->stream));
        EL_BHIP(b, launchAll());
        EL_BHIP(b, hipEventRecord(b->e1, b->stream));
    }
    const unsigned long long* const h = stage->tallies;
    EL_BHIP(b, readTallies(stage, ctr));
    float t = 0;
    EL_BHIP(b, hipEventElapsedTime(&t, b->e0, b->e1));
    *ms = t;
    for (size_t i = 0; i < S; i++) {
        el_ctx* c = b->scenes[i];
        c->sampleBase = sppCap ? std::min(sppCap, b->spp[i]) : b->spp[i];
        c->accSeed = b->seed[i];
        c->accDepth = depth;
        c->accPending = false;
        c->accMixed = true;   // batch RNG streams carry the scene index: no el_adjoint on them
        c->recValid = false;
    }
    b->stats = el_stats{};
    b->stats.rays = tally(h, kStatRays);
    b->stats.vertices = tally(h, kStatVerts);
    b->stats.paths = tally(h, kStatPaths);
    b->stats.render_ms = t;
    b->stats.bvh_width = (uint32_t)width;
    b->stats.extend_launches = gens.size() * depth;
    if (tally(h, kStatOverflow)) return bfail(b, EL_ERR_RANGE, "traversal stack or queue overflow (results incomplete)");
    return EL_OK;
}

extern "C" int el_batch_render(el_batch* b, const el_batch_params* p) {
    if (!b || !p) return bfail(b, EL_ERR_ARG, "null argument");
    double ms = 0;
    return batchRender(b, p, 0, &ms);
}

// Coordinate descent over BVH width, queue capacity, traversal block size
// and refill threshold, each trial rendering every scene at min(spp,
// trial_spp) samples; keeps the fastest setting of each knob in turn.
// A setting replaces the current best only if its trial is this much faster.
constexpr double kTuneMargin = 0.98;

extern "C" int el_batch_tune(el_batch* b, el_batch_params* io, uint32_t trial_spp) {
    if (!b || !io) return bfail(b, EL_ERR_ARG, "null argument");
    if (trial_spp == 0) trial_spp = 2;
    el_batch_params best = *io;
    best.flags &= ~EL_BATCH_GRAPH;
    // explicit defaults, so a sweep value equal to the default is not retried
    if (!best.bvh_width) best.bvh_width = (uint32_t)b->width;
    if (!best.block) best.block = kDefaultBlock;
    if (!best.refill) best.refill = kDefaultRefill;
    std::ostringstream log;
    auto trial = [&](const el_batch_params& p, double* ms) -> int {
        double t = 0;
        int rc = batchRender(b, &p, trial_spp, &t);   // warm (BVH repack, buffers)
        if (rc) return rc;
        rc = batchRender(b, &p, trial_spp, &t);
        if (rc) return rc;
        *ms = t;
        log << "width " << (p.bvh_width ? p.bvh_width : 4) << " queue " << p.queue_cap << " block "
            << (p.block ? p.block : kDefaultBlock) << " refill " << (p.refill ? p.refill : kDefaultRefill) << ": "
            << t << " ms\n";
        return EL_OK;
    };
    double bestMs = 0;
    int rc = trial(best, &bestMs);
    if (rc) return rc;
    auto sweep = [&](uint32_t el_batch_params::*field, std::vector<uint32_t> values) -> int {
        for (uint32_t v : values) {
            el_batch_params p = best;
            p.*field = v;
            if (p.*field == best.*field) continue;
            double ms = 0;
            int r = trial(p, &ms);
            if (r) return r;
            if (ms < bestMs * kTuneMargin) {   // trials closer than the margin are noise
                bestMs = ms;
                best = p;
            }
        }
        return EL_OK;
    };
    if ((rc = sweep(&el_batch_params::bvh_width, {4, 8}))) return rc;
    if ((rc = sweep(&el_batch_params::queue_cap, {1u << 22, 1u << 24, 1u << 26, 0}))) return rc;
    if ((rc = sweep(&el_batch_params::block, {64, 128, 256}))) return rc;
    if ((rc = sweep(&el_batch_params::refill, {8, 16, 32, 64}))) return rc;
    log << "chosen: width " << (best.bvh_width ? best.bvh_width : 4) << " queue " << best.queue_cap << " block "
        << (best.block ? best.block : kDefaultBlock) << " refill " << (best.refill ? best.refill : kDefaultRefill)
        << " (" << bestMs << " ms per trial)\n";
    b->log = log.str();
    best.flags = io->flags;
    *io = best;
    return EL_OK;
}
