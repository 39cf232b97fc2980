// api_internal.h — host-side state shared by the C ABI translation units
// (api.cpp: scenes and single-request tracing; server.cpp: the request loop).
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>
#include <string>
#include <vector>

#include "rt_layout.h"
#include "wavefront.h"

namespace rt {

// Records msg as the calling thread's last error (reina_rt_last_error) and
// returns code.
int fail(int code, const std::string& msg);

#define HIP_TRY(expr)                                                                   \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess)                                                           \
            return fail(REINA_RT_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Live paths at or below which reina_rt_trace ends the frame in one tail
// launch where tail_paths is REINA_RT_TAIL_AUTO: with next-event estimation,
// or the options that count or time the extend kernel, which then has to run
// (and a server's default) ...
constexpr uint32_t kDefaultTailPaths = 1u << 20;
// ... and in every other trace: a frame of up to 2^22 paths is one tail launch
// from its first ray on.
// The tail keeps a pixel's state and ray in registers, where a bounce
// iteration moves ~200 bytes per ray through HBM and ends with its slowest
// waves. ms at 2^20 | 2^22 | 2^24: 1080p 64 spp, 327,686 triangles
// 88.8 | 72.8 | 72.3; 1080x1350 8.30 | 7.57 | 7.48; 1080p 2 spp, 1.05M
// instanced triangles 2.20 | 1.33 | 1.28, 40 triangles 1.98 | 1.55 | 1.55.
// Above, frames start as bounce iterations: 3840x2160 8 spp, 500,000 triangles
// 29.4 | 28.7 | 30.5, instanced 14.6 | 14.3 | 14.7, 40 triangles
// 27.4 | 25.6 | 20.7; 1080p in 8 sample groups 7.60 | 7.55 | 8.52. With
// next-event estimation the tail's lockstep steps lose as often as they win
// (1080p 8 spp at 2^20 | 2^22: icosphere 23.8 | 29.0, lobes 26.8 | 28.4,
// textured 30.5 | 26.3).
constexpr uint32_t kDefaultTailPathsPlain = 1u << 22;

// Kernel parameters of one vkCmdTraceRaysKHR-equivalent render.
inline TraceParams make_trace_params(const RtPushConsts* pc, uint32_t W, uint32_t H) {
    TraceParams P;
    std::memcpy(P.cam.invView, pc->invView, 64);
    std::memcpy(P.cam.invProj, pc->invProjection, 64);
    P.cam.focusDist = pc->focusDist;
    P.cam.defocus = pc->defocusMultiplier;
    P.cam.W = (float)(int32_t)W;
    P.cam.H = (float)(int32_t)H;
    P.cam.right = normalize(v3(pc->invView[0], pc->invView[1], pc->invView[2]));
    P.cam.up = normalize(v3(pc->invView[4], pc->invView[5], pc->invView[6]));
    P.W = W;
    P.H = H;
    P.spp = pc->samplesPerPixel;
    P.maxBounces = pc->maxBounces;
    P.sampleBatch = pc->sampleBatch;
    P.directClamp = pc->directClamp;
    P.nee = 0;
    P.fixes = 0;
    P.groups = 1;
    return P;
}

}  // namespace rt

// A scene resident in HBM (reina_rt_scene_create).
struct ReinaScene {
    int device = 0;
    rt::SceneView sv{};
    void* arena = nullptr;              // everything but the tree
    void* tree = nullptr;               // nodes, then leaf-ordered triangles
    uint64_t tree_tris = 0;             // byte offset of the triangles
    ReinaSceneInfo info{};
    bool quantized = false;
    // light-sampling tables (next-event estimation)
    std::vector<rt::EmissiveInst> emi;
    std::vector<float> tri_cdf;
    std::vector<int32_t> inst_emi;
    std::vector<uint8_t> tri_flags;
    // trace buffers (grown on demand)
    uint64_t cap_px = 0;
    void* tbuf = nullptr;
    rt::PathState S{};
    rt::Queues Q{};
    rt::Ctrl* ctrl = nullptr;
    unsigned long long* stats = nullptr;
    uint32_t* fetch = nullptr;
    uint32_t* h_count = nullptr;        // pinned: [2 readbacks][partition * kLine] queue lengths
    rt::Tuning tune{16, 16, 0, 0, 0, 0};
    hipEvent_t cev[2] = {};             // queue-length readbacks
    uint32_t tail_count = 0;            // 1 if the last trace ended with a tail launch
    hipEvent_t tev0 = nullptr, tev1 = nullptr;   // around the tail launch
    uint32_t min_stack = 8;             // smallest legal stack depth for this BVH
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    bool traced = false;
    uint32_t options = 0;
    std::vector<hipEvent_t> xev;        // extend event pairs (REINA_RT_TRACE_TIME_EXTEND)
    uint32_t xev_used = 0;
    uint32_t last_iters = 0;
    bool trace_ready = false;           // control words and events created
    hipStream_t last_stream = nullptr;
};

using rt::fail;
