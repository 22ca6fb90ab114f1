// kpt_kernels.hip — traversal and megakernel path-tracing kernels for gfx950,
// with their host launch wrappers.
#include "kpt_integrator.h"
#include "kpt_launch.h"
#include "kpt_temporal.h"

namespace kpt {

// ------------------------------------------------------------------ traversal
// 8 waves per SIMD (64 VGPRs): 1125 us a million incoherent rays, 1181 at 7,
// 1179 unconstrained (69 VGPRs).
template <bool COUNT>
__global__ __launch_bounds__(TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(8))) void k_trace_closest(SceneView S, const kpt_ray* __restrict__ rays,
                                                               kpt_hit* __restrict__ hits, int64_t n,
                                                               int32_t* overflow,
                                                               unsigned long long* counters) {
    __shared__ uint32_t s_stack[LDS_STACK][TRACE_BLOCK];
    const int64_t i = (int64_t)blockIdx.x * TRACE_BLOCK + threadIdx.x;
    TraceCounts c = {0, 0, 0, 0, 0};
    uint32_t spill[SPILL_STACK];
    ClosestTrav tr;
    tr.idle();
    if (i < n) {
        const kpt_ray r = rays[i];
        tr.init(S, make_ray(mk3(r.org[0], r.org[1], r.org[2]), mk3(r.dir[0], r.dir[1], r.dir[2])), r.tmin, r.tmax,
                StackShape{&s_stack[0][threadIdx.x], TRACE_BLOCK, LDS_STACK}, spill);
    }
    tr.template run<COUNT>(S, &c);   // all lanes: the triangles of a leaf spread over the wave
    if (i < n) {
        const Hit h = tr.hit();
        kpt_hit o;
        o.t = h.t;
        if (h.slot >= 0) {
            o.prim_id = S.tris[h.slot].prim;
            o.inst_id = h.inst;
            o.bary[0] = 1.0f - h.u - h.v;
            o.bary[1] = h.u;
            o.bary[2] = h.v;
        } else {
            o.prim_id = -1; o.inst_id = -1; o.bary[0] = 0.0f; o.bary[1] = 0.0f; o.bary[2] = 0.0f;
        }
        hits[i] = o;
        if (tr.st.overflow()) atomicOr(overflow, 1);
    }
    if (COUNT) {
        // wave-level reduction, then one atomic per wave and counter
        uint32_t v[5] = {c.interior, c.leaf, c.tri, c.entries, c.tlas};
        for (int k = 0; k < 5; ++k) {
            unsigned long long x = v[k];
            for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
            if ((threadIdx.x & 63) == 0) atomicAdd(&counters[k], x);
        }
    }
}

__global__ __launch_bounds__(TRACE_BLOCK) void k_trace_any(SceneView S, const kpt_ray* __restrict__ rays,
                                                           int32_t* __restrict__ occluded, int64_t n,
                                                           int32_t* overflow) {
    __shared__ uint32_t s_stack[LDS_STACK][TRACE_BLOCK];
    const int64_t i = (int64_t)blockIdx.x * TRACE_BLOCK + threadIdx.x;
    uint32_t spill[SPILL_STACK];
    AnyTrav tr;
    tr.idle();
    if (i < n) {
        const kpt_ray r = rays[i];
        tr.init(S, make_ray(mk3(r.org[0], r.org[1], r.org[2]), mk3(r.dir[0], r.dir[1], r.dir[2])), r.tmin, r.tmax,
                StackShape{&s_stack[0][threadIdx.x], TRACE_BLOCK, LDS_STACK}, spill);
    }
    tr.template run<false>(S, nullptr);
    if (i < n) {
        occluded[i] = tr.any() ? 1 : 0;
        if (tr.st.overflow()) atomicOr(overflow, 1);
    }
}

hipError_t launch_trace_closest(hipStream_t s, const SceneView& S, const kpt_ray* rays, kpt_hit* hits, int64_t n,
                                int32_t* overflow, kpt_trace_counters* counters) {
    if (n <= 0) return hipSuccess;
    dim3 grid((unsigned)((n + TRACE_BLOCK - 1) / TRACE_BLOCK));
    if (counters) {
        hipLaunchKernelGGL(k_trace_closest<true>, grid, dim3(TRACE_BLOCK), 0, s, S, rays, hits, n, overflow,
                           reinterpret_cast<unsigned long long*>(counters));
    } else {
        hipLaunchKernelGGL(k_trace_closest<false>, grid, dim3(TRACE_BLOCK), 0, s, S, rays, hits, n, overflow,
                           (unsigned long long*)nullptr);
    }
    return hipGetLastError();
}

hipError_t launch_trace_any(hipStream_t s, const SceneView& S, const kpt_ray* rays, int32_t* occluded, int64_t n,
                            int32_t* overflow) {
    if (n <= 0) return hipSuccess;
    dim3 grid((unsigned)((n + TRACE_BLOCK - 1) / TRACE_BLOCK));
    hipLaunchKernelGGL(k_trace_any, grid, dim3(TRACE_BLOCK), 0, s, S, rays, occluded, n, overflow);
    return hipGetLastError();
}

// ------------------------------------------------------------------ megakernel
// computePathTraceSamplesMegaKernel (kernels.cu:385-451) with static
// accumulation (Integrator::addSample, integrator.cuh:406-416) or temporal
// reprojection (reprojectAccumulate, kernels.cu:299-338).  16x16 pixel
// tiles, XCD-swizzled tile order.  4 waves per SIMD (128 VGPRs): a 640x360
// frame of depth 3 takes 937 us, 1017 at 3 waves, 983 at 5, 996 at 6 (1067 at
// 4 with the shadow rays traced before the next vertex's rays, wave by wave).
constexpr int TILE = 16;

__global__ __launch_bounds__(TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_megakernel(SceneView S, FrameConst fc, int32_t frame,
                                                            FrameBuffers fb, int32_t* overflow) {
    __shared__ uint32_t s_stack[LDS_STACK][TRACE_BLOCK];
    const uint32_t tiles_x = (fc.width + TILE - 1) / TILE;
    const uint32_t tiles_y = (fc.height + TILE - 1) / TILE;
    const uint32_t tile = xcd_swizzle(blockIdx.x, tiles_x * tiles_y);
    const int px = (int)((tile % tiles_x) * TILE + (threadIdx.x % TILE));
    const int py = (int)((tile / tiles_x) * TILE + (threadIdx.x / TILE));
    const bool inside = px < fc.width && py < fc.height;
    const int64_t idx = (int64_t)py * fc.width + px;
    uint32_t seed = init_seed(px, py, fc.width, frame, fc.seed_mode);
    // BoxFilter::sample consumes two numbers whose jitter is discarded (kernels.cu:397-402)
    (void)rng1(seed);
    (void)rng1(seed);
    Ray ray = camera_ray(fc, px, py);
    VisOut vs;
    vs.albedo = mk3(0.0f, 0.0f, 0.0f); vs.normal = mk3(0.0f, 0.0f, 0.0f); vs.pos = mk3(0.0f, 0.0f, 0.0f);
    vs.depth = __builtin_inff(); vs.inst = -1; vs.prim = -1;
    bool ovf = false;
    v3 L = li_path(S, fc, inside, ray, seed, StackShape{&s_stack[0][threadIdx.x], TRACE_BLOCK, LDS_STACK}, &ovf, &vs);
    if (!inside) return;
    L = (mk3(1.0f, 1.0f, 1.0f) * 1.0f) * L;
    L = clamp_output(L);
    write_pixel(S, fc, fb, frame, idx, px, py, L, vs.albedo, vs.normal, vs.depth, vs.inst, vs.prim, vs.pos);
    if (ovf) atomicOr(overflow, 1);
}

hipError_t launch_megakernel(hipStream_t s, const SceneView& S, const FrameConst& fc, int32_t frame,
                             const FrameBuffers& fb, int32_t* overflow) {
    const uint32_t tiles = ((fc.width + TILE - 1) / TILE) * ((fc.height + TILE - 1) / TILE);
    hipLaunchKernelGGL(k_megakernel, dim3(tiles), dim3(TRACE_BLOCK), 0, s, S, fc, frame, fb, overflow);
    return hipGetLastError();
}

__global__ void k_clear4(float4* p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

hipError_t launch_clear(hipStream_t s, float4* p, int64_t n) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_clear4, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

}  // namespace kpt
