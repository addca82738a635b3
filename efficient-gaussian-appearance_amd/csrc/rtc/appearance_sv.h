// Soft spherical-Voronoi residual (EFGS_MODEL == 2): R(v) = sum_k softmax_k(-tau_k |site_k - v|) c_k with
// 7 raw parameters per site [site xyz | log tau | rgb], evaluated as a single-pass online softmax.
// Reference: B/rasterization/rtc/appearance_sv.cuh:26-139.
#pragma once

namespace efgs {

constexpr float sv_eps = 1e-12f;
constexpr float sv_log2e = 1.44269504088896340736f, sv_ln2 = 0.69314718055994530942f;

// Site arithmetic on the hardware's exp2, reciprocal and reciprocal square root (1 ulp each), each with one Newton step
// or its argument's rounding compensated, and fused multiply-adds; the softmax takes one exponential per site (the
// larger of the running maximum and the new logit has weight 1). Against 64 bits, colours and gradients are as close as
// with the library's exp and correctly rounded divides and square roots (50k primitives of 8 sites, two draws: median and
// 99th percentile of the error 0.97 to 1.02 of the old ones, 1.04 to 1.2 without the steps), which were most of a site's
// instructions (150k primitives at 1237 x 823, 8 sites: forward 30.6 -> 27.8 us, backward 35.0 -> 32.5 us; the step of
// 223 us is the same with and without the Newton steps).

// exp x (x at most 88, no NaN and no infinity) with the rounding of x log2 e compensated
__device__ __forceinline__ float sv_exp_bounded(float x) {
    const float t = x * sv_log2e;
    const float r = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, sv_log2e, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return __builtin_fmaf(e, r * sv_ln2, e);
}
// any x: clamped to the range of finite, normal results (NaN: the largest)
__device__ __forceinline__ float sv_exp(float x) { return sv_exp_bounded(fmaxf(fminf(x, 88.0f), -87.0f)); }
// exp x for x <= 0 (NaN: 1); the clamp keeps the compensation finite
__device__ __forceinline__ float sv_weight(float x) { return sv_exp_bounded(fmaxf(fminf(x, 0.0f), -200.0f)); }

// 1 / x, the hardware's reciprocal with one Newton step (0 and infinities: NaN)
__device__ __forceinline__ float sv_rcp(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
}
// 1 / sqrt(x) (x positive; infinity: 0) and sqrt(x) (x at least FLT_MIN, finite), each with one Newton step
__device__ __forceinline__ float sv_rsqrt(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    return __builtin_fmaf(0.5f * y, fmaxf(__builtin_fmaf(-x * y, y, 1.0f), -1.0f), y);
}
__device__ __forceinline__ float sv_sqrt(float x) {
    const float y = __builtin_amdgcn_rsqf(x), s = x * y;
    return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
}

__device__ __forceinline__ float sv_dot(float x, float y, float z) { return __builtin_fmaf(z, z, __builtin_fmaf(y, y, x * x)); }

// a site: its unit direction minus the view direction, their distance, its sharpness and the logit
struct SvSite {
    float inv, dx, dy, dz, dist, tau, logit;
};
__device__ __forceinline__ SvSite sv_site(const float* p, float3 d) {
    SvSite s;
    s.inv = sv_rsqrt(fmaxf(sv_dot(p[0], p[1], p[2]), sv_eps * sv_eps));
    s.dx = __builtin_fmaf(s.inv, p[0], -d.x);
    s.dy = __builtin_fmaf(s.inv, p[1], -d.y);
    s.dz = __builtin_fmaf(s.inv, p[2], -d.z);
    s.dist = sv_sqrt(fmaxf(sv_dot(s.dx, s.dy, s.dz), 1.17549435e-38f));
    s.tau = sv_exp(p[3]);
    s.logit = -s.tau * s.dist;
    return s;
}

// running softmax over the sites
struct SvState {
    float max_logit = -1e30f, wsum = 0.0f, r = 0.0f, g = 0.0f, b = 0.0f;
};

template <int RES_ACT>
__device__ __forceinline__ void sv_add_sites(SvState& v, const float* p, float3 d, uint32_t sites) {
    for (uint32_t s = 0; s < sites; s++, p += 7) {
        const float logit = sv_site(p, d).logit;
        const bool higher = logit > v.max_logit;
        const float e = sv_weight(-fabsf(logit - v.max_logit));
        const float rescale = higher ? e : 1.0f, w = higher ? 1.0f : e;
        v.wsum = __builtin_fmaf(v.wsum, rescale, w);
        v.r = __builtin_fmaf(v.r, rescale, w * residual_activation<RES_ACT>(p[4]));
        v.g = __builtin_fmaf(v.g, rescale, w * residual_activation<RES_ACT>(p[5]));
        v.b = __builtin_fmaf(v.b, rescale, w * residual_activation<RES_ACT>(p[6]));
        v.max_logit = higher ? logit : v.max_logit;
    }
}

__device__ __forceinline__ float3 sv_color(const SvState& v) {
    const float wr = sv_rcp(v.wsum);
    return make_float3(wr * v.r, wr * v.g, wr * v.b);
}

// writes dL/d(site parameters) of the active sites and returns dL/dmean through the view direction. A site's
// parameters are read before its gradients are written, and no later step reads them, so gp may be p0 itself.
template <int RES_ACT>
__device__ inline float3 sv_residual_backward(const float* p0, float3 gc, float* gp, float3 d, float norm_rcp, uint32_t sites) {
#pragma clang fp contract(fast)
    if (sites == 0) return make_float3(0.0f, 0.0f, 0.0f);
    SvState v;
    sv_add_sites<RES_ACT>(v, p0, d, sites);
    const float wr = sv_rcp(v.wsum);
    const float gmean = wr * (gc.x * v.r + gc.y * v.g + gc.z * v.b);
    float3 gd = make_float3(0.0f, 0.0f, 0.0f);
    const float* p = p0;
    for (uint32_t s = 0; s < sites; s++, p += 7, gp += 7) {
        const SvSite q = sv_site(p, d);
        const float w = sv_weight(q.logit - v.max_logit) * wr;
        const float cr = residual_activation<RES_ACT>(p[4]);
        const float cg = residual_activation<RES_ACT>(p[5]);
        const float cb = residual_activation<RES_ACT>(p[6]);
        const float3 site = make_float3(q.inv * p[0], q.inv * p[1], q.inv * p[2]);
        gp[4] = w * gc.x * residual_activation_grad<RES_ACT>(cr);
        gp[5] = w * gc.y * residual_activation_grad<RES_ACT>(cg);
        gp[6] = w * gc.z * residual_activation_grad<RES_ACT>(cb);
        const float glogit = w * ((gc.x * cr + gc.y * cg + gc.z * cb) - gmean);
        gp[3] = -q.dist * q.tau * glogit;
        const float f = -q.tau * glogit * sv_rcp(fmaxf(q.dist, sv_eps));
        const float gx = f * q.dx, gy = f * q.dy, gz = f * q.dz;
        const float dd = gx * site.x + gy * site.y + gz * site.z;
        gp[0] = (gx - dd * site.x) * q.inv;
        gp[1] = (gy - dd * site.y) * q.inv;
        gp[2] = (gz - dd * site.z) * q.inv;
        gd.x -= gx;
        gd.y -= gy;
        gd.z -= gz;
    }
    return direction_grad_to_mean(gd, d, norm_rcp);
}

}  // namespace efgs
