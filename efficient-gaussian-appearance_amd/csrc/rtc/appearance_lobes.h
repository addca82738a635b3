// Normalised anisotropic spherical Gaussian lobes: NASG (EFGS_MODEL == 3, 8 raw parameters per lobe) and
// NASGabor (EFGS_MODEL == 4, 9 per lobe, an extra Gabor factor (1 + cos(k v_x)) / 2).
//   raw [0..2] -> tanh -> cos(theta), cos(phi), cos(tau) of the lobe frame
//   raw [3]    -> exp  -> sharpness lambda (<= 1e4)       raw [4] -> exp -> anisotropy a (<= 1e4)
//   NASGabor raw [5] -> k = 20 (tanh + 1)                 last 3 -> residual activation -> rgb amplitude
//   K = (v.z + 1)/2, K_e = eps + a (v.x)^2 / (1 - (v.z)^2), E = K^K_e,
//   N = lambda sqrt(1 + a) / (2 pi (1 + eps_n - exp(-2 lambda))), pdf = exp(2 lambda (E K - 1)) E [G] N
// Reference: B/rasterization/rtc/appearance_nasg.cuh:164-350, appearance_nasgabor.cuh:25-223.
#pragma once

namespace efgs {

constexpr float lobe_two_pi = 6.28318530717958647692f;
constexpr float lobe_eps = 5e-6f;
constexpr float lobe_eps_norm = 1e-8f;
constexpr float lobe_cos_limit = 0.999999f;
constexpr float lobe_sin_limit = 1.41421321e-3f;  // sqrt(1 - lobe_cos_limit^2)
constexpr float lobe_pole_limit = 0.99999988f;
constexpr float lobe_min_om = 2.38418579e-7f;  // 1 - lobe_pole_limit^2
constexpr float lobe_shape_limit = 1e4f;
constexpr float lobe_freq_scale = 20.0f;
constexpr float lobe_log2e = 1.44269504088896340736f, lobe_ln2 = 0.69314718055994530942f;

// Lobe arithmetic on the hardware's exp2, log2, reciprocal and square root (1 ulp each) and fused multiply-adds: the
// lobe kernels issued 6.6e7 (forward) and 1.16e8 (backward) VALU instructions for 8 lobes on 1M Gaussians, most of them
// in the library's tanh, exp and log and in correctly rounded divides and square roots. Against 64 bits, values and
// gradients are as close as those were, or closer (50k Gaussians of 8 lobes, three draws; median and 99th percentile of
// the error, as a share of the old one: raw angles of deviation 1, values 0.93 and 1.00, sharpness gradients 0.86 and 0.99,
// angle gradients 0.83 and 0.99; deviation 0.01, values 0.94 and 0.90; deviation 3, values 0.15 and 0.11; sharpness of
// e^4, values 0.90 and 0.98), because of three things that cost a few instructions each: tanh and sech of small angles
// by polynomial (as 1 - 2 u^2 / (1 + u^2) at all angles, tanh has an absolute error of 6e-8 where it should have a
// relative one, and angle gradients were 1.4 to 1.6 times as far off), sech x instead of sqrt(1 - tanh^2 x) for large
// ones, and lobe_view below. With them NASG on 1M Gaussians at 1080p takes 95 us forward and 148 us backward, 90 and 145
// without (213 us backward on the library's functions, with the row staging of the time).

// tanh x and sech x = sqrt(1 - tanh^2 x). |x| < 0.7: polynomials in x^2 (x + x^3 P and 1 + x^2 Q; P and Q fitted for the least
// largest relative error of the result, 2e-8); above, from u = exp(-|x|): sech x = 2 u / (1 + u^2) and tanh |x| =
// 1 - u sech x. (Up to 0.5 with one coefficient less: the same time, errors 3 to 6 % larger.)
__device__ __forceinline__ float lobe_tanh(float x, float& sech) {
    const float z = x * x;
    float p = __builtin_fmaf(z, -5.13866186e-3f, 2.00919697e-2f);
    p = __builtin_fmaf(z, p, -5.35588611e-2f);
    p = __builtin_fmaf(z, p, 1.33291107e-1f);
    p = __builtin_fmaf(z, p, -3.33331899e-1f);
    float q = __builtin_fmaf(z, -8.05757752e-3f, 3.15411327e-2f);
    q = __builtin_fmaf(z, q, -8.40721233e-2f);
    q = __builtin_fmaf(z, q, 2.08265854e-1f);
    q = __builtin_fmaf(z, q, -4.99997688e-1f);
    const float u = __builtin_amdgcn_exp2f(-lobe_log2e * fabsf(x));
    const float s = (u + u) * __builtin_amdgcn_rcpf(__builtin_fmaf(u, u, 1.0f));
    const bool small = fabsf(x) < 0.7f;
    sech = small ? __builtin_fmaf(z, q, 1.0f) : s;
    return small ? __builtin_fmaf(x * z, p, x) : __builtin_copysignf(__builtin_fmaf(-u, s, 1.0f), x);
}

// exp x with the rounding of x log2 e compensated (x clamped to the range of finite, normal results; NaN: the largest)
__device__ __forceinline__ float lobe_exp(float x) {
    x = fmaxf(fminf(x, 88.0f), -87.0f);
    const float t = x * lobe_log2e;
    const float r = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, lobe_log2e, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return __builtin_fmaf(e, r * lobe_ln2, e);
}

struct LobeFrame {
    float3 x, z;
    float ct, cp, cu, st, sp, su;
};

// frame of the raw angles; th, tp, tu receive their tanh before the clamp
__device__ __forceinline__ LobeFrame build_lobe_frame(float a, float b, float c, float& th, float& tp, float& tu) {
    LobeFrame f;
    th = lobe_tanh(a, f.st);
    tp = lobe_tanh(b, f.sp);
    tu = lobe_tanh(c, f.su);
    f.ct = clampf(th, -lobe_cos_limit, lobe_cos_limit);
    f.cp = clampf(tp, -lobe_cos_limit, lobe_cos_limit);
    f.cu = clampf(tu, -lobe_cos_limit, lobe_cos_limit);
    f.st = fmaxf(f.st, lobe_sin_limit);
    f.sp = fmaxf(f.sp, lobe_sin_limit);
    f.su = fmaxf(f.su, lobe_sin_limit);
    const float cc = f.cp * f.cu;
    f.x = make_float3(__builtin_fmaf(f.ct, cc, -f.st * f.su), __builtin_fmaf(f.st, cc, f.ct * f.su), -f.sp * f.cu);
    f.z = make_float3(f.ct * f.sp, f.st * f.sp, f.cp);
    return f;
}

__device__ __forceinline__ float lobe_dot(float3 a, float3 b) { return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.y, b.y, a.x * b.x)); }

// The view direction in a lobe's frame: vx, vz (vzc: within the pole limits), om = 1 - vz^2 and K = (1 + vz) / 2. Towards
// the antipole both differences cancel, and the lobe holds their quotient and the logarithm of K: there om is the sum of
// the other components' squares, and K follows from it (flat lobes, whose values near the antipole count: values 0.1
// to 0.2 times as far off, gradients 0.01). Elsewhere both come from vz: on the lobe's own side om and log K are nearly
// proportional, and the error that they then share drops out of K_e log K (taken from the squares there too, sharpness
// gradients were 1.4 times as far off).
struct LobeView {
    float vx, vz, vzc, om, K;
};
__device__ __forceinline__ LobeView lobe_view(const LobeFrame& f, float3 d) {
    LobeView v;
    v.vz = lobe_dot(d, f.z);
    v.vx = lobe_dot(d, f.x);
    v.vzc = clampf(v.vz, -lobe_pole_limit, lobe_pole_limit);
    const float cs = f.cp * f.su;
    const float yx = __builtin_fmaf(f.ct, cs, f.st * f.cu), yy = __builtin_fmaf(f.ct, f.cu, -f.st * cs);
    const float vy = __builtin_fmaf(d.z, f.sp * f.su, __builtin_fmaf(d.y, yy, -d.x * yx));
    const float om = fmaxf(__builtin_fmaf(v.vx, v.vx, vy * vy), lobe_min_om);
    const bool away = v.vzc < -0.75f;
    v.om = away ? om : __builtin_fmaf(-v.vzc, v.vzc, 1.0f);
    v.K = away ? 0.5f * om * __builtin_amdgcn_rcpf(1.0f - v.vzc) : __builtin_fmaf(0.5f, v.vzc, 0.5f);
    return v;
}

// cos and sin of 2 pi t (t in revolutions): t reduced to [-1/2, 1/2] exactly, then to the nearest quarter, and Taylor
// polynomials of the remaining angle, at most pi / 4
__device__ __forceinline__ void lobe_sincos_revolutions(float t, float& s, float& c) {
    t -= __builtin_rintf(t);
    const float q = __builtin_rintf(4.0f * t);
    const float y = __builtin_fmaf(-0.25f, q, t) * lobe_two_pi, z = y * y;
    const float sy = __builtin_fmaf(y * z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 2.75573192e-6f, -1.98412698e-4f), 8.33333333e-3f), -1.66666667e-1f), y);
    const float cy = __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 2.48015873e-5f, -1.38888889e-3f), 4.16666667e-2f), -0.5f), 1.0f);
    const int k = static_cast<int>(q);
    const bool swap = (k & 1) != 0;
    const float a = swap ? cy : sy, b = swap ? sy : cy;
    s = (k & 2) != 0 ? -a : a;
    c = ((k + 1) & 2) != 0 ? -b : b;
}

constexpr float lobe_rev_scale = lobe_freq_scale / lobe_two_pi;

template <int RES_ACT, bool GABOR>
__device__ inline float3 lobe_residual(const float* p, float3 d, uint32_t lobes) {
    constexpr int stride = GABOR ? 9 : 8;
    constexpr int wo = GABOR ? 6 : 5;
    float r = 0.0f, g = 0.0f, b = 0.0f;
    for (uint32_t l = 0; l < lobes; l++, p += stride) {
        float th, tp, tu;
        const LobeFrame f = build_lobe_frame(p[0], p[1], p[2], th, tp, tu);
        const float lambda = fminf(lobe_exp(p[3]), lobe_shape_limit);
        const float an = fminf(lobe_exp(p[4]), lobe_shape_limit);
        const LobeView view = lobe_view(f, d);
        const float vx = view.vx, vz = view.vz, K = view.K;
        const float Ke = __builtin_fmaf(an * (vx * vx), __builtin_amdgcn_rcpf(view.om), lobe_eps);
        const float E = __builtin_amdgcn_exp2f(Ke * __builtin_amdgcn_logf(K));  // K^Ke (K in (0, 1], Ke > 0)
        const float l2 = 2.0f * lobe_log2e * lambda;
        const float N = lambda * __builtin_amdgcn_sqrtf(1.0f + an) * __builtin_amdgcn_rcpf(lobe_two_pi * (1.0f + lobe_eps_norm - __builtin_amdgcn_exp2f(-l2)));
        const float P = __builtin_amdgcn_exp2f(l2 * __builtin_fmaf(E, K, -1.0f));
        float v = P * E * N;
        if (GABOR) {
            float sech, skv, ckv;
            lobe_sincos_revolutions((lobe_tanh(p[5], sech) + 1.0f) * lobe_rev_scale * vx, skv, ckv);
            v *= __builtin_fmaf(0.5f, ckv, 0.5f);
        }
        const float pdf = vz >= lobe_pole_limit ? 1.0f : (vz > -lobe_pole_limit ? v : 0.0f);
        r = __builtin_fmaf(pdf, residual_activation<RES_ACT>(p[wo]), r);
        g = __builtin_fmaf(pdf, residual_activation<RES_ACT>(p[wo + 1]), g);
        b = __builtin_fmaf(pdf, residual_activation<RES_ACT>(p[wo + 2]), b);
    }
    return make_float3(r, g, b);
}

template <int RES_ACT, bool GABOR>
__device__ inline float3 lobe_residual_backward(const float* p, float3 gc, float* gp, float3 d, float norm_rcp, uint32_t lobes) {
#pragma clang fp contract(fast)
    constexpr int stride = GABOR ? 9 : 8;
    constexpr int wo = GABOR ? 6 : 5;
    float3 gd = make_float3(0.0f, 0.0f, 0.0f);
    for (uint32_t l = 0; l < lobes; l++, p += stride, gp += stride) {
        float th, tp, tu;
        const LobeFrame f = build_lobe_frame(p[0], p[1], p[2], th, tp, tu);
        const float lu = lobe_exp(p[3]), au = lobe_exp(p[4]);
        const float lambda = fminf(lu, lobe_shape_limit), an = fminf(au, lobe_shape_limit);
        float sk = 0.0f, k = 0.0f;
        if (GABOR) k = lobe_tanh(p[5], sk) + 1.0f;
        const float w0 = residual_activation<RES_ACT>(p[wo]);
        const float w1 = residual_activation<RES_ACT>(p[wo + 1]);
        const float w2 = residual_activation<RES_ACT>(p[wo + 2]);
        const LobeView view = lobe_view(f, d);
        const float vx = view.vx, vz = view.vz, K = view.K;
        const float rom = __builtin_amdgcn_rcpf(view.om);
        const float vx2 = vx * vx, avr = an * vx * rom;
        const float Ke = __builtin_fmaf(an * vx2, rom, lobe_eps);
        const float logK2 = __builtin_amdgcn_logf(K);
        const float E = __builtin_amdgcn_exp2f(Ke * logK2);  // K^Ke (K in (0, 1], Ke > 0)
        const float l2 = 2.0f * lobe_log2e * lambda;
        const float em2l = __builtin_amdgcn_exp2f(-l2);
        const float rnd = __builtin_amdgcn_rcpf(lobe_two_pi * (1.0f + lobe_eps_norm - em2l));
        const float rs1a = __builtin_amdgcn_rsqf(1.0f + an);
        const float s1a = (1.0f + an) * rs1a;
        const float N = lambda * s1a * rnd;
        const float EK1 = __builtin_fmaf(E, K, -1.0f);
        const float P = __builtin_amdgcn_exp2f(l2 * EK1);
        float skv = 0.0f, ckv = 1.0f;
        if (GABOR) lobe_sincos_revolutions(k * lobe_rev_scale * vx, skv, ckv);
        const float G = GABOR ? __builtin_fmaf(0.5f, ckv, 0.5f) : 1.0f;
        const bool valid = fabsf(vz) < lobe_pole_limit;
        const float PE = P * E, PEN = PE * N, v = GABOR ? PEN * G : PEN;
        const float pdf = vz >= lobe_pole_limit ? 1.0f : (valid ? v : 0.0f);
        gp[wo] = gc.x * pdf * residual_activation_grad<RES_ACT>(w0);
        gp[wo + 1] = gc.y * pdf * residual_activation_grad<RES_ACT>(w1);
        gp[wo + 2] = gc.z * pdf * residual_activation_grad<RES_ACT>(w2);
        const float gpdf = valid ? (gc.x * w0 + gc.y * w1 + gc.z * w2) : 0.0f;
        // gv: the gradient with respect to the lobe's logarithm; every factor's derivative is taken as one of its logarithm
        // (d log P = 2 (E K - 1) d lambda + 2 lambda (K dE + E dK), d log E = d (Ke log K), d log N, d log G)
        const float gv = gpdf * v;
        const float dlogN_dl = 1.0f - lambda * 2.0f * lobe_two_pi * em2l * rnd;  // lambda d log N / d lambda
        gp[3] = lu >= lobe_shape_limit ? 0.0f : gv * (2.0f * lambda * EK1 + dlogN_dl);
        const float logK = logK2 * lobe_ln2;
        const float both = 1.0f + 2.0f * lambda * K * E;  // d log (P E) / d log E
        gp[4] = au >= lobe_shape_limit ? 0.0f : gv * (both * logK * (vx2 * rom) + 0.5f * rs1a * rs1a) * an;
        float gvx = gv * both * logK * (2.0f * avr);
        if (GABOR) {
            const float gG = gpdf * PEN * (-0.5f * skv);  // d pdf / d (k vx)
            gp[5] = gG * vx * lobe_freq_scale * (sk * sk);
            gvx += gG * (k * lobe_freq_scale);
        }
        const float dKe_dvz = avr * vx * 2.0f * vz * rom;
        const float gvz = gv * (both * (0.5f * Ke * __builtin_amdgcn_rcpf(K) + logK * dKe_dvz) + lambda * E);
        const float gxx = gvx * d.x, gxy = gvx * d.y, gxz = gvx * d.z;
        const float gzx = gvz * d.x, gzy = gvz * d.y, gzz = gvz * d.z;
        gd.x += gvx * f.x.x + gvz * f.z.x;
        gd.y += gvx * f.x.y + gvz * f.z.y;
        gd.z += gvx * f.x.z + gvz * f.z.z;
        // d cos = sin^2 d raw for each angle, and d sin = -(cos / sin) d cos: one sin of the sin^2 cancels the quotient (the
        // three reciprocals and products of the quotients 152 -> 148 us)
        const float cc = f.cp * f.cu, q = gxx * f.ct + gxy * f.st;
        const float gt = f.st * (gxx * cc + gxy * f.su + gzx * f.sp) - f.ct * (gxy * cc - gxx * f.su + gzy * f.sp);
        const float gph = f.sp * (q * f.cu + gzz) - f.cp * (gzx * f.ct + gzy * f.st - gxz * f.cu);
        const float gta = f.su * (q * f.cp - gxz * f.sp) - f.cu * (gxy * f.ct - gxx * f.st);
        gp[0] = fabsf(th) >= lobe_cos_limit ? 0.0f : gt * f.st;
        gp[1] = fabsf(tp) >= lobe_cos_limit ? 0.0f : gph * f.sp;
        gp[2] = fabsf(tu) >= lobe_cos_limit ? 0.0f : gta * f.su;
    }
    return direction_grad_to_mean(gd, d, norm_rcp);
}

}  // namespace efgs
