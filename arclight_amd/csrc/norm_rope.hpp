// Per-head RMSNorm, weight and rotary embedding of 128-float rows, 8 lanes
// to a row (gfx950): the arithmetic of the attention-input producers,
// shared by the stand-alone kernels and the decode kernel that folds them
// into its prologue, so that both give the same bits.
//   rms_norm  nnml/src/ops/ops.cpp:680-726
//   mul       nnml/src/ops/ops.cpp:1248-1250
//   rope_ext  nnml/src/ops/ops.cpp:728-777, 871-962
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Rotation constants of the rope_ext op, resolved on the host as the
// reference's rope op computes them (rope_yarn_corr_dims, the YaRN mscale).
struct RopeConsts {
    float theta_scale, freq_scale, ext_factor, corr0, corr1, mscale;
};

// Dims of pair i. MODE: 0 no rotation, 1 pairs (2i, 2i + 1), 2 NEOX pairs
// (i, i + 64).
template <int MODE> __device__ __forceinline__ int rope_d0(const int i) { return MODE == 1 ? 2 * i : i; }
template <int MODE> __device__ __forceinline__ int rope_d1(const int i) { return MODE == 1 ? 2 * i + 1 : i + 64; }

// The sum of v over groups of 8 lanes, in every lane of the group (DPP:
// lanes within a quad, then the two quads of 8 lanes mirrored).
template <int CTRL>
__device__ __forceinline__ double dpp_move(const double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) (uint32_t) b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) (uint32_t) (b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, (uint64_t) lo | (uint64_t) hi << 32);
}
__device__ __forceinline__ double sum8(double v) {
    v += dpp_move<0xb1>(v);                      // quad_perm [1, 0, 3, 2]
    v += dpp_move<0x4e>(v);                      // quad_perm [2, 3, 0, 1]
    v += dpp_move<0x141>(v);                     // row_half_mirror
    return v;
}

// x of lane l times scale, l times over, each product rounded: step k runs
// with the lanes above k enabled, one vector instruction a step (as selects
// the 63 steps were three each). Needs all 64 lanes of the wave.
__device__ __forceinline__ void rope_angle_steps(float & x, const float scale) {
    uint64_t all;
    asm volatile("s_mov_b64 %1, exec\n\t"
                 ".rept 63\n\t"
                 "s_lshl_b64 exec, exec, 1\n\t"
                 "v_mul_f32 %0, %2, %0\n\t"
                 ".endr\n\t"
                 "s_mov_b64 exec, %1"
                 : "+v"(x), "=&s"(all)
                 : "s"(scale)
                 : "scc");
}

// cos / sin (times mscale) of the lane's pair at position pos (ops.cpp:743-772);
// every lane of the wave takes part.
template <int MODE>
__device__ __forceinline__ void rope_cos_sin(const RopeConsts & r, const int32_t pos, const int lane, float & c,
                                             float & s) {
    // every product and sum rounded on its own, as the reference's C source
    // reads: at angles of thousands of radians one ulp of theta moves the
    // output by ~1e-4, so a fused multiply-add there would not match
#pragma clang fp contract(off)
    c = 1.0f;
    s = 0.0f;
    if constexpr (MODE != 0) {
        float theta_extrap = (float) pos;
        rope_angle_steps(theta_extrap, r.theta_scale);
        const float theta_interp = r.freq_scale * theta_extrap;
        float theta = theta_interp;
        if (r.ext_factor != 0.0f) {
            const float yv = ((float) lane - r.corr0) / fmaxf(0.001f, r.corr1 - r.corr0);
            const float ramp = 1.0f - fminf(1.0f, fmaxf(0.0f, yv));
            const float mix = ramp * r.ext_factor;
            theta = theta_interp * (1.0f - mix) + theta_extrap * mix;
        }
        sincosf(theta, &s, &c);
        c *= r.mscale;
        s *= r.mscale;
    }
}

// RMSNorm, weight and rotation of rows held by groups of 8 lanes (lanes
// 8i..8i+7 of a wave hold one row), each lane with 8 rotation pairs: lo[k]
// and hi[k] are the two dims of the lane's pair k, w_lo / w_hi their
// weights (1 where there is no weight, which leaves the product bit for bit
// unchanged), rot[k] the pair's (cos, sin). The row's sum of squares is
// taken in double; which pairs a lane holds decides the order of its terms,
// so two layouts can differ only where the partial sums are not exact in
// double, by rounding in the double's last bits, far below the f32 mean's
// resolution. Every lane of the wave takes part (the sum's moves).
template <int MODE>
__device__ __forceinline__ void norm_rope_group8(const float (&lo)[8], const float (&hi)[8], const float (&w_lo)[8],
                                                 const float (&w_hi)[8], const float eps, const float2 (&rot)[8],
                                                 float (&y_lo)[8], float (&y_hi)[8]) {
#pragma clang fp contract(off)
    double part[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float a = lo[k] * lo[k], b = hi[k] * hi[k];
        part[k] = (double) a + (double) b;
    }
#pragma unroll
    for (int h = 4; h >= 1; h /= 2)
#pragma unroll
        for (int k = 0; k < h; ++k) part[k] += part[k + h];
    const double sum = sum8(part[0]);
    const float mean = (float) (sum / 128.0);
    const float scale = 1.0f / sqrtf(mean + eps);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float n0 = (lo[k] * scale) * w_lo[k], n1 = (hi[k] * scale) * w_hi[k];
        y_lo[k] = n0;
        y_hi[k] = n1;
        if constexpr (MODE != 0) {
            y_lo[k] = n0 * rot[k].x - n1 * rot[k].y;
            y_hi[k] = n0 * rot[k].y + n1 * rot[k].x;
        }
    }
}
