// Producers of the attention operands for gfx950 (include/arclight_prologue.h):
// per-head RMSNorm, the norm weight and the rotary embedding of Q and K in
// one pass, K optionally straight into the f16 KV cache.
//
// Semantics: nnml_compute_forward_rms_norm_f32 (nnml/src/ops/ops.cpp:
// 680-726: squares summed in double, mean and scale in float), the f32 mul,
// and nnml_compute_forward_rope_f32 (ops.cpp:871-962) with rope_yarn and the
// rotation cache (ops.cpp:743-772): the angle of pair i is the position
// multiplied i times by theta_scale in float, exactly as the cache loop
// carries it.
//
// One wavefront takes 8 heads of one token, 8 lanes to a row of 128 floats:
// lane j of 8 holds dims 4j..4j+3 of each 32, so that a load or store of the
// wave covers whole 128-byte lines; the norm's sum is three DPP moves, and a
// row's rotation needs no other lane's values. The rotation's 64 (cos, sin)
// pairs are computed one per lane, once for the 8 rows, and handed over
// through LDS within the wave.
//
// What bounds it: for many tokens memory, for few the chain position ->
// angle (63 products in series) -> sine -> rows. One row per wave repeated
// that chain for every row and was bound by its vector instructions.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/arclight_prologue.h"
#include "fattn_kernels.hpp"
#include "kv_write.hpp"
#include "norm_rope.hpp"
#include "runtime.hpp"

namespace {

struct NormRopeParams {
    const char * x;     int64_t x_nb1, x_nb2;      // row (head h, token t) at x + h nb1 + t nb2
    const float * w;                               // [128] or null
    const int32_t * pos;                           // [T]
    char * y;           int64_t y_nb1, y_nb2;      // f32 rows, or the f16 cache (nb1 = row bytes)
    const char * rows;  int64_t rows_nb0;          // cache rows [T] or null
    int32_t rows64;
    int64_t n_rows_dst;
    int32_t y_vec;                                 // cache rows 8-byte aligned
    int32_t H, T;
    float eps;
    RopeConsts rope;
    int * err;                                     // [2]: first out-of-range cache row
};

constexpr int kRows = 8;                         // rows of a wave: heads of one token
constexpr int kWaves = 4;                        // waves of a workgroup: tokens

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

// Rows of heads h0 .. h0 + 7 of token t, one wavefront; rot: the wave's 64
// (cos, sin) pairs in LDS. MODE: 0 no rotation, 1 pairs (2i, 2i + 1), 2 NEOX
// pairs (i, i + 64).
template <int MODE, bool CACHE>
__device__ __forceinline__ void norm_rope_rows(const NormRopeParams & p, const int h0, const int t, const int lane,
                                               float2 * rot) {
    if (h0 >= p.H) return;
    const int l8 = lane & 7, h = h0 + (lane >> 3);
    const float * xr = (const float *) (p.x + (int64_t) min(h, p.H - 1) * p.x_nb1 + (int64_t) t * p.x_nb2);
    float4u x[4], w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = *(const float4u *) (xr + 32 * j + 4 * l8);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = p.w ? *(const float4u *) (p.w + 32 * j + 4 * l8) : float4u{1.0f, 1.0f, 1.0f, 1.0f};
    // pair k of the lane: in place (k % 4) of piece k / 4 and of the piece 64
    // dims on, or (MODE 1) values 2 (k % 2), 2 (k % 2) + 1 of piece k / 2
    float lo[8], hi[8], wl[8], wh[8];
    float2 cs[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int j = MODE == 1 ? k / 2 : k / 4, e = MODE == 1 ? 2 * (k % 2) : k % 4;
        lo[k] = x[j][e];
        hi[k] = MODE == 1 ? x[j][e + 1] : x[j + 2][e];
        wl[k] = w[j][e];
        wh[k] = MODE == 1 ? w[j][e + 1] : w[j + 2][e];
    }
    if constexpr (MODE != 0) {
        float c, s;
        rope_cos_sin<MODE>(p.rope, p.pos[t], lane, c, s);
        rot[lane] = float2{c, s};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            const int first = MODE == 1 ? 16 * (k / 2) + 2 * l8 : 32 * (k / 4) + 4 * l8 + k % 4;   // its pair
            const float4 v = *(const float4 *) (rot + first);
            cs[k] = float2{v.x, v.y};
            cs[k + 1] = float2{v.z, v.w};
        }
    }
    float yl[8], yh[8];
    norm_rope_group8<MODE>(lo, hi, wl, wh, p.eps, cs, yl, yh);
    float4u y[4];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int j = MODE == 1 ? k / 2 : k / 4, e = MODE == 1 ? 2 * (k % 2) : k % 4;
        y[j][e] = yl[k];
        if constexpr (MODE == 1) y[j][e + 1] = yh[k];
        else y[j + 2][e] = yh[k];
    }
    if constexpr (CACHE) {
        const char * ip = p.rows + (int64_t) t * p.rows_nb0;
        const int64_t r = p.rows64 ? *(const int64_t *) ip : (int64_t) *(const int32_t *) ip;
        if (r < 0 || r >= p.n_rows_dst) {
            if (lane == 0 && atomicCAS(p.err, 0, 1) == 0) p.err[1] = (int) r;
            return;
        }
        if (h >= p.H) return;
        _Float16 * yr = (_Float16 *) (p.y + r * p.y_nb1) + (int64_t) h * 128;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const half4 v = {(_Float16) y[j][0], (_Float16) y[j][1], (_Float16) y[j][2], (_Float16) y[j][3]};
            _Float16 * d = yr + 32 * j + 4 * l8;
            if (p.y_vec) {
                *(half4 *) d = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = v[e];
            }
        }
    } else {
        if (h >= p.H) return;
        float * yr = (float *) (p.y + (int64_t) h * p.y_nb1 + (int64_t) t * p.y_nb2);
#pragma unroll
        for (int j = 0; j < 4; ++j) *(float4u *) (yr + 32 * j + 4 * l8) = y[j];
    }
}

template <int MODE, bool CACHE>
__global__ __launch_bounds__(64 * kWaves) void norm_rope_kernel(const NormRopeParams p) {
    __shared__ __attribute__((aligned(16))) float2 rot[kWaves][64];
    prefetch_params(p);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x * kWaves + wave;
    if (t < p.T) norm_rope_rows<MODE, CACHE>(p, blockIdx.y * kRows, t, threadIdx.x & 63, rot[wave]);
}

// The attention inputs of one layer in one launch: blockIdx.y < yq are Q
// rows, then yk of K rows into the cache, then yv of the tokens' V rows.
// Traced, us per launch, one row per wave before: 512 tokens of 32 + 8 heads
// 14.3 -> 5.3, 1024 tokens of 64 + 8 heads 41.5 -> 13.2 (5.9 TB/s), 4 tokens
// of 32 + 8 heads 3.7 -> 2.5.
template <int MODE>
__global__ __launch_bounds__(64 * kWaves) void attn_inputs_kernel(const NormRopeParams q, const NormRopeParams k,
                                                                  const SetRowsParams v, const int yq, const int yk,
                                                                  const int yv) {
    __shared__ __attribute__((aligned(16))) float2 rot[kWaves][64];
    prefetch_params(q, k, v, yq, yk, yv);
    const int by = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x * kWaves + wave;
    if (t >= q.T) return;
    if (by < yq) norm_rope_rows<MODE, false>(q, by * kRows, t, lane, rot[wave]);
    else if (by < yq + yk) norm_rope_rows<MODE, true>(k, (by - yq) * kRows, t, lane, rot[wave]);
    else set_rows_row(v, t, 0, 0, (by - yq - yk) * 64 + lane, yv * 64);
}

template <int MODE>
hipError_t launch_mode(const NormRopeParams & p, bool cache, hipStream_t stream) {
    const dim3 grid((unsigned) ((p.T + kWaves - 1) / kWaves), (unsigned) ((p.H + kRows - 1) / kRows));
    if (cache) hipLaunchKernelGGL((norm_rope_kernel<MODE, true>), grid, dim3(64 * kWaves), 0, stream, p);
    else       hipLaunchKernelGGL((norm_rope_kernel<MODE, false>), grid, dim3(64 * kWaves), 0, stream, p);
    return hipGetLastError();
}

// YaRN correction dimension for a rotation count (ops.cpp:728-730).
float yarn_corr_dim(int n_dims, int n_ctx_orig, float n_rot, float base) {
    const double pi = 3.14159265358979323846;
    return n_dims * logf(n_ctx_orig / (n_rot * 2 * (float) pi)) / (2 * logf(base));
}

// Checks the operands as al_rms_norm_rope_f32 documents them and fills p
// and the rotation mode (0 none, 1 normal, 2 NEOX).
int norm_rope_params(const al_tensor * x, const al_tensor * w, const al_tensor * pos, float eps,
                     const al_rope_params * rope, const al_tensor * y, const al_tensor * rows, NormRopeParams * out,
                     int * mode_out) {
    if (!x || !pos || !y) return al_fail(AL_ERR_INVALID, "rms_norm_rope: x, pos and y required");
    if (x->type != AL_TYPE_F32 || x->ne[0] != 128 || x->nb[0] != 4 || x->ne[3] != 1)
        return al_fail(AL_ERR_UNSUPPORTED, "rms_norm_rope: x must be f32 [128, H, T, 1] with nb0 = 4");
    const int64_t H = x->ne[1], T = x->ne[2];
    if (H <= 0 || T <= 0 || T > INT32_MAX / 2 || H > 65535 * 4) return al_fail(AL_ERR_INVALID, "rms_norm_rope: bad H %lld or T %lld", (long long) H, (long long) T);
    if (!(eps >= 0.0f)) return al_fail(AL_ERR_INVALID, "rms_norm_rope: eps %g < 0 (ops.cpp:697)", (double) eps);
    if (w && (w->type != AL_TYPE_F32 || w->ne[0] < 128 || w->nb[0] != 4 || !w->data))
        return al_fail(AL_ERR_INVALID, "rms_norm_rope: w must be f32 [128]");
    if (pos->type != AL_TYPE_I32 || pos->ne[0] != T || pos->nb[0] != 4 || !pos->data)
        return al_fail(AL_ERR_INVALID, "rms_norm_rope: pos must be i32 [T] (tensor.cpp:1014-1019)");
    int mode = 0;
    NormRopeParams p;
    memset(&p, 0, sizeof(p));
    if (rope) {
        if (rope->n_dims != 128) return al_fail(AL_ERR_UNSUPPORTED, "rms_norm_rope: n_dims %d (only the full head, 128)", rope->n_dims);
        if (rope->mode == AL_ROPE_NEOX) mode = 2;
        else if (rope->mode == AL_ROPE_NORMAL) mode = 1;
        else return al_fail(AL_ERR_UNSUPPORTED, "rms_norm_rope: rope mode %d", rope->mode);
        // host-side constants exactly as the reference's rope op computes them
        p.rope.theta_scale = powf(rope->freq_base, -2.0f / rope->n_dims);
        const float start = floorf(yarn_corr_dim(rope->n_dims, rope->n_ctx_orig, rope->beta_fast, rope->freq_base));
        const float end = ceilf(yarn_corr_dim(rope->n_dims, rope->n_ctx_orig, rope->beta_slow, rope->freq_base));
        p.rope.corr0 = fmaxf(0.0f, start);
        p.rope.corr1 = fminf((float) (rope->n_dims - 1), end);
        p.rope.freq_scale = rope->freq_scale;
        p.rope.ext_factor = rope->ext_factor;
        p.rope.mscale = rope->attn_factor;
        if (rope->ext_factor != 0.0f) p.rope.mscale *= 1.0f + 0.1f * logf(1.0f / rope->freq_scale);
    }
    p.x = (const char *) x->data; p.x_nb1 = (int64_t) x->nb[1]; p.x_nb2 = (int64_t) x->nb[2];
    p.w = w ? (const float *) w->data : nullptr;
    p.pos = (const int32_t *) pos->data;
    p.H = (int32_t) H; p.T = (int32_t) T;
    p.eps = eps;
    const bool cache = rows != nullptr;
    if (cache) {
        if (y->type != AL_TYPE_F16 || y->ne[0] != 128 * H || y->nb[0] != 2 || (int64_t) y->nb[1] < 256 * H)
            return al_fail(AL_ERR_INVALID, "rms_norm_rope: cache must be f16 [128*H, n_rows] with contiguous rows");
        if ((rows->type != AL_TYPE_I64 && rows->type != AL_TYPE_I32) || rows->ne[0] != T || !rows->data)
            return al_fail(AL_ERR_INVALID, "rms_norm_rope: rows must be i64 / i32 [T]");
        p.rows = (const char *) rows->data;
        p.rows_nb0 = (int64_t) rows->nb[0];
        p.rows64 = rows->type == AL_TYPE_I64;
        p.n_rows_dst = y->ne[1];
        p.y_nb1 = (int64_t) y->nb[1];
        int rc = al_device_error_flag(&p.err);
        if (rc != AL_OK) return rc;
    } else {
        if (y->type != AL_TYPE_F32 || y->ne[0] != 128 || y->ne[1] != H || y->ne[2] != T || y->nb[0] != 4)
            return al_fail(AL_ERR_INVALID, "rms_norm_rope: y must be f32 [128, H, T] with nb0 = 4");
        p.y_nb1 = (int64_t) y->nb[1];
        p.y_nb2 = (int64_t) y->nb[2];
    }
    p.y = (char *) y->data;
    p.y_vec = (((uintptr_t) p.y | (uintptr_t) p.y_nb1) & 7u) == 0;
    if (!p.x || !p.y) return al_fail(AL_ERR_INVALID, "rms_norm_rope: null data");
    *out = p;
    *mode_out = mode;
    return AL_OK;
}

}  // namespace

// The checks of al_attn_inputs_f32, then what the decode kernel needs to fold
// the inputs into its prologue (one token, operands it can move by 16-byte
// DMA); fills *out and the rotation mode.
int attn_inputs_decode(const al_attn_inputs_args * a, DecodeInputs * out, int * mode_out) {
    if (!a) return al_fail(AL_ERR_INVALID, "attn_inputs: null arguments");
    NormRopeParams q, k;
    int mq = 0, mk = 0;
    int rc = norm_rope_params(&a->q, a->q_w.data ? &a->q_w : nullptr, &a->pos, a->eps, a->rope, &a->q_out, nullptr, &q, &mq);
    if (rc != AL_OK) return rc;
    rc = norm_rope_params(&a->k, a->k_w.data ? &a->k_w : nullptr, &a->pos, a->eps, a->rope, &a->k_cache, &a->rows, &k, &mk);
    if (rc != AL_OK) return rc;
    if (q.T != k.T) return al_fail(AL_ERR_INVALID, "attn_inputs: q has %d tokens, k %d", q.T, k.T);
    if (a->v.ne[1] != q.T || a->v.ne[2] != 1 || a->v.ne[3] != 1)
        return al_fail(AL_ERR_INVALID, "attn_inputs: v must be f32 [n, T] with the tokens of q");
    SetRowsParams v;
    bool empty = false;
    rc = set_rows_params(&a->v_cache, &a->v, &a->rows, &v, &empty);
    if (rc != AL_OK) return rc;
    if (empty) return al_fail(AL_ERR_INVALID, "attn_inputs: empty v");
    auto al16 = [](const void * ptr) { return ((uintptr_t) ptr & 15u) == 0; };
    const int64_t esz = k.rows64 ? 8 : 4;
    if (q.T != 1 || v.nc != 128 * k.H || v.n_dst != k.n_rows_dst || k.rows_nb0 != esz ||
        !al16(k.x) || k.x_nb1 % 16 || k.x_nb2 % 16 || !al16(v.src) || v.s_nb1 % 16 || !al16(k.rows) || !al16(k.pos) ||
        (q.w && !al16(q.w)) || (k.w && !al16(k.w)))
        return al_fail(AL_ERR_UNSUPPORTED, "attn_inputs: operands the fused decode prologue cannot take");
    DecodeInputs d;
    memset(&d, 0, sizeof(d));
    d.q_w = (const char *) q.w;
    d.k = k.x; d.k_nb1 = k.x_nb1; d.k_nb2 = k.x_nb2;
    d.k_w = (const char *) k.w;
    d.v = v.src; d.v_nb1 = v.s_nb1;
    d.pos = q.pos;
    d.rows = k.rows; d.rows_nb0 = k.rows_nb0; d.rows64 = k.rows64;
    d.T = q.T;
    d.q_out = q.y; d.qo_nb1 = q.y_nb1; d.qo_nb2 = q.y_nb2;
    d.k_cache = k.y; d.kc_nb1 = k.y_nb1;
    d.v_cache = v.dst; d.vc_nb1 = v.d_nb1;
    d.n_rows = k.n_rows_dst;
    d.eps = a->eps;
    d.rope = q.rope;
    *out = d;
    *mode_out = mq;
    return AL_OK;
}

extern "C" int al_rms_norm_rope_f32(const al_tensor * x, const al_tensor * w, const al_tensor * pos, float eps,
                                    const al_rope_params * rope, const al_tensor * y, const al_tensor * rows,
                                    void * stream) {
    NormRopeParams p;
    int mode = 0;
    const int rc = norm_rope_params(x, w, pos, eps, rope, y, rows, &p, &mode);
    if (rc != AL_OK) return rc;
    const bool cache = rows != nullptr;
    hipStream_t s = (hipStream_t) stream;
    hipError_t e;
    switch (mode) {
        case 2: e = launch_mode<2>(p, cache, s); break;
        case 1: e = launch_mode<1>(p, cache, s); break;
        default: e = launch_mode<0>(p, cache, s); break;
    }
    return e == hipSuccess ? AL_OK : al_hip_fail(e, "rms_norm_rope: launch");
}

extern "C" int al_attn_inputs_f32(const al_attn_inputs_args * a, void * stream) {
    if (!a) return al_fail(AL_ERR_INVALID, "attn_inputs: null arguments");
    NormRopeParams q, k;
    int mq = 0, mk = 0;
    int rc = norm_rope_params(&a->q, a->q_w.data ? &a->q_w : nullptr, &a->pos, a->eps, a->rope, &a->q_out, nullptr, &q, &mq);
    if (rc != AL_OK) return rc;
    rc = norm_rope_params(&a->k, a->k_w.data ? &a->k_w : nullptr, &a->pos, a->eps, a->rope, &a->k_cache, &a->rows, &k, &mk);
    if (rc != AL_OK) return rc;
    if (q.T != k.T) return al_fail(AL_ERR_INVALID, "attn_inputs: q has %d tokens, k %d", q.T, k.T);
    if (a->v.ne[1] != q.T || a->v.ne[2] != 1 || a->v.ne[3] != 1)
        return al_fail(AL_ERR_INVALID, "attn_inputs: v must be f32 [n, T] with the tokens of q");
    SetRowsParams v;
    bool empty = false;
    rc = set_rows_params(&a->v_cache, &a->v, &a->rows, &v, &empty);
    if (rc != AL_OK) return rc;
    if (empty) return al_fail(AL_ERR_INVALID, "attn_inputs: empty v");
    // V: 256 values of a row to a wave (one load each lane), at most 8 waves
    const int yq = (q.H + kRows - 1) / kRows, yk = (k.H + kRows - 1) / kRows;
    const int yv = std::max(1, std::min(8, (v.nc + 255) / 256));
    const dim3 grid((unsigned) ((q.T + kWaves - 1) / kWaves), (unsigned) (yq + yk + yv));
    hipStream_t s = (hipStream_t) stream;
    switch (mq) {
        case 2: hipLaunchKernelGGL(attn_inputs_kernel<2>, grid, dim3(64 * kWaves), 0, s, q, k, v, yq, yk, yv); break;
        case 1: hipLaunchKernelGGL(attn_inputs_kernel<1>, grid, dim3(64 * kWaves), 0, s, q, k, v, yq, yk, yv); break;
        default: hipLaunchKernelGGL(attn_inputs_kernel<0>, grid, dim3(64 * kWaves), 0, s, q, k, v, yq, yk, yv); break;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AL_OK : al_hip_fail(e, "attn_inputs: launch");
}
