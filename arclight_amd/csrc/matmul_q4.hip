// The attention output projection (WO) with Q4_0 weights for gfx950
// (include/arclight_matmul.h).
//
// Semantics: nnml_compute_forward_mul_mat for src0 Q4_0 / src1 f32
// (nnml/src/ops/ops.cpp:1252-1274, forward_mul_mat_generic,
// nnml/src/ops/arm/common.cpp:120-...): each activation row is quantized to
// Q8_0 (quantize_row_q8_0, arm.cpp:1819-1848: d = amax / 127, q = x / d
// rounded to nearest even), and y[t][n] = sum over blocks of
// (sumi * d_w) * d_x with sumi the integer dot product of the block's
// weights minus 8 and its Q8_0 values (nnml_vec_dot_q4_0_q8_0, arm.cpp:401).
//
// Up to 8 tokens (decode, speculative verify) take one launch,
// gemv_q4_fused_kernel: one wavefront per output row, every row resident at
// once; each workgroup issues its rows' weight loads, quantizes all T
// activation rows into LDS meanwhile (the activations are small and
// L2-resident), then lane l forms the dot products of the row's blocks
// l*BPL .. l*BPL + BPL - 1 (a contiguous 36-byte-aligned run of 18-byte
// blocks held in registers) with 8 v_dot4_i32_i8 per block on the unsigned
// nibbles, the weights' offset of 8 folded into one multiply by the block's
// value sum; lane sums meet in a DPP wave reduction.
// Longer inputs (up to 64 tokens) take two launches: quantize_q8_kernel
// (into library scratch, laid out as MFMA operands) and gemm_q4_kernel, whose
// integer dot products run on the matrix cores. The 4-bit weights, 18 bytes
// per 32, are read from memory once; with more than 16 tokens every tile of
// 16 reads them again from the caches.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>

#include "../../include/arclight_matmul.h"
#include "kernel_args.hpp"
#include "runtime.hpp"

namespace {

constexpr int kMaxT = 64;

// Cross-lane moves on the VALU (DPP): within rows of 16 lanes, then the
// broadcasts of a row's last lane into the next row(s).
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xf, false));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kRowHalfMirror = 0x141, kRowMirror = 0x140, kRowBcast15 = 0x142,
              kRowBcast31 = 0x143, kRowRor8 = 0x128;

// Sum over the wavefront; the total is valid in lane 63 only.
__device__ __forceinline__ float wave_sum_to_last(float v) {
    v += dpp<kQuadXor1>(v);
    v += dpp<kQuadXor2>(v);
    v += dpp<kRowHalfMirror>(v);                                       // lane i <-> 7 - i of its 8
    v += dpp<kRowMirror>(v);                                           // lane i <-> 15 - i of its 16
    v += dpp<kRowBcast15, 0xa>(v);                                     // rows 1, 3 += last lane of rows 0, 2
    v += dpp<kRowBcast31, 0xc>(v);                                     // rows 2, 3 += lane 31
    return v;
}

// Q4_0 block j (0 .. BPL-1) of a lane's chunk of 18-byte blocks held as
// 9 * BPL / 2 dwords: its scale and its 16 bytes of nibbles as 4 dwords.
template <int BPL>
__device__ __forceinline__ void block_of(const uint32_t (&c)[9 * BPL / 2], const int j, float & d, uint32_t (&q)[4]) {
    const int byte = 18 * j;                                           // even
    const int w0 = byte >> 2;
    if ((byte & 3) == 0) {
        d = (float) __builtin_bit_cast(_Float16, (uint16_t) (c[w0] & 0xffff));
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = __builtin_amdgcn_alignbyte(c[w0 + i + 1], c[w0 + i], 2);
    } else {
        d = (float) __builtin_bit_cast(_Float16, (uint16_t) (c[w0] >> 16));
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = c[w0 + 1 + i];
    }
}

// The four 16-lane groups' values of x (group d's in out[d], in all lanes).
__device__ __forceinline__ void gather_groups(const float x, float (&out)[4]) {
    const int xi = __builtin_bit_cast(int, x);
    const auto h = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
    const auto a = __builtin_amdgcn_permlane16_swap((int) h[0], (int) h[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap((int) h[1], (int) h[1], false, false);
    out[0] = __builtin_bit_cast(float, (int) a[0]);
    out[1] = __builtin_bit_cast(float, (int) a[1]);
    out[2] = __builtin_bit_cast(float, (int) b[0]);
    out[3] = __builtin_bit_cast(float, (int) b[1]);
}
// q[d] of 16-lane group g <-> q[g] of group d (a 4 x 4 transpose).
__device__ __forceinline__ void transpose_groups(uint32_t (&q)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap((int) q[0], (int) q[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap((int) q[1], (int) q[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap((int) a[0], (int) b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap((int) a[1], (int) b[1], false, false);
    q[0] = (uint32_t) c[0]; q[1] = (uint32_t) c[1];
    q[2] = (uint32_t) d[0]; q[3] = (uint32_t) d[1];
}

constexpr int min_c(int a, int b) { return a < b ? a : b; }
constexpr int kTile = 16;                        // tokens of an MFMA tile
constexpr int kGemmWaves = 8;                    // waves of a workgroup, each with 1/8 of K

// Activations as gemm_q4_kernel's MFMA operands: one wavefront per (16-token
// tile, pair of Q8_0 blocks), lane 16 g + t holding token t's values
// 4g..4g+3 and 16+4g..16+4g+3 of both blocks (the nibble order of a Q4_0
// dword), 16 bytes per lane, so operand loads and stores are whole 1 KiB
// lines; the block scales (f16, as the format stores them) as
// [tile][block][token]. Tokens past T are zeros.
// Latency-bound (one load round; reads are whole 128-byte lines per token).
__global__ __launch_bounds__(256) void quantize_q8_kernel(const char * __restrict__ x, int64_t x_nb1, int nb, int T,
                                                          int n_items, uint4 * __restrict__ frag, _Float16 * __restrict__ dx) {
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= n_items) return;
    const int tile = item / (nb / 2), pair = item - tile * (nb / 2);
    const int g = lane >> 4, tok = tile * kTile + (lane & 15);
    float4 f[2][2] = {};
    if (tok < T) {
        const float * xr = (const float *) (x + (int64_t) tok * x_nb1) + 64 * pair + 4 * g;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            f[k][0] = *(const float4 *) (xr + 32 * k);
            f[k][1] = *(const float4 *) (xr + 32 * k + 16);
        }
    }
    uint32_t words[4];
    float d[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float v[8] = {f[k][0].x, f[k][0].y, f[k][0].z, f[k][0].w, f[k][1].x, f[k][1].y, f[k][1].z, f[k][1].w};
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
        float gm[4];
        gather_groups(amax, gm);
        amax = fmaxf(fmaxf(gm[0], gm[1]), fmaxf(gm[2], gm[3]));
        d[k] = amax / 127.0f;
        const float id = d[k] != 0.0f ? 1.0f / d[k] : 0.0f;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            words[2 * k + w] = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)                                    // ties to even, as vcvtnq
                words[2 * k + w] |= (uint32_t) ((int) rintf(v[4 * w + e] * id) & 0xff) << (8 * e);
        }
    }
    frag[(int64_t) item * 64 + lane] = uint4{words[0], words[1], words[2], words[3]};
    if (g < 2) dx[((int64_t) tile * nb + 2 * pair + g) * kTile + (lane & 15)] = (_Float16) (g ? d[1] : d[0]);
}

// 9 to 64 tokens: a workgroup takes 16 weight rows and a tile of 16 tokens,
// each of its 8 waves 1/8 of K. One MFMA 16x16x32 i8 is one block's integer
// dot products of 16 tokens and 16 rows, exact, as the format needs them;
// its 4 results per lane then cost a conversion, a product and an FMA each.
// Nothing is saturated: at K 8192, N 5120 and 48 tokens the 896 vector
// instructions of a wave take 11.2 of the launch's 19.4 us, the MFMAs 1.6, the
// LDS 4.6, the 28 MB from memory 6; the rest is waiting, in two rounds of
// workgroups (960 for 512 places, two a CU by their 106 registers) that each
// start with their loads exposed. A workgroup takes one token tile: more
// would unpack the weights once for several tiles, but leave CUs idle (21.4
// us with one tile, 27.9 with three; 64 tokens: 25.7 with one, 27.5 with two,
// 33.0 with four).
// In a step the workgroup takes 64 blocks of every row, a wave 8: lanes 4 r
// .. 4 r + 3 load row r's 144 bytes of them (a pair of blocks each), so that
// a load touches few lines, and a permute brings row r's pair g to lane 16 g
// + r (loaded there directly, 16 rows to a load's every quarter: 23.8
// instead of 21.1 us). A block's MFMA operand wants dword g of it in group
// g, which a transpose across the four groups gives for the four groups'
// blocks together (4 permlane swaps). Nibbles become signed bytes of 16
// times the weight (xor 8, shifted high), the 1/16 goes into the block scale
// (both exact), so no sum of activations is needed. The activations come
// straight from L2, 1 KiB per wave load, their scales through LDS (as vector
// loads they took twice the operands' issue: 26.4 -> 24.0 us). The product of
// two f16 scales is exact in f32, so a block adds one rounding; each block of
// a step (at K = 4096 each pair) has a sum of its own and the waves' sums
// meet in LDS in a tree, which keeps the error against the exact result at
// that of one wave per row (2-norm 7.80e-8 at K = 8192, 7.37e-8 at 4096).
// Measured, us per call with the quantization launch (before: one wave per
// row, the tokens in series): K 8192, N 5120: 48 tokens 232 -> 21.9, 16
// tokens 15.5; K 4096, N 2560: 37 tokens 39 -> 9.2, 16 tokens 22 -> 7.4; K
// 4096, N 4096: 12 tokens 22 -> 7.5.
template <int BL>
__global__ __launch_bounds__(kGemmWaves * 64, 4) void gemm_q4_kernel(const char * w, int64_t w_nb1, int N, const uint4 * frag,
                                                                  const uint4 * dx, int T, char * y, int64_t y_nb1) {
    constexpr int NB = 32 * BL;                                        // blocks of a row
    constexpr int kSteps = NB / (8 * kGemmWaves);
    constexpr int kDx = NB * kTile * 2, kRed = kGemmWaves * 4 * 256;
    __shared__ __align__(16) char lds[kDx > kRed ? kDx : kRed];        // the scales, then the waves' sums
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, tile = blockIdx.y;
    // the wave's blocks: 8 of every 64, group g's pair of those of step s
    auto block = [&](const int s, const int d) { return (s * kGemmWaves + wave) * 8 + 2 * d; };
    frag += (int64_t) tile * (NB / 2) * 64;
    dx += (int64_t) tile * NB * 2;

    // the wave's scales (it alone reads them: no barrier), 16-byte pieces
    for (int i = lane; i < 16 * kSteps; i += 64) {
        const int o = block(i >> 4, 0) * 2 + (i & 15);
        ((uint4 *) lds)[o] = dx[o];
    }
    // A step's weights and operands go out together, kDepth steps ahead (a
    // wave's loads return in order).
    constexpr int kDepth = min_c(kSteps, 2);
    uint32_t c[kDepth][9];
    uint4 a[kDepth][4];
    const char * wr = w + (int64_t) min(n0 + (lane >> 2), N - 1) * w_nb1;
    auto issue = [&](const int s) {
        const uint32_t * ws = (const uint32_t *) (wr + block(s, lane & 3) * 18);
#pragma unroll
        for (int i = 0; i < 9; ++i) c[s % kDepth][i] = ws[i];
#pragma unroll
        for (int d = 0; d < 4; ++d) a[s % kDepth][d] = frag[block(s, d) / 2 * 64 + lane];
        asm volatile("" ::: "memory");                                 // keeps the issue order
    };
#pragma unroll
    for (int s = 0; s < kDepth; ++s) issue(s);

    typedef int int4v __attribute__((ext_vector_type(4)));
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    constexpr int kSums = kSteps > 2 ? 8 : 4;                          // sums a lane keeps per output: per block of a step, or pair
    float acc[kSums / 4][4][4] = {};
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
        uint32_t cs[9], q[2][4];
        float dw[2][4];
#pragma unroll
        for (int i = 0; i < 9; ++i) cs[i] = (uint32_t) __builtin_amdgcn_ds_bpermute(16 * r + 4 * g, (int) c[st % kDepth][i]);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float d;
            block_of<2>(cs, k, d, q[k]);
            gather_groups(d * 0.0625f, dw[k]);
            transpose_groups(q[k]);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {                                  // the blocks of group d: b, b + 1
            const int b = block(st, d);
            const uint4 f = a[st % kDepth][d];
            const long av[2] = {(long) ((uint64_t) f.x | (uint64_t) f.y << 32), (long) ((uint64_t) f.z | (uint64_t) f.w << 32)};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t x = q[k][d] ^ 0x88888888u;
                const long wv = (long) ((uint64_t) ((x << 4) & 0xf0f0f0f0u) | (uint64_t) (x & 0xf0f0f0f0u) << 32);
                const half4 s = *(const half4 *) (lds + ((b + k) * kTile + 4 * g) * 2);
                const int4v sumi = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[k], wv, int4v{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[k % (kSums / 4)][d][i] = __builtin_fmaf((float) sumi[i], dw[k][d] * (float) s[i], acc[k % (kSums / 4)][d][i]);
            }
        }
        if (st + kDepth < kSteps) issue(st + kDepth);
    }
    __syncthreads();                                                   // every wave is past its scales
    float (*red)[4][64] = (float (*)[4][64]) lds;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) v[d] = kSums == 8 ? acc[0][d][i] + acc[kSums / 4 - 1][d][i] : acc[0][d][i];
        red[wave][i][lane] = (v[0] + v[1]) + (v[2] + v[3]);
    }
    __syncthreads();
    // wave i < 4: token 4 (lane / 16) + i of the tile, row lane % 16
    if (wave < 4) {
        float v[kGemmWaves];
#pragma unroll
        for (int u = 0; u < kGemmWaves; ++u) v[u] = red[u][wave][lane];
#pragma unroll
        for (int h = kGemmWaves / 2; h >= 1; h /= 2)
#pragma unroll
            for (int u = 0; u < h; ++u) v[u] += v[u + h];
        const int tok = tile * kTile + 4 * g + wave;
        if (tok < T && n0 + r < N) *(float *) (y + (int64_t) tok * y_nb1 + (int64_t) (n0 + r) * 4) = v[0];
    }
}

// 1 / d as the IEEE division rounds it, for a Q8_0 block scale d >= 0 (0
// for d = 0, as quantize_row_q8_0 takes it): for d in [2^-126, 2^126) the
// v_rcp_f32 estimate and one Newton step give that quotient
// (al_mul_mat_q4_0_check_inverse counts the floats where they do not);
// zero, denormal d and the top two binades take the division.
__device__ __forceinline__ float q8_inverse(const float d) {
    if (d >= 0x1p-126f && d < 0x1p126f) {
        const float r = __builtin_amdgcn_rcpf(d);
        return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
    }
    return d != 0.0f ? 1.0f / d : 0.0f;
}

// Every non-negative float bit pattern up to +inf (grid-stride): counts the
// ones where q8_inverse differs from the division, bit for bit.
__global__ __launch_bounds__(256) void q8_inverse_check_kernel(unsigned long long * bad) {
    unsigned long long n = 0;
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u <= 0x7f800000u; u += stride) {
        const float d = __uint_as_float(u);
        const float ref = d != 0.0f ? 1.0f / d : 0.0f;
        n += __float_as_uint(q8_inverse(d)) != __float_as_uint(ref);
        if (u > 0x7f800000u - stride) break;
    }
    if (n) atomicAdd(bad, n);
}

// Eight values of a Q8_0 block (part 0..3 of it, the four parts in the four
// lanes of a quad) quantized into LDS.
__device__ __forceinline__ void quantize_part(const float4 f0, const float4 f1, const int part, int8_t * qdst,
                                              float2 * sdst) {
    const float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    amax = fmaxf(amax, dpp<kQuadXor1>(amax));
    amax = fmaxf(amax, dpp<kQuadXor2>(amax));
    // d = amax / 127 as the IEEE division rounds it: amax r with r = RN(1/127)
    // and one FMA correction, which gives the correctly rounded quotient for
    // every finite non-negative float (all 2^31 checked against the division);
    // an infinite amax passes through as the division would give it
    constexpr float kR127 = 1.0f / 127.0f;
    const float q0 = amax * kR127;
    const float dq = __builtin_fmaf(__builtin_fmaf(-q0, 127.0f, amax), kR127, q0);
    const float d = amax <= 3.40282347e+38f ? dq : amax;
    const float id = q8_inverse(d);
    uint32_t words[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        uint32_t y[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // rint(v * id), ties to even as vcvtnq: the product (|p| <= 127)
            // plus 1.5 * 2^23 rounds to the integer k + 1.5 * 2^23, whose
            // float holds k in its low bits (two's complement in the low byte);
            // the product is kept out of a fused multiply-add
            float pr = v[4 * j + k] * id;
            asm volatile("" : "+v"(pr));
            y[k] = __float_as_uint(pr + 12582912.0f);
        }
        // the four low bytes into one word (v_perm: bytes of y0, y1 | of y2, y3)
        words[j] = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0400u) | __builtin_amdgcn_perm(y[3], y[2], 0x04000c0cu);
    }
    // the eight values' sum: the signed bytes dotted with ones
    const int sum = __builtin_amdgcn_sdot4((int) words[1], 0x01010101, __builtin_amdgcn_sdot4((int) words[0], 0x01010101, 0, false), false);
    float fs = (float) sum;                                             // |sum| <= 1016: exact in f32
    fs += dpp<kQuadXor1>(fs);
    fs += dpp<kQuadXor2>(fs);
    *(uint2 *) qdst = uint2{words[0], words[1]};
    if (part == 0) *sdst = float2{(float) (_Float16) d, fs};           // the block scale as stored (f16), the sum
}

// Eight per-lane values (tokens 0..7) summed over the wavefront, scattered:
// token t's total ends in lanes 8t .. 8t + 7. Lanes exchange half of their
// values with lane ^ 32, then ^ 16 (permlane swaps), then ^ 8 (DPP row
// rotate), each time keeping the tokens of their side, then sum within
// their 8 lanes: 18 instructions instead of a wave sum per token.
__device__ __forceinline__ float wave_sum8_scatter(const float (&v)[8], const int lane) {
    float a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {       // lanes 0..31 keep tokens k, lanes 32..63 tokens 4 + k
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v[k]), __builtin_bit_cast(int, v[4 + k]),
                                                        false, false);
        a[k] = __builtin_bit_cast(float, (int) r[0]) + __builtin_bit_cast(float, (int) r[1]);
    }
    float b[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {       // lane bit 4 clear keeps a[k], set keeps a[k + 2]
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, a[k]), __builtin_bit_cast(int, a[k + 2]),
                                                        false, false);
        b[k] = __builtin_bit_cast(float, (int) r[0]) + __builtin_bit_cast(float, (int) r[1]);
    }
    const bool odd = (lane & 8) != 0;   // lane bit 3 set keeps b[1]
    const float keep = odd ? b[1] : b[0], send = odd ? b[0] : b[1];
    float c = keep + dpp<kRowRor8>(send);
    c += dpp<kQuadXor1>(c);
    c += dpp<kQuadXor2>(c);
    c += dpp<kRowHalfMirror>(c);
    return c;
}

// One launch for decode and verify (T <= TMAX): every workgroup issues its
// rows' weight loads, quantizes all T activation rows into LDS meanwhile
// (they are small and L2-resident after the first workgroup touches them;
// each thread issues the loads of all T tokens of its part of a block before
// using any), then runs the dot products from LDS. One wavefront per row; with several tokens the rows' per-lane sums of all of
// them meet in one scattering wave reduction.
template <int BPL, int TMAX>
__global__ __launch_bounds__(1024) void gemv_q4_fused_kernel(const char * w, int64_t w_nb1, int N, int K,
                                                             const char * x, int64_t x_nb1, int T,
                                                             char * __restrict__ y, int64_t y_nb1) {
    extern __shared__ __align__(16) char lds[];
    prefetch_params(w_nb1, y_nb1, blockDim.x);
    const int nb = K / 32;
    int8_t * qs = (int8_t *) lds;                                       // [T][K]
    float2 * sc = (float2 *) (lds + T * K);                             // [T][nb]: (block scale, value sum)
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int b0 = lane * BPL;
    // LDS holds block b at slot (b % BPL) * 64 + b / BPL, so that the dot
    // products' reads (lane l, its j-th block) are lane-consecutive
    auto block_at = [](const int slot) { return (slot & 63) * BPL + (slot >> 6); };
    auto load_weights = [&](uint32_t (&c)[9 * BPL / 2]) {
        const int r = row < N ? row : N - 1;
        const uint32_t * wr = (const uint32_t *) (w + (int64_t) r * w_nb1 + (int64_t) b0 * 18);
#pragma unroll
        for (int i = 0; i < 9 * BPL / 2; ++i) c[i] = wr[i];           // (non-temporal loads measured slower)
    };
    uint32_t c[9 * BPL / 2];

    // (block, part) items of the activations, a uniform number of rounds per
    // thread; loads are unconditional (indices clamped in bounds) so that no
    // branch makes the compiler wait for outstanding loads early
    const int items = 4 * nb;
    const int rounds = (items + blockDim.x - 1) / blockDim.x;
    constexpr int PRE = TMAX == 1 ? 2 : 1;                             // rounds whose loads go out first
    float4 f[PRE][TMAX][2];
    auto load_item = [&](const int item, float4 (&g)[TMAX][2]) {
        const int it = item < items ? item : items - 1;
        const int b = block_at(it >> 2), part = it & 3;
#pragma unroll
        for (int t = 0; t < TMAX; ++t) {                                // rows past T re-read row T-1
            const int tr = t < T ? t : T - 1;
            const float4 * xb = (const float4 *) ((const float *) (x + (int64_t) tr * x_nb1) + 32 * b + 8 * part);
            g[t][0] = xb[0];
            g[t][1] = xb[1];
        }
    };
    auto quantize_item = [&](const int item, const float4 (&g)[TMAX][2]) {
        if (item < items) {
            const int sl = item >> 2, part = item & 3;
#pragma unroll
            for (int t = 0; t < TMAX; ++t)
                if (t < T) quantize_part(g[t][0], g[t][1], part, qs + t * K + 32 * sl + 8 * part, sc + t * nb + sl);
        }
    };
    // the first rounds' activations (L2) before the weights (HBM): the
    // quantization then waits only for the former
#pragma unroll
    for (int k = 0; k < PRE; ++k) load_item(threadIdx.x + k * blockDim.x, f[k]);
    asm volatile("" ::: "memory");                                     // keeps the issue order
    load_weights(c);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < PRE; ++k)
        if (k < rounds) quantize_item(threadIdx.x + k * blockDim.x, f[k]);
    for (int k = PRE; k < rounds; ++k) {
        load_item(threadIdx.x + k * blockDim.x, f[0]);
        quantize_item(threadIdx.x + k * blockDim.x, f[0]);
    }
    __syncthreads();
    if (row >= N) return;

    float dw[BPL];
    uint32_t lo[BPL][4], hi[BPL][4];
#pragma unroll
    for (int j = 0; j < BPL; ++j) {
        uint32_t q[4];
        block_of<BPL>(c, j, dw[j], q);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[j][i] = q[i] & 0x0f0f0f0fu;
            hi[j][i] = (q[i] >> 4) & 0x0f0f0f0fu;
        }
    }
    // the row's dot product with token t's activations (this lane's blocks)
    auto dot_t = [&](const int t) {
        float part = 0.0f;
#pragma unroll
        for (int j = 0; j < BPL; ++j) {
            const int sl = j * 64 + lane;                                // block b0 + j
            const uint4 * ab = (const uint4 *) (qs + t * K + 32 * sl);
            const uint4 a0 = ab[0], a1 = ab[1];
            const float2 s2 = sc[t * nb + sl];
            const uint32_t a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            int dot = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dot = __builtin_amdgcn_sdot4((int) lo[j][i], (int) a[i], dot, false);
                dot = __builtin_amdgcn_sdot4((int) hi[j][i], (int) a[4 + i], dot, false);
            }
            const int sumi = dot - 8 * (int) s2.y;
            part += ((float) sumi * dw[j]) * s2.x;
        }
        return part;
    };
    if constexpr (TMAX > 1) {
        float part[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) part[t] = t < TMAX && t < T ? dot_t(t) : 0.0f;
        const float tot = wave_sum8_scatter(part, lane);
        const int t = lane >> 3;
        if ((lane & 7) == 0 && t < T) *(float *) (y + (int64_t) t * y_nb1 + (int64_t) row * 4) = tot;
    } else {
        for (int t = 0; t < T; ++t) {
            const float part = wave_sum_to_last(dot_t(t));
            if (lane == 63) *(float *) (y + (int64_t) t * y_nb1 + (int64_t) row * 4) = part;
        }
    }
}

// Most tokens of the one-launch kernel. Against the two launches for more
// tokens (us per call): K 4096, N 4096: 7.0 / 8.2 at 5 tokens, 8.3 / 8.2 at 8;
// K 8192, N 5120: 13.2 / 15.8 at 4, 17.9 / 15.6 at 5, 21.7 / 15.7 at 8. At K
// 8192 the line for time alone would be 4; calls of 5 to 8 tokens, as verify
// steps make them, stay here because this kernel needs no scratch, so that
// they can be captured into a graph whatever ran before.
constexpr int kFusedMaxT = 8;

size_t fused_lds_bytes(int64_t K, int64_t T) { return (size_t) (T * K + 8 * T * (K / 32)); }   // <= 160 KiB

template <int BPL, int TMAX>
int launch_fused(const al_tensor * w, const al_tensor * x, const al_tensor * y, int N, int K, int T, hipStream_t st) {
    int n_cu = 0;
    int rc = al_device_cu_count(&n_cu);
    if (rc != AL_OK) return rc;
    // one wavefront per row, all rows resident at once: the fewest workgroups
    // per CU that keep a workgroup at 16 waves or fewer
    const int per_cu = (N + 16 * n_cu - 1) / (16 * n_cu);
    const int waves = std::max(1, (N + per_cu * n_cu - 1) / (per_cu * n_cu));
    const size_t lds = fused_lds_bytes(K, T);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *) gemv_q4_fused_kernel<BPL, TMAX>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        if (e != hipSuccess) return al_hip_fail(e, "mul_mat_q4_0: LDS attribute");
    }
    hipLaunchKernelGGL((gemv_q4_fused_kernel<BPL, TMAX>), dim3((unsigned) ((N + waves - 1) / waves)), dim3(64 * waves), lds, st,
                       (const char *) w->data, (int64_t) w->nb[1], N, K, (const char *) x->data, (int64_t) x->nb[1], T,
                       (char *) y->data, (int64_t) y->nb[1]);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? AL_OK : al_hip_fail(e, "mul_mat_q4_0: fused launch");
}

template <int BPL>
int launch_fused_t(const al_tensor * w, const al_tensor * x, const al_tensor * y, int N, int K, int T, hipStream_t st) {
    // Every wave loads and quantizes its share of TMAX rows, those past T for
    // nothing: at 2 to 4 tokens the kernel for 8 took, us per call, K 4096, N
    // 4096: 5.9 (4 tokens) and 5.2 (2) against 5.3 and 4.3; K 8192, N 5120: 15.9
    // (4) and 14.5 (3) against 12.7 and 11.5. Same bits.
    if (T == 1) return launch_fused<BPL, 1>(w, x, y, N, K, T, st);
    return T <= 4 ? launch_fused<BPL, 4>(w, x, y, N, K, T, st) : launch_fused<BPL, kFusedMaxT>(w, x, y, N, K, T, st);
}

template <int BL>
int launch_gemm(const al_tensor * w, const al_tensor * y, int N, int tiles, int T, const uint4 * frag, const uint4 * dx,
                hipStream_t st) {
    const dim3 grid((unsigned) ((N + 15) / 16), (unsigned) tiles);
    hipLaunchKernelGGL(gemm_q4_kernel<BL>, grid, dim3(kGemmWaves * 64), 0, st, (const char *) w->data, (int64_t) w->nb[1], N,
                       frag, dx, T, (char *) y->data, (int64_t) y->nb[1]);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AL_OK : al_hip_fail(e, "mul_mat_q4_0: launch");
}

// Per-device scratch for the quantized activations; the first allocation
// has room for every call (64 tokens of K = 16384: 1.1 MB), so that none
// grows it, which would fail inside a capture.
struct Scratch {
    void * p = nullptr;
    size_t bytes = 0;
};
std::mutex g_mu;
Scratch g_scratch[64];

int scratch(size_t bytes, void ** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return al_hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= 64) return al_fail(AL_ERR_INVALID, "mul_mat_q4_0: device %d", dev);
    std::lock_guard<std::mutex> lk(g_mu);
    Scratch & s = g_scratch[dev];
    if (s.bytes < bytes) {
        if (s.p) {
            e = hipDeviceSynchronize();
            if (e == hipSuccess) e = hipFree(s.p);
            if (e != hipSuccess) return al_hip_fail(e, "mul_mat_q4_0: scratch free");
            s.p = nullptr;
            s.bytes = 0;
        }
        const size_t sz = std::max(bytes, (size_t) 2 << 20);
        e = hipMalloc(&s.p, sz);
        if (e != hipSuccess) return al_hip_fail(e, "mul_mat_q4_0: scratch");
        s.bytes = sz;
    }
    *out = s.p;
    return AL_OK;
}

}  // namespace

extern "C" int al_mul_mat_q4_0_check_inverse(unsigned long long * mismatches) {
    if (!mismatches) return al_fail(AL_ERR_INVALID, "al_mul_mat_q4_0_check_inverse: mismatches required");
    unsigned long long * dev = nullptr;
    hipError_t e = hipMalloc(&dev, sizeof(unsigned long long));
    if (e != hipSuccess) return al_hip_fail(e, "check_inverse: hipMalloc");
    e = hipMemset(dev, 0, sizeof(unsigned long long));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(q8_inverse_check_kernel, dim3(4096), dim3(256), 0, (hipStream_t) 0, dev);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(mismatches, dev, sizeof(unsigned long long), hipMemcpyDeviceToHost);
    const hipError_t f = hipFree(dev);
    if (e != hipSuccess) return al_hip_fail(e, "check_inverse");
    if (f != hipSuccess) return al_hip_fail(f, "check_inverse: hipFree");
    return AL_OK;
}

extern "C" int al_mul_mat_q4_0_f32(const al_tensor * w, const al_tensor * x, const al_tensor * y, void * stream) {
    if (!w || !x || !y || !w->data || !x->data || !y->data) return al_fail(AL_ERR_INVALID, "mul_mat_q4_0: w, x and y required");
    if (w->type != AL_TYPE_Q4_0 || x->type != AL_TYPE_F32 || y->type != AL_TYPE_F32)
        return al_fail(AL_ERR_UNSUPPORTED, "mul_mat_q4_0: types %d x %d -> %d (Q4_0 x f32 -> f32 only)", w->type, x->type, y->type);
    const int64_t K = w->ne[0], N = w->ne[1], T = x->ne[1];
    if (x->ne[0] != K || y->ne[0] != N || y->ne[1] != T || x->ne[2] != 1 || x->ne[3] != 1 || w->ne[2] != 1 || w->ne[3] != 1)
        return al_fail(AL_ERR_INVALID, "mul_mat_q4_0: shapes w [%lld, %lld], x [%lld, %lld], y [%lld, %lld]",
                       (long long) K, (long long) N, (long long) x->ne[0], (long long) T, (long long) y->ne[0], (long long) y->ne[1]);
    if (K % 4096 != 0 || K > 16384) return al_fail(AL_ERR_UNSUPPORTED, "mul_mat_q4_0: K %lld (4096, 8192, 12288 or 16384)", (long long) K);
    if (T < 1 || T > kMaxT) return al_fail(AL_ERR_UNSUPPORTED, "mul_mat_q4_0: %lld tokens (1 .. %d)", (long long) T, kMaxT);
    if (N < 1 || N > (int64_t) 65535 * 4) return al_fail(AL_ERR_INVALID, "mul_mat_q4_0: N %lld", (long long) N);
    const int64_t nb = K / 32;
    if ((int64_t) w->nb[1] != nb * 18 || x->nb[0] != 4 || y->nb[0] != 4 || ((uintptr_t) w->data & 3) || ((uintptr_t) x->data & 15) ||
        (x->nb[1] & 15) || x->nb[1] < (uint64_t) K * 4 || y->nb[1] < (uint64_t) N * 4 || ((uintptr_t) y->data & 3))
        return al_fail(AL_ERR_INVALID, "mul_mat_q4_0: w rows must be contiguous blocks (nb1 = K/32*18, 4-byte aligned), x rows 16-byte aligned, rows not overlapping");
    hipStream_t st = (hipStream_t) stream;
    if (T <= kFusedMaxT) {
        switch (nb / 64) {
            case 2: return launch_fused_t<2>(w, x, y, (int) N, (int) K, (int) T, st);
            case 4: return launch_fused_t<4>(w, x, y, (int) N, (int) K, (int) T, st);
            case 6: return launch_fused_t<6>(w, x, y, (int) N, (int) K, (int) T, st);
            case 8: return launch_fused_t<8>(w, x, y, (int) N, (int) K, (int) T, st);
            default: return al_fail(AL_ERR_UNSUPPORTED, "mul_mat_q4_0: K %lld", (long long) K);
        }
    }
    const int tiles = (int) ((T + kTile - 1) / kTile);
    const size_t qs_bytes = (size_t) tiles * kTile * (size_t) K, f_bytes = (size_t) tiles * kTile * (size_t) nb * 2;
    void * s = nullptr;
    int rc = scratch(qs_bytes + f_bytes, &s);
    if (rc != AL_OK) return rc;
    uint4 * frag = (uint4 *) s;
    _Float16 * dx = (_Float16 *) ((char *) s + qs_bytes);
    const int items = tiles * (int) (nb / 2);
    hipLaunchKernelGGL(quantize_q8_kernel, dim3((unsigned) ((items + 3) / 4)), dim3(256), 0, st,
                       (const char *) x->data, (int64_t) x->nb[1], (int) nb, (int) T, items, frag, dx);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return al_hip_fail(e, "mul_mat_q4_0: quantize launch");
    switch (nb / 128) {
        case 1: return launch_gemm<4>(w, y, (int) N, tiles, (int) T, frag, (const uint4 *) dx, st);
        case 2: return launch_gemm<8>(w, y, (int) N, tiles, (int) T, frag, (const uint4 *) dx, st);
        case 3: return launch_gemm<12>(w, y, (int) N, tiles, (int) T, frag, (const uint4 *) dx, st);
        case 4: return launch_gemm<16>(w, y, (int) N, tiles, (int) T, frag, (const uint4 *) dx, st);
        default: return al_fail(AL_ERR_UNSUPPORTED, "mul_mat_q4_0: K %lld", (long long) K);
    }
}
