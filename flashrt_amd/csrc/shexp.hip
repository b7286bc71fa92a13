// The shared expert in the model's own GGUF type, and the slot path of a layer (per-slot expert
// outputs, then a combine) that it and the shapes outside the templated decode kernels take.
//
// The reference computes the shared expert with ggml's linear() on whatever type the model file
// ships (arch/qwen4exp/moe_ref.cu:117-123; moe_fast.cu:1056-1068; moe_stream.cu:169-173), then adds
// it, gated by sigmoid(ffn_gate_inp_shexp . x), in the combine (moe_fast.cu:498-542). Here:
//   - k_shexp_mv: rows of a dense ggml matrix (F32, F16, BF16 or Q8_0, row-major as in the GGUF
//     file) against a tile of TT tokens, one wave per row: gate and up together with the SwiGLU
//     (h = g / (1 + exp(-g)) * u), or the down product. Q8_0 weights take Q8_0 activations (x and
//     h quantized per 32 as the CPU path does, q8_0 . q8_0 per block as an exact integer dot, then
//     scaled by d_w d_a); the other types take the fp32 activations.
//     More than 8 tokens go to k_shexp_mm, the same products on the matrix cores, save for short calls of
//     little work (shexp_on_mfma).
//   - the layer with such a shared expert: windows of up to 8 tokens of a shape that the decode kernels
//     are templated for run the window kernels with the shared expert's outputs in slot K; else router
//     logits -> route_topk -> the routed experts as per-slot outputs (moe_hits for windows of up to 8
//     tokens, moe_q2::run for prefill chunks) -> the shared expert -> k_slot_combine (the routed slots
//     in ascending expert id, then the shared expert times sigmoid(gate), then the residual:
//     moe_cpu.cpp:63-80 and moe_ref.cu:90-97).
#include "common.hpp"
#include "../../include/flashrt_moe.h"

#include <type_traits>

namespace frt {

namespace {

constexpr int kShNT = 256;   // 4 waves: one row each
constexpr int kShTT = 4;     // tokens per workgroup
constexpr int kShMaxCols = 4096;

// 32 weights of row r, block b (32 columns), as floats (dense types) -> w[32]
template <int TYPE>
__device__ __forceinline__ void dense_block(const uint8_t* row, int b, float (&w)[32]) {
    if (TYPE == FRT_GGML_F32) {
        const float4* p = reinterpret_cast<const float4*>(row) + b * 8;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 v = p[i];
            w[4 * i] = v.x;
            w[4 * i + 1] = v.y;
            w[4 * i + 2] = v.z;
            w[4 * i + 3] = v.w;
        }
    } else {
        const uint4* p = reinterpret_cast<const uint4*>(row) + b * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint4 v = p[i];
            const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint16_t lo = uint16_t(d[k] & 0xffffu), hi = uint16_t(d[k] >> 16);
                if (TYPE == FRT_GGML_F16) {
                    w[8 * i + 2 * k] = h2f(lo);
                    w[8 * i + 2 * k + 1] = h2f(hi);
                } else {   // bf16: the upper half of an fp32
                    w[8 * i + 2 * k] = __uint_as_float(uint32_t(lo) << 16);
                    w[8 * i + 2 * k + 1] = __uint_as_float(uint32_t(hi) << 16);
                }
            }
        }
    }
}

// A pair of Q8_0 blocks 2p, 2p + 1 of a row (68 bytes from a 4-byte aligned offset): their codes as
// 8 + 8 dwords and their scales.
__device__ __forceinline__ void q8_pair(const uint8_t* row, int p, uint32_t (&q0)[8], uint32_t (&q1)[8], float& d0,
                                        float& d1) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(row + size_t(p) * 68);
    uint32_t v[17];
#pragma unroll
    for (int i = 0; i < 17; ++i) v[i] = w[i];
    d0 = h2f(uint16_t(v[0] & 0xffffu));
#pragma unroll
    for (int i = 0; i < 8; ++i) q0[i] = __builtin_amdgcn_alignbyte(v[i + 1], v[i], 2);   // bytes 2 .. 33
    d1 = h2f(uint16_t(v[8] >> 16));
#pragma unroll
    for (int i = 0; i < 8; ++i) q1[i] = v[9 + i];   // bytes 36 .. 67
}

// rows r of W1 (and W2, DUAL) against TT tokens t0 .. : out[t][r] = W1 a_t (DUAL: silu(W1 a_t) * W2 a_t).
// a: fp32 [T][cols] (dense types; Q8_0 down, which quantizes its h while staging it) or Q8_0 codes aq
// [T][cols] with scales ad [T][cols/32] (Q8_0 gate / up). out rows are out_ld apart.
template <int TYPE, bool DUAL>
__global__ void __launch_bounds__(kShNT) k_shexp_mv(const uint8_t* __restrict__ W1, const uint8_t* __restrict__ W2,
                                                     int rows, int cols, const float* __restrict__ af,
                                                     const int8_t* __restrict__ aq, const float* __restrict__ ad, int T,
                                                     float* __restrict__ out, size_t out_ld) {
    constexpr bool Q8 = TYPE == FRT_GGML_Q8_0;
    __shared__ __align__(16) float s_af[Q8 ? 1 : kShTT * kShMaxCols];
    __shared__ __align__(16) int8_t s_aq[Q8 ? kShTT * kShMaxCols : 16];
    __shared__ float s_ad[Q8 ? kShTT * kShMaxCols / kQ8 : 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int t0 = blockIdx.y * kShTT, tn = min(kShTT, T - t0);
    // the token tile's activations into LDS
    if (Q8 && !DUAL) {
        // h to Q8_0 (the values of k_quant_q8): eight lanes to a block of 32, four values each, four loads in
        // flight. Every workgroup does this for itself, so it has to be short: a block per half wave and a
        // load at a time took 28 us of a call at 4 tokens of 512 with a shared expert of 4096 (84 us; a
        // launch of its own before this one 56 us; this 55 us).
        const float4* src = reinterpret_cast<const float4*>(af + size_t(t0) * cols);
        const int nv = tn * cols / 4;   // (a multiple of 16: a block's lanes are all within it or all past it)
        for (int i0 = 0; i0 < nv; i0 += 4 * kShNT) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[min(i0 + u * kShNT + tid, nv - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (i0 + u * kShNT >= nv) break;   // (uniform)
                const int i = i0 + u * kShNT + tid;
                float am = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
                am = fmaxf(am, __shfl_xor(am, 1));
                am = fmaxf(am, __shfl_xor(am, 2));
                am = fmaxf(am, __shfl_xor(am, 4));
                const float d = q8_scale(am), id = q8_inv(d);
                const int q[4] = {q8_code(v[u].x, id), q8_code(v[u].y, id), q8_code(v[u].z, id), q8_code(v[u].w, id)};
                if (i < nv) {
                    reinterpret_cast<uint32_t*>(s_aq)[i] = uint32_t(uint8_t(int8_t(q[0]))) | uint32_t(uint8_t(int8_t(q[1]))) << 8 |
                                                           uint32_t(uint8_t(int8_t(q[2]))) << 16 | uint32_t(uint8_t(int8_t(q[3]))) << 24;
                    if (i % 8 == 0) s_ad[i / 8] = f16_round(d);
                }
            }
        }
    } else if (Q8) {
        const int nw = tn * cols / 4;
        for (int i = tid; i < nw; i += kShNT)
            reinterpret_cast<uint32_t*>(s_aq)[i] = reinterpret_cast<const uint32_t*>(aq + size_t(t0) * cols)[i];
        for (int i = tid; i < tn * cols / kQ8; i += kShNT) s_ad[i] = ad[size_t(t0) * (cols / kQ8) + i];
    } else {
        const int nw = tn * cols / 4;
        for (int i = tid; i < nw; i += kShNT)
            reinterpret_cast<float4*>(s_af)[i] = reinterpret_cast<const float4*>(af + size_t(t0) * cols)[i];
    }
    __syncthreads();
    const int r = blockIdx.x * 4 + wave;
    if (r >= rows) return;
    float acc1[kShTT], acc2[kShTT];
#pragma unroll
    for (int t = 0; t < kShTT; ++t) acc1[t] = acc2[t] = 0.0f;
    if (Q8) {
        const size_t rb = size_t(cols / kQ8) * 34;
        const uint8_t* row1 = W1 + size_t(r) * rb;
        const uint8_t* row2 = DUAL ? W2 + size_t(r) * rb : nullptr;
        for (int p = lane; p < cols / 64; p += 64) {
            uint32_t qa[8], qb[8];
            float da, db;
            q8_pair(row1, p, qa, qb, da, db);
            uint32_t ua[8], ub[8];
            float ea = 0.0f, eb = 0.0f;
            if (DUAL) q8_pair(row2, p, ua, ub, ea, eb);
#pragma unroll
            for (int t = 0; t < kShTT; ++t) {
                if (t >= tn) break;
                const int* xa = reinterpret_cast<const int*>(s_aq + t * cols + 64 * p);
                int s0 = 0, s1 = 0, v0 = 0, v1 = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    s0 = dot4(int(qa[i]), xa[i], s0);
                    s1 = dot4(int(qb[i]), xa[8 + i], s1);
                    if (DUAL) {
                        v0 = dot4(int(ua[i]), xa[i], v0);
                        v1 = dot4(int(ub[i]), xa[8 + i], v1);
                    }
                }
                const float x0 = s_ad[t * (cols / kQ8) + 2 * p], x1 = s_ad[t * (cols / kQ8) + 2 * p + 1];
                acc1[t] = acc1[t] + float(s0) * (da * x0);
                acc1[t] = acc1[t] + float(s1) * (db * x1);
                if (DUAL) {
                    acc2[t] = acc2[t] + float(v0) * (ea * x0);
                    acc2[t] = acc2[t] + float(v1) * (eb * x1);
                }
            }
        }
    } else {
        const size_t rb = size_t(cols) * (TYPE == FRT_GGML_F32 ? 4 : 2);
        const uint8_t* row1 = W1 + size_t(r) * rb;
        const uint8_t* row2 = DUAL ? W2 + size_t(r) * rb : nullptr;
        for (int b = lane; b < cols / 32; b += 64) {
            float w1[32], w2[32];
            dense_block<TYPE>(row1, b, w1);
            if (DUAL) dense_block<TYPE>(row2, b, w2);
#pragma unroll
            for (int t = 0; t < kShTT; ++t) {
                if (t >= tn) break;
                const float4* xp = reinterpret_cast<const float4*>(s_af + t * cols + 32 * b);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float4 xv = xp[i];
                    const float xs[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        acc1[t] = fmaf(w1[4 * i + k], xs[k], acc1[t]);
                        if (DUAL) acc2[t] = fmaf(w2[4 * i + k], xs[k], acc2[t]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < kShTT; ++t) {
        if (t >= tn) break;
        const float g = wave_sum_tree(acc1[t]);
        if (DUAL) {
            const float u = wave_sum_tree(acc2[t]);
            if (lane == 0) out[size_t(t0 + t) * out_ld + r] = g / (1.0f + expf(-g)) * u;
        } else if (lane == 0) {
            out[size_t(t0 + t) * out_ld + r] = g;
        }
    }
}

// ---- the same products for more tokens, on the matrix cores
//
// A workgroup takes 64 weight rows (DUAL: 32 gate rows and the same 32 up rows) against 16 NC tokens;
// its four waves split K in quarters and add their sums in LDS as (q0 + q1) + (q2 + q3), so that a
// chunk of a few hundred tokens still has several waves per SIMD and no wave runs a long serial K loop.
// Operands go straight from global memory (each weight row is read by one wave; the activations come
// from L2) into registers, one K-step ahead; no barrier in the K loop, and LDS only for a wave's own Q8_0 block
// scales, from the lanes that load them to those that use them. The activations are kept in
// the MFMA's own order, a 16-token tile's K-step as 64 lanes x 16 bytes, so that a load's four consecutive
// lanes read 64 bytes: the L1 takes a clock per 64-byte piece, and in rows (16 tokens x 64 bytes, another
// token in every lane) a 1 KB load takes 64 clocks instead of 16. The weights stay in the file's rows.
//   bf16 planes [3][tiles][K / 32][64 lanes][8]: lane 16 g + j holds K 8 g .. 8 g + 7 of token j.
//   Q8_0 codes [tiles][K / 64][64 lanes][16]: lane 16 g + j holds codes 8 g .. of both blocks of the pair;
//   scales [tiles][K / 64][2][16].
//   F32, F16, BF16 weights: the fp32 activations are split exactly into three bf16 planes
//     (k_split3: 8 + 8 + 8 significant bits by truncation), the weights into one (BF16), two (F16) or
//     three (F32), and every pair of parts is one v_mfma_f32_16x16x32_bf16: exact products, fp32 sums (three,
//     see Precision), as the fmaf chains of k_shexp_mv.
//   Q8_0 weights: v_mfma_i32_16x16x32_i8 per 32-block, an exact integer dot, then + float(s) * (d_w d_a),
//     the terms of k_shexp_mv.
// Precision: the products of the leading parts and the small ones have sums of their own, and the leading
// ones two (even and odd K-steps; Q8_0: a pair's two blocks), added at the end. With one sum for all, every
// small product rounds the full sum: rms error against float64 2.5e-7 (k_shexp_mv) -> 4.2e-7 (BF16), 6.2e-7
// (F32) at 2560 / 640; with these 2.0e-7, at no cost (a layer of 200 tokens 224 us, 1024 tokens 469 us both).
// What bounds it: latency at a few hundred tokens. The weights loaded four lanes to a row's 64 bytes and
// turned through the wave's LDS instead (a quarter of the L1's clocks) changed nothing: a layer of 200 tokens
// 224 us, of 1024 tokens 449-471 us both ways.
typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16v __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int intx4 __attribute__((ext_vector_type(4)));

// v = hi + mid + lo exactly, each with at most 8 significant bits (truncations: no part overflows);
// an infinity or a NaN stays in hi alone (its products with the other operand's zero parts are NaN where
// the value's own are not: k_shexp_mm forms such sums again, dot_chain)
__device__ __forceinline__ void split3(float v, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const uint32_t b = __float_as_uint(v);
    hi = b & 0xffff0000u;
    const float r = v - __uint_as_float(hi);
    mid = __float_as_uint(r) & 0xffff0000u;
    lo = __float_as_uint(r - __uint_as_float(mid));
    if ((b & 0x7f800000u) == 0x7f800000u) {
        if (b & 0x007fffffu) hi |= 0x00400000u;
        mid = lo = 0;
    }
}
// the upper halves of two floats' bits as one dword (a below b)
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// element offset of (token t, value k) in a bf16 plane of rows of cols; planes are up16(T) * cols apart
__host__ __device__ __forceinline__ size_t plane_at(int t, int k, int cols) {
    return ((size_t(t >> 4) * (cols / 32) + (k >> 5)) * 64 + ((k & 31) >> 3) * 16 + (t & 15)) * 8 + (k & 7);
}
__host__ __device__ __forceinline__ size_t up16(int t) { return size_t((t + 15) & ~15); }

// the planes of x [T][n]: eight values per thread (tokens past T in the last tile are left as they are: their
// columns of the products are never stored)
__global__ void __launch_bounds__(256) k_split3(const float* __restrict__ xr, int T, int n, uint16_t* __restrict__ planes) {
    const size_t e = (size_t(blockIdx.x) * 256 + threadIdx.x) * 8;
    if (e >= size_t(T) * n) return;
    const float* x = xr + e;
    const size_t i = plane_at(int(e / n), int(e % n), n), count = up16(T) * n;
    uint32_t w[3][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t a[3], b[3];
        split3(x[2 * q], a[0], a[1], a[2]);
        split3(x[2 * q + 1], b[0], b[1], b[2]);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p][q] = pack_hi(a[p], b[p]);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
        *reinterpret_cast<uint4*>(planes + p * count + i) = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

template <int TYPE>
struct ShDense {
    static constexpr int parts = TYPE == FRT_GGML_F32 ? 3 : TYPE == FRT_GGML_F16 ? 2 : 1;
    static constexpr int words = TYPE == FRT_GGML_F32 ? 8 : 4;   // dwords of 8 weights
    // the bf16 parts of 8 weights held as raw dwords
    static __device__ __forceinline__ void split(const uint32_t (&raw)[words], bf16x8 (&out)[parts]) {
        uint32_t w[parts][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (TYPE == FRT_GGML_BF16) {
                w[0][q] = raw[q];
            } else {
                float a, b;
                if constexpr (TYPE == FRT_GGML_F32) {
                    a = __uint_as_float(raw[2 * q]);
                    b = __uint_as_float(raw[2 * q + 1]);
                } else {
                    a = h2f(uint16_t(raw[q] & 0xffffu));
                    b = h2f(uint16_t(raw[q] >> 16));
                }
                uint32_t pa[3], pb[3];
                split3(a, pa[0], pa[1], pa[2]);   // (fp16: 11 significant bits, the third part is 0)
                split3(b, pb[0], pb[1], pb[2]);
#pragma unroll
                for (int p = 0; p < parts; ++p) w[p][q] = pack_hi(pa[p], pb[p]);
            }
        }
#pragma unroll
        for (int p = 0; p < parts; ++p) out[p] = __builtin_bit_cast(bf16x8, make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]));
    }
};

// Row `row` of weights (TYPE) against token t of the planes, as one chain of fused multiply-adds.
template <int TYPE>
__device__ __forceinline__ float dot_chain(const uint8_t* row, const uint16_t* ap, size_t plane, int t, int cols) {
    float s = 0.0f;
#pragma unroll 1
    for (int k = 0; k < cols; ++k) {
        float w;
        if constexpr (TYPE == FRT_GGML_F32) w = reinterpret_cast<const float*>(row)[k];
        else if constexpr (TYPE == FRT_GGML_F16) w = h2f(reinterpret_cast<const uint16_t*>(row)[k]);
        else w = __uint_as_float(uint32_t(reinterpret_cast<const uint16_t*>(row)[k]) << 16);
        const uint16_t* a = ap + plane_at(t, k, cols);
        float x = 0.0f;   // lo, mid, hi: exact
#pragma unroll
        for (int p = 2; p >= 0; --p) x += __uint_as_float(uint32_t(a[p * plane]) << 16);
        s = fmaf(w, x, s);
    }
    return s;
}

// out (DUAL): dense types the planes of h = silu(gate) * up, Q8_0 its codes hq and scales hd (both as the
// input's); else of [T][rows] fp32. aq / ad or ap (planes): the input.
template <int TYPE, bool DUAL, int NC>
__global__ void __launch_bounds__(256) k_shexp_mm(const uint8_t* __restrict__ W1, const uint8_t* __restrict__ W2, int rows,
                                                  int cols, const uint16_t* __restrict__ ap, const int8_t* __restrict__ aq,
                                                  const float* __restrict__ ad, int T, float* __restrict__ of,
                                                  uint16_t* __restrict__ op, int8_t* __restrict__ hq,
                                                  float* __restrict__ hd) {
    constexpr bool Q8 = TYPE == FRT_GGML_Q8_0;
    __shared__ __align__(16) floatx4 part[4][NC][4][64];
    __shared__ __align__(16) float s_dw[Q8 ? 4 : 1][4][2][16];   // per wave: the row tiles' block scales
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int t0 = blockIdx.y * 16 * NC;
    const int r0 = blockIdx.x * (DUAL ? 32 : 64);
    size_t tile[NC];   // token tiles; past the end the last again, not written
#pragma unroll
    for (int c = 0; c < NC; ++c) tile[c] = size_t(min(t0 / 16 + c, (T - 1) / 16));
    constexpr int kHi = 2, NA = Q8 ? 2 : kHi + 1;   // sums: see "Precision" above
    floatx4 acc[NA][4][NC];
#pragma unroll
    for (int k = 0; k < NA; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[k][i][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (Q8) {
        // K-steps of 64: a pair of Q8_0 blocks, 68 bytes of a row. Lane group lg takes codes 8 lg .. 8 lg + 7
        // of each block: bytes 2 + 8 lg (dwords 2 lg .. 2 lg + 2, shifted by two bytes) and 36 + 8 lg.
        const size_t rb = size_t(cols / kQ8) * 34;
        const int steps = cols / 64, s0 = steps * wave / 4, s1 = steps * (wave + 1) / 4;
        const uint8_t* row[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            row[i] = DUAL ? (i < 2 ? W1 : W2) + size_t(r0 + 16 * (i & 1) + li) * rb : W1 + size_t(r0 + 16 * i + li) * rb;
        struct Step {
            uint32_t a[4][5];
            uint4 b[NC];
            float d[NC][2];
        };
        auto load = [&](int st, Step& s) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t* p = reinterpret_cast<const uint32_t*>(row[i] + size_t(st) * 68);
#pragma unroll
                for (int q = 0; q < 3; ++q) s.a[i][q] = p[2 * lg + q];
#pragma unroll
                for (int q = 0; q < 2; ++q) s.a[i][3 + q] = p[9 + 2 * lg + q];
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const size_t at = tile[c] * steps + st;
                s.b[c] = *reinterpret_cast<const uint4*>(aq + (at * 64 + lane) * 16);
                s.d[c][0] = ad[at * 32 + li];
                s.d[c][1] = ad[at * 32 + 16 + li];
            }
        };
        auto mac = [&](const Step& s) {
            // d_w of the pair's blocks by row: the first's in dword 0 (lane group 0), the second's in the
            // upper half of dword 8 (lane group 3), through the wave's LDS to the lanes of rows 4 lg ..
            float* sw = &s_dw[wave][0][0][0];
            asm volatile("" ::: "memory");   // (a wave's LDS operations complete in order)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (lg == 0) sw[(i * 2) * 16 + li] = h2f(uint16_t(s.a[i][0] & 0xffffu));
                if (lg == 3) sw[(i * 2 + 1) * 16 + li] = h2f(uint16_t(s.a[i][2] >> 16));
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const long a0 = __builtin_bit_cast(long, make_uint2(__builtin_amdgcn_alignbyte(s.a[i][1], s.a[i][0], 2),
                                                                    __builtin_amdgcn_alignbyte(s.a[i][2], s.a[i][1], 2)));
                const long a1 = __builtin_bit_cast(long, make_uint2(s.a[i][3], s.a[i][4]));
                const float4 d0 = *reinterpret_cast<const float4*>(sw + (i * 2) * 16 + 4 * lg);
                const float4 d1 = *reinterpret_cast<const float4*>(sw + (i * 2 + 1) * 16 + 4 * lg);
                const float w0[4] = {d0.x, d0.y, d0.z, d0.w}, w1[4] = {d1.x, d1.y, d1.z, d1.w};
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const intx4 z = {0, 0, 0, 0};
                    const intx4 v0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a0, __builtin_bit_cast(long, make_uint2(s.b[c].x, s.b[c].y)), z, 0, 0, 0);
                    const intx4 v1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a1, __builtin_bit_cast(long, make_uint2(s.b[c].z, s.b[c].w)), z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc[0][i][c][r] = fmaf(float(v0[r]), w0[r] * s.d[c][0], acc[0][i][c][r]);
                        acc[1][i][c][r] = fmaf(float(v1[r]), w1[r] * s.d[c][1], acc[1][i][c][r]);
                    }
                }
            }
        };
        Step a, b;
        if (s0 < s1) load(s0, a);
        for (int st = s0; st < s1; st += 2) {
            load(min(st + 1, s1 - 1), b);
            mac(a);
            if (st + 1 < s1) {
                load(min(st + 2, s1 - 1), a);
                mac(b);
            }
        }
    } else {
        using D = ShDense<TYPE>;
        constexpr int es = TYPE == FRT_GGML_F32 ? 4 : 2;   // bytes per weight
        const int steps = cols / 32, s0 = steps * wave / 4, s1 = steps * (wave + 1) / 4;
        const uint8_t* row[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            row[i] = (DUAL ? (i < 2 ? W1 : W2) + size_t(r0 + 16 * (i & 1) + li) * cols * es
                           : W1 + size_t(r0 + 16 * i + li) * cols * es) + 8 * lg * es;
        const size_t plane = up16(T) * cols;
        const uint16_t* xp[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) xp[c] = ap + (tile[c] * (cols / 32) * 64 + lane) * 8;
        struct Step {
            uint32_t a[4][D::words];
            bf16x8 b[NC][3];
        };
        auto load = [&](int st, Step& s) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < D::words / 4; ++q) {
                    const uint4 v = reinterpret_cast<const uint4*>(row[i] + size_t(st) * 32 * es)[q];
                    s.a[i][4 * q] = v.x;
                    s.a[i][4 * q + 1] = v.y;
                    s.a[i][4 * q + 2] = v.z;
                    s.a[i][4 * q + 3] = v.w;
                }
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int p = 0; p < 3; ++p) s.b[c][p] = *reinterpret_cast<const bf16x8*>(xp[c] + p * plane + size_t(st) * 512);
        };
        auto mac = [&](const Step& s, auto hi) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bf16x8 a[D::parts];
                D::split(s.a[i], a);
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int pa = D::parts - 1; pa >= 0; --pa)   // the small products first
#pragma unroll
                        for (int pb = 2; pb >= 0; --pb) {
                            floatx4& t = acc[pa + pb ? kHi : hi][i][c];
                            t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16v, a[pa]),
                                                                        __builtin_bit_cast(bf16v, s.b[c][pb]), t, 0, 0, 0);
                        }
            }
        };
        Step a, b;
        if (s0 < s1) load(s0, a);
        for (int st = s0; st < s1; st += 2) {
            load(min(st + 1, s1 - 1), b);
            mac(a, std::integral_constant<int, 0>());
            if (st + 1 < s1) {
                load(min(st + 2, s1 - 1), a);
                mac(b, std::integral_constant<int, kHi - 1>());
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            floatx4 v = acc[0][i][c] + acc[1][i][c];
            if constexpr (NA > 2) v += acc[2][i][c];
            part[wave][c][i][lane] = v;
        }
    __syncthreads();
    if (wave >= NC) return;
    // wave c finishes token column c: lane (token li, rows 16 i + 4 lg + r)
    const int c = wave, t = t0 + 16 * c + li;
    floatx4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (part[0][c][i][lane] + part[1][c][i][lane]) + (part[2][c][i][lane] + part[3][c][i][lane]);
    if constexpr (!Q8) {   // an infinity or a NaN among the operands: never a finite sum (split3)
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) bad |= !(fabsf(v[i][r]) < INFINITY);
        if (__builtin_expect(bad && t < T, 0)) {   // (the sums go through LDS so that the loop stays small)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[0][c][i][lane] = v[i];
#pragma unroll 1
            for (int q = 0; q < 16; ++q) {
                const int i = q >> 2, row = r0 + 16 * (DUAL ? i & 1 : i) + 4 * lg + (q & 3);
                float* p = reinterpret_cast<float*>(&part[0][c][i][lane]) + (q & 3);
                if (!(fabsf(*p) < INFINITY))
                    *p = dot_chain<TYPE>((DUAL && i >= 2 ? W2 : W1) + size_t(row) * cols * (TYPE == FRT_GGML_F32 ? 4 : 2), ap,
                                         up16(T) * cols, t, cols);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = part[0][c][i][lane];
        }
    }
    if constexpr (!DUAL) {
        if (t < T)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<floatx4*>(of + size_t(t) * rows + r0 + 16 * i + 4 * lg) = v[i];
        return;
    }
    float h[2][4];
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float g = v[i][r], u = v[2 + i][r];
            h[i][r] = g / (1.0f + expf(-g)) * u;
            am = fmaxf(am, fabsf(h[i][r]));
        }
    if constexpr (Q8) {   // the 32 rows are one Q8_0 block of h: its maximum over the four lanes of a token
        am = fmaxf(am, __shfl_xor(am, 16, 64));
        am = fmaxf(am, __shfl_xor(am, 32, 64));
        const float d = q8_scale(am), id = q8_inv(d);
        if (t < T) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                uint32_t q = 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) q |= uint32_t(uint8_t(int8_t(q8_code(h[i][r], id)))) << (8 * r);
                *reinterpret_cast<uint32_t*>(hq + shexp_code_at(t, r0 + 16 * i + 4 * lg, rows)) = q;
            }
            if (lg == 0) hd[shexp_scale_at(t, r0 / 32, rows)] = f16_round(d);
        }
    } else if (t < T) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t p[4][3];
#pragma unroll
            for (int r = 0; r < 4; ++r) split3(h[i][r], p[r][0], p[r][1], p[r][2]);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uint2*>(op + q * up16(T) * rows + plane_at(t, r0 + 16 * i + 4 * lg, rows)) =
                    make_uint2(pack_hi(p[0][q], p[1][q]), pack_hi(p[2][q], p[3][q]));
        }
    }
}

// hit lists of moe_hits from routing ids: hit_ptr[t][k] = arena + ids[t][k] * stride for k < K, and,
// with a shared blob, hit_ptr[t][K] = shared; hit_n[t] = the slots per token (K or K + 1)
__global__ void k_hits_from_ids(const int32_t* __restrict__ ids, int T, int K, const uint8_t* arena, size_t stride,
                                const uint8_t* shared, const uint8_t** hit_ptr, int32_t* hit_n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int S = shared ? K + 1 : K;
    if (i < T * S) {
        const int t = i / S, k = i % S;
        hit_ptr[i] = k < K ? arena + size_t(ids[t * K + k]) * stride : shared;
    }
    if (i < T) hit_n[i] = S;
}

// out[t][i] = (resid) + (sum over the token's K slots in ascending expert id of w * Y[slot][i]
// + sh[t][i] * sigmoid(gate[t])). Y: per-slot rows, S slots per token, slot t * S + k in rank order
// (moe_hits' yh or moe_q2::run's yd); sh: the shared expert's row of token t at sh + t * sh_stride.
__global__ void __launch_bounds__(256) k_slot_combine(int T, int K, int S, int n, const int32_t* __restrict__ ids,
                                                      const float* __restrict__ wts, const float* __restrict__ Y,
                                                      const float* __restrict__ sh, size_t sh_stride,
                                                      const float* __restrict__ gate,
                                                      const float* __restrict__ resid, float* __restrict__ out) {
    __shared__ int s_ord[32];
    __shared__ float s_w[32];
    const int t = blockIdx.y;
    const int tid = threadIdx.x;
    if (tid < K) {   // the slot of rank r in ascending id (ids of one token are distinct)
        const int id = ids[t * K + tid];
        int r = 0;
        for (int k = 0; k < K; ++k) r += int(ids[t * K + k] < id);
        s_ord[r] = tid;
        s_w[r] = wts[t * K + tid];
    }
    __syncthreads();
    const float g = 1.0f / (1.0f + expf(-gate[t]));
    const int i = (blockIdx.x * 256 + tid) * 2;   // (n is even)
    if (i >= n) return;
    const float2 s = *reinterpret_cast<const float2*>(sh + size_t(t) * sh_stride + i);
    float a0 = 0.0f, a1 = 0.0f;
    for (int r0 = 0; r0 < K; r0 += 8) {   // eight slots' rows in flight
        float2 y[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            y[q] = *reinterpret_cast<const float2*>(Y + (size_t(t) * S + s_ord[min(r0 + q, K - 1)]) * n + i);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (r0 + q < K) {
                const float w = s_w[r0 + q];
                const float p0 = w * y[q].x, p1 = w * y[q].y;
                a0 = a0 + p0;
                a1 = a1 + p1;
            }
    }
    const float p0 = s.x * g, p1 = s.y * g;
    float o0 = a0 + p0, o1 = a1 + p1;
    if (resid) {
        o0 = resid[size_t(t) * n + i] + o0;
        o1 = resid[size_t(t) * n + i + 1] + o1;
    }
    out[size_t(t) * n + i] = o0;
    out[size_t(t) * n + i + 1] = o1;
}

}  // namespace

// ---------------------------------------------------------------- host side

bool shexp_type_ok(int type) {
    return type == FRT_GGML_F32 || type == FRT_GGML_F16 || type == FRT_GGML_BF16 || type == FRT_GGML_Q8_0;
}
bool shexp_shape_ok(int n, int ffs) {
    return n >= 64 && ffs >= 64 && n % 64 == 0 && ffs % 64 == 0 && n <= kShMaxCols && ffs <= kShMaxCols;
}

// W (rows x cols) against T tokens; DUAL: W1, W2 and the SwiGLU.
static int shexp_mv(int type, bool dual, const void* W1, const void* W2, int rows, int cols, const float* af,
                    const int8_t* aq, const float* ad, int T, float* out, size_t out_ld, hipStream_t stream) {
    const dim3 grid((rows + 3) / 4, (T + kShTT - 1) / kShTT);
    const uint8_t* w1 = static_cast<const uint8_t*>(W1);
    const uint8_t* w2 = static_cast<const uint8_t*>(W2);
#define FRT_SH(TY)                                                                                                  \
    if (dual) k_shexp_mv<TY, true><<<grid, kShNT, 0, stream>>>(w1, w2, rows, cols, af, aq, ad, T, out, out_ld);             \
    else k_shexp_mv<TY, false><<<grid, kShNT, 0, stream>>>(w1, w2, rows, cols, af, aq, ad, T, out, out_ld);
    switch (type) {
        case FRT_GGML_F32: FRT_SH(FRT_GGML_F32) break;
        case FRT_GGML_F16: FRT_SH(FRT_GGML_F16) break;
        case FRT_GGML_BF16: FRT_SH(FRT_GGML_BF16) break;
        case FRT_GGML_Q8_0: FRT_SH(FRT_GGML_Q8_0) break;
        default: return set_error(kErrShape, "shared expert: ggml type %d (F32, F16, BF16 or Q8_0)", type);
    }
#undef FRT_SH
    FRT_LAUNCHED("shared expert");
    return kOk;
}

// Whether a call of T tokens runs on the matrix cores (k_shexp_mm). F32 and F16 weights cost nine and six
// products each there and the activations a launch for their planes, and a few workgroups share the work, so that
// a short call of little work is faster on k_shexp_mv, whose time goes with the tokens. A whole layer, k_shexp_mv / k_shexp_mm in us, F16, shared width x
// hidden size: 4096 x 512 58 / 91 at 9 tokens, 81 / 92 at 20, 101 / 93 at 32; 4096 x 1024 70 / 108 at 9,
// 105 / 107 at 20, 117 / 106 at 24; 2048 x 1536 at 24 97 / 91; 2048 x 4096 122 / 147 at 9, 158 / 148 at 16.
// BF16 and Q8_0, three products and one, are faster on the matrix cores from 9 tokens on (0.64 to 0.85 and 0.65
// to 0.77 of the time).
static bool shexp_on_mfma(int type, int T, int n, int ffs) {
    if (T < kShMmMinT) return false;
    if (type != FRT_GGML_F32 && type != FRT_GGML_F16) return true;
    return T > 20 || int64_t(T) * n * ffs >= 72000000;
}

size_t shexp_ws_bytes(int T, int n, int ffs) {
    const size_t mv = up256(size_t(T) * ffs * 4);
    if (T < kShMmMinT) return mv;
    const size_t mm = up256(up16(T) * n * 6) + up256(up16(T) * ffs * 6);   // the bf16 planes of x and h
    return mv > mm ? mv : mm;
}

template <int TYPE, bool DUAL>
static void shexp_mm(const uint8_t* W1, const uint8_t* W2, int rows, int cols, const uint16_t* ap, const int8_t* aq,
                     const float* ad, int T, float* of, uint16_t* op, int8_t* hq, float* hd, hipStream_t stream) {
    const int gx = rows / (DUAL ? 32 : 64);
    // 32 tokens per workgroup halve the weights' L1 reads, where that leaves two workgroups per CU
    if (gx * ((T + 31) / 32) >= 512)
        k_shexp_mm<TYPE, DUAL, 2><<<dim3(gx, (T + 31) / 32), 256, 0, stream>>>(W1, W2, rows, cols, ap, aq, ad, T, of, op, hq, hd);
    else
        k_shexp_mm<TYPE, DUAL, 1><<<dim3(gx, (T + 15) / 16), 256, 0, stream>>>(W1, W2, rows, cols, ap, aq, ad, T, of, op, hq, hd);
}

template <int TYPE>
static int shexp_run_mm(const void* g, const void* u, const void* d, int n, int ffs, const float* x, const int8_t* xq,
                        const float* xd, int T, float* sh, void* ws, hipStream_t stream) {
    const uint8_t *wg = static_cast<const uint8_t*>(g), *wu = static_cast<const uint8_t*>(u), *wd = static_cast<const uint8_t*>(d);
    uint8_t* p = static_cast<uint8_t*>(ws);
    if (TYPE == FRT_GGML_Q8_0) {
        int8_t* hq = reinterpret_cast<int8_t*>(p);
        float* hd = reinterpret_cast<float*>(p + up256(up16(T) * ffs));
        shexp_mm<TYPE, true>(wg, wu, ffs, n, nullptr, xq, xd, T, nullptr, nullptr, hq, hd, stream);
        shexp_mm<TYPE, false>(wd, nullptr, n, ffs, nullptr, hq, hd, T, sh, nullptr, nullptr, nullptr, stream);
    } else {
        uint16_t* xp = reinterpret_cast<uint16_t*>(p);
        uint16_t* hp = reinterpret_cast<uint16_t*>(p + up256(up16(T) * n * 6));
        k_split3<<<unsigned((size_t(T) * n / 8 + 255) / 256), 256, 0, stream>>>(x, T, n, xp);
        shexp_mm<TYPE, true>(wg, wu, ffs, n, xp, nullptr, nullptr, T, nullptr, hp, nullptr, nullptr, stream);
        shexp_mm<TYPE, false>(wd, nullptr, n, ffs, hp, nullptr, nullptr, T, sh, nullptr, nullptr, nullptr, stream);
    }
    FRT_LAUNCHED("shared expert");
    return kOk;
}

// sh (rows of n, sh_ld apart; n from kShMmMinT tokens on) = the shared expert of type `type` on x [T][n];
// xq / xd: x's Q8_0 (Q8_0 type only; from kShMmMinT tokens on in the order of shexp_code_at and
// shexp_scale_at, for whole tiles of 16 tokens). ws: shexp_ws_bytes.
int shexp_run(int type, const void* g, const void* u, const void* d, int n, int ffs, const float* x, const int8_t* xq,
              const float* xd, int T, float* sh, size_t sh_ld, void* ws, hipStream_t stream) {
    if (!shexp_type_ok(type)) return set_error(kErrShape, "shared expert: ggml type %d (F32, F16, BF16 or Q8_0)", type);
    if (!shexp_shape_ok(n, ffs)) return set_error(kErrShape, "shared expert: n=%d ffs=%d", n, ffs);
    const bool mm = shexp_on_mfma(type, T, n, ffs);
    if (mm && sh_ld != size_t(n)) return set_error(kErrShape, "shared expert: row distance %zu", sh_ld);
    if (mm) switch (type) {
        case FRT_GGML_F32: return shexp_run_mm<FRT_GGML_F32>(g, u, d, n, ffs, x, xq, xd, T, sh, ws, stream);
        case FRT_GGML_F16: return shexp_run_mm<FRT_GGML_F16>(g, u, d, n, ffs, x, xq, xd, T, sh, ws, stream);
        case FRT_GGML_BF16: return shexp_run_mm<FRT_GGML_BF16>(g, u, d, n, ffs, x, xq, xd, T, sh, ws, stream);
        default: return shexp_run_mm<FRT_GGML_Q8_0>(g, u, d, n, ffs, x, xq, xd, T, sh, ws, stream);
    }
    // h [T][ffs] fp32; the down product quantizes it (Q8_0) or takes it as it is
    float* h = static_cast<float*>(ws);
    const bool q8 = type == FRT_GGML_Q8_0;
    if (int rc = shexp_mv(type, true, g, u, ffs, n, q8 ? nullptr : x, xq, xd, T, h, size_t(ffs), stream)) return rc;
    return shexp_mv(type, false, d, nullptr, n, ffs, h, nullptr, nullptr, T, sh, sh_ld, stream);
}

int hits_from_ids(const int32_t* ids, int T, int K, const uint8_t* arena, size_t stride, const uint8_t* shared,
                  const uint8_t** hit_ptr, int32_t* hit_n, hipStream_t stream) {
    const int cnt = T * (K + 1);
    k_hits_from_ids<<<(cnt + 255) / 256, 256, 0, stream>>>(ids, T, K, arena, stride, shared, hit_ptr, hit_n);
    FRT_LAUNCHED("hit lists");
    return kOk;
}

int slot_combine(int T, int K, int S, int n, const int32_t* ids, const float* wts, const float* Y, const float* sh,
                 size_t sh_stride, const float* gate, const float* resid, float* out, hipStream_t stream) {
    if (K < 1 || K > 32) return set_error(kErrShape, "combine: K=%d", K);
    const dim3 grid((n + 511) / 512, T);
    k_slot_combine<<<grid, 256, 0, stream>>>(T, K, S, n, ids, wts, Y, sh, sh_stride, gate, resid, out);
    FRT_LAUNCHED("combine");
    return kOk;
}

}  // namespace frt
