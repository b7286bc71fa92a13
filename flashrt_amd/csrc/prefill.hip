// Prefill MoE: routed (token, slot) pairs sorted by expert, then grouped GEMMs on fp16 MFMA
// (kernels/cuda/moe_q2.cu:514-548 is the reference's int8 counterpart).
//
// Dispatch (moe_q2.cu:83-168 semantics: a stable sort of slots s = t*K + k by ids[s]). Up to 4096 slots
// and 1024 experts k_pf_dispatch1, one workgroup; beyond:
//   k_pf_hist     per chunk of 256 slots, an LDS histogram of experts (integer atomics only)
//   k_pf_colscan  per expert, its column's prefix over the chunks
//   k_pf_scan     one workgroup: bounds, the tile list
//   k_pf_place    one wave per chunk walks its slots in order, 64 at a time; each lane's rank among
//               equal experts in the batch comes from ballots (a wave64 match-any), so the
//               placement is stable and needs no atomics.
//   The shared expert, when present, is group E holding every token in order (rows T*K + t, written
//   by the workgroups of k_pf_place past the chunks).
//
// GEMMs (k_pf_gemm, below): Q2_0 weights dequantized exactly to fp16 in registers, activations
// as exact fp16 (hi, lo) pairs (gate/up) or fp16 (down), fp32 accumulation on MFMA; tiles of up to 16
// or of up to 64 tokens of one group; the gate/up epilogue applies SwiGLU and the Q8_0 quantization of h.
//   k_pf_combine out[t] = sum_k (in expert order) w * yd[t*K+k] + yd[shared t] * sigmoid(gate)
#include "common.hpp"

#include <hip/hip_bf16.h>

#include <algorithm>
#include <type_traits>

namespace frt {

constexpr int kTN = 64;        // tokens per GEMM tile
constexpr int kChunk = 256;    // slots per dispatch chunk (one wave of k_pf_place walks one)

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

namespace {

// ---------------------------------------------------------------- dispatch

__global__ void __launch_bounds__(256) k_pf_hist(const int32_t* __restrict__ ids, int S, int E, int32_t* __restrict__ cnt) {
    extern __shared__ int32_t h[];
    for (int e = threadIdx.x; e < E; e += blockDim.x) h[e] = 0;
    __syncthreads();
    const int s0 = blockIdx.x * kChunk, s1 = min(S, s0 + kChunk);
    for (int s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
        const int e = ids[s];
        if (unsigned(e) < unsigned(E)) atomicAdd(&h[e], 1);   // ids outside [0, E) are dropped
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[size_t(blockIdx.x) * E + e] = h[e];
}

// Per expert (a wave each): cnt[b][e] becomes the exclusive prefix over the chunks b' < b (the
// chunk's first row within the expert's group), rows[e] the group's size. Lane l takes the chunks
// l P .. l P + P - 1 in order; the lanes' sums are scanned across the wave.
__global__ void __launch_bounds__(256) k_pf_colscan(int32_t* __restrict__ cnt, int nchunk, int E,
                                                    int32_t* __restrict__ rows) {
    const int e = int(blockIdx.x) * 4 + int(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (e >= E) return;   // whole waves
    const int P = (nchunk + 63) / 64, b0 = lane * P, b1 = min(nchunk, b0 + P);
    int sum = 0;
    for (int b = b0; b < b1; ++b) sum += cnt[size_t(b) * E + e];
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    int run = incl - sum;
    for (int b = b0; b < b1; ++b) {
        const int v = cnt[size_t(b) * E + e];
        cnt[size_t(b) * E + e] = run;
        run += v;
    }
    if (lane == 63) rows[e] = incl;
}

// Exclusive prefix sums over the workgroup of N ints per thread at once (and the totals): a shuffle
// scan within each wave, then wave 0 scans the wave totals in parallel. ws: (nwaves + 1) * N ints.
template <int N>
__device__ __forceinline__ void block_excl_scan_v(const int (&v)[N], int (&r)[N], int (&total)[N], int* ws) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int incl[N];
#pragma unroll
    for (int i = 0; i < N; ++i) incl[i] = v[i];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int y = __shfl_up(incl[i], o, 64);
            if (lane >= o) incl[i] += y;
        }
    if (lane == 63)
#pragma unroll
        for (int i = 0; i < N; ++i) ws[wave * N + i] = incl[i];
    __syncthreads();
    if (wave == 0) {   // the wave totals: lane w < nw holds wave w's, scanned across the lanes
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int x = lane < nw ? ws[lane * N + i] : 0;
            int c = x;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const int y = __shfl_up(c, o, 64);
                if (lane >= o) c += y;
            }
            if (lane < nw) ws[lane * N + i] = c - x;
            if (lane == nw - 1) ws[nw * N + i] = c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        r[i] = ws[wave * N + i] + incl[i] - v[i];
        total[i] = ws[nw * N + i];
    }
    __syncthreads();
}

// 1024 threads. bounds[e] holds each group's rows (k_pf_colscan) and becomes its first row.
// Tiles are listed longest first (4 token columns of 16, then 3, 2, 1; by expert within a class),
// so that the grouped GEMMs start the long tiles first and finish on short ones.
__device__ __forceinline__ int tile_class(int rows) { return (rows + 15) / 16; }   // 1..4

// The body of k_pf_scan for a 1024-thread workgroup: s_rows[e] (LDS) holds group e's rows on entry
// and its first row on exit; bounds[e] gets the same first rows (bounds[E] = T K, bounds[E + 1] =
// T K + T with the shared group), tiles and n_tiles the tile list.
__device__ void pf_scan_body(int* s_rows, int E, int T, int shared, int32_t* __restrict__ bounds,
                             int2* __restrict__ tiles, int32_t* __restrict__ n_tiles) {
    __shared__ int ws[17 * 5];
    static_assert(1024 / 64 <= 16, "the wave-total scan covers 16 waves");
    // tiles of each class of group e (rows c): c / 64 full tiles (class 4) and one of class (c % 64)
    auto count = [&](int c, int (&n)[5]) {
        n[1] = n[2] = n[3] = n[4] = 0;
        n[4] = c / kTN;
        if (c % kTN) ++n[tile_class(c % kTN)];
    };
    // pass 1: tiles per class over all groups (the shared group E included)
    int total[5] = {0, 0, 0, 0, 0};
    for (int e0 = 0; e0 < E; e0 += blockDim.x) {
        const int e = e0 + threadIdx.x;
        int n[5];
        count(e < E ? s_rows[e] : 0, n);
        const int v[4] = {n[1], n[2], n[3], n[4]};
        int r[4], tot[4];
        block_excl_scan_v<4>(v, r, tot, ws);
        for (int k = 1; k <= 4; ++k) total[k] += tot[k - 1];
    }
    int sh[5] = {0, 0, 0, 0, 0};
    if (shared) {
        count(T, sh);
        for (int k = 1; k <= 4; ++k) total[k] += sh[k];
    }
    int base[5];   // first tile of each class
    base[4] = 0;
    for (int k = 3; k >= 1; --k) base[k] = base[k + 1] + total[k + 1];
    // pass 2: bounds, chunk offsets for k_pf_place, and the tiles
    int run_rows = 0;
    for (int e0 = 0; e0 < E; e0 += blockDim.x) {
        const int e = e0 + threadIdx.x;
        const int c = e < E ? s_rows[e] : 0;   // (each thread reads and then writes only its own groups')
        int n[5], at[5];
        count(c, n);
        const int v[5] = {c, n[1], n[2], n[3], n[4]};
        int r[5], tot[5];
        block_excl_scan_v<5>(v, r, tot, ws);
        const int off = r[0] + run_rows, tot_rows = tot[0];
        for (int k = 1; k <= 4; ++k) {
            at[k] = r[k] + base[k];
            base[k] += tot[k];
        }
        if (e < E) {
            bounds[e] = off;
            s_rows[e] = off;
            for (int i = 0; i < c / kTN; ++i) tiles[at[4] + i] = make_int2(e, i * kTN);
            if (c % kTN) {
                const int k = tile_class(c % kTN);
                tiles[at[k] + (k == 4 ? n[4] - 1 : 0)] = make_int2(e, (c / kTN) * kTN);
            }
        }
        run_rows += tot_rows;
    }
    if (threadIdx.x == 0) {
        bounds[E] = run_rows;   // = T * K
        if (shared) {
            bounds[E + 1] = run_rows + T;
            for (int i = 0; i < T / kTN; ++i) tiles[base[4] + i] = make_int2(E, i * kTN);
            if (T % kTN) {
                const int k = tile_class(T % kTN);
                tiles[base[k] + (k == 4 ? sh[4] - 1 : 0)] = make_int2(E, (T / kTN) * kTN);
            }
        }
        n_tiles[0] = total[1] + total[2] + total[3] + total[4];
        n_tiles[1] = total[2] + total[3] + total[4];   // the one-column tiles come last
    }
    __syncthreads();
}

__global__ void __launch_bounds__(1024) k_pf_scan(int E, int T, int shared, int32_t* __restrict__ bounds,
                                                  int2* __restrict__ tiles, int32_t* __restrict__ n_tiles) {
    __shared__ int s_rows[4096];   // (E <= 4096)
    for (int e = threadIdx.x; e < E; e += blockDim.x) s_rows[e] = bounds[e];   // (k_pf_colscan's group sizes)
    __syncthreads();
    pf_scan_body(s_rows, E, T, shared, bounds, tiles, n_tiles);
}

// one wave per chunk; stable ranks from a ballot match-any over the expert id bits
__global__ void __launch_bounds__(64) k_pf_place(const int32_t* __restrict__ ids, int S, int K, int E, int id_bits,
                                                 const int32_t* __restrict__ cnt, const int32_t* __restrict__ bounds,
                                                 int32_t* __restrict__ tok_of, int32_t* __restrict__ slot_of, int shared_T) {
    extern __shared__ int32_t next[];
    const int lane = threadIdx.x;
    const int nchunk = (S + kChunk - 1) / kChunk;
    if (int(blockIdx.x) >= nchunk) {   // the workgroups past the chunks: the shared group's rows S + t
        const int t = (int(blockIdx.x) - nchunk) * 64 + lane;
        if (t < shared_T) {
            tok_of[S + t] = t;
            slot_of[S + t] = S + t;
        }
        return;
    }
    for (int e = lane; e < E; e += 64) next[e] = bounds[e] + cnt[size_t(blockIdx.x) * E + e];
    __syncthreads();
    const int s0 = blockIdx.x * kChunk, s1 = min(S, s0 + kChunk);
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int b = s0; b < s1; b += 64) {
        const int s = b + lane;
        const int e0 = s < s1 ? ids[s] : -1;
        const bool valid = unsigned(e0) < unsigned(E);
        const int e = valid ? e0 : 0;
        uint64_t peers = __ballot(valid);
        for (int bit = 0; bit < id_bits; ++bit) {
            const bool on = (e >> bit) & 1;
            const uint64_t m = __ballot(on);
            peers &= on ? m : ~m;
        }
        if (valid) {
            const int rank = __popcll(peers & lt);
            const int row = next[e] + rank;
            tok_of[row] = s / K;
            slot_of[row] = s;
            if (rank == 0) next[e] += __popcll(peers);   // the first lane of each expert
        }
        __syncthreads();
    }
}

// The whole dispatch of a short chunk in one workgroup: up to 256 slots per wave (kSmallSlots in all), E <=
// 1024 (a thread per expert). Wave w ranks its slots in order by ballots against its own histogram
// (hist [16][E]), the histograms are summed over the waves per expert, one scan gives the groups' first
// rows and the tiles, and each slot goes to its place: the same bounds, tiles and rows as the four
// kernels above. What bounds either is launches and latency: 21 -> 6 us for 370 slots. (Longer chunks keep
// the four kernels: one workgroup would walk them serially, 36 against 24 us at 20480 slots.)
constexpr int kSmallSlots = 4096;
// The tokens per tile of a chunk of S slots (k_pf_dispatch1's tn): with few slots there are fewer
// workgroups than the chip holds, and a 64-token tile's serial K loop (32 stages) sets the time; tiles of
// 16 tokens are more and shorter, at the price of weights dequantized once per 16 tokens. Layers of 37
// and 64 tokens (skewed) of 10 out of 512 experts: 78.5 -> 64.1 and 81.3 -> 73.1 us; 93 (even): unchanged; 140:
// 145.0 -> 146.1 skewed, 190.4 -> 181.7 with 16 hot experts; 200: 162 -> 169; 340: 194 -> 206. With few experts
// each weight is dequantized up to four times as often, but there are fewer tiles still. The expert products
// alone, tiles of 64 -> of 16, 8 experts (the same within 5% with 16): 160 slots 51.5 -> 32.7 us (2048 / 512),
// 62.7 -> 37.5 (2560 / 640); 512 slots 56.3 -> 39.6, 68.9 -> 46.3; 1024 slots 60.3 -> 53.7, 74.4 -> 64.8, but at 1024 /
// 1024 46.1 -> 47.4; 1536 slots 63.1 -> 59.9, 79.0 -> 83.4, 50.5 -> 55.2: the line for few experts lies near it too.
constexpr int kTile16Slots = 1536;
static int pf_tile_tokens(int S) { return S <= kTile16Slots ? 16 : kTN; }
__global__ void __launch_bounds__(1024) k_pf_dispatch1(const int32_t* __restrict__ ids, int S, int K, int E, int id_bits, int T,
                                                       int shared, int tn, int32_t* __restrict__ bounds, int2* __restrict__ tiles,
                                                       int32_t* __restrict__ n_tiles, int32_t* __restrict__ tok_of,
                                                       int32_t* __restrict__ slot_of) {
    extern __shared__ int32_t hist[];
    __shared__ int s_row[1024];
    __shared__ int ws[17 * 5];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int32_t* const h = hist + wave * E;
    for (int e = lane; e < E; e += 64) h[e] = 0;
    const int nb = (S + 1023) / 1024;   // batches of 64 slots per wave (1..4)
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int ex[4], pos[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int s = (wave * nb + b) * 64 + lane;
        ex[b] = b < nb && s < S ? ids[s] : -1;
        if (unsigned(ex[b]) >= unsigned(E)) ex[b] = -1;   // ids outside [0, E) are dropped
    }
    asm volatile("" ::: "memory");   // (a wave's LDS operations complete in order)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        pos[b] = 0;
        if (b >= nb) break;
        const bool valid = ex[b] >= 0;
        const int e = valid ? ex[b] : 0;
        uint64_t peers = __ballot(valid);
        for (int bit = 0; bit < id_bits; ++bit) {
            const bool on = (e >> bit) & 1;
            const uint64_t m = __ballot(on);
            peers &= on ? m : ~m;
        }
        const int rank = __popcll(peers & lt);
        const int seen = h[e];
        pos[b] = seen + rank;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) h[e] = seen + __popcll(peers);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    int rows = 0;
    if (tid < E)
        for (int w = 0; w < 16; ++w) {
            const int c = hist[w * E + tid];
            hist[w * E + tid] = rows;
            rows += c;
        }
    // tiles per class (as pf_scan_body counts them; tn = 16: all of class 1) and rows, scanned together.
    // full tiles are of class 4 (tn = 64) or 1, the rest tile of class kr; a class ends with the shared
    // group's tiles.
    const int fc = tn == kTN ? 4 : 1;
    const int full = rows / tn, rest = rows % tn, kr = rest ? tile_class(rest) : 0;
    const int v[5] = {rows, int(kr == 1) + (fc == 1 ? full : 0), int(kr == 2), int(kr == 3), int(kr == 4) + (fc == 4 ? full : 0)};
    int r[5], tot[5];
    block_excl_scan_v<5>(v, r, tot, ws);
    const int sfull = shared ? T / tn : 0, srest = shared ? T % tn : 0, sk = srest ? tile_class(srest) : 0;
    int base[5], at[5];   // first tile of each class ([0]: their number); this group's first tile of each
    base[4] = 0;
    for (int k = 3; k >= 0; --k) base[k] = base[k + 1] + tot[k + 1] + (fc == k + 1 ? sfull : 0) + int(sk == k + 1);
    for (int k = 1; k <= 4; ++k) at[k] = base[k] + r[k];
    if (tid < E) {
        bounds[tid] = r[0];
        s_row[tid] = r[0];
        for (int i = 0; i < full; ++i) tiles[(fc == 4 ? at[4] : at[1]) + i] = make_int2(tid, i * tn);
        if (kr) {
            const int p = kr == 4 ? at[4] : kr == 3 ? at[3] : kr == 2 ? at[2] : at[1];
            tiles[p + (kr == fc ? full : 0)] = make_int2(tid, full * tn);
        }
    }
    if (tid == 0) {
        bounds[E] = tot[0];
        if (shared) {
            bounds[E + 1] = tot[0] + T;
            const int p = fc == 4 ? base[4] + tot[4] : base[1] + tot[1];
            for (int i = 0; i < sfull; ++i) tiles[p + i] = make_int2(E, i * tn);
            if (sk) {
                const int q = sk == 4 ? base[4] + tot[4] : sk == 3 ? base[3] + tot[3] : sk == 2 ? base[2] + tot[2] : base[1] + tot[1];
                tiles[q + (sk == fc ? sfull : 0)] = make_int2(E, sfull * tn);
            }
        }
        n_tiles[0] = base[0];
        n_tiles[1] = base[1];
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (b < nb && ex[b] >= 0) {
            const int s = (wave * nb + b) * 64 + lane, row = s_row[ex[b]] + h[ex[b]] + pos[b];
            tok_of[row] = s / K;
            slot_of[row] = s;
        }
    if (shared)
        for (int t = tid; t < T; t += 1024) {   // rows S + t (S = T K: every slot holds a valid id)
            tok_of[S + t] = t;
            slot_of[S + t] = S + t;
        }
}

// ---------------------------------------------------------------- grouped GEMMs (gate + up, down)
//
// Operands enter the MFMA exactly, so the products are exact and only the fp32 accumulation rounds:
//   A (weights): (q - 1) * d_w in fp16, dequantized in registers from the code dwords.
//   B (activations a = code * d_a, Q8_0: up to 18 significant bits), in NP fp16 parts:
//     NP = 2 (gate/up): hi = fp16(a), lo = fp16(a - hi); every 32-deep MFMA step is issued for
//            both parts into one fp32 accumulator (gfx950's MFMA keeps the fp16 subnormals that
//            the lo parts can be). Exactness matters here because h is requantized to Q8_0 after
//            SwiGLU: a rounding difference would move h codes across rounding boundaries.
//     NP = 1 (down): fp16(a), 2^-12 relative per element, with no requantization after it.
//   No per-block scaling happens on the VALU.
//
// Dequantization: code k of a weight dword sits at bits 2k, 2k+1. Masked in place (p = 2k mod 8
// within each 16-bit half) and OR'ed with the fp16 bits of M = 2^(10-p), whose ulp is 2^(p-10),
// it reads as M + q exactly; (M + q) - (M + 1) = q - 1 and the product with d_w are exact too.
// Codes 4..7 of each half are shifted down by 8 first. Per pair of weights: one v_and_or_b32,
// one v_pk_add_f16 and one v_pk_mul_f16 (plus one shift per 16 weights).
//
// k_pf_gemm<DOWN, SMALL>: 256 threads, 64 weight rows (A) per wave against the tokens (B) of one tile.
// Gate/up: wave w takes ff rows f0 + 32 w .. of gate and the same 32 of up, so SwiGLU and the Q8_0 of a
// 32-row block of h (quant/q2_0/moe_cpu.cpp:43-61) stay in the wave; h = code * d is written as fp16
// for the down GEMM. Down: wave w takes output rows r0 + 64 w .., K = ff.
//   SMALL = false: tiles of 17-64 tokens, v_mfma_f32_32x32x16_f16 (two row tiles x one or two token
//                  columns of 32), activation stages of K = 64. A 32x32 product holds the matrix core
//                  32 cycles and the issue port about 10, so five of the dequantization's VALU
//                  instructions hide behind each (a 16x16 one: 16 and 9, two); both measured with
//                  chains of independent products and VALU instructions. In the kernel the two add up
//                  all the same: MFMA 47% and VALU 43% of the SIMD cycles at 2048 tokens.
//   SMALL = true:  tiles of up to 16 tokens, v_mfma_f32_16x16x32_f16 (four row tiles), stages of
//                  K = 256; bound by the dequantization (26 VALU instructions per 16 x 64 weights).
//
// K order (perm256_pos): within each 256-element stretch, MFMA lane group g (16x16: four groups; 32x32:
// two, of blocks 2 p + g for p = 0, 1) takes one block's 16-byte code chunk, dword by dword.
//
// Weights go through the wave's own LDS (no barrier): 64 rows x 64 bytes of codes and 64 x 4 scales per
// stretch by direct global-to-LDS loads whose four consecutive lanes read one row's 64 bytes. Loaded
// straight into the MFMA's registers, each lane of a quad is another row, and the L1 takes one clock
// per lane instead of one per 64 bytes: 17 against 59 bytes per clock and CU (measured, L2-resident
// rows). Chunk c of row r sits at c ^ ((r >> 2) & 3), so that the sixteen lanes of a read phase hit
// distinct banks. A stretch's weights are read
// into registers at its start; the next stretch's then load into the same LDS.
//
// Activations go through LDS too: stages in a ring of slots filled by direct global-to-LDS loads
// (global_load_lds: each lane's 16 bytes land at the wave's LDS base + 16 lane, no registers), issued
// `ahead` stages ahead; one workgroup barrier per stage. Slot layout:
//   [NP][tokens][cpt chunks of 8 fp16], chunk kc of token j at j * cpt + (kc ^ swz(j)) (GemmShape).
// Issue order of k_pf_gemm's loads, as stages s of the same pattern: stage s issues the weights of
// stretch s / sps + 1 when s is a stretch's first (s % sps == 0: "A"), then the activations of stage
// s + ahead ("B"). The prologue is the stages s = -max(ahead, sps) .. -1 of that pattern (A of
// stretch 0 at s = -sps; B stage s + ahead for s >= -ahead), so every stage's wait counts the same.
constexpr int gu_mod(int a, int m) { return ((a % m) + m) % m; }
// The vmcnt of stage st's wait: the loads issued after B stage st (at stage st - ahead), by stages
// st - ahead + 1 .. st - 1: ahead - 1 B stages and the A of each stretch's first among them.
constexpr int gu_wait(int h, int ahead, int sps, int kDB, int kDA) {
    int c = (ahead - 1) * kDB;
    for (int d = 1; d < ahead; ++d) c += gu_mod(h - d, sps) == 0 ? kDA : 0;
    return c;
}
// The same count by listing the issues of the prologue and stages 0 .. st - 1 (1 = an A, 2 + s = B
// stage s) and counting what follows B stage st.
constexpr int gu_after_b(int st, int ahead, int sps, int kDB, int kDA) {
    int seq[96] = {};
    int n = 0;
    const int first = -(ahead > sps ? ahead : sps);
    for (int s = first; s < st; ++s) {
        if (gu_mod(s, sps) == 0 && s / sps + 1 >= 0 && s >= -sps) seq[n++] = 1;
        if (s >= -ahead) seq[n++] = 2 + s + ahead;
    }
    int after = 0;
    bool seen = false;
    for (int i = 0; i < n; ++i) {
        if (seen) after += seq[i] == 1 ? kDA : kDB;
        if (seq[i] == 2 + st) seen = true;
    }
    return after;
}
constexpr bool gu_waits_ok(int ahead, int sps, int kDB, int kDA) {
    for (int st = 0; st < 16; ++st)
        if (gu_after_b(st, ahead, sps, kDB, kDA) != gu_wait(gu_mod(st, sps), ahead, sps, kDB, kDA)) return false;
    return true;
}
template <bool DOWN, bool SMALL>
struct GemmShape {
    static constexpr int parts = DOWN ? 1 : 2;            // activation parts (h as one fp16 value, x as hi and lo)
    static constexpr int tokens = SMALL ? 16 : kTN;       // activation rows in LDS
    static constexpr int rows = DOWN ? 256 : 128;         // output rows (down) / ff rows (gate/up) per workgroup
    static constexpr int stage_k = SMALL ? 256 : 64;      // K per activation stage
    static constexpr int sps = 256 / stage_k;             // stages per weight stretch
    static constexpr int cpt = stage_k / 8;               // 16-byte chunks per token per stage
    static constexpr int slot_b = tokens * stage_k * 2;   // bytes per part per slot
    static constexpr int stages = SMALL ? 2 : DOWN ? 4 : 2;   // activation ring slots
    static constexpr int ahead = stages - 1;              // stages issued ahead
    static constexpr int ring_b = stages * parts * slot_b;
    static constexpr int wave_a = 64 * 64 + 64 * 16;      // a wave's weights: codes of one stretch, scales of two
    static constexpr int smem = ring_b + 4 * wave_a;
    // chunk kc of token j sits at kc ^ swz(j): the sixteen tokens of a 256-byte read phase (64 banks) take
    // sixteen different 16-byte columns (two tokens of 128 bytes share a row of the banks when cpt = 8)
    static __device__ __forceinline__ int swz(int j) { return (cpt == 8 ? j >> 1 : j) & (cpt - 1); }
    static constexpr int dma = tokens * cpt / 256;        // activation loads per lane per part
    static constexpr int kDB = dma * parts, kDA = 6;      // loads per stage (activations) and stretch (weights)
    static_assert(sps <= 4 && gu_waits_ok(ahead, sps, kDB, kDA), "the wait counts of k_pf_gemm");
    static_assert(!DOWN || tokens * (256 + 4) * (SMALL ? 4 : 2) <= smem, "the down epilogue's staging");
};


typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* gbl_ptr_t;
// direct global -> LDS load of 16 bytes per lane to lds_base + 16 lane (lds_base uniform)
__device__ __forceinline__ void ldsdma16(const void* g, void* lds_base) {
    __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)lds_base, 16, 0, 0);
}
// the same with 4 bytes per lane, to lds_base + 4 lane
__device__ __forceinline__ void ldsdma4(const void* g, void* lds_base) {
    __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)lds_base, 4, 0, 0);
}
// A workgroup barrier that does not wait for outstanding global loads (__syncthreads' release fence
// would wait for all of them, the ring's later stages included): this wave's LDS accesses complete,
// then s_barrier. The wait is the builtin (so the compiler's own wait insertion knows the LDS reads
// before it are complete); the empty asm statements keep memory accesses from moving across.
__device__ __forceinline__ void ring_barrier() {
    __builtin_amdgcn_sched_barrier(0);   // nothing is scheduled across (register math included)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0); vmcnt and expcnt not waited for
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// this wave's LDS reads have returned, before anything after this is issued (direct global-to-LDS loads
// may then overwrite what they read)
__device__ __forceinline__ void lds_reads_done() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// s_waitcnt with vmcnt = N (gfx9 encoding; expcnt and lgkmcnt not waited for)
template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70 | 0xF00);
}
// (x & mask) | bits as one v_and_or_b32 (with literal operands the compiler splits it in two)
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t bits) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
    return r;
}

// The fp16 bits of 2^(10 - 2m) in both halves, m = 0..3, held in VGPRs
struct DqMagic {
    uint32_t v[4];
};
__device__ __forceinline__ DqMagic dq_magic() {
    DqMagic r;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        r.v[m] = (0x6400u - 0x0800u * m) * 0x00010001u;
        asm volatile("" : "+v"(r.v[m]));
    }
    return r;
}

// The 8 A operand values of K-step h of one weight row's code dword: pass cw for h = 0 and cw >> 8
// for h = 1; dd = the row's block scale in both halves.
__device__ __forceinline__ half8 dequant8(uint32_t c, half2v dd, const DqMagic& mg) {
    half8 a;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const _Float16 off = _Float16(float((1 << (10 - 2 * m)) + 1));
        const half2v offs = {off, off};
        half2v v = __builtin_bit_cast(half2v, and_or(c, 0x00030003u << (2 * m), mg.v[m]));
        v = (v - offs) * dd;
        a[2 * m] = v[0];
        a[2 * m + 1] = v[1];
    }
    return a;
}

__device__ __forceinline__ int lane_xor16(int v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (threadIdx.x & 16) ? int(r[0]) : int(r[1]);
}
__device__ __forceinline__ int lane_xor32(int v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32) ? int(r[0]) : int(r[1]);
}

__device__ __forceinline__ floatx4 mfma_acc(half8 a, half8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx16 mfma_acc(half8 a, half8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }


// 4 consecutive per-slot outputs as float, fp16 or bf16 (round to nearest even)
__device__ __forceinline__ void store4(float* p, floatx4 v) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void store4(_Float16* p, floatx4 v) {
    typedef _Float16 half4v __attribute__((ext_vector_type(4)));
    const half4v h = {_Float16(v[0]), _Float16(v[1]), _Float16(v[2]), _Float16(v[3])};
    *reinterpret_cast<half4v*>(p) = h;
}
__device__ __forceinline__ void store4(__hip_bfloat16* p, floatx4 v) {
    p[0] = __float2bfloat16(v[0]);
    p[1] = __float2bfloat16(v[1]);
    p[2] = __float2bfloat16(v[2]);
    p[3] = __float2bfloat16(v[3]);
}

// One workgroup's part of one tile: row slice `slice` of tile `tile`.
template <bool DOWN, bool SMALL, typename OutT>
__device__ __forceinline__ void pf_tile(uint8_t* smem, int* sRow, const int2 tile, int slice, const uint8_t* __restrict__ arena,
                                        size_t stride, int E, const uint8_t* __restrict__ shared_blob, int n, int kp, int hblk,
                                        int ff, const _Float16* __restrict__ bh, const _Float16* __restrict__ bl,
                                        const int32_t* __restrict__ row_of, const int32_t* __restrict__ bounds,
                                        OutT* __restrict__ out) {
    using Sh = GemmShape<DOWN, SMALL>;
    constexpr int NP = Sh::parts;
    const int grp = tile.x;
    const int row0 = bounds[grp] + tile.y;
    const int cnt = min(Sh::tokens, bounds[grp + 1] - row0);
    const uint8_t* blob = grp < E ? arena + size_t(grp) * stride : shared_blob;
    const int nbk = (DOWN ? ff : n) / kBlock;   // weight blocks per row (even: n and ff are multiples of 128)
    const int mrows = DOWN ? n : ff;            // rows of the matrix
    const size_t mb = mat_bytes(ff, n);
    const int rbase = slice * Sh::rows;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // the activation row of each tile token (gate/up: its token's; down: its own); past the group's end
    // the last repeats (never written)
    if (tid < Sh::tokens) {
        const int r = row0 + min(tid, cnt - 1);
        sRow[tid] = DOWN ? r : row_of[r];
    }
    __syncthreads();

    // weight loads of stretch q: lane l takes chunk position l % 4 of rows 16 p + l / 4, p = 0..3 (codes).
    // Scales come for two stretches at a time (16 bytes a row: block pair l % 4 of row 16 p + l / 4), half
    // of the rows with each stretch before. Wave rows: gate/up 0..31 gate, 32..63 up; down: 64
    // consecutive rows (past the matrix's end the last repeats, never written). K runs to kp; a block
    // past the row's last is read as its last, whose finite products with the zeros are 0.
    uint8_t* const sA = smem + Sh::ring_b + wave * Sh::wave_a;
    const uint8_t* const mat = DOWN ? blob + 2 * mb : blob;
    const uint32_t scale_off = uint32_t(mrows) * nbk * 16;
    auto row_at = [&](int rl) {   // (matrix offset, row) of wave row rl
        return DOWN ? min(rbase + 64 * wave + rl, mrows - 1) : rbase + 32 * wave + (rl & 31);
    };
    uint32_t coff[4], soff[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t m = !DOWN && p >= 2 ? uint32_t(mb) : 0u, r = uint32_t(row_at(16 * p + (lane >> 2))) * nbk;
        coff[p] = m + r * 16;
        soff[p] = m + scale_off + r * 2;
    }
    const int cchunk = (lane & 3) ^ ((lane >> 4) & 3);   // the chunk at this lane's position: c ^ ((row >> 2) & 3)
    auto issue_scales = [&](int pair, int half) {
        const uint32_t so = uint32_t(min(4 * pair + (lane & 3), nbk / 2 - 1)) * 4;
#pragma unroll
        for (int p = 0; p < 2; ++p) ldsdma4(mat + ((half ? soff[2 + p] : soff[p]) + so), sA + 4096 + half * 512 + p * 256);
    };
    auto issue_a = [&](int q) {   // stretch q's codes; half the rows' scales of the pair of stretches after q's
        const uint32_t bo = uint32_t(min(4 * q + cchunk, nbk - 1)) * 16;
#pragma unroll
        for (int p = 0; p < 4; ++p) ldsdma16(mat + (coff[p] + bo), sA + p * 1024);
        issue_scales((q + 1) >> 1, (q & 1) ^ 1);
    };
    // this thread's activation chunks of a stage: LDS positions P = 256 p + tid (token P / cpt)
    size_t boff[Sh::dma];   // element offsets
#pragma unroll
    for (int p = 0; p < Sh::dma; ++p) {
        const int P = 256 * p + tid, j = P / Sh::cpt, kc = (P % Sh::cpt) ^ Sh::swz(j);
        boff[p] = size_t(sRow[j]) * kp + kc * 8;
    }
    auto issue_b = [&](int st, int slot) {
        uint8_t* b = smem + slot * NP * Sh::slot_b + wave * 1024;
#pragma unroll
        for (int p = 0; p < Sh::dma; ++p) {
            ldsdma16(bh + boff[p] + size_t(st) * Sh::stage_k, b + p * 4096);
            if constexpr (NP == 2) ldsdma16(bl + boff[p] + size_t(st) * Sh::stage_k, b + Sh::slot_b + p * 4096);
        }
    };
    // the MFMA shape: RT row tiles of MR rows, lanes (row or token lr, group lg), PG blocks per lane and stretch
    constexpr int MR = SMALL ? 16 : 32, RT = 64 / MR, MC = Sh::tokens / MR, PG = SMALL ? 1 : 2;
    const int lr = lane & (MR - 1), lg = lane / MR;
    using Acc = std::conditional_t<SMALL, floatx4, floatx16>;
    Acc acc[RT][MC];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int c = 0; c < MC; ++c)
#pragma unroll
            for (int r = 0; r < MR * MR / 64; ++r) acc[i][c][r] = 0.0f;
    const DqMagic mg = dq_magic();
    half8 cw[RT][PG];        // (read as the activations are: bits of code dwords)
    _Float16 sc[RT][PG], sc1[RT][PG];   // scales of this stretch and, in an even one, of the next
    auto read_a = [&](bool even) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int p = 0; p < PG; ++p) {
                const int rl = MR * i + lr, c = (SMALL ? 0 : 2 * p) + lg;
                cw[i][p] = reinterpret_cast<const half8*>(sA)[rl * 4 + (c ^ ((rl >> 2) & 3))];
                sc[i][p] = sc1[i][p];
                if (even) {
                    sc[i][p] = reinterpret_cast<const _Float16*>(sA + 4096)[rl * 8 + c];
                    sc1[i][p] = reinterpret_cast<const _Float16*>(sA + 4096)[rl * 8 + 4 + c];
                }
            }
    };

    // Stage st (K = stage_k st ..) is part h = st % sps of stretch st / sps. Per stage st, after its
    // barrier: A stretch st / sps + 1 (first stage of a stretch, h = 0, once the current stretch's
    // weights are in registers), then B stage st + ahead (the issue pattern of gu_wait). Waiting for B
    // stage st (vmcnt: the loads issued after it may stay outstanding) covers everything issued before
    // it, A stretch st / sps included. The pattern is the same for every stage: past the end, the last
    // stretch / stage is loaded again (into LDS that nothing reads any more), so the wait counts are
    // constants.
    const int nst = kp / Sh::stage_k;   // stages
    const int nq = kp / 256;            // stretches
    auto run = [&](auto nc) {
        constexpr int NC = decltype(nc)::value;
        // K-step t of the stage in slot sb (t: its 32-deep chunk group), block pair half p (32x32 only)
        auto rd = [&](const half8* sb, int t, int p, half8(&b)[NC][NP]) {
            const int kc = t * 4 + (SMALL ? 0 : 2 * p) + lg;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j = c * MR + lr;
#pragma unroll
                for (int part = 0; part < NP; ++part)
                    b[c][part] = sb[part * (Sh::slot_b / 16) + j * Sh::cpt + (kc ^ Sh::swz(j))];
            }
        };
        // the loads of stages -max(ahead, sps) .. -1 of the steady-state pattern below
#pragma unroll
        for (int s = -(Sh::ahead > Sh::sps ? Sh::ahead : Sh::sps); s < 0; ++s) {
            if (gu_mod(s, Sh::sps) == 0 && s >= -Sh::sps) {
                issue_scales(0, 0);
                issue_a(0);   // (with the other half's scales)
            }
            if (s >= -Sh::ahead) issue_b(min(s + Sh::ahead, nst - 1), s + Sh::ahead);
        }
        int slot = 0, slot_in = Sh::ahead;   // the slots of stages st and st + ahead
        for (int q = 0; q < nq; ++q) {
#pragma unroll
            for (int h = 0; h < Sh::sps; ++h) {
                const int st = Sh::sps * q + h;
                // loads issued after B stage st (by stages st - ahead + 1 .. st - 1) may stay outstanding
                switch (h) {
                    case 0: wait_vm<gu_wait(0, Sh::ahead, Sh::sps, Sh::kDB, Sh::kDA)>(); break;
                    case 1: wait_vm<gu_wait(1, Sh::ahead, Sh::sps, Sh::kDB, Sh::kDA)>(); break;
                    case 2: wait_vm<gu_wait(2, Sh::ahead, Sh::sps, Sh::kDB, Sh::kDA)>(); break;
                    default: wait_vm<gu_wait(3, Sh::ahead, Sh::sps, Sh::kDB, Sh::kDA)>(); break;
                }
                ring_barrier();   // stage st is in LDS for every wave; every wave is done with stage st - 1
                if (h == 0) {
                    read_a((q & 1) == 0);
                    lds_reads_done();   // the wave's weights are in registers: their LDS may be written
                    issue_a(min(q + 1, nq - 1));
                }
                issue_b(min(st + Sh::ahead, nst - 1), slot_in);   // into stage st - 1's slot
                const half8* sb = reinterpret_cast<const half8*>(smem + slot * NP * Sh::slot_b);
                slot = slot + 1 == Sh::stages ? 0 : slot + 1;
                slot_in = slot_in + 1 == Sh::stages ? 0 : slot_in + 1;
                constexpr int steps = Sh::stage_k / 32 * PG;
                half8 b[2][NC][NP];
                rd(sb, 0, 0, b[0]);
#pragma unroll
                for (int u = 0; u < steps; ++u) {
                    const int tt = Sh::stage_k / 32 * h + u / PG, p = u % PG;   // the step's place in the stretch
                    if (u + 1 < steps) rd(sb, (u + 1) / PG, (u + 1) % PG, b[(u + 1) & 1]);
#pragma unroll
                    for (int i = 0; i < RT; ++i) {
                        const uint32_t x = __builtin_bit_cast(u32x4_t, cw[i][p])[tt >> 1];
                        const half8 av = dequant8((tt & 1) ? x >> 8 : x, half2v{sc[i][p], sc[i][p]}, mg);
#pragma unroll
                        for (int c = 0; c < NC; ++c)
#pragma unroll
                            for (int part = 0; part < NP; ++part) acc[i][c] = mfma_acc(av, b[u & 1][c][part], acc[i][c]);
                    }
                }
            }
        }
    };
    if constexpr (SMALL) {
        run(std::integral_constant<int, 1>{});
    } else {
        if (cnt <= 32) run(std::integral_constant<int, 1>{});
        else run(std::integral_constant<int, 2>{});
    }
    wait_vm<0>();      // the ring's last direct-to-LDS loads (repeats past the end) have landed
    __syncthreads();   // and every wave is past its last LDS read

    // Lane (token lr, group lg) holds MFMA rows 4 lg + 8 a + b (32x32: a, b = 0..3) or 4 lg + b (16x16) of
    // each row tile, as register 4 a + b.
    if constexpr (DOWN) {
        // through LDS, a column of tokens at a time, so that each token's 256 outputs leave in one run
        constexpr int ld = 256 + 4;
        float* sy = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int c = 0; c < MC; ++c) {
            if (c * MR >= cnt) break;   // (uniform)
            if (c) __syncthreads();
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int a = 0; a < MR * MR / 256; ++a)
                    *reinterpret_cast<floatx4*>(sy + lr * ld + 64 * wave + MR * i + 8 * a + 4 * lg) =
                        floatx4{acc[i][c][4 * a], acc[i][c][4 * a + 1], acc[i][c][4 * a + 2], acc[i][c][4 * a + 3]};
            __syncthreads();
            for (int j = wave; j < min(MR, cnt - c * MR); j += 4) {
                const int r = rbase + 4 * lane;
                if (r < n)   // (n % 4 == 0)
                    store4(out + size_t(row_of[row0 + c * MR + j]) * n + r, *reinterpret_cast<const floatx4*>(sy + j * ld + 4 * lane));
            }
        }
    } else {
        // ff rows fbase .. fbase + 31 (one Q8_0 block of h) of token column c: gate in the first half of
        // the row tiles, up in the second
        const int ffp = (ff + 255) & ~255;   // h row length
        const int fbase = rbase + 32 * wave;
        constexpr int HT = RT / 2, NR = MR * MR / 64;   // gate row tiles; values per lane of each
#pragma unroll
        for (int c = 0; c < MC; ++c) {
            const int col = c * MR + lr;
            float hv[HT][NR];
            float am = 0.0f;
#pragma unroll
            for (int i = 0; i < HT; ++i)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    hv[i][r] = silu_mul(acc[i][c][r], acc[HT + i][c][r]);
                    am = fmaxf(am, fabsf(hv[i][r]));
                }
            if (SMALL) am = fmaxf(am, __builtin_bit_cast(float, lane_xor16(__builtin_bit_cast(int, am))));
            am = fmaxf(am, __builtin_bit_cast(float, lane_xor32(__builtin_bit_cast(int, am))));
            if (hblk == 64) {   // ff rows 64 m .. 64 m + 63 are waves 2m' and 2m' + 1 (rbase is a multiple of 128)
                float* sam = reinterpret_cast<float*>(smem);
                if (c) __syncthreads();   // (uniform: hblk is a kernel argument)
                if (lg == 0) sam[wave * MR + lr] = am;
                __syncthreads();
                am = fmaxf(am, sam[(wave ^ 1) * MR + lr]);
            }
            const float d = q8_scale(am);
            const float id = q8_inv(d);
            const float dr = f16_round(d);
            if (col < cnt) {
                // f = fbase + 16 s + 4 e + b: 16x16 s = i, e = lg; 32x32 s = a / 2, e = 2 (a % 2) + lg. In
                // perm256 order (s, b / 2) are the four consecutive values at the position of (s = 0, e, b % 2).
                _Float16* dst = out + size_t(row0 + col) * ffp + (fbase & ~255);
#pragma unroll
                for (int e = 0; e < (SMALL ? 1 : 2); ++e)
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        _Float16 v[4];
#pragma unroll
                        for (int s = 0; s < 2; ++s)
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const float x = SMALL ? hv[s % HT][(b + 2 * u) % NR] : hv[0][(4 * (2 * s + e) + b + 2 * u) % NR];
                                v[2 * s + u] = _Float16(float(q8_code(x, id)) * dr);
                            }
                        typedef _Float16 half4v __attribute__((ext_vector_type(4)));
                        const int f = (fbase & 255) + 4 * (SMALL ? lg : 2 * e + lg) + b;
                        *reinterpret_cast<half4v*>(dst + perm256_pos(f)) = half4v{v[0], v[1], v[2], v[3]};
                    }
            }
        }
        // h rows are ffp = ff rounded up to 256 long (whole perm256 stretches for the down GEMM); the
        // slice holding the last rows also writes zeros at the pad's positions, so that the down GEMM's
        // products there are 0 (its weights for the pad are any finite values of the row)
        if (ffp > ff && rbase + Sh::rows >= ff) {
            const int np = ffp - ff;   // pad elements per row: f = ff .. ffp - 1
            for (int i = tid; i < cnt * np; i += 256) {
                const int col = i / np, f = ff + i % np;
                out[size_t(row0 + col) * ffp + (f & ~255) + perm256_pos(f & 255)] = _Float16(0.0f);
            }
        }
    }
}

// DOWN: bh is h [S][kp] (kp = ff rounded up to 256, zeros in the pad), out is yd [slot][n]. Gate/up: bh and
// bl are the x pairs [T][kp] (kp = n rounded up to 512, zeros past n), out is h.
// Both tile shapes in one launch, in an order that mixes them: the small tiles stream weights from HBM
// (each expert's once), the larger ones are bound by the matrix cores, and side by side each fills what
// the other leaves idle.
template <bool DOWN, typename OutT>
__global__ void __launch_bounds__(256, 3)
k_pf_gemm(const uint8_t* __restrict__ arena, size_t stride, int E, const uint8_t* __restrict__ shared_blob, int n,
          int kp, int hblk, int ff, const _Float16* __restrict__ bh, const _Float16* __restrict__ bl,
          const int32_t* __restrict__ row_of, const int32_t* __restrict__ bounds, const int2* __restrict__ tiles,
          const int32_t* __restrict__ n_tiles, OutT* __restrict__ out) {
    // A 1-D grid of gx row slices x tiles (tiles rounded up to a multiple of 8). Workgroup L runs on
    // XCD L % 8, so the slices of a tile are placed 8 apart: they run on the same XCD at about the same
    // time, and the tile's activations come into that XCD's L2 once.
    const int gx = DOWN ? (n + 255) / 256 : ff / GemmShape<DOWN, false>::rows;
    const int L = blockIdx.x, r8 = L >> 3;
    const int slice = r8 % gx, t = (L & 7) + 8 * (r8 / gx);
    // n_tiles[0]: tiles in all; n_tiles[1] = B: the first tile of up to 16 tokens (the list is ordered
    // longest first). The first M places of the order hold the B large tiles evenly spread, the rest
    // are small, so that the launch ends on short tiles.
    const int N = n_tiles[0], B = n_tiles[1];
    if (t >= N) return;
    const int M = max(1, B + (N - B) * 3 / 4);
    const int before = t < M ? int(int64_t(t) * B / M) : B, upto = t < M ? int(int64_t(t + 1) * B / M) : B;
    const bool big = upto > before;
    const int2 tile = tiles[big ? before : B + t - before];
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int sRow[kTN];
    if (big)
        pf_tile<DOWN, false, OutT>(smem, sRow, tile, slice, arena, stride, E, shared_blob, n, kp, hblk, ff, bh, bl, row_of, bounds, out);
    else
        pf_tile<DOWN, true, OutT>(smem, sRow, tile, slice, arena, stride, E, shared_blob, n, kp, hblk, ff, bh, bl, row_of, bounds, out);
}

// ---------------------------------------------------------------- combine

// out[t][i] = sum over the token's K slots in ascending expert id of w * yd (+ shared * sigmoid(g));
// grid (ceil(n / 1024), T), 4 consecutive outputs per thread
template <typename InT>
__global__ void __launch_bounds__(256) k_pf_combine(const InT* __restrict__ yd, const int32_t* __restrict__ ids,
                                                    const float* __restrict__ wts, const float* __restrict__ gate, int T,
                                                    int K, int n, int shared, const float* __restrict__ resid,
                                                    float* __restrict__ out) {
    __shared__ int order[32];
    const int t = blockIdx.y;
    if (threadIdx.x < K) {   // rank of slot k by expert id (the ids of one token are distinct)
        const int e = ids[t * K + threadIdx.x];
        int r = 0;
        for (int k = 0; k < K; ++k) r += ids[t * K + k] < e ? 1 : 0;
        order[r] = threadIdx.x;
    }
    __syncthreads();
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n) return;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int r = 0; r < K; ++r) {
        const int k = order[r];
        const float w = wts[t * K + k];
        const InT* src = yd + (size_t(t) * K + k) * n + i;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float p = w * float(src[q]);
            acc[q] = acc[q] + p;
        }
    }
    float o[4] = {acc[0], acc[1], acc[2], acc[3]};
    if (shared) {
        const float g = 1.0f / (1.0f + expf(-gate[t]));
        const InT* src = yd + (size_t(T) * K + t) * n + i;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float p = float(src[q]) * g;
            o[q] = acc[q] + p;
        }
    }
    if (resid)
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = resid[size_t(t) * n + i + q] + o[q];
    *reinterpret_cast<float4*>(out + size_t(t) * n + i) = make_float4(o[0], o[1], o[2], o[3]);
}

}  // namespace

// ---------------------------------------------------------------- host side

struct PfWs {
    int32_t *cnt, *bounds, *tok_of, *slot_of, *n_tiles;
    int2* tiles;
    _Float16 *xhi, *xlo;   // x = code * d as an exact fp16 pair, perm256 order [T][n]
    _Float16* h16;         // h = code * d as fp16, perm256 order [S][ffp], ffp = ff rounded up to 256
    _Float16* yd;   // fp16 per-slot outputs of a whole layer (combined by k_pf_combine)
    size_t bytes;
};

static int pf_max_tiles(int S, int G) { return (S + pf_tile_tokens(S) - 1) / pf_tile_tokens(S) + G; }
// The tile list's length in a workspace: never less than a shorter chunk's (whose tiles are of 16 tokens), so
// that a workspace sized for the longest call holds every other.
static size_t pf_tile_list(int S, int G) {
    return size_t(S <= kTile16Slots ? pf_max_tiles(S, G) : std::max(pf_max_tiles(S, G), pf_max_tiles(kTile16Slots, G)));
}
// the gate/up GEMM's K extent: n rounded up to whole pairs of 256-element stretches
static int pf_np(int n) { return (n + 511) & ~511; }

static PfWs pf_carve(void* base, int T, int K, int n, int ff, int E, bool shared, bool own_yd) {
    PfWs w{};
    uint8_t* p = static_cast<uint8_t*>(base);
    auto take = [&](size_t b) {
        uint8_t* r = p;
        p += up256(b);
        return r;
    };
    const int S = T * K + (shared ? T : 0);
    const int G = E + (shared ? 1 : 0);
    const int nchunk = (T * K + kChunk - 1) / kChunk;
    w.cnt = reinterpret_cast<int32_t*>(take(size_t(nchunk) * E * 4));
    w.bounds = reinterpret_cast<int32_t*>(take(size_t(E + 2) * 4));
    w.tok_of = reinterpret_cast<int32_t*>(take(size_t(S) * 4));
    w.slot_of = reinterpret_cast<int32_t*>(take(size_t(S) * 4));
    w.n_tiles = reinterpret_cast<int32_t*>(take(8));   // [0] tiles, [1] first tile of one column
    w.tiles = reinterpret_cast<int2*>(take(pf_tile_list(S, G) * 8));
    w.xhi = reinterpret_cast<_Float16*>(take(size_t(T) * pf_np(n) * 2));
    w.xlo = reinterpret_cast<_Float16*>(take(size_t(T) * pf_np(n) * 2));
    w.h16 = reinterpret_cast<_Float16*>(take(size_t(S) * ((ff + 255) & ~255) * 2));
    // (fp32 when ff > 1024: pf_moe)
    w.yd = own_yd ? reinterpret_cast<_Float16*>(take(size_t(S) * n * (ff > 1024 ? 4 : 2))) : nullptr;
    w.bytes = size_t(p - static_cast<uint8_t*>(base));
    return w;
}

size_t pf_workspace_bytes(int T, int K, int n, int ff, int E, bool shared, bool own_yd) {
    return pf_carve(nullptr, T, K, n, ff, E, shared, own_yd).bytes + 256;
}

int quantize_pairs(const float* x, int rows, int n, int np, int blk, _Float16* xhi, _Float16* xlo, int8_t* xq, float* xd,
                   hipStream_t stream);
int norm_pairs(const float* x, int rows, int n, int np, float* u, _Float16* xhi, _Float16* xlo, int8_t* xq, float* xd,
               hipStream_t stream);

int pf_check(int T, int K, int n, int ff, int E) {
    if (T < 1 || K < 1 || K > 32 || E < 1 || E > 4096 || K > E) return set_error(kErrShape, "prefill: T=%d K=%d E=%d", T, K, E);
    // n and ff multiples of 128 (moe_q2.cu:516-517): gate/up takes slices of 128 ff rows, and a row's 64-blocks
    // come in pairs
    if (n % 128 || n < 128 || n > 65536 || ff % 128 || ff < 128 || ff > 4096)
        return set_error(kErrShape, "prefill: n=%d ff=%d (n and ff multiples of 128; ff at most 4096)", n, ff);
    return kOk;
}

template <bool DOWN, typename OutT>
static int pf_gemm(const char* name, const uint8_t* arena, size_t stride, int E, const uint8_t* shared_blob, int n, int kp,
                   int ff, int blk, const _Float16* bh, const _Float16* bl, const int32_t* row_of, const PfWs& w, int mt,
                   OutT* out, hipStream_t stream) {
    constexpr int big = GemmShape<DOWN, false>::smem, small = GemmShape<DOWN, true>::smem, smem = big > small ? big : small;
    static_assert(3 * (smem + 4 * kTN) <= 160 * 1024, "three workgroups per CU");
    static bool done = false;   // per process; the attribute is a property of the kernel
    if (!done) {
        FRT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_gemm<DOWN, OutT>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, smem));
        done = true;
    }
    const unsigned grid = unsigned(DOWN ? (n + 255) / 256 : ff / GemmShape<DOWN, false>::rows) * unsigned((mt + 7) / 8 * 8);
    launch_timed(name, k_pf_gemm<DOWN, OutT>, dim3(grid), dim3(256), smem, stream, arena, stride, E, shared_blob, n, kp, blk,
                 ff, bh, bl, row_of, (const int32_t*)w.bounds, (const int2*)w.tiles, (const int32_t*)w.n_tiles, out);
    return kOk;
}

// The two grouped GEMMs: gate/up on the exact x pairs, SwiGLU and Q8_0 of h in the epilogue; down on
// h -> yd per slot as OutT.
template <typename OutT>
static int pf_expert_gemms(const uint8_t* arena, size_t stride, int E, const uint8_t* shared_blob, int n, int ff,
                           int blk, const PfWs& w, int mt, OutT* ydf, hipStream_t stream) {
    const int ffp = (ff + 255) / 256 * 256;   // h row length
    // (the kernels take any ff: 16-bit outputs of longer sums are refused as a matter of precision)
    if (ffp > 1024 && !std::is_same<OutT, float>::value)
        return set_error(kErrShape, "prefill: ff=%d above 1024 needs fp32 per-slot outputs", ff);
    if (int rc = pf_gemm<false>("pf_gateup", arena, stride, E, shared_blob, n, pf_np(n), ff, blk,
                                (const _Float16*)w.xhi, (const _Float16*)w.xlo, (const int32_t*)w.tok_of, w, mt, w.h16, stream))
        return rc;
    timing_mark(stream, "pf_gateup");
    return pf_gemm<true>("pf_down", arena, stride, E, shared_blob, n, ffp, ff, blk, (const _Float16*)w.h16,
                         (const _Float16*)nullptr, (const int32_t*)w.slot_of, w, mt, ydf, stream);
}

// The dispatch of S = T K slots (and the shared group's T rows): bounds, tiles, tok_of and slot_of.
static int pf_dispatch_run(const int32_t* ids, int T, int K, int E, bool shared, int32_t* cnt, int32_t* bounds, int2* tiles,
                           int32_t* n_tiles, int32_t* tok_of, int32_t* slot_of, hipStream_t stream) {
    int id_bits = 1;
    while ((1 << id_bits) < E) ++id_bits;
    const int S = T * K, nchunk = (S + kChunk - 1) / kChunk;
    if (S <= kSmallSlots && E <= 1024) {
        const size_t lds = size_t(16) * E * 4;
        static bool done = false;   // per process; the attribute is a property of the kernel
        if (!done) {
            FRT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pf_dispatch1),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 16 * 1024 * 4));
            done = true;
        }
        launch_timed("pf_dispatch1", k_pf_dispatch1, dim3(1), dim3(1024), lds, stream, ids, S, K, E, id_bits, T, shared ? 1 : 0,
                     pf_tile_tokens(shared ? S + T : S), bounds, tiles, n_tiles, tok_of, slot_of);
        return kOk;
    }
    launch_timed("pf_hist", k_pf_hist, dim3(nchunk), dim3(256), size_t(E) * 4, stream, ids, S, E, cnt);
    launch_timed("pf_colscan", k_pf_colscan, dim3((E + 3) / 4), dim3(256), 0, stream, cnt, nchunk, E, bounds);
    launch_timed("pf_scan", k_pf_scan, dim3(1), dim3(1024), 0, stream, E, T, shared ? 1 : 0, bounds, tiles, n_tiles);
    launch_timed("pf_place", k_pf_place, dim3(nchunk + (shared ? (T + 63) / 64 : 0)), dim3(64), size_t(E) * 4, stream, ids, S,
                 K, E, id_bits, (const int32_t*)cnt, (const int32_t*)bounds, tok_of, slot_of, shared ? T : 0);
    return kOk;
}

// The grouped expert products for routed ids (+ optionally the shared expert as group E).
// yd_kind: 0 float, 1 bf16 (moe_q2::run's yd_bf16), 2 fp16 (a whole layer's, combined here)
static int pf_experts(const uint8_t* arena, size_t stride, int E, const uint8_t* shared_blob, int n, int ff,
                      const float* x, const int32_t* ids, int T, int K, void* yd, int yd_kind, int blk, const PfWs& w,
                      bool pairs_done, hipStream_t stream) {
    const bool shared = shared_blob != nullptr;
    const int S = T * K + (shared ? T : 0);
    const int G = E + (shared ? 1 : 0);
    if (!pairs_done)
        if (int rc = quantize_pairs(x, T, n, pf_np(n), blk, w.xhi, w.xlo, nullptr, nullptr, stream)) return rc;
    timing_mark(stream, "pf_quant_x");
    if (int rc = pf_dispatch_run(ids, T, K, E, shared, w.cnt, w.bounds, w.tiles, w.n_tiles, w.tok_of, w.slot_of, stream)) return rc;
    timing_mark(stream, "pf_dispatch");
    const int mt = pf_max_tiles(S, G);
    int rc = kOk;
    if (yd_kind == 1) rc = pf_expert_gemms(arena, stride, E, shared_blob, n, ff, blk, w, mt, static_cast<__hip_bfloat16*>(yd), stream);
    else if (yd_kind == 2) rc = pf_expert_gemms(arena, stride, E, shared_blob, n, ff, blk, w, mt, static_cast<_Float16*>(yd), stream);
    else rc = pf_expert_gemms(arena, stride, E, shared_blob, n, ff, blk, w, mt, static_cast<float*>(yd), stream);
    if (rc) return rc;
    timing_mark(stream, "pf_down");
    FRT_LAUNCHED("prefill experts");
    return kOk;
}

// The GEMMs' x pairs ahead of a pf_run (shared, own_yd false) or pf_moe (true) call on the same workspace
// (its pairs_done): with norm_u, of x * rms scale, which also goes to norm_u. xq, xd (or null): the Q8_0
// codes and scales of the same values.
int pf_pairs(const float* x, int T, int K, int n, int ff, int E, bool shared, bool own_yd, void* ws, size_t ws_bytes,
             float* norm_u, int8_t* xq, float* xd, hipStream_t stream) {
    if (int rc = pf_check(T, K, n, ff, E)) return rc;
    const PfWs w = pf_carve(ws, T, K, n, ff, E, shared, own_yd);
    if (w.bytes > ws_bytes) return set_error(kErrWorkspace, "prefill: workspace %zu < %zu", ws_bytes, w.bytes);
    if (norm_u) return norm_pairs(x, T, n, pf_np(n), norm_u, w.xhi, w.xlo, xq, xd, stream);
    return quantize_pairs(x, T, n, pf_np(n), 32, w.xhi, w.xlo, xq, xd, stream);
}

// moe_q2::run (kernels/cuda/moe_q2.h:20-30): yd [T*K][n] per slot
int pf_run(const uint8_t* experts, size_t stride, int E, int n, int ff, const float* x, const int32_t* ids, int T, int K,
           void* yd, void* ws, size_t ws_bytes, hipStream_t stream, int block64, int yd_bf16, bool pairs_done) {
    if (int rc = pf_check(T, K, n, ff, E)) return rc;
    if (!experts || !x || !ids || !yd || !ws) return set_error(kErrNull, "moe_q2::run: null pointer");
    const PfWs w = pf_carve(ws, T, K, n, ff, E, false, false);
    if (w.bytes > ws_bytes) return set_error(kErrWorkspace, "moe_q2::run: workspace %zu < %zu", ws_bytes, w.bytes);
    // block64: x and h quantized in Q8_0 blocks of 64 values rather than 32 (moe_q2.cu's AB = 64)
    return pf_experts(experts, stride, E, nullptr, n, ff, x, ids, T, K, yd, yd_bf16 ? 1 : 0, block64 ? 64 : 32, w, pairs_done,
                      stream);
}

// The whole prefill layer after routing: ids/wts [T][K], gate [T] -> out [T][n] (+ resid)
int pf_moe(const uint8_t* arena, size_t stride, int E, const uint8_t* shared_blob, int n, int ff, const float* x,
           const int32_t* ids, const float* wts, const float* gate, int T, int K, const float* resid, float* out,
           void* ws, size_t ws_bytes, bool pairs_done, hipStream_t stream) {
    if (int rc = pf_check(T, K, n, ff, E)) return rc;
    const PfWs w = pf_carve(ws, T, K, n, ff, E, true, true);
    if (w.bytes > ws_bytes) return set_error(kErrWorkspace, "prefill: workspace %zu < %zu", ws_bytes, w.bytes);
    if (ff > 1024) {   // fp32 per-slot outputs: fp16 ones would be a precision less than these layers have
        if (int rc = pf_experts(arena, stride, E, shared_blob, n, ff, x, ids, T, K, w.yd, 0, 32, w, pairs_done, stream)) return rc;
        launch_timed("pf_combine", k_pf_combine<float>, dim3((n + 1023) / 1024, T), dim3(256), 0, stream,
                     (const float*)w.yd, ids, wts, gate, T, K, n, 1, resid, out);
        timing_mark(stream, "pf_combine");
        FRT_LAUNCHED("prefill combine");
        return kOk;
    }
    if (int rc = pf_experts(arena, stride, E, shared_blob, n, ff, x, ids, T, K, w.yd, 2, 32, w, pairs_done, stream)) return rc;
    launch_timed("pf_combine", k_pf_combine<_Float16>, dim3((n + 1023) / 1024, T), dim3(256), 0, stream,
                 (const _Float16*)w.yd, ids, wts, gate, T, K, n, 1, resid, out);
    timing_mark(stream, "pf_combine");
    FRT_LAUNCHED("prefill combine");
    return kOk;
}

size_t pf_dispatch_ws_bytes(int T, int K, int E) {
    const int nchunk = (T * K + kChunk - 1) / kChunk;
    return up256(size_t(nchunk) * E * 4) + up256(pf_tile_list(T * K, E) * 8) + 256;
}
// expose the dispatch alone (tests compare the permutation with the oracle)
int pf_dispatch(const int32_t* ids, int T, int K, int E, int32_t* bounds, int32_t* tok_of, int32_t* slot_of, void* ws,
                size_t ws_bytes, hipStream_t stream) {
    if (T < 1 || K < 1 || E < 1 || E > 4096) return set_error(kErrShape, "dispatch: T=%d K=%d E=%d", T, K, E);
    const int nchunk = (T * K + kChunk - 1) / kChunk;
    const size_t need = pf_dispatch_ws_bytes(T, K, E);
    if (ws_bytes < need) return set_error(kErrWorkspace, "dispatch: workspace %zu < %zu", ws_bytes, need);
    uint8_t* p = static_cast<uint8_t*>(ws);
    int32_t* cnt = reinterpret_cast<int32_t*>(p);
    p += up256(size_t(nchunk) * E * 4);
    int2* tiles = reinterpret_cast<int2*>(p);
    p += up256(pf_tile_list(T * K, E) * 8);
    int32_t* n_tiles = reinterpret_cast<int32_t*>(p);
    if (int rc = pf_dispatch_run(ids, T, K, E, false, cnt, bounds, tiles, n_tiles, tok_of, slot_of, stream)) return rc;
    FRT_LAUNCHED("dispatch");
    return kOk;
}

}  // namespace frt
