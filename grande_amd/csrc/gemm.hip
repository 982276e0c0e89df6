// Dequant-fused MFMA GEMMs for the linear layers (matmul.wgsl and
// matmul_gated.wgsl's job): Y[M,N] = f16(X)[M,K] . deq(W)[N,K]^T with f32
// accumulation on v_mfma_f32_32x32x16_f16.
//
// Row-owner tiles: NW wave64s per workgroup over a BM x BN output tile,
// BM = 32 * MI activation rows.  Each wave owns 32 * NJ weight rows (gated:
// half of them rows of the gate matrix and half the same rows of the up
// matrix) across all BM rows, so every weight row is decoded by exactly one
// wave of the tile, straight from its codes into MFMA operand registers.  K
// advances 64 at a time ("stages").  The X tile of a stage (f16 [BM][64])
// goes by LDS DMA into a ring of NS slots; the weights come from the tiled
// copy (one contiguous packet of codes per 32 rows and stage, and one of
// scales) into the registers of the wave that owns the rows.  The DMA holds
// no registers for what is in flight, the stage's K offset rides in the
// instruction's scalar offset, so the per-lane offsets are fixed for the
// whole loop, and there is one barrier per stage.  The decode rounds
// (q - 8) * d (or q * d) to f16 once, the reference's f16 rounding point
// (shaders/weight.wgsl:40-54).
//
// Three kernels with the same sums: gemm32_kernel (fragments of a whole stage
// at a time; short products, where a tile's own latency counts),
// gemm32w_kernel (fragments one k-step ahead, so twice the tile in the same
// registers; products of more than one round of tiles) and gemm32l_kernel
// (f16 weights, which have nothing to decode: they go through LDS like X and
// every wave of a tile reads them from there).
//
// X tiles are 128 B per row with the 16 B chunk c of row r stored at
// c ^ ((r >> 1) & 7), so the rows of one fragment read hit distinct banks.
//
// MFMA operand layout (32x32x16 f16): lane l supplies A[l % 32][8*(l/32)..+8)
// and B[8*(l/32)..+8)[l % 32]; D[8*q + 4*(l/32) + r][l % 32] of the f32
// result lands in element 4 q + r of the lane's sixteen.  The weight fragment
// is the A operand and the activation fragment the B operand, so D =
// (X W^T)^T and each lane ends up with runs of four consecutive output
// columns of one row: the epilogue stores them as vectors.
//
// Bounds: every global read is a buffer load on a per-tile resource, so rows
// past M or N read as zero in hardware; in the K tail (K % 64 == 32) the X
// lanes past K are sent out of range by their lane offset (a zero activation
// times the packet's zero padding).
#include <algorithm>
#include <climits>
#include <string>
#include <utility>

#include "common.h"
#include "kern_common.h"

namespace omg {

constexpr int G_BK = 64;  // k per stage
constexpr int G_ROW = G_BK * 2;  // bytes per LDS tile row
constexpr uint32_t OOB = 0x7ffffff0u;  // an offset past every resource

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Epilogues: what a tile does with its f32 accumulators.
//   EPI_F32        y[m][n] = acc (f32)
//   EPI_GELU_TANH  y[m][n] = f16(gelu_tanh(acc_gate) * acc_up)  (gated)
//   EPI_GELU_ERF   y[m][n] = f16(gelu_erf(acc_gate) * acc_up)   (gated)
//   EPI_RELU_F16   y[m][n] = f16(max(acc + bias[n], 0))
//   EPI_QKV        the fused [q | k | v] projection of a bidirectional
//                  encoder, scattered per head as f16 (see QkvHeads)
//   EPI_QKPREP     the decoder's [q | k | v] projection with qk_prep's
//                  work (per-head RMS norm, RoPE, query scale; q as f16
//                  rows, k and V^T into the f16 cache), head_dim 256
constexpr int EPI_F32 = 0, EPI_GELU_TANH = 1, EPI_GELU_ERF = 2, EPI_RELU_F16 = 3, EPI_QKV = 4, EPI_QKPREP = 5;

struct GemmArgs {
    const half_t* x;
    int64_t ldx, m;
    DevWeight w0, w1;  // w1: the up projection of the gated kernel
    void* y;
    int64_t ldy;
    const uint16_t* bias;  // f16 per output column (EPI_RELU_F16; EPI_QKV, may be null)
    QkvHeads qkv;          // EPI_QKV
    QkArgs qk;             // EPI_QKPREP (its qkv / qkv_stride unused)
    // Split K (EPI_F32): blockIdx.y = split z sums K range
    // [z K / ksplit, (z + 1) K / ksplit) into y + z * part_stride.
    int ksplit = 1;
    int64_t part_stride = 0;
    // EPI_F32 with FOLD: K pieces of kfold stages counted
    // from the split's first stage; see launch_gemm_splitk.
    int kfold = 0;
    // EPI_QKPREP: row tiles start at BM * i - mshift (0 <= mshift < BM)
    int64_t mshift = 0;
};

constexpr int RSRC_FLAGS = 0x00020000;  // raw (untyped) 32-bit buffer

__device__ inline __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
    const int64_t n = bytes < 0 ? 0 : (bytes > 0x7fffffff ? 0x7fffffff : bytes);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, int(n), RSRC_FLAGS);
}

__device__ inline int swz(int r) { return (r >> 1) & 7; }

// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding:
// vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ inline void wait_vm() {
    static_assert(N >= 0 && N <= 63, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// LDS operations done (s_waitcnt lgkmcnt(0), other counters left alone),
// then the workgroup barrier, between compiler fences for memory.  Written
// with builtins rather than inline assembly so that the compiler's own
// wait-count tracking knows the LDS counter is clear afterwards.
__device__ inline void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// matmul_gated.wgsl:117-129: exact GELU, 0.5 x (1 + erf(x / sqrt 2)), with
// erf from Abramowitz & Stegun 7.1.26 (|error| < 1.5e-7), the form the
// reference evaluates.
__device__ inline float gelu_erf(float x) {
    const float z = x * 0.7071067811865476f;
    const float a = fabsf(z);
    const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * a);
    const float poly = ((((1.061405429f * t - 1.453152027f) * t + 1.421413741f) * t - 0.284496736f) * t +
                        0.254829592f) * t;
    const float e = __builtin_amdgcn_exp2f(-a * a * 1.4426950408889634f);  // e^(-a^2)
    const float y = 1.0f - poly * e;
    return 0.5f * x * (1.0f + (z < 0.0f ? -y : y));
}

// matmul_gated.wgsl:126-134: tanh GELU with the argument clamped to +-15,
// through the identity 0.5 (1 + tanh z) = 1 / (1 + e^(-2z)) evaluated with
// the hardware exp2 and reciprocal.
__device__ inline float gelu_tanh(float x) {
    float z = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    z = fminf(15.0f, fmaxf(-15.0f, z));
    const float e = __builtin_amdgcn_exp2f(z * -2.8853900817779268f);  // e^(-2z)
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// ------------------------------------------------------ 32x32x16 tiles

// gemm32_kernel, on v_mfma_f32_32x32x16_f16, which issues at full rate on gfx950 with one or
// two accumulation chains per wave (16x16x32 needs about sixteen).  Row-
// owner scheme: each wave owns 32 * NJ weight rows across all BM = 32 * MI
// activation rows, so its weights are private to it and go straight from
// their stage tiles (kernels.h) into registers: per stage and row block
// one coalesced 16-byte-per-lane load of the packet (lane 32 h + r gets
// row r's four k-steps of half h) and one 4-byte load of the row's block
// scales.  Only the activation tile, which every wave reads, goes through
// LDS.  Per 64-wide K stage, four 16-wide steps: lane l supplies A = the
// decoded weight word of row l % 32 at k 16 s + 8 (l / 32) (one Q4 word,
// two Q8 words or 16 bytes of f16), B = X row l % 32 of each activation
// block at the same k (one 16-byte LDS read), and holds D for activation
// row l % 32 at weight rows 8 j + 4 (l / 32) + i: four consecutive output
// columns per j, stored as one vector.  The K order (stage, step) does not
// depend on the tile shape, so every dispatch gives every output element
// the same sums: rows of a pass are the same whatever else it holds.
//
// Pipeline, iteration kt (stage kt):
//   wait for stage kt + 1's X DMA (this wave's), barrier (everyone's; and
//       everyone has finished reading the ring slot of stage kt - 1);
//   DMA stage kt + NS - 1's X tile into that slot;
//   read stage kt + 1's X fragments from LDS into registers;
//   decode + MFMA stage kt (X fragments read one iteration earlier,
//       weights loaded NS - 1 iterations earlier);
//   load stage kt + NS - 1's weights into the register slot just used.
// Every wave issues the same memory instructions in every iteration (past
// the end they read empty resources), so the wait counts are constants.
template <int QUANT, int MI, int NJ, int EPI, int NS, int NW_ = 4, bool PAIR_ = false>
struct Cfg32 {
    static constexpr bool GATED = EPI == EPI_GELU_TANH || EPI == EPI_GELU_ERF;
    // PAIR: a gated tile whose waves hold one matrix each, the first half
    // the gate blocks and the second half the matching up blocks; the gate
    // sums go through LDS to the up waves, which finish the tile.
    static constexpr bool PAIR = PAIR_;
    static constexpr int NW = NW_, T = NW * WAVE;
    static constexpr int BM = 32 * MI;
    static constexpr int WR = 32 * NJ;                 // weight rows per wave
    static constexpr int BNW = NW * WR;                // weight rows per tile
    static constexpr int BN = GATED ? BNW / 2 : BNW;   // output columns per tile
    static constexpr int PM = BN / 32;                 // row blocks per matrix
    static constexpr int PK = tile_packet_bytes(QUANT);
    static constexpr int CL = PK / 1024;               // 16-byte code loads per row block and stage
    static constexpr int X_CH = BM * 8, X_I = (X_CH + T - 1) / T;
    static constexpr int WL = NJ * (CL + (QUANT == F16_DT ? 0 : 1));  // weight loads per wave and stage
    static constexpr int C = X_I + WL;                 // memory instructions per wave and stage
    static constexpr int R = NS - 1;                   // weight register slots
    static constexpr int U = R % 2 == 0 ? R : 2 * R;   // loop unroll: X fragments alternate two sets
    static constexpr int X_BYTES = X_I * T * 16;
    // EPI_QKPREP stages the f32 tile [BM][256] (rows padded to 260
    // floats), eight partial sums of squares and a scale per row in LDS
    // after the K loop.
    static constexpr int QK_LDS = EPI == EPI_QKPREP ? BM * (260 + 17) * 4 : 0;  // + [BM][16] sums, [BM] scales
    static constexpr int PAIR_LDS = PAIR ? (NW / 2) * MI * NJ * 16 * WAVE * 4 : 0;  // the gate waves' sums
    static constexpr int EPI_LDS = QK_LDS > PAIR_LDS ? QK_LDS : PAIR_LDS;           // LDS after the K loop
    static constexpr int LDS = NS * X_BYTES > EPI_LDS ? NS * X_BYTES : EPI_LDS;
    static_assert(EPI != EPI_QKPREP || (BN == 256 && (NW == 4 || NW == 8)),
                  "the q/k/v epilogue: one 256-wide head on four or eight waves");
    static_assert(LDS <= 160 * 1024, "ring larger than the LDS");
    static_assert(!PAIR || (GATED && NW % 2 == 0), "paired tiles: gated, gate and up waves in pairs");
    static_assert(!GATED || PAIR || NJ % 2 == 0, "gated tiles pair gate and up row blocks");
    static_assert(NS >= 3, "ring needs >= 3 slots: one read into registers, one landing, one in flight");
    static_assert(WL + (NS - 2) * C <= 63, "vmcnt range");
};

// The q/k/v epilogue (EPI_QKPREP) for row blocks C0 .. C0 + RB - 1 of a
// 256-column tile (one head); m0: the first row of those blocks; qpos: the
// rope row of each of the thread's rows (row p * NW * 2 + tid / 32 of the
// blocks at p).
constexpr int QK_TS = 260;  // floats per staged row
template <int MI, int NJ, int NW, int C0, int RB>
__device__ inline void finish_qkprep(const GemmArgs& g, const floatx16 (&acc)[MI][NJ], int64_t m0, int64_t n0,
                                     uint8_t* smem, int wave, int lane, const int* qpos) {
    // Every multiply-add that rounds once is an explicit fmaf and every
    // f16 comes from an f32 value (nothing for the compiler to fuse in
    // one tile shape and not another): a row's outputs are the same
    // bits from the four-wave and the eight-wave tile.
    // qk_prep.wgsl:66-114 on the tile's rows, without cross-lane
    // traffic: each lane's sums of squares over its 16 accumulators of
    // a row in each 32-column block go to LDS with the f32 tile (the
    // ring is free: every DMA landed, every read done); a row's RMS is
    // the sum of its sixteen partials (block, lane half) in a fixed
    // order, whichever wave held which block.  q and k heads: 32 threads per row,
    // thread c holding head dimensions 4c..4c+3 and their RoPE partners
    // 128 + 4c..: RMS norm with the head's weight, RoPE, query scale,
    // f16 q rows or k cache rows.  v head: (optional) RMS norm, then
    // the V^T tiles of the cache in whole 16-byte chunks of 8 keys, 8
    // lanes per 128-byte dimension row (the caller aligns the row tiles
    // to 32 cache rows, so every chunk belongs to one tile; at the
    // pass's edges a chunk keeps the cache's other keys).
    constexpr int HD = 256, TS = QK_TS, HALF = HD / 2, BM = 32 * RB, WR = 32 * NJ;
    constexpr int QK_RP = NW * WAVE / 32, QK_PASSES = BM / QK_RP;  // 32 threads per row
    const int tid = wave * WAVE + lane, lr = lane % 32, lh = lane / 32;
    const int64_t M = g.m;
    auto row_ok = [&](int64_t r) { return m0 + r >= 0 && m0 + r < M; };
    const QkArgs& a = g.qk;
    float* T = reinterpret_cast<float*>(smem);
    float* ssp = T + BM * TS;  // [BM][16] partial sums of squares
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float ss = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                *reinterpret_cast<float4*>(T + (i * 32 + lr) * TS + wave * WR + j * 32 + 8 * q + 4 * lh) =
                    make_float4(acc[C0 + i][j][4 * q], acc[C0 + i][j][4 * q + 1], acc[C0 + i][j][4 * q + 2], acc[C0 + i][j][4 * q + 3]);
#pragma unroll
                for (int r = 0; r < 4; ++r) ss = fmaf(acc[C0 + i][j][4 * q + r], acc[C0 + i][j][4 * q + r], ss);
            }
            ssp[(i * 32 + lr) * 16 + 2 * (wave * NJ + j) + lh] = ss;
        }
    const int slot = int(n0 / HD);
    const int H = a.heads, KV = a.kv_heads;
    const bool is_v = slot >= H + KV;
    const int c = tid % 32, d0 = 4 * c;
    // The rope pairs of every pass now, while the tile is staged.
    float4 r01[QK_PASSES], r23[QK_PASSES];
    if (!is_v) {
#pragma unroll
        for (int p = 0; p < QK_PASSES; ++p) {
            const float4* rt = reinterpret_cast<const float4*>(a.rope + int64_t(qpos[p]) * HALF + d0);
            r01[p] = rt[0];
            r23[p] = rt[1];
        }
    }
    lds_barrier();
    // Each row's scale once, from the sum of its sixteen partials in
    // order; the passes below read it.
    float* rinv = ssp + BM * 16;  // [BM] row scales
    if (tid < BM) {
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k) ss += ssp[tid * 16 + k];
        rinv[tid] = 1.0f / sqrtf(ss / float(HD) + a.eps);
    }
    lds_barrier();
    if (!is_v) {
        const bool is_q = slot < H;
        const int head = is_q ? slot : slot - H;
        const float* wn = is_q ? a.q_norm : a.k_norm;
        const float4 wl = *reinterpret_cast<const float4*>(wn + d0), wh = *reinterpret_cast<const float4*>(wn + HALF + d0);
        const float w_lo[4] = {wl.x, wl.y, wl.z, wl.w}, w_hi[4] = {wh.x, wh.y, wh.z, wh.w};
        const float sc = is_q ? a.q_scale : 1.0f;
        const int rot = int(a.rope_dims / 2);
#pragma unroll
        for (int p = 0; p < QK_PASSES; ++p) {
            const int r = p * QK_RP + tid / 32;
            if (!row_ok(r)) continue;
            const float inv = rinv[r];
            const float4 vl = *reinterpret_cast<const float4*>(T + r * TS + d0);
            const float4 vh = *reinterpret_cast<const float4*>(T + r * TS + HALF + d0);
            const float v_lo[4] = {vl.x, vl.y, vl.z, vl.w}, v_hi[4] = {vh.x, vh.y, vh.z, vh.w};
            const float cs[4] = {r01[p].x, r01[p].z, r23[p].x, r23[p].z};
            const float sn[4] = {r01[p].y, r01[p].w, r23[p].y, r23[p].w};
            float o_lo[4], o_hi[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float y0 = v_lo[k] * inv * w_lo[k], y1 = v_hi[k] * inv * w_hi[k];
                if (d0 + k < rot) {
                    o_lo[k] = fmaf(y0, cs[k], -(y1 * sn[k]));
                    o_hi[k] = fmaf(y1, cs[k], y0 * sn[k]);
                } else {
                    o_lo[k] = y0;
                    o_hi[k] = y1;
                }
            }
            const int64_t tok = m0 + r, row = a.base + tok;
            half_t* dst = is_q ? a.q16 + (tok * H + head) * HD : a.kc + (int64_t(head) * a.cap_pad + row) * HD;
            *reinterpret_cast<half4*>(dst + d0) =
                half4{f16_rounded(o_lo[0] * sc), f16_rounded(o_lo[1] * sc), f16_rounded(o_lo[2] * sc),
                      f16_rounded(o_lo[3] * sc)};
            *reinterpret_cast<half4*>(dst + HALF + d0) =
                half4{f16_rounded(o_hi[0] * sc), f16_rounded(o_hi[1] * sc), f16_rounded(o_hi[2] * sc),
                      f16_rounded(o_hi[3] * sc)};
        }
        return;
    }
    // V head: per 32-key half of the tile, item (dim, chunk cc) for
    // 256 dims x 4 chunks; chunk 4 hf + cc of a 64-key cache tile holds
    // keys 32 hf + 4 cc + {0..3, 16..19} (vt_col).
    const int head = slot - H - KV;
#pragma unroll
    for (int hh = 0; hh < BM / 32; ++hh) {
        const int64_t kh = a.base + m0 + 32 * hh;  // first cache row of this half (a multiple of 32)
        if (m0 + 32 * hh + 32 <= 0 || m0 + 32 * hh >= M) continue;
        const int64_t t0 = kh / 64 * 64;
        const int hf = int((kh % 64) / 32);
#pragma unroll
        for (int u = 0; u < 1024 / (NW * WAVE); ++u) {
            const int item = tid + NW * WAVE * u;
            const int dim = item / 4, cc = item % 4;
            half_t* dst = a.vt + ((int64_t(head) * (a.cap_pad / 64) + t0 / 64) * HD + dim) * 64 + 8 * (4 * hf + cc);
            half_t h[8];
            bool all = true;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int r = 32 * hh + 4 * cc + 16 * (e / 4) + e % 4;  // tile row of key e
                const bool in = row_ok(r);
                all = all && in;
                const float v = T[r * TS + dim];
                h[e] = f16_rounded(a.v_norm ? v * rinv[r] : v);
            }
            if (!all) {
                // a pass edge: the chunk's other keys keep the cache's values
                const half8 old = *reinterpret_cast<const half8*>(dst);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int r = 32 * hh + 4 * cc + 16 * (e / 4) + e % 4;
                    if (!row_ok(r)) h[e] = old[e];
                }
            }
            *reinterpret_cast<half8*>(dst) = half8{h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7]};
        }
    }
}

// A pair of four-value f16 groups, columns c .. c + 3 in lanes l < 32 and
// c + 4 .. c + 7 in lanes l + 32 for group a (c) and group b (c + 8), turned
// into eight consecutive columns per lane: c .. c + 7 of the row in lanes
// l < 32, c + 8 .. c + 15 in lanes l + 32.
__device__ inline uint4 wide8(half4 a, half4 b) {
    const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
    const auto x = __builtin_amdgcn_permlane32_swap(ua.x, ub.x, false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(ua.y, ub.y, false, false);
    return uint4{uint32_t(x[0]), uint32_t(y[0]), uint32_t(x[1]), uint32_t(y[1])};
}

// What the 32x32 tiles do with their sums: lane (lr, lh) holds, for
// activation row m0 + 32 i + lr, columns nw0 + 32 j + 8 q + 4 lh + 0..3 of
// weight block j in elements 4 q .. 4 q + 3 (gated: blocks NJ / 2 .. of the
// up matrix).  Every f16 is converted from a value first rounded to f32 and
// every multiply-add that rounds once is an explicit fmaf, so the outputs of
// a row do not depend on the tile shape that computed it.
template <int MI, int NJ, int EPI, bool W8 = false>
__device__ inline void finish32(const GemmArgs& g, const floatx16 (&acc)[MI][NJ], int64_t m0, int64_t nw0, int lane) {
    constexpr bool GATED = EPI == EPI_GELU_TANH || EPI == EPI_GELU_ERF;
    constexpr int NO = GATED ? NJ / 2 : NJ;
    const int lr = lane % 32, lh = lane / 32;
    const int64_t M = g.m, N = g.w0.rows;
    if constexpr (EPI == EPI_QKV) {
        // The wave's 64 columns are one head of q, k or v.  RoPE pairs dims
        // (c, c + 32): blocks 0 and 1 of the same lane and element.
        static_assert(NJ == 2, "one 64-wide head per wave");
        const QkvHeads& o = g.qkv;
        if (nw0 >= N) return;
        const int sec = int(nw0 / o.dq);
        const int64_t head = (nw0 % o.dq) / 64;
        float bias[2][16];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                bias[j][e] = g.bias ? float(__builtin_bit_cast(half_t, g.bias[nw0 + 32 * j + 8 * (e / 4) + 4 * lh + e % 4]))
                                    : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int64_t m = m0 + 32 * i + lr;
            const bool live = m >= 0 && m < M;
            float v[2][16];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) v[j][e] = acc[i][j][e] + bias[j][e];
            if (sec < 2) {
                if (o.rope) {
                    // rope_bi.wgsl:30-49: a' = a cos - b sin, b' = b cos + a sin,
                    // each with a's product inside the fmaf (the other order
                    // moves one q or k in 20,000 by an f16 ulp, which the
                    // encoder's 22 layers turn into 1e-3 of its logits).
                    const float2* rp = o.rope + int64_t(live ? o.meta[4 * m] : 0) * 32 + 4 * lh;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 c01 = *reinterpret_cast<const float4*>(rp + 8 * q);
                        const float4 c23 = *reinterpret_cast<const float4*>(rp + 8 * q + 2);
                        const float cs[4] = {c01.x, c01.z, c23.x, c23.z}, sn[4] = {c01.y, c01.w, c23.y, c23.w};
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float a = v[0][4 * q + r], b = v[1][4 * q + r];
                            v[0][4 * q + r] = fmaf(a, cs[r], -(b * sn[r]));
                            v[1][4 * q + r] = fmaf(a, sn[r], b * cs[r]);
                        }
                    }
                }
                const float sc = sec == 0 ? o.qscale : 1.0f;
                half_t* dst = (sec == 0 ? o.q16 : o.k16) + (head * o.tpad + m) * 64;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; q += 2) {
                        half4 h[2];
#pragma unroll
                        for (int u = 0; u < 2; ++u)
                            h[u] = half4{f16_rounded(v[j][4 * (q + u)] * sc), f16_rounded(v[j][4 * (q + u) + 1] * sc),
                                         f16_rounded(v[j][4 * (q + u) + 2] * sc), f16_rounded(v[j][4 * (q + u) + 3] * sc)};
                        const uint4 w = wide8(h[0], h[1]);
                        if (live) *reinterpret_cast<uint4*>(dst + 32 * j + 8 * (q + lh)) = w;
                    }
            } else {
                // V^T: lanes 2 k and 2 k + 1 hold neighbouring keys of a
                // dimension, two f16 of one word; the even lane writes the
                // pair of one dimension, the odd lane the next one's.
                half_t* dst = o.vt + (head * (o.tpad / 32) + m / 32) * (64 * 32) + vt_col32(lr & ~1);
                const bool odd = lane & 1;
                const bool pair = __shfl_xor(int(live), 1, WAVE) && live;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; e += 2) {
                        const uint32_t a = __builtin_bit_cast(uint16_t, f16_rounded(v[j][e]));
                        const uint32_t b = __builtin_bit_cast(uint16_t, f16_rounded(v[j][e + 1]));
                        const int dim = 32 * j + 8 * (e / 4) + 4 * lh + e % 4;
                        const uint32_t got = uint32_t(__builtin_amdgcn_update_dpp(0, int(odd ? a : b), 0xb1, 0xf, 0xf, false));
                        const uint32_t w = odd ? (got | b << 16) : (a | got << 16);
                        if (pair) {
                            *reinterpret_cast<uint32_t*>(dst + (dim + int(odd)) * 32) = w;
                        } else if (live) {  // the pass's last key: alone
                            dst[dim * 32 + int(odd)] = __builtin_bit_cast(half_t, uint16_t(a));
                            dst[(dim + 1) * 32 + int(odd)] = __builtin_bit_cast(half_t, uint16_t(b));
                        }
                    }
            }
        }
        return;
    }
    float cbias[EPI == EPI_RELU_F16 ? NO : 1][16];
    if constexpr (EPI == EPI_RELU_F16) {
#pragma unroll
        for (int j = 0; j < NO; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t n = nw0 + 32 * j + 8 * (e / 4) + 4 * lh + e % 4;
                cbias[j][e] = n < N ? float(__builtin_bit_cast(half_t, g.bias[n])) : 0.0f;
            }
    }
    auto value = [&](int i, int j, int x) {
        if constexpr (EPI == EPI_GELU_TANH)
            return gelu_tanh(acc[i][j][x]) * acc[i][j + NJ / 2][x];
        else if constexpr (EPI == EPI_GELU_ERF)
            return gelu_erf(acc[i][j][x]) * acc[i][j + NJ / 2][x];
        else if constexpr (EPI == EPI_RELU_F16)
            return fmaxf(acc[i][j][x] + cbias[j][x], 0.0f);
        else
            return acc[i][j][x];
    };
    // f16 rows: whole 32-column blocks of 16-byte-aligned rows go out eight
    // columns per store, others as the lane's own four.
    const bool aligned = EPI != EPI_F32 && g.ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(g.y) & 15) == 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int64_t m = m0 + 32 * i + lr;
        const bool live = m >= 0 && m < M;
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int64_t n0 = nw0 + 32 * j;
            if constexpr (EPI == EPI_F32) {
                if (!live) continue;
                float* dst = static_cast<float*>(g.y) + int64_t(blockIdx.y) * g.part_stride + m * g.ldy;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int64_t n = n0 + 8 * q + 4 * lh;
                    if (n + 3 < N) {
                        *reinterpret_cast<float4*>(dst + n) = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                                          acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (n + r < N) dst[n + r] = acc[i][j][4 * q + r];
                    }
                }
            } else if (W8 && aligned && n0 + 32 <= N) {
                half_t* dst = static_cast<half_t*>(g.y) + m * g.ldy;
#pragma unroll
                for (int q = 0; q < 4; q += 2) {
                    half4 h[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int r = 0; r < 4; ++r) h[u][r] = f16_rounded(value(i, j, 4 * (q + u) + r));
                    const uint4 w = wide8(h[0], h[1]);
                    if (live) *reinterpret_cast<uint4*>(dst + n0 + 8 * (q + lh)) = w;
                }
            } else {
                if (!live) continue;
                half_t* dst = static_cast<half_t*>(g.y) + m * g.ldy;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int64_t n = n0 + 8 * q + 4 * lh;
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = value(i, j, 4 * q + r);
                    if (n + 3 < N) {
                        *reinterpret_cast<half4*>(dst + n) =
                            half4{f16_rounded(v[0]), f16_rounded(v[1]), f16_rounded(v[2]), f16_rounded(v[3])};
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (n + r < N) dst[n + r] = f16_rounded(v[r]);
                    }
                }
            }
        }
    }
}

template <class F, size_t... I>
__device__ inline bool run_phases(F& f, std::index_sequence<I...>) {
    return (f(std::integral_constant<int, int(I)>{}) && ...);
}

template <class F, size_t... I>
__device__ inline void run_all(F& f, std::index_sequence<I...>) {
    (f(std::integral_constant<int, int(I)>{}), ...);
}

// f(phase) for nk stages, phase = stage % U; f returns whether a stage is
// left.  Whole groups of U without an exit among them, then the rest: with
// an exit after every stage the compiler gave the loop one latch for all of
// them, could no longer tell which stages' loads were out at the loop head,
// and waited there for nearly all of them (vmcnt 0 to 4), once every U
// stages.
template <int U, class F>
__device__ inline void run_stages(F& f, int nk) {
    for (int n = nk / U; n > 0; --n) run_all(f, std::make_index_sequence<U>{});
    if (nk % U) run_phases(f, std::make_index_sequence<U>{});
}

// XR (resident X): the workgroup's whole X tile (BM rows x its K range)
// lands in LDS in the prologue, one slot per stage, and the K loop runs
// with no barrier and no X wait (the weights are each wave's own).  Same
// MFMA sequence, same sums; chosen per launch when the tile fits.
template <int QUANT, int MI, int NJ, int EPI, int NS, int NW_, bool FOLD, bool XR, bool PAIR>
__global__ __launch_bounds__(NW_ * WAVE) void gemm32_kernel(GemmArgs g) {
    using P = Cfg32<QUANT, MI, NJ, EPI, NS, NW_, PAIR>;
    static_assert(!FOLD || EPI == EPI_F32, "K chunks: f32 products only");
    constexpr bool GATED = P::GATED;
    constexpr int NW = P::NW, BM = P::BM, BN = P::BN, WR = P::WR, PK = P::PK, PM = P::PM, R = P::R;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = int(threadIdx.x), lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);

    // XCD-aware tile order: workgroups reach the eight XCDs in turn, so each
    // XCD is given a contiguous run of tiles (which share rows in its L2).
    // Row tiles start at BM * i - mshift (mshift < BM: the first tile is
    // short), so a caller can align the tiles to its own row grid.
    const int64_t N = g.w0.rows, K = g.w0.cols, M = g.m;
    const int ntn = int((N + BN - 1) / BN);
    const int ntiles = ntn * int((M + g.mshift + BM - 1) / BM);
    const int per_xcd = int(gridDim.x) / 8;
    const int tile = (int(blockIdx.x) % 8) * per_xcd + int(blockIdx.x) / 8;
    if (tile >= ntiles) return;
    const int64_t n0 = int64_t(tile % ntn) * BN, m0 = int64_t(tile / ntn) * BM - g.mshift;
    const int kbeg = int(blockIdx.y) * int(K / g.ksplit);
    const int nk = int((K / g.ksplit + G_BK - 1) / G_BK);
    const int K32 = int(K);
    auto row_ok = [&](int64_t r) { return m0 + r >= 0 && m0 + r < M; };  // tile row r is a row of the pass

    // X lanes: row m0 + r of the whole matrix (rows before 0 or from M on
    // are out of range, so they read as zeros).
    uint32_t xoff[P::X_I];
    int xcol[P::X_I];
#pragma unroll
    for (int i = 0; i < P::X_I; ++i) {
        const int slot = (i * NW + wave) * WAVE + lane;
        const int r = slot / 8, lc = (slot % 8) ^ swz(r);
        xcol[i] = lc * 8;
        xoff[i] = slot < P::X_CH && row_ok(r) ? uint32_t(((m0 + r) * g.ldx + lc * 8) * 2) : OOB;
    }

    // This wave's row blocks: j < NJ / 2 of the gate matrix and the rest of
    // the up matrix when gated (PAIR: all NJ of the gate matrix in the
    // first half of the waves, of the up matrix in the second, wave w and
    // w + NW / 2 on the same blocks).  Block j's packet of stage st sits at
    // st * PK + bj * stages * PK from the matrix's first block of the tile.
    const int64_t stages = g.w0.stages, rblocks = (N + 31) / 32, rb0 = n0 / 32;
    const int64_t live_blocks = rblocks - rb0;  // > 0: the tile starts inside N
    const int pw = PAIR ? wave % (NW / 2) : wave;  // the wave's place among the waves of its matrix
    auto mat_of = [&](int j) { return PAIR ? (wave >= NW / 2 ? 1 : 0) : (GATED && j >= NJ / 2 ? 1 : 0); };
    auto blk_of = [&](int j) {
        return PAIR ? pw * NJ + j : (GATED ? wave * (NJ / 2) + (j % (NJ / 2)) : wave * NJ + j);
    };
    uint32_t coff[NJ], scoff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        coff[j] = blk_of(j) < live_blocks ? uint32_t(blk_of(j) * stages * PK + lane * (PK / 64)) : OOB;
        scoff[j] = blk_of(j) < live_blocks ? uint32_t(blk_of(j) * stages * TILE_SCALE_BYTES + (lane % 32) * 4) : OOB;
    }

    // Stages past the end repeat the last one (in range, never consumed),
    // so the resources and lane offsets stay the same for every stage and
    // only the scalar stage offset moves.
    auto slot_base = [&](int s) { return smem + (XR ? unsigned(s) : unsigned(s) % unsigned(NS)) * P::X_BYTES; };
    const int last = nk - 1;
    const int64_t xbytes = M * g.ldx * 2;
    const bool ktail = (K32 & (G_BK - 1)) != 0;  // K % 64 == 32: the last stage masks lanes
    // X tile of stage s into its ring slot.
    auto issue_x = [&](int s) {
        uint8_t* base = slot_base(s);
        const int k0 = __builtin_amdgcn_readfirstlane(kbeg + (s < last ? s : last) * G_BK);  // a scalar offset
        const bool tail = ktail && k0 + G_BK > K32;
#pragma unroll
        for (int i = 0; i < P::X_I; ++i) {
            const uint32_t o = tail && xcol[i] >= K32 - k0 ? OOB : xoff[i];
            const __amdgpu_buffer_rsrc_t r = rsrc(g.x, xbytes);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(base + (i * NW + wave) * WAVE * 16), 16, o,
                                                     k0 * 2, 0, 0);
        }
    };

    // A stage's weights in registers.
    struct WRegs {
        uint4 code[NJ][P::CL];
        uint32_t sc[NJ];
    };
    const int st0 = kbeg / G_BK;  // this split's first stage
    auto issue_w = [&](int s, WRegs& w) {
        const int st = __builtin_amdgcn_readfirstlane(st0 + (s < last ? s : last));
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const DevWeight& wt = mat_of(j) ? g.w1 : g.w0;
            const __amdgpu_buffer_rsrc_t r = rsrc(wt.tiles + rb0 * stages * PK, live_blocks * stages * PK);
#pragma unroll
            for (int c = 0; c < P::CL; ++c)
                w.code[j][c] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             r, coff[j] + 16 * c, st * PK, 0));
            if constexpr (QUANT != F16_DT) {
                const __amdgpu_buffer_rsrc_t rs = rsrc(wt.tscales + rb0 * stages * TILE_SCALE_BYTES,
                                                       live_blocks * stages * TILE_SCALE_BYTES);
                w.sc[j] = __builtin_amdgcn_raw_buffer_load_b32(rs, scoff[j], st * TILE_SCALE_BYTES, 0);
            }
        }
    };

    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};
    // FOLD: the products of each K piece (g.kfold stages) accumulate from
    // zero in acc and the piece sums are added into tot in K order — the
    // sums of a pass that runs every piece in a workgroup of its own and
    // adds the partials in order (the residual norm's runs).
    floatx16 tot[FOLD ? MI : 1][FOLD ? NJ : 1];
    int kleft = g.kfold;  // stages left in the current piece (FOLD)
    bool folded = false;
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                tot[i][j] = folded ? tot[i][j] + acc[i][j] : acc[i][j];
                acc[i][j] = floatx16{};
            }
        folded = true;
    };

    const int lr = lane % 32, lh = lane / 32;
    int foff[4];  // the lane's X fragment offset within a 32-row block, per k-step
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) foff[ks] = lr * G_ROW + (((2 * ks + lh) ^ swz(lr)) * 16);

    struct XRegs {
        half8 x[4][MI];
    };
    auto read_x = [&](int s, XRegs& f) {
        const uint8_t* X = slot_base(s);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int i = 0; i < MI; ++i) f.x[ks][i] = *reinterpret_cast<const half8*>(X + i * 32 * G_ROW + foff[ks]);
    };
    auto compute = [&](const XRegs& f, const WRegs& w) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            half8 wf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if constexpr (QUANT == F16_DT) {
                    wf[j] = __builtin_bit_cast(half8, w.code[j][ks]);
                } else {
                    // k-steps 0, 1 are the stage's first block, 2, 3 its second
                    const half_t d = __builtin_bit_cast(half_t, uint16_t(w.sc[j] >> (16 * (ks / 2))));
                    if constexpr (QUANT == Q4_DT) {
                        const uint4 u = w.code[j][0];
                        const uint32_t word = ks == 0 ? u.x : ks == 1 ? u.y : ks == 2 ? u.z : u.w;
                        wf[j] = dq4_word(word, half2v{d, d});
                    } else {
                        const uint4 u = w.code[j][ks / 2];
                        wf[j] = ks % 2 == 0 ? dq8_words(u.x, u.y, half2v{d, d}) : dq8_words(u.z, u.w, half2v{d, d});
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[j], f.x[ks][i], acc[i][j], 0, 0, 0);
        }
    };

    // EPI_QKPREP, q and k heads: the rope rows of the rows this thread
    // finishes (RP rows per pass of the workgroup, row p * RP + tid / 32),
    // loaded now so their latency hides behind the K loop.  Every thread
    // loads the position of a row of the pass (its own row, clamped into the
    // pass); rows outside the pass and the v head take position 0 in
    // clamp_pos, once the first stages have landed: with the choice made
    // here the compiler put each load in a branch of its own with its wait.
    constexpr int QK_RP = NW * WAVE / 32;  // rows per pass: 32 threads per row
    constexpr int QK_PASSES = EPI == EPI_QKPREP ? BM / QK_RP : 1;
    int qpos[QK_PASSES];
    if constexpr (EPI == EPI_QKPREP) {
#pragma unroll
        for (int p = 0; p < QK_PASSES; ++p) {
            const int r = p * QK_RP + tid / 32;
            const int64_t m = m0 + r < 0 ? 0 : (m0 + r < M ? m0 + r : M - 1);
            qpos[p] = g.qk.meta[4 * (g.qk.base + m)];
        }
    }
    auto clamp_pos = [&] {
        if constexpr (EPI == EPI_QKPREP) {
            const bool qk_head = n0 / 256 < g.qk.heads + g.qk.kv_heads;
#pragma unroll
            for (int p = 0; p < QK_PASSES; ++p) asm volatile("" : "+v"(qpos[p]));
#pragma unroll
            for (int p = 0; p < QK_PASSES; ++p) {
                const int v = qpos[p] < 0 ? 0 : (qpos[p] >= g.qk.rope_rows ? int(g.qk.rope_rows - 1) : qpos[p]);
                qpos[p] = qk_head && row_ok(p * QK_RP + tid / 32) ? v : 0;
            }
        }
    };

    WRegs wr[R];
    XRegs xa, xb;
    int kt = 0;
    if constexpr (XR) {
        // Prologue: every stage's X, then weight stages 0 .. R - 1; all of
        // it landed (everyone's X: one barrier), then stage 0's fragments.
        for (int s = 0; s < nk; ++s) issue_x(s);
#pragma unroll
        for (int s = 0; s < R; ++s) issue_w(s, wr[s]);
        wait_vm<0>();
        clamp_pos();
        lds_barrier();
        read_x(0, xa);
        auto xstep = [&](auto phase) {
            constexpr int PH = decltype(phase)::value;
            XRegs& cur = PH % 2 == 0 ? xa : xb;
            XRegs& nxt = PH % 2 == 0 ? xb : xa;
            // Stage kt's weights (issued R iterations ago) landed: at most
            // the R - 1 later stages' loads are still out.
            wait_vm<(R - 1) * P::WL>();
            if (kt + 1 < nk) read_x(kt + 1, nxt);
            compute(cur, wr[PH % R]);
            issue_w(kt + R, wr[PH % R]);
            if constexpr (FOLD) {
                if (--kleft == 0 || kt + 1 == nk) {
                    kleft = g.kfold;
                    fold();
                }
            }
            return ++kt < nk;
        };
        run_stages<P::U>(xstep, nk);
    }
    // Prologue: stages 0 .. NS - 2 in the same order as the loop issues
    // them (X, then weights), then stage 0's X fragments.
    if constexpr (!XR) {
#pragma unroll
    for (int s = 0; s < R; ++s) {
        issue_x(s);
        issue_w(s, wr[s]);
    }
    wait_vm<P::WL + (NS - 2) * P::C>();
    clamp_pos();
    lds_barrier();
    read_x(0, xa);
    }
    auto step = [&](auto phase) {
        constexpr int PH = decltype(phase)::value;
        XRegs& cur = PH % 2 == 0 ? xa : xb;
        XRegs& nxt = PH % 2 == 0 ? xb : xa;
        // Stage kt + 1's X landed: after it this wave issued its weights
        // and NS - 3 whole stages.
        wait_vm<P::WL + (NS - 3) * P::C>();
        lds_barrier();
        issue_x(kt + NS - 1);
        if (kt + 1 < nk) read_x(kt + 1, nxt);
        compute(cur, wr[PH % R]);
        issue_w(kt + NS - 1, wr[PH % R]);
        if constexpr (FOLD) {
            if (--kleft == 0 || kt + 1 == nk) {
                kleft = g.kfold;
                fold();
            }
        }
        return ++kt < nk;
    };
    if constexpr (!XR) {
        run_stages<P::U>(step, nk);
    }
    wait_vm<0>();
    if constexpr (FOLD) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = tot[i][j];
    }

    if constexpr (EPI == EPI_QKPREP) {
        finish_qkprep<MI, NJ, NW, 0, MI>(g, acc, m0, n0, smem, wave, lane, qpos);
        return;
    }

    // PAIR: the gate waves' sums to the up waves, element for element (the
    // same lane layout), through LDS that every wave has finished with.
    if constexpr (PAIR) {
        float* E = reinterpret_cast<float*>(smem);
        lds_barrier();
        if (wave < NW / 2) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) E[(((pw * MI + i) * NJ + j) * 16 + e) * WAVE + lane] = acc[i][j][e];
        }
        lds_barrier();
        if (wave < NW / 2) return;
        floatx16 both[MI][2 * NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                both[i][NJ + j] = acc[i][j];
#pragma unroll
                for (int e = 0; e < 16; ++e) both[i][j][e] = E[(((pw * MI + i) * NJ + j) * 16 + e) * WAVE + lane];
            }
        finish32<MI, 2 * NJ, EPI>(g, both, m0, n0 + pw * WR, lane);
    } else if constexpr (EPI != EPI_QKPREP) {
        finish32<MI, NJ, EPI>(g, acc, m0, n0 + (GATED ? wave * (WR / 2) : wave * WR), lane);
    }
}

// Wide tiles for long passes: the same products, operand layouts and K order
// as gemm32_kernel (so the same sums), with 128 x 64 results per wave.  A
// 32-row block per wave reads each X fragment from LDS for one MFMA, which
// takes the LDS its whole bandwidth; two blocks halve that and share the
// decode over four row blocks.  The accumulators take half the registers,
// so the X fragments and the decoded weights are double buffered one k-step
// (16 K) at a time instead of a stage.  Iteration kt, k-step ks:
//   read the fragments and decode the weights of the next k-step (of stage
//   kt + 1 after a wait for its X DMA and a barrier, which also frees stage
//   kt's ring slot: the DMA of stage kt + NS goes out), between the MFMAs
//   of this one; after the last decode, load stage kt + 2's weights.
template <int QUANT, int MI, int NJ, int EPI, int NS, int NW_, bool FOLD>
__global__ __launch_bounds__(NW_ * WAVE, 2) void gemm32w_kernel(GemmArgs g) {
    using P = Cfg32<QUANT, MI, NJ, EPI, NS, NW_, false>;
    constexpr bool GATED = P::GATED;
    constexpr int NW = P::NW, BM = P::BM, BN = P::BN, WR = P::WR, PK = P::PK;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = int(threadIdx.x), lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int64_t N = g.w0.rows, K = g.w0.cols, M = g.m;
    const int ntn = int((N + BN - 1) / BN);
    const int ntiles = ntn * int((M + g.mshift + BM - 1) / BM);
    const int per_xcd = int(gridDim.x) / 8;
    const int tile = (int(blockIdx.x) % 8) * per_xcd + int(blockIdx.x) / 8;
    if (tile >= ntiles) return;
    const int64_t n0 = int64_t(tile % ntn) * BN, m0 = int64_t(tile / ntn) * BM - g.mshift;
    const int kbeg = int(blockIdx.y) * int(K / g.ksplit);
    const int nk = int((K / g.ksplit + G_BK - 1) / G_BK);
    const int K32 = int(K), last = nk - 1;

    uint32_t xoff[P::X_I];
    int xcol[P::X_I];
#pragma unroll
    for (int i = 0; i < P::X_I; ++i) {
        const int slot = (i * NW + wave) * WAVE + lane;
        const int r = slot / 8, lc = (slot % 8) ^ swz(r);
        xcol[i] = lc * 8;
        xoff[i] = slot < P::X_CH && m0 + r >= 0 && m0 + r < M ? uint32_t(((m0 + r) * g.ldx + lc * 8) * 2) : OOB;
    }
    const int64_t stages = g.w0.stages, rblocks = (N + 31) / 32, rb0 = n0 / 32;
    const int64_t live_blocks = rblocks - rb0;
    auto mat_of = [&](int j) { return GATED && j >= NJ / 2 ? 1 : 0; };
    auto blk_of = [&](int j) { return GATED ? wave * (NJ / 2) + (j % (NJ / 2)) : wave * NJ + j; };
    uint32_t coff[NJ], scoff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        coff[j] = blk_of(j) < live_blocks ? uint32_t(blk_of(j) * stages * PK + lane * (PK / 64)) : OOB;
        scoff[j] = blk_of(j) < live_blocks ? uint32_t(blk_of(j) * stages * TILE_SCALE_BYTES + (lane % 32) * 4) : OOB;
    }
    auto slot_base = [&](int s) { return smem + (unsigned(s) % unsigned(NS)) * P::X_BYTES; };
    const int64_t xbytes = M * g.ldx * 2;
    const bool ktail = (K32 & (G_BK - 1)) != 0;
    auto issue_x = [&](int s) {
        uint8_t* base = slot_base(s);
        const int k0 = __builtin_amdgcn_readfirstlane(kbeg + (s < last ? s : last) * G_BK);
        const bool tail = ktail && k0 + G_BK > K32;
#pragma unroll
        for (int i = 0; i < P::X_I; ++i) {
            const uint32_t o = tail && xcol[i] >= K32 - k0 ? OOB : xoff[i];
            const __amdgpu_buffer_rsrc_t r = rsrc(g.x, xbytes);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(base + (i * NW + wave) * WAVE * 16), 16, o,
                                                     k0 * 2, 0, 0);
        }
    };
    struct WRegs {
        uint4 code[NJ][P::CL];
        uint32_t sc[NJ];
    };
    const int st0 = kbeg / G_BK;
    auto issue_w = [&](int s, WRegs& w) {
        const int st = __builtin_amdgcn_readfirstlane(st0 + (s < last ? s : last));
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const DevWeight& wt = mat_of(j) ? g.w1 : g.w0;
            const __amdgpu_buffer_rsrc_t r = rsrc(wt.tiles + rb0 * stages * PK, live_blocks * stages * PK);
#pragma unroll
            for (int c = 0; c < P::CL; ++c)
                w.code[j][c] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             r, coff[j] + 16 * c, st * PK, 0));
            if constexpr (QUANT != F16_DT) {
                const __amdgpu_buffer_rsrc_t rs = rsrc(wt.tscales + rb0 * stages * TILE_SCALE_BYTES,
                                                       live_blocks * stages * TILE_SCALE_BYTES);
                w.sc[j] = __builtin_amdgcn_raw_buffer_load_b32(rs, scoff[j], st * TILE_SCALE_BYTES, 0);
            }
        }
    };
    // The memory instructions' order (X of a stage, then weights) is what the
    // wait counts rely on: compiler fences keep it.
    auto fence = [] { asm volatile("" ::: "memory"); };

    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};
    // FOLD: K pieces of g.kfold stages from zero, added in K order (as in
    // gemm32_kernel).
    floatx16 tot[FOLD ? MI : 1][FOLD ? NJ : 1];
    bool folded = false;
    int kleft = g.kfold;
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                tot[i][j] = folded ? tot[i][j] + acc[i][j] : acc[i][j];
                acc[i][j] = floatx16{};
            }
        folded = true;
    };
    const int lr = lane % 32, lh = lane / 32;
    int foff[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) foff[ks] = lr * G_ROW + (((2 * ks + lh) ^ swz(lr)) * 16);

    struct Frag {
        half8 x[MI], w[NJ];
    };
    auto read_x = [&](int s, int ks, Frag& f) {
        const uint8_t* X = slot_base(s);
#pragma unroll
        for (int i = 0; i < MI; ++i) f.x[i] = *reinterpret_cast<const half8*>(X + i * 32 * G_ROW + foff[ks]);
    };
    auto decode = [&](const WRegs& w, int ks, Frag& f) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (QUANT == F16_DT) {
                f.w[j] = __builtin_bit_cast(half8, w.code[j][ks]);
            } else {
                const half_t d = __builtin_bit_cast(half_t, uint16_t(w.sc[j] >> (16 * (ks / 2))));
                if constexpr (QUANT == Q4_DT) {
                    const uint4 u = w.code[j][0];
                    f.w[j] = dq4_word(ks == 0 ? u.x : ks == 1 ? u.y : ks == 2 ? u.z : u.w, half2v{d, d});
                } else {
                    const uint4 u = w.code[j][ks / 2];
                    f.w[j] = ks % 2 == 0 ? dq8_words(u.x, u.y, half2v{d, d}) : dq8_words(u.z, u.w, half2v{d, d});
                }
            }
        }
    };
    auto mfmas = [&](const Frag& f) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[j], f.x[i], acc[i][j], 0, 0, 0);
    };

    constexpr int VPM = (NJ * (QUANT == F16_DT ? 0 : 14) + MI * NJ - 1) / (MI * NJ) + 1;  // decode per MFMA
    WRegs wr[2];
    Frag fa, fb;
    issue_x(0);
    fence();
#pragma unroll
    for (int s = 1; s < NS; ++s) {
        issue_x(s);
        fence();
        if (s >= NS - 2) {
            issue_w(s - (NS - 2), wr[s - (NS - 2)]);
            fence();
        }
    }
    wait_vm<(NS - 1) * P::X_I>();  // stage 0's X: at least the other stages' follow it
    lds_barrier();
    read_x(0, 0, fa);
    decode(wr[0], 0, fa);
    int kt = 0;
    auto step = [&](auto phase) {
        constexpr int PH = decltype(phase)::value;
        WRegs& cw = wr[PH];
        WRegs& nw = wr[1 - PH];
        // One k-step: the next one's fragment reads first, its decode spread
        // between this one's MFMAs; nothing moves across its ends (the
        // compiler would otherwise pull a later decode, and with it the wait
        // for its weights, ahead of these MFMAs).
        auto kstep = [&](const WRegs& w, int s, int ks, const Frag& cur, Frag& nxt) {
            read_x(s, ks, nxt);
            decode(w, ks, nxt);
            mfmas(cur);
            __builtin_amdgcn_sched_group_barrier(0x100, MI, 0);  // LDS reads
#pragma unroll
            for (int u = 0; u < MI * NJ; ++u) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);  // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        kstep(cw, kt, 1, fa, fb);
        kstep(cw, kt, 2, fb, fa);
        kstep(cw, kt, 3, fa, fb);
        // Stage kt + 1's X landed (this wave's; past the barrier everyone's,
        // and everyone holds stage kt's last fragments).
        fence();
        wait_vm<(NS - 2) * P::C>();
        lds_barrier();
        issue_x(kt + NS);
        fence();
        issue_w(kt + 2, cw);
        fence();
        __builtin_amdgcn_sched_barrier(0);
        kstep(nw, kt + 1, 0, fb, fa);
        ++kt;
        if constexpr (FOLD) {
            if (--kleft == 0 || kt == nk) {
                kleft = g.kfold;
                fold();
            }
        }
    };
    // (Two stages per iteration and no exit between them: with one, the
    // compiler's wait counts have to hold on a path that skips a stage.)
    for (int left = nk; left >= 2; left -= 2) {
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
    }
    if (nk & 1) step(std::integral_constant<int, 0>{});
    wait_vm<0>();
    if constexpr (EPI == EPI_QKPREP) {
        // One 32-row block at a time: the staged tile then fits the ring.
        auto block = [&](auto c) {
            constexpr int C = decltype(c)::value;
            int pos[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int64_t r = m0 + 32 * C + 8 * p + tid / 32;
                const int v = g.qk.meta[4 * (g.qk.base + (r < 0 ? 0 : (r < M ? r : M - 1)))];
                pos[p] = v < 0 ? 0 : (v >= g.qk.rope_rows ? int(g.qk.rope_rows - 1) : v);
            }
            finish_qkprep<MI, NJ, NW, C, 1>(g, acc, m0 + 32 * C, n0, smem, wave, lane, pos);
            return true;
        };
        run_phases(block, std::make_index_sequence<MI>{});
    } else {
        if constexpr (FOLD)
            finish32<MI, NJ, EPI, true>(g, tot, m0, n0 + wave * WR, lane);
        else
            finish32<MI, NJ, EPI, true>(g, acc, m0, n0 + (GATED ? wave * (WR / 2) : wave * WR), lane);
    }
}

// f16 weights.  Nothing is decoded, so no wave has to own its weight rows:
// both operands of a stage go by LDS DMA into a ring slot and 2 x 2 waves
// each take 32 MI rows by 32 NJ weight rows of the tile.  With the weights in
// registers (gemm32w_kernel) three row blocks were the most that fit and every
// weight passed L2 once per 96 rows.  The same products, operand layouts and K
// order as the other two, so the same sums.  Fragments are read one k-step
// ahead, and a slot is refilled as soon as everyone holds its last fragments:
// two workgroups share a CU and cover each other's waits.
//
// Isolated products (16x16x32 tiles with the weights through LDS / weights in
// registers -> this): erf-gated, N 2 x 1,152, K 768: 49,152 rows 199 / 230 ->
// 193 us, 8,192 41 / 49 -> 41, 500 10.8 / 11.4 -> 8.4; [q | k | v] heads, N
// 2,304, K 768: 49,152 rows 343 / 265 -> 235, 300 11.0 / 12.5 -> 9.0; f32, N
// 768, K 1,152, 49,152 rows 135 (128 x 128, weights in registers) / 137 ->
// 115; tanh-gated, N 2 x 6,912, K 1,152, 2,384 rows 135 / 122 -> 86.
//
// A weight packet's lane runs (kernels.h: 64 bytes of lane l at 64 l) keep
// their place, with the run's four 16-byte k-steps at ks ^ ((l >> 2) & 3): the
// sixteen lanes of a read's quarter then hit distinct banks.
template <int MI, int NJ, int EPI, int NS, int WM, int WN>
struct CfgL {
    static constexpr bool GATED = EPI == EPI_GELU_TANH || EPI == EPI_GELU_ERF;
    static constexpr int NW = WM * WN, T = NW * WAVE;
    static constexpr int BM = 32 * MI * WM;
    static constexpr int WR = 32 * NJ;                // weight rows per wave
    static constexpr int BNW = WN * WR;               // weight rows per tile
    static constexpr int BN = GATED ? BNW / 2 : BNW;  // output columns per tile
    static constexpr int PK = tile_packet_bytes(F16_DT);
    static constexpr int X_CH = BM * 8, X_I = (X_CH + T - 1) / T, X_BYTES = X_I * T * 16;
    static constexpr int W_BYTES = BNW / 32 * PK, W_I = W_BYTES / (T * 16);
    static constexpr int C = X_I + W_I;               // memory instructions per wave and stage
    static constexpr int STAGE = X_BYTES + W_BYTES, LDS = NS * STAGE;
    static_assert(!GATED || NJ % 2 == 0, "gated tiles pair gate and up row blocks");
    static_assert(W_BYTES % (T * 16) == 0, "whole DMA instructions per stage of weights");
    static_assert(LDS <= 160 * 1024, "ring larger than the LDS");
    static_assert(NS >= 2 && (NS - 1) * C <= 63, "vmcnt range");
};

template <int MI, int NJ, int EPI, int NS, int WM, int WN>
__global__ __launch_bounds__(WM * WN * WAVE, 2) void gemm32l_kernel(GemmArgs g) {
    using P = CfgL<MI, NJ, EPI, NS, WM, WN>;
    constexpr bool GATED = P::GATED;
    constexpr int NW = P::NW, BM = P::BM, BN = P::BN, WR = P::WR, PK = P::PK;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = int(threadIdx.x), lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = wave % WM, wn = wave / WM;
    const int64_t N = g.w0.rows, K = g.w0.cols, M = g.m;
    const int ntn = int((N + BN - 1) / BN);
    const int ntiles = ntn * int((M + BM - 1) / BM);
    const int per_xcd = int(gridDim.x) / 8;
    const int tile = (int(blockIdx.x) % 8) * per_xcd + int(blockIdx.x) / 8;
    if (tile >= ntiles) return;
    const int64_t n0 = int64_t(tile % ntn) * BN, m0 = int64_t(tile / ntn) * BM;
    const int kbeg = int(blockIdx.y) * int(K / g.ksplit);
    const int nk = int((K / g.ksplit + G_BK - 1) / G_BK);
    const int K32 = int(K), last = nk - 1;

    uint32_t xoff[P::X_I];
    int xcol[P::X_I];
#pragma unroll
    for (int i = 0; i < P::X_I; ++i) {
        const int slot = (i * NW + wave) * WAVE + lane;
        const int r = slot / 8, lc = (slot % 8) ^ swz(r);
        xcol[i] = lc * 8;
        xoff[i] = slot < P::X_CH && m0 + r < M ? uint32_t(((m0 + r) * g.ldx + lc * 8) * 2) : OOB;
    }
    // Weight blocks of the tile in LDS: wave column wn's NJ in order (gated:
    // its gate blocks, then the same blocks of the up matrix).  A DMA
    // instruction moves a quarter of one, 1 KB.
    const int64_t stages = g.w0.stages, rblocks = (N + 31) / 32, rb0 = n0 / 32;
    const int64_t live_blocks = rblocks - rb0;  // > 0: the tile starts inside N
    uint32_t woff[P::W_I];
    bool wup[P::W_I];
#pragma unroll
    for (int i = 0; i < P::W_I; ++i) {
        const int q = i * NW + wave, b = q / 4, j = b % NJ;
        wup[i] = GATED && j >= NJ / 2;
        const int blk = GATED ? b / NJ * (NJ / 2) + j % (NJ / 2) : b;
        woff[i] = blk < live_blocks ? uint32_t(blk * stages * PK + (q % 4) * 1024 + (lane / 4) * 64 +
                                               ((lane % 4) ^ ((lane / 16) & 3)) * 16)
                                    : OOB;
    }
    // Stages past the end repeat the last one (in range, never consumed), so
    // every wave always issues P::C instructions per stage.
    auto slot_base = [&](int s) { return smem + (unsigned(s) % unsigned(NS)) * P::STAGE; };
    const int64_t xbytes = M * g.ldx * 2;
    const bool ktail = (K32 & (G_BK - 1)) != 0;
    const int st0 = kbeg / G_BK;
    auto issue = [&](int s) {
        uint8_t* base = slot_base(s);
        const int sc = s < last ? s : last;
        const int k0 = __builtin_amdgcn_readfirstlane(kbeg + sc * G_BK);
        const bool tail = ktail && k0 + G_BK > K32;
#pragma unroll
        for (int i = 0; i < P::X_I; ++i) {
            const uint32_t o = tail && xcol[i] >= K32 - k0 ? OOB : xoff[i];
            const __amdgpu_buffer_rsrc_t r = rsrc(g.x, xbytes);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(base + (i * NW + wave) * WAVE * 16), 16, o,
                                                     k0 * 2, 0, 0);
        }
        // (The offset is a named value: read from its array in the call, the
        // host-side compile drops this kernel.)
        const int st = __builtin_amdgcn_readfirstlane(st0 + sc);
#pragma unroll
        for (int i = 0; i < P::W_I; ++i) {
            const uint32_t o = woff[i];
            const DevWeight& wt = wup[i] ? g.w1 : g.w0;
            const __amdgpu_buffer_rsrc_t r = rsrc(wt.tiles + rb0 * stages * PK, live_blocks * stages * PK);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                r, (lds_ptr_t)(base + P::X_BYTES + (i * NW + wave) * WAVE * 16), 16, o, st * PK, 0, 0);
        }
    };
    auto fence = [] { asm volatile("" ::: "memory"); };

    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};
    const int lr = lane % 32, lh = lane / 32;
    int foff[4], goff[4];  // the lane's X and weight fragment offsets per k-step
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        foff[ks] = (wm * MI * 32 + lr) * G_ROW + (((2 * ks + lh) ^ swz(lr)) * 16);
        goff[ks] = P::X_BYTES + wn * NJ * PK + lane * 64 + (ks ^ ((lane / 4) & 3)) * 16;
    }
    struct Frag {
        half8 x[MI], w[NJ];
    };
    auto read = [&](int s, int ks, Frag& f) {
        const uint8_t* S = slot_base(s);
#pragma unroll
        for (int j = 0; j < NJ; ++j) f.w[j] = *reinterpret_cast<const half8*>(S + goff[ks] + j * PK);
#pragma unroll
        for (int i = 0; i < MI; ++i) f.x[i] = *reinterpret_cast<const half8*>(S + foff[ks] + i * 32 * G_ROW);
    };
    // One k-step: the next one's fragment reads spread over this one's
    // products; nothing moves across its ends.
    auto kstep = [&](int s, int ks, const Frag& cur, Frag& nxt) {
        read(s, ks, nxt);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.w[j], cur.x[i], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < MI + NJ; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                     // LDS read
            __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ / (MI + NJ), 0);  // MFMA
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    Frag fa, fb;
#pragma unroll
    for (int s = 0; s < NS; ++s) issue(s);
    fence();
    wait_vm<(NS - 1) * P::C>();
    lds_barrier();
    read(0, 0, fa);
    for (int kt = 0; kt < nk; ++kt) {
        kstep(kt, 1, fa, fb);
        kstep(kt, 2, fb, fa);
        kstep(kt, 3, fa, fb);
        // Stage kt + 1 landed (this wave's part; past the barrier
        // everyone's, and everyone holds stage kt's last fragments).
        fence();
        wait_vm<(NS - 2) * P::C>();
        lds_barrier();
        issue(kt + NS);
        fence();
        __builtin_amdgcn_sched_barrier(0);
        kstep(kt + 1, 0, fb, fa);
    }
    wait_vm<0>();  // no DMA into LDS outlives the workgroup
    finish32<MI, NJ, EPI, true>(g, acc, m0 + wm * MI * 32, n0 + (GATED ? wn * (WR / 2) : wn * WR), lane);
}

// Resident X tiles up to this many bytes of LDS (one workgroup per CU
// above half of it).
constexpr int XR_MAX_LDS = 96 * 1024;

template <int QUANT, int MI, int NJ, int EPI, int NS, int NW = 4, bool FOLD = false, bool PAIR = false>
static void run32(hipStream_t s, const GemmArgs& g) {
    using P = Cfg32<QUANT, MI, NJ, EPI, NS, NW, PAIR>;
    for (const DevWeight* w : {&g.w0, &g.w1})
        if (!w->tiles || w->stages != (w->cols + G_BK - 1) / G_BK || (QUANT != F16_DT && !w->tscales))
            fail(E_INVALID, "gemm: weight without stage tiles");
    static bool lds_set = false;
    if (!lds_set) {
        OMG_HIP(hipFuncSetAttribute(
            reinterpret_cast<const void*>(&gemm32_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD, false, PAIR>),
            hipFuncAttributeMaxDynamicSharedMemorySize, P::LDS));
        OMG_HIP(hipFuncSetAttribute(
            reinterpret_cast<const void*>(&gemm32_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD, true, PAIR>),
            hipFuncAttributeMaxDynamicSharedMemorySize, XR_MAX_LDS > P::EPI_LDS ? XR_MAX_LDS : P::EPI_LDS));
        lds_set = true;
    }
    const int64_t N = g.w0.rows;
    if (g.mshift < 0 || g.mshift >= P::BM) fail(E_INVALID, "gemm: row tile shift out of range");
    const int64_t tiles = ((N + P::BN - 1) / P::BN) * ((g.m + g.mshift + P::BM - 1) / P::BM);
    const dim3 grid(unsigned((tiles + 7) / 8 * 8), unsigned(g.ksplit));
    const int64_t nk = (g.w0.cols / g.ksplit + G_BK - 1) / G_BK;
    const int64_t xr_lds = nk * P::X_BYTES;
    if (xr_lds <= XR_MAX_LDS) {
        const int lds = int(xr_lds > P::EPI_LDS ? xr_lds : P::EPI_LDS);
        gemm32_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD, true, PAIR><<<grid, dim3(P::T), lds, s>>>(g);
    } else {
        gemm32_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD, false, PAIR><<<grid, dim3(P::T), P::LDS, s>>>(g);
    }
    OMG_HIP(hipGetLastError());
}

template <int QUANT, int MI, int NJ, int EPI, int NS, int NW = 4, bool FOLD = false>
static void run32w(hipStream_t s, const GemmArgs& g) {
    static_assert(!FOLD || EPI == EPI_F32, "K pieces: f32 products only");
    using P = Cfg32<QUANT, MI, NJ, EPI, NS, NW, false>;
    for (const DevWeight* w : {&g.w0, &g.w1})
        if (!w->tiles || w->stages != (w->cols + G_BK - 1) / G_BK || (QUANT != F16_DT && !w->tscales))
            fail(E_INVALID, "gemm: weight without stage tiles");
    constexpr int QK = EPI == EPI_QKPREP ? 32 * (QK_TS + 17) * 4 : 0, RING = NS * P::X_BYTES;
    constexpr int LDS = QK > RING ? QK : RING;
    static bool lds_set = false;
    if (!lds_set) {
        OMG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm32w_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        lds_set = true;
    }
    if (FOLD != (g.kfold > 0)) fail(E_INVALID, "gemm: K pieces");
    const int64_t tiles = ((g.w0.rows + P::BN - 1) / P::BN) * ((g.m + g.mshift + P::BM - 1) / P::BM);
    const dim3 grid(unsigned((tiles + 7) / 8 * 8), unsigned(g.ksplit));
    gemm32w_kernel<QUANT, MI, NJ, EPI, NS, NW, FOLD><<<grid, dim3(P::T), LDS, s>>>(g);
    OMG_HIP(hipGetLastError());
}

template <int MI, int NJ, int EPI, int NS, int WM = 2, int WN = 2>
static void run32l(hipStream_t s, const GemmArgs& g) {
    using P = CfgL<MI, NJ, EPI, NS, WM, WN>;
    for (const DevWeight* w : {&g.w0, &g.w1})
        if (!w->tiles || w->stages != (w->cols + G_BK - 1) / G_BK) fail(E_INVALID, "gemm: weight without stage tiles");
    if (g.mshift != 0 || g.kfold != 0) fail(E_INVALID, "gemm: row shift or K pieces");
    static bool lds_set = false;
    if (!lds_set) {
        OMG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm32l_kernel<MI, NJ, EPI, NS, WM, WN>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, P::LDS));
        lds_set = true;
    }
    const int64_t tiles = ((g.w0.rows + P::BN - 1) / P::BN) * ((g.m + P::BM - 1) / P::BM);
    const dim3 grid(unsigned((tiles + 7) / 8 * 8), unsigned(g.ksplit));
    gemm32l_kernel<MI, NJ, EPI, NS, WM, WN><<<grid, dim3(P::T), P::LDS, s>>>(g);
    OMG_HIP(hipGetLastError());
}

// Row blocks (of 32) of the wide tile, at least LO: a workgroup of MI blocks
// takes about 1 + MI units of time whatever the product, and ROUND tiles run
// at a time, so the MI with the least rounds x (1 + MI) is taken (the larger
// of equals: less decode and weight traffic).  With 256 to a round it picks
// the fastest MI or one within 3% of it over 19 shapes from 300 to 49,152
// rows, K 640 to 2,560; the q/k/v tile, whose epilogue of one workgroup runs
// beside the K loop of the next on its CU, fits 512 (eight passes of 930 to
// 16,320 rows, K 1,152 to 2,560).  f16 weights take twice the registers of
// Q8 ones and stop at three blocks.
template <int QUANT, int LO, int ROUND>
static int wide_blocks(int64_t m, int64_t ntn) {
    int best = LO;
    int64_t cost = INT64_MAX;
    for (int mi = QUANT == F16_DT ? 3 : 4; mi >= LO; --mi) {
        const int64_t tiles = (m + 32 * mi - 1) / (32 * mi) * ntn, c = (tiles + ROUND - 1) / ROUND * (1 + mi);
        if (c < cost) cost = c, best = mi;
    }
    return best;
}

// 32 MI rows x 256 weight rows on four waves.
template <int QUANT, int EPI, int LO = 1, int ROUND = 256>
static void run_wide(hipStream_t s, const GemmArgs& g, int64_t cols_per_tile) {
    const int mi = wide_blocks<QUANT, LO, ROUND>(g.m, (g.w0.rows + cols_per_tile - 1) / cols_per_tile * g.ksplit);
    if constexpr (QUANT != F16_DT)
        if (mi == 4) return run32w<QUANT, 4, 2, EPI, 3, 4>(s, g);
    if (mi == 3) return run32w<QUANT, 3, 2, EPI, 3, 4>(s, g);
    if constexpr (LO == 1)
        if (mi == 1) return run32w<QUANT, 1, 2, EPI, 4, 4>(s, g);
    return run32w<QUANT, 2, 2, EPI, 4, 4>(s, g);
}

// f16 weights through LDS: 64, 128 or 192 rows x 128 weight rows.  64 while
// those tiles make one round of the 256 CUs; past it the two large tiles run
// two to a CU, 512 at a time, and take about three and four units: the least
// rounds x units (the larger tile of equals).  Over 34 products from 900 to
// 49,152 rows (erf-gated, q/k/v heads, bias + ReLU, f32, tanh-gated) it picks
// the faster of the two or one within 6% of it.
template <int EPI, bool SHORT = true>
static void run_lds(hipStream_t s, const GemmArgs& g, int64_t cols_per_tile) {
    const int64_t ntn = (g.w0.rows + cols_per_tile - 1) / cols_per_tile * g.ksplit;
    auto tiles = [&](int64_t rows) { return (g.m + rows - 1) / rows * ntn; };
    if constexpr (SHORT)
        if (tiles(64) <= 256) return run32l<1, 2, EPI, 3>(s, g);
    if (4 * ((tiles(192) + 511) / 512) <= 3 * ((tiles(128) + 511) / 512)) return run32l<3, 2, EPI, 2>(s, g);
    run32l<2, 2, EPI, 2>(s, g);
}

// Tile choice, measured on MI355X (tiles are activation rows x weight rows;
// every kernel gives every output element the same sums, so rows never
// depend on M).  gemm32_kernel, whose K loop has the shorter stages, while
// its tiles make one round of the 256 CUs; above that the wide tiles, or for
// f16 weights the ones through LDS (figures there).  Isolated products,
// 16x16x32 tiles / gemm32_kernel before -> now:
//   [q | k | v] heads, N 2,304, K 768, Q8: 49,152 rows 303 -> 236 us, 6,000
//   53 -> 33, 3,000 32 -> 21, 500 18.5 -> 9.8; erf-gated, N 2 x 1,152: 226
//   -> 204, 53 -> 28, 33 -> 17, 12.1 -> 9.1; o, N 768: 84 -> 79, 20.8 ->
//   16.3, 14.5 -> 11.0; tanh-gated, N 2 x 10,240, K 2,560, Q4, 16,320 rows:
//   1,557 -> 1,444; N 2 x 6,912, K 1,152, Q8, 384 rows: 32.5 -> 20.8.
// Long products are bound by power: the card runs the 16,320-row one at
// 1.6 GHz with its matrix cores 67% busy (a library f16 product of 8,192^3:
// 1.4 GHz, 89%).
template <int QUANT, int EPI>
static void dispatch(hipStream_t s, const GemmArgs& g) {
    const int64_t N = g.w0.rows, K = g.w0.cols, M = g.m;
    auto tiles = [&](int64_t rows, int64_t cols) { return (M + rows - 1) / rows * ((N + cols - 1) / cols) * g.ksplit; };
    auto rounds = [&](int64_t rows, int64_t cols) { return (tiles(rows, cols) + 255) / 256; };
    if constexpr (EPI == EPI_QKV) {
        // a 64-wide head per wave
        if constexpr (QUANT == F16_DT) return run_lds<EPI>(s, g, 128);
        if constexpr (QUANT != F16_DT) {
            if (tiles(32, 256) <= 256) return run32<QUANT, 1, 2, EPI, 4, 4>(s, g);
            if (tiles(64, 256) <= 256) return run32<QUANT, 2, 2, EPI, 4, 4>(s, g);
            return run_wide<QUANT, EPI>(s, g, 256);
        }
    } else if constexpr (EPI == EPI_RELU_F16) {
        // 32 x 64 on two waves for the fewest rows (N 3,072, K 768, 32 x 128
        // on four waves -> this: 12 rows f16 7.8 -> 6.0 us, Q4 7.0 -> 6.4, Q8
        // 7.1 -> 6.6); f16 64 x 64 through LDS up to a round of those (150
        // rows 9.3 -> 7.5, 300 11.2 -> 8.0).
        if constexpr (QUANT == F16_DT) {
            if (M <= 64) return run32<QUANT, 1, 1, EPI, 4, 2>(s, g);
            if (tiles(64, 64) <= 256) return run32l<1, 1, EPI, 4>(s, g);
            return run_lds<EPI>(s, g, 128);
        } else {
            if (tiles(32, 64) <= 256) return run32<QUANT, 1, 1, EPI, 4, 2>(s, g);
            if (tiles(32, 128) <= 256) return run32<QUANT, 1, 1, EPI, 4, 4>(s, g);
            return run_wide<QUANT, EPI>(s, g, 256);
        }
    } else if constexpr (EPI == EPI_QKPREP) {
        // One head on eight waves of one 32-row weight block each (half the
        // decode per wave and K stage of the four-wave tile): short passes,
        // and long ones whose 64-row X tile stays resident (K <= 768; the
        // 270M model's cold q/k/v 15.9 -> 13.3 us, its cold pass -3.2%).
        // Longer K: 64 rows on four waves of the short stages while the wide
        // rule would take no more and two workgroups per CU hold them all
        // (1B, K 1,152, Q4: 992 rows 17.0 us against 15.7, 2,352 18.1 against
        // 16.8, f16 23.2 against 19.5; 4B, K 2,560, Q4, 1,980 rows 49.9
        // against 49.3), past that wide tiles (16,320 rows 355 -> 324, 4,100
        // 109 -> 96).
        if (M <= 512) return run32<QUANT, 1, 1, EPI, 4, 8>(s, g);
        if (K <= 768) return run32<QUANT, 2, 1, EPI, 4, 8>(s, g);
        if (tiles(64, 256) <= 512 && wide_blocks<QUANT, 2, 512>(M, (N + 255) / 256) == 2)
            return run32<QUANT, 2, 2, EPI, 4, 4>(s, g);
        return run_wide<QUANT, EPI, 2, 512>(s, g, 256);
    } else if constexpr (EPI == EPI_F32) {
        if (g.kfold > 0) {
            // K pieces added in registers (the totals take what a second
            // weight block would).  A round of 64, 96 or 128 rows x 128 takes
            // about 50, 62 or 84 units, one alone 65, 80 or 95, and the least
            // sum is taken.  N 2,560, K 10,240, Q4 (96 rows of the short
            // stages / of the wide kernel -> this): 560 rows 76 / 77 -> 63 us,
            // 1,600 120 / 122 -> 107, 1,980 122 / 126 -> 122, 2,663 194 / 171
            // -> 158, 16,320 904 / 871 -> 859; f16, 930 rows 74 / 109 -> 74.
            // The wide kernel's 96 rows only past four rounds, where it is 4%
            // the faster, and not on Q8, where it is 3% the slower.
            if (M <= 512) return run32<QUANT, 1, 1, EPI, 4, 4, true>(s, g);
            const int64_t r96 = rounds(96, 128);
            const int64_t c64 = std::max<int64_t>(65, 50 * rounds(64, 128)), c96 = std::max<int64_t>(80, 62 * r96),
                          c128 = std::max<int64_t>(95, 84 * rounds(128, 128));
            if (c64 < c96 && c64 < c128) return run32<QUANT, 2, 1, EPI, 4, 4, true>(s, g);
            if (c128 <= c96) return run32w<QUANT, 4, 1, EPI, 3, 4, true>(s, g);
            if (QUANT == Q8_DT || r96 <= 4) return run32<QUANT, 3, 1, EPI, 4, 4, true>(s, g);
            if constexpr (QUANT != Q8_DT) return run32w<QUANT, 3, 1, EPI, 3, 4, true>(s, g);
        }
        if (M <= 512 && tiles(32, 128) <= 512) return run32<QUANT, 1, 1, EPI, 4, 4>(s, g);
        if ((g.ksplit > 1 || (QUANT == F16_DT && tiles(64, 128) > 256)) && tiles(96, 128) <= 256)
            return run32<QUANT, 3, 1, EPI, 4, 4>(s, g);
        if (g.ksplit == 1 && tiles(64, 128) <= 256) return run32<QUANT, 2, 1, EPI, 4, 4>(s, g);
        if constexpr (QUANT == F16_DT) return run_lds<EPI, false>(s, g, 128);
        if constexpr (QUANT != F16_DT) {
            // A round of 64 x 128 of the short stages takes 37 units, of 96 x
            // 128 48, of 128 x 256 100.  N 2,560, K 2,048, Q4 (96 x 128 ->
            // this): 1,350 rows 27.1 -> 21.8 us, 1,600 28.3 -> 24.7, 2,663
            // 39.6 -> 37.1, 16,320 183 -> 169.
            const int64_t c64 = 37 * rounds(64, 128), c96 = 48 * rounds(96, 128), c256 = 100 * rounds(128, 256);
            if (c64 < c96 && c64 < c256) return run32<QUANT, 2, 1, EPI, 4, 4>(s, g);
            if (c96 < c256) return run32w<QUANT, 3, 1, EPI, 3, 4>(s, g);
            return run32w<QUANT, 4, 2, EPI, 3, 4>(s, g);
        }
    } else {
        // Branch-sized passes (M <= 64) pair the waves (a gate and an up
        // wave per 32 columns: half the decode per wave and stage; flushed
        // one-branch passes, same box, against 32 x 128 on four waves of
        // gate and up each: the 270M model's gate/up 9.2 -> 7.4 us and pass
        // 1.064 -> 1.027 ms, the 4B model's 23.9 -> 21.4 us and 3.60 -> 3.50
        // ms).  With X resident (K <= 1,024) nine slots of weights (four:
        // 7.9 us); through the ring 64 rows on four waves, four slots (32
        // rows on two: 21.8 us; five to nine slots 26-29 us).
        if (M <= 64 && EPI == EPI_GELU_TANH) {
            if (K <= 1024) return run32<QUANT, 1, 1, EPI, 9, 2, false, true>(s, g);
            return run32<QUANT, 2, 1, EPI, 4, 4, false, true>(s, g);
        }
        if constexpr (QUANT == F16_DT) return run_lds<EPI>(s, g, 64);
        if constexpr (QUANT != F16_DT) {
            // (the encoder's short gated product on two waves while those
            // tiles make one round: N 1,152, K 768, 100 rows, Q4 9.2 -> 8.2
            // us, Q8 9.8 -> 8.5)
            if constexpr (EPI == EPI_GELU_ERF)
                if (tiles(32, 64) <= 256) return run32<QUANT, 1, 2, EPI, 4, 2>(s, g);
            if (tiles(32, 128) <= 256) return run32<QUANT, 1, 2, EPI, 4, 4>(s, g);
            return run_wide<QUANT, EPI>(s, g, 128);
        }
    }
}

template <int EPI>
static void dispatch_dtype(hipStream_t s, const GemmArgs& g) {
    switch (g.w0.dtype) {
        case F16_DT: return dispatch<F16_DT, EPI>(s, g);
        case Q8_DT: return dispatch<Q8_DT, EPI>(s, g);
        default: return dispatch<Q4_DT, EPI>(s, g);
    }
}

static void check(const half_t* x, int64_t ldx, const DevWeight& w, int64_t ldy, int64_t m) {
    if (m < 0) fail(E_INVALID, "gemm: negative M");
    if (w.cols % 32 != 0) fail(E_INVALID, "gemm: K must be a multiple of 32");
    if (ldx < w.cols || ldx % 8 != 0) fail(E_INVALID, "gemm: X row stride must be >= K and a multiple of 8");
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w.data) % 16 != 0)
        fail(E_INVALID, "gemm: operands must be 16-byte aligned");
    if (ldy < w.rows) fail(E_INVALID, "gemm: Y row stride must be >= N");
    if (ldy % 4 != 0) fail(E_INVALID, "gemm: Y row stride must be a multiple of 4");
    if (w.dtype != F16_DT && (!w.scales || w.sld < (w.cols / 32 + 1) / 2 * 2))
        fail(E_INVALID, "gemm: quantized weight without padded scales");
    // Buffer offsets are 32-bit.
    if (m * ldx * 2 >= 0x7fff0000LL || w.rows * w.cols * 2 >= 0x7fff0000LL)
        fail(E_INVALID, "gemm: operand of 2 GiB or more");
}

void launch_gemm(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& w, float* y, int64_t ldy,
                 int64_t m) {
    check(x, ldx, w, ldy, m);
    if (m == 0) return;
    dispatch_dtype<EPI_F32>(s, GemmArgs{x, ldx, m, w, w, y, ldy, nullptr, {}});
}

void launch_gemm_splitk(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& w, float* y, int64_t ldy,
                       int64_t m, int parts, int64_t part_stride, int kfold) {
    check(x, ldx, w, ldy, m);
    if (parts < 1 || (parts > 1 && w.cols % (int64_t(G_BK) * parts) != 0))
        fail(E_INVALID, "gemm_splitk: K must split into parts of whole 64-wide stages");
    if (kfold < 0) fail(E_INVALID, "gemm_splitk: negative K piece length");
    if (parts > 1 && part_stride < m * ldy) fail(E_INVALID, "gemm_splitk: partial outputs overlap");
    if (m == 0) return;
    GemmArgs g{x, ldx, m, w, w, y, ldy, nullptr, {}};
    g.ksplit = parts;
    g.part_stride = part_stride;
    g.kfold = kfold;
    dispatch_dtype<EPI_F32>(s, g);
}

void launch_gemm_geglu(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& wg,
                       const DevWeight& wu, half_t* act, int64_t ldact, int64_t m, bool erf) {
    check(x, ldx, wg, ldact, m);
    if (wu.rows != wg.rows || wu.cols != wg.cols || wu.dtype != wg.dtype || wu.sld != wg.sld)
        fail(E_INVALID, "gemm_geglu: gate and up must share shape and storage type");
    if (m == 0) return;
    const GemmArgs g{x, ldx, m, wg, wu, act, ldact, nullptr, {}};
    if (erf) return dispatch_dtype<EPI_GELU_ERF>(s, g);
    dispatch_dtype<EPI_GELU_TANH>(s, g);
}

void launch_gemm_bias_relu(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& w,
                           const uint16_t* bias, half_t* y, int64_t ldy, int64_t m) {
    check(x, ldx, w, ldy, m);
    if (!bias) fail(E_INVALID, "gemm_bias_relu: bias required");
    if (m == 0) return;
    dispatch_dtype<EPI_RELU_F16>(s, GemmArgs{x, ldx, m, w, w, y, ldy, bias, {}});
}

void launch_gemm_qkprep(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& w, const QkArgs& a, int64_t m) {
    check(x, ldx, w, w.rows, m);
    const int64_t slots = a.heads + (a.has_kv ? 2 * a.kv_heads : 0);
    if (a.hd != 256 || a.heads <= 0 || a.kv_heads <= 0 || w.rows != slots * 256)
        fail(E_INVALID, "gemm_qkprep: head_dim 256 and N = (heads + 2 kv_heads) x 256 (heads x 256 without K/V)");
    if (a.base < 0 || a.base + m > a.cap_pad || a.cap_pad % 64) fail(E_INVALID, "gemm_qkprep: cache rows out of range");
    if (a.rope_rows <= 0 || a.rope_dims > a.hd || !a.rope || !a.meta || !a.q_norm || !a.q16)
        fail(E_INVALID, "gemm_qkprep: rope table, row meta, q norm and q output required");
    if (a.has_kv && (!a.k_norm || !a.kc || !a.vt)) fail(E_INVALID, "gemm_qkprep: K/V layer without k norm or cache");
    if (m == 0) return;
    GemmArgs g{x, ldx, m, w, w, nullptr, 0, nullptr, {}};
    g.qk = a;
    g.mshift = a.base % 32;  // row tiles on the cache's 32-row grid: whole V^T chunks per tile
    dispatch_dtype<EPI_QKPREP>(s, g);
}

void launch_gemm_qkv_heads(hipStream_t s, const half_t* x, int64_t ldx, const DevWeight& w,
                           const uint16_t* bias, const QkvHeads& o, int64_t m) {
    check(x, ldx, w, w.rows, m);
    if (o.dq <= 0 || o.dq % 64 != 0 || w.rows != 3 * o.dq)
        fail(E_INVALID, "gemm_qkv_heads: N must be 3 x the q width, a multiple of 64");
    if (o.tpad < m || o.tpad % 32 != 0) fail(E_INVALID, "gemm_qkv_heads: padded rows must cover M, multiple of 32");
    if (!o.q16 || !o.k16 || !o.vt || (o.rope && !o.meta)) fail(E_INVALID, "gemm_qkv_heads: missing output");
    if (m == 0) return;
    dispatch_dtype<EPI_QKV>(s, GemmArgs{x, ldx, m, w, w, nullptr, 0, bias, o});
}

}  // namespace omg
