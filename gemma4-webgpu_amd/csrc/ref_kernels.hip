// The six gemma4-webgpu attention kernels, one HIP kernel each, with the
// reference's semantics, dispatch grids and reduction order:
//
//   fusedPerHeadNormRope    shaders/fused_per_head_norm_rope.wgsl:20-64
//   perHeadRmsNormNoWeight  shaders/per_head_rms_norm_no_weight.wgsl:13-38
//   kvCacheStore            shaders/kv_cache_store.wgsl:8-18     (f16 cache)
//   attnScore               shaders/attn_score.wgsl:15-40        (f16 cache)
//   softmax                 shaders/softmax.wgsl:7-46
//   attnOutput              shaders/attn_output.wgsl:7-23        (f16 cache)
//
// attnScore, softmax and attnOutput also have forms for the sizes the engine
// dispatches (k_attn_score_tile, k_softmax_reg, k_attn_output_chain): the same
// operations in the same order on every value, so the same bits, with the work
// of one value spread differently over threads and memory.
//
// They are the per-kernel drop-in surface (the engine's capture points
// postRopeQ/K and attnOut sit between them, src/engine.ts:2086-2095) and the
// unfused comparison path for the fused kernels. Arithmetic: every f32
// operation rounds separately (no FMA contraction), sqrt and division are
// IEEE correctly rounded, and pow/sin/cos/exp return the f32 nearest to the
// exact value (evaluated in f64), so results are reproducible bit for bit on
// any IEEE machine that evaluates the same expressions.
#include "launch_rules.h"
#include "ref_math.h"

namespace g4 {

__global__ __launch_bounds__(kWG) void k_fused_per_head_norm_rope(float* __restrict__ data,
                                                                  const uint16_t* __restrict__ weight,
                                                                  const uint16_t* __restrict__ rope_freqs,
                                                                  g4_norm_rope_params p) {
    __shared__ float scratch[kNormScratch];
    const unsigned head = blockIdx.x;
    if (head >= p.num_heads) return;
    head_norm_rope(data + head * p.head_dim, weight, true, rope_freqs, p.head_dim, p.eps, p.position, p.theta,
                   p.apply_divisor, scratch);
}

__global__ __launch_bounds__(kWG) void k_per_head_rms_norm_no_weight(float* __restrict__ data, g4_norm_params p) {
    __shared__ float scratch[kNormScratch];
    const unsigned head = blockIdx.x;
    if (head >= p.num_heads) return;
    head_norm_rope(data + head * p.head_dim, nullptr, false, nullptr, p.head_dim, p.eps, 0, 0.0f, 0, scratch);
}

__global__ __launch_bounds__(kWG) void k_kv_cache_store(const float* __restrict__ k_in, const float* __restrict__ v_in,
                                                        uint16_t* __restrict__ k_cache,
                                                        uint16_t* __restrict__ v_cache, g4_kv_store_params p) {
    const unsigned i = blockIdx.x * kWG + threadIdx.x;
    const unsigned total = p.num_kv_heads * p.head_dim;
    if (i >= total) return;
    const unsigned head = i / p.head_dim;
    const unsigned d = i % p.head_dim;
    const uint64_t cache_idx = (uint64_t)p.position * total + head * p.head_dim + d;
    k_cache[cache_idx] = f2h(k_in[i]);
    v_cache[cache_idx] = f2h(v_in[i]);
}

__global__ __launch_bounds__(kWG) void k_attn_score(const float* __restrict__ q, const uint16_t* __restrict__ k_cache,
                                                    float* __restrict__ scores, g4_attn_score_params p) {
    const uint64_t idx = (uint64_t)blockIdx.x * kWG + threadIdx.x;
    const uint64_t total = (uint64_t)p.num_q_heads * p.seq_len;
    if (idx >= total) return;
    const unsigned head = (unsigned)(idx / p.seq_len);
    const unsigned pos = (unsigned)(idx % p.seq_len);
    const uint64_t score_idx = (uint64_t)head * p.seq_len + pos;
    if (p.sliding_window != 0u) {
        const unsigned current_pos = p.seq_len - 1u;
        const unsigned window_start =
            (current_pos + 1u > p.sliding_window) ? current_pos + 1u - p.sliding_window : 0u;
        if (pos < window_start) {
            scores[score_idx] = -1e30f;
            return;
        }
    }
    const unsigned kv_head = head * p.num_kv_heads / p.num_q_heads;
    const unsigned q_offset = head * p.head_dim;
    const unsigned kv_stride = p.num_kv_heads * p.head_dim;
    const uint64_t k_offset = (uint64_t)pos * kv_stride + kv_head * p.head_dim;
    float dot = 0.0f;
    for (unsigned d = 0; d < p.head_dim; d++) dot = dot + q[q_offset + d] * h2f(k_cache[k_offset + d]);
    scores[score_idx] = dot * p.scale;
}

// x * y rounded once, x an f16 value widened exactly: v_fma_mix_f32 with an
// addend of -0 (x y + -0 is x y, its sign of zero included), one instruction
// where widening and multiplying take two. `neg_zero` comes from opaque_neg_zero,
// which keeps the compiler from folding the addition away.
__device__ __forceinline__ float opaque_neg_zero() {
    float z = -0.0f;
    asm volatile("" : "+v"(z));
    return z;
}
__device__ __forceinline__ float mul_f16(f16 x, float y, float neg_zero) { return __builtin_fmaf((float)x, y, neg_zero); }

// t[e] = k[e] * q[e] for 8 f16 values in a register quad and 8 uniform f32 values. One block, so that a
// product is never used by the very next instruction (left to itself the compiler puts a wait state there).
__device__ __forceinline__ void mul8_f16(float (&t)[8], u32x4 k, const float* q, float neg_zero) {
#pragma unroll
    for (int h = 0; h < 2; h++)
        asm("v_fma_mix_f32 %0, %4, %6, %10 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %1, %4, %7, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %2, %5, %8, %10 op_sel_hi:[1,0,0]\n\t"
            "v_fma_mix_f32 %3, %5, %9, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=&v"(t[4 * h]), "=&v"(t[4 * h + 1]), "=&v"(t[4 * h + 2]), "=&v"(t[4 * h + 3])
            : "v"(k[2 * h]), "v"(k[2 * h + 1]), "s"(q[4 * h]), "s"(q[4 * h + 1]), "s"(q[4 * h + 2]), "s"(q[4 * h + 3]),
              "v"(neg_zero));
}

// attnScore with the K rows staged through LDS: one workgroup takes
// kScoreRows rows and 4 query heads of one kv head, one wave per head and one
// row per lane, so a row is read from memory once per 4 heads, coalesced. Each
// dot keeps the shader's order (d = 0, 1, ...: products and sums rounded, one
// chain per thread), and that chain is the bound: 2 VALU instructions per
// element (the q value is uniform, read through the scalar cache). Rows are
// padded by 16 bytes in LDS, so the lanes' 16-byte reads meet no bank conflict.
// Measured at 8 heads, head_dim 512, 2048 rows: 113.1 us as one strided global
// read per element and thread, 7.5 us here.
constexpr unsigned kScoreRows = 64;
constexpr unsigned kScoreHeads = 4;

template <int HD>
__global__ __launch_bounds__(kWG) void k_attn_score_tile(const float* __restrict__ q, const uint16_t* __restrict__ k_cache,
                                                         float* __restrict__ scores, g4_attn_score_params p) {
    constexpr unsigned kPieces = HD / 8;                                  // 16-byte pieces of a row
    constexpr unsigned kStride = HD + 8;                                  // f16 elements between LDS rows
    constexpr unsigned kLoads = kScoreRows * kPieces / kWG;               // pieces per thread
    __shared__ f16 tile[kScoreRows * kStride];
    const unsigned group = p.num_q_heads / p.num_kv_heads;
    const unsigned hblocks = (group + kScoreHeads - 1) / kScoreHeads;
    const unsigned kvh = blockIdx.y / hblocks;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const unsigned hg = (blockIdx.y % hblocks) * kScoreHeads + wave;      // head within the group
    const unsigned row0 = blockIdx.x * kScoreRows;
    const unsigned first = p.sliding_window != 0u && p.seq_len > p.sliding_window ? p.seq_len - p.sliding_window : 0u;
    const unsigned pos = row0 + lane;
    const bool live = hg < group && pos < p.seq_len;
    float* dst = scores + (uint64_t)(kvh * group + hg) * p.seq_len + pos;
    if (row0 + kScoreRows <= first) {  // uniform: every row of the tile is before the window
        if (live) *dst = -1e30f;
        return;
    }
    const uint64_t stride = (uint64_t)p.num_kv_heads * HD;
    const uint16_t* krows = k_cache + (uint64_t)kvh * HD;
    f16x8 v[kLoads];
#pragma unroll
    for (unsigned i = 0; i < kLoads; i++) {
        const unsigned c = threadIdx.x + i * kWG;
        v[i] = ldg<f16x8>(krows + min(row0 + c / kPieces, p.seq_len - 1u) * stride + (c % kPieces) * 8);
    }
#pragma unroll
    for (unsigned i = 0; i < kLoads; i++) {
        const unsigned c = threadIdx.x + i * kWG;
        *reinterpret_cast<f16x8*>(tile + (c / kPieces) * kStride + (c % kPieces) * 8) = v[i];
    }
    __syncthreads();
    if (hg >= group) return;
    const float* __restrict__ qh = q + (uint64_t)(kvh * group + hg) * HD;
    const f16* row = tile + lane * kStride;
    const float nz = opaque_neg_zero();
    // Two sets of operands in turn: a set is requested when the other has arrived (scalar loads return in
    // any order, so only a full wait tells), and is in flight under the other's chain.
    u32x4 ka[4], kb[4];
    float qa[32], qb[32], dot = 0.0f;
    auto load = [&](u32x4(&k8)[4], float(&qd)[32], unsigned d) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
#pragma unroll
        for (unsigned i = 0; i < 4; i++) k8[i] = *reinterpret_cast<const u32x4*>(row + d + 8 * i);
#pragma unroll
        for (unsigned i = 0; i < 32; i++) qd[i] = qh[d + i];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto chain = [&](const u32x4(&k8)[4], const float(&qd)[32]) {
#pragma unroll
        for (unsigned i = 0; i < 32; i += 8) {
            float t[8];
            mul8_f16(t, k8[i / 8], qd + i, nz);
#pragma unroll
            for (unsigned e = 0; e < 8; e++) dot = dot + t[e];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    load(ka, qa, 0);
    for (unsigned d = 0; d < HD; d += 64) {
        load(kb, qb, d + 32);
        chain(ka, qa);
        load(ka, qa, (d + 64) % HD);
        chain(kb, qb);
    }
    if (live) *dst = pos < first ? -1e30f : dot * p.scale;
}

__global__ __launch_bounds__(kWG) void k_softmax(float* __restrict__ scores, g4_softmax_params p) {
    __shared__ float shared_max[kWG];
    __shared__ float shared_sum[kWG];
    const unsigned tid = threadIdx.x;
    const unsigned head = blockIdx.x;
    if (head >= p.num_heads) return;
    const uint64_t base = (uint64_t)head * p.seq_len;
    float local_max = -1e30f;
    for (unsigned i = tid; i < p.seq_len; i += kWG) local_max = wgsl_max(local_max, scores[base + i]);
    shared_max[tid] = local_max;
    __syncthreads();
    const float max_val = wg_tree_max(shared_max, tid);
    float local_sum = 0.0f;
    for (unsigned i = tid; i < p.seq_len; i += kWG) {
        float e = (float)exp((double)(scores[base + i] - max_val));
        scores[base + i] = e;
        local_sum = local_sum + e;
    }
    shared_sum[tid] = local_sum;
    __syncthreads();
    const float sum_val = wg_tree_sum(shared_sum, tid);
    for (unsigned i = tid; i < p.seq_len; i += kWG) scores[base + i] = scores[base + i] / sum_val;
}

// softmax of heads of up to 1024 R scores: each thread keeps its R scores in
// registers, so memory is read and written once (the loop form above passes over
// it three times, a memory round trip per pass and 256 scores), and 1024 threads
// share the f64 exponentials. The sum keeps the shader's order: exponentials pass
// through LDS to the 256 partials, each added in index order, then the 128 -> 1
// tree. Bound by its chain of latencies. Measured at 8 heads of 2048 scores:
// 8.2 us -> 5.0 us.
constexpr unsigned kSoftThreads = 1024;

template <int R>
__global__ __launch_bounds__(kSoftThreads) void k_softmax_reg(float* __restrict__ scores, g4_softmax_params p) {
    __shared__ float e_all[kSoftThreads * R];
    __shared__ float red[kWG + 1];
    const unsigned tid = threadIdx.x;
    float* base = scores + (uint64_t)blockIdx.x * p.seq_len;
    float x[R];
    float local_max = -1e30f;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned i = tid + r * kSoftThreads;
        x[r] = i < p.seq_len ? base[i] : -1e30f;
        local_max = wgsl_max(local_max, x[r]);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) local_max = wgsl_max(local_max, __shfl_xor(local_max, m));  // no NaN: any order
    if ((tid & 63) == 0) red[tid >> 6] = local_max;
    __syncthreads();
    float max_val = red[0];
#pragma unroll
    for (unsigned w = 1; w < kSoftThreads / 64; w++) max_val = wgsl_max(max_val, red[w]);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned i = tid + r * kSoftThreads;
        x[r] = (float)exp((double)(x[r] - max_val));
        if (i < p.seq_len) e_all[i] = x[r];
    }
    __syncthreads();  // also: every thread has read the wave maxima
    if (tid < kWG) {
        float sum = 0.0f;
        for (unsigned i = tid; i < p.seq_len; i += kWG) sum = sum + e_all[i];
        red[tid] = sum;
    }
    __syncthreads();
    if (tid < 64) {  // strides 128, 64, then 32 .. 1 within the wave: wg_tree_sum's operand pairs
        float s = (red[tid] + red[tid + 128]) + (red[tid + 64] + red[tid + 192]);
        s = wave_tree_sum(s);
        if (tid == 0) red[kWG] = s;
    }
    __syncthreads();
    const float sum_val = red[kWG];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned i = tid + r * kSoftThreads;
        if (i < p.seq_len) base[i] = x[r] / sum_val;
    }
}

__global__ __launch_bounds__(kWG) void k_attn_output(const float* __restrict__ probs,
                                                     const uint16_t* __restrict__ v_cache, float* __restrict__ out,
                                                     g4_attn_output_params p) {
    const unsigned idx = blockIdx.x * kWG + threadIdx.x;
    const unsigned total = p.num_q_heads * p.head_dim;
    if (idx >= total) return;
    const unsigned head = idx / p.head_dim;
    const unsigned d = idx % p.head_dim;
    const unsigned kv_head = head * p.num_kv_heads / p.num_q_heads;
    const unsigned kv_stride = p.num_kv_heads * p.head_dim;
    float sum = 0.0f;
    for (unsigned pos = 0; pos < p.seq_len; pos++) {
        float prob = probs[(uint64_t)head * p.seq_len + pos];
        const uint64_t v_idx = (uint64_t)pos * kv_stride + kv_head * p.head_dim + d;
        sum = sum + prob * h2f(v_cache[v_idx]);
    }
    out[(uint64_t)head * p.head_dim + d] = sum;
}

// attnOutput for head_dims of whole 64-column blocks. An output's sum is one
// chain over the rows (each product and sum rounded, in row order), so what
// bounds the kernel is the chain's length; the form above puts two dependent
// loads, a conversion and a product on every link. Here the workgroup's wave 0
// holds the 64 chains and does nothing but add: the other seven waves read
// V and the probabilities two rounds ahead (16 bytes a lane, 8 rows a load),
// multiply, and leave the products in LDS, four rows of a column side by side
// (one 16-byte read per four additions).
// A block of rows whose products are all zero is not added: the sum starts at +0
// and never becomes -0, so adding a zero of either sign returns its bits (rows
// before a sliding window have probability 0; 0 * inf is NaN and is added).
// Measured at 8 heads, head_dim 512, 2048 rows: 502.3 us -> 12.8 us.
constexpr unsigned kOutMul = 7;    // multiplying waves
constexpr unsigned kOutRows = 32;  // rows of a multiplying wave per round
constexpr unsigned kOutRound = kOutMul * kOutRows;
constexpr unsigned kOutQuad = 288;  // floats of 4 rows of products: 8 groups of 8 columns x 4 rows, 4 floats between
                                    // groups (the multiplying lanes' 64 stores then fall in 64 different banks)

struct OutSmem {
    f32x4 prod[2][kOutMul][kOutRows / 4][kOutQuad / 4];  // [round parity][wave][row / 4]
    uint32_t live[2][kOutMul];                           // some product of the block is not zero
};

// A multiplying wave's operands of one round: lane (r, c) = 8 r + c holds rows 8 i + r, columns 8 c .. + 7.
struct OutRows {
    f16x8 v[kOutRows / 8];
    float p[kOutRows / 8];
};

__device__ __forceinline__ void out_load(OutRows& x, const uint16_t* v, uint64_t stride, const float* probs, unsigned row0,
                                         unsigned rows, unsigned lane) {
#pragma unroll
    for (unsigned i = 0; i < kOutRows / 8; i++) {
        const unsigned row = min(row0 + 8 * i + (lane >> 3), rows - 1);  // clamped: see out_multiply
        x.p[i] = ldg<float>(probs + row);
        x.v[i] = ldg<f16x8>(v + row * stride + (lane & 7) * 8);
    }
}

__device__ __forceinline__ void out_multiply(const OutRows& x, OutSmem& sm, unsigned par, unsigned wave, unsigned lane,
                                             unsigned row0, unsigned rows, float nz) {
    uint32_t any = 0;
#pragma unroll
    for (unsigned i = 0; i < kOutRows / 8; i++) {
        const unsigned r = 8 * i + (lane >> 3);
        const bool in = row0 + r < rows;  // rows past the end: 0 * 0, which adds +0
        const float p = in ? x.p[i] : 0.0f;
        const f16x8 v = in ? x.v[i] : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
        float* dst = reinterpret_cast<float*>(sm.prod[par][wave][r / 4]) + (lane & 7) * 36 + r % 4;
#pragma unroll
        for (unsigned e = 0; e < 8; e++) {
            const float y = mul_f16(v[e], p, nz);
            any |= __float_as_uint(y);
            dst[4 * e] = y;
        }
    }
    const bool nonzero = __any((any << 1) != 0);
    if (lane == 0) sm.live[par][wave] = nonzero;
}

__global__ __launch_bounds__(64 * (kOutMul + 1)) void k_attn_output_chain(const float* __restrict__ probs,
                                                                          const uint16_t* __restrict__ v_cache,
                                                                          float* __restrict__ out,
                                                                          g4_attn_output_params p) {
    __shared__ OutSmem sm;
    const unsigned lane = threadIdx.x & 63;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned head = blockIdx.y, d = blockIdx.x * 64 + lane, rows = p.seq_len;
    const unsigned kv_head = head / (p.num_q_heads / p.num_kv_heads);
    const uint64_t stride = (uint64_t)p.num_kv_heads * p.head_dim;
    const unsigned rounds = (rows + kOutRound - 1) / kOutRound;
    if (wave == 0) {
        __builtin_amdgcn_s_setprio(3);  // one multiplying wave shares its SIMD
        float sum = 0.0f;
        for (unsigned t = 0; t < rounds; t++) {
            __syncthreads();
            const unsigned par = t & 1;
            uint64_t todo = __ballot(lane < kOutMul && sm.live[par][min(lane, kOutMul - 1)] != 0);
            if (!todo) continue;  // uniform, as every branch here
            f32x4 x[kOutRows / 4], y[kOutRows / 4];  // a block is read from LDS under the additions of the one before
            auto take = [&](f32x4(&to)[kOutRows / 4]) {
                const unsigned w = (unsigned)__builtin_ctzll(todo);
#pragma unroll
                for (unsigned r = 0; r < kOutRows / 4; r++) to[r] = sm.prod[par][w][r][lane + lane / 8];
                todo &= todo - 1;
                __builtin_amdgcn_sched_barrier(0);
            };
            auto add = [&](const f32x4(&from)[kOutRows / 4]) {
#pragma unroll
                for (unsigned r = 0; r < kOutRows / 4; r++)
#pragma unroll
                    for (unsigned e = 0; e < 4; e++) sum = sum + from[r][e];
                __builtin_amdgcn_sched_barrier(0);
            };
            take(x);
            while (true) {
                if (!todo) {
                    add(x);
                    break;
                }
                take(y);
                add(x);
                if (!todo) {
                    add(y);
                    break;
                }
                take(x);
                add(y);
            }
        }
        out[(uint64_t)head * p.head_dim + d] = sum;
        return;
    }
    const unsigned mw = wave - 1;
    const uint16_t* v = v_cache + (uint64_t)kv_head * p.head_dim + blockIdx.x * 64;
    const float* pr = probs + (uint64_t)head * rows;
    const float nz = opaque_neg_zero();
    OutRows a, b;
    unsigned row0 = mw * kOutRows;
    out_load(a, v, stride, pr, row0, rows, lane);
    out_load(b, v, stride, pr, row0 + kOutRound, rows, lane);
    // Barrier t (the adding wave's t-th) follows the multiplication of round t; a buffer is written
    // again after the next barrier, which the adding wave reaches when it is done with it.
    for (unsigned t = 0; t < rounds; t += 2) {
        out_multiply(a, sm, 0, mw, lane, row0, rows, nz);
        out_load(a, v, stride, pr, row0 + 2 * kOutRound, rows, lane);
        __syncthreads();
        if (t + 1 < rounds) {  // uniform
            out_multiply(b, sm, 1, mw, lane, row0 + kOutRound, rows, nz);
            out_load(b, v, stride, pr, row0 + 3 * kOutRound, rows, lane);
            __syncthreads();
        }
        row0 += 2 * kOutRound;
    }
}

__global__ __launch_bounds__(kWG) void k_zero(uint32_t* __restrict__ dst, uint64_t words, uint8_t* tail,
                                              unsigned tail_bytes) {
    const uint64_t stride = (uint64_t)gridDim.x * kWG;
    for (uint64_t i = (uint64_t)blockIdx.x * kWG + threadIdx.x; i < words; i += stride) dst[i] = 0u;
    if (blockIdx.x == 0 && threadIdx.x < tail_bytes) tail[threadIdx.x] = 0;
}

}  // namespace g4

using namespace g4;

static inline unsigned ceil_div_u(uint64_t a, uint64_t b) { return (unsigned)((a + b - 1) / b); }

extern "C" {

int g4_fused_per_head_norm_rope(float* data, const uint16_t* weight, const uint16_t* rope_freqs,
                                g4_norm_rope_params p, void* stream) {
    if (!data || !weight) return fail(G4_EINVAL, "fusedPerHeadNormRope: NULL data/weight");
    if (p.apply_divisor && !rope_freqs) return fail(G4_EINVAL, "fusedPerHeadNormRope: apply_divisor needs rope_freqs");
    if (p.head_dim == 0 || p.head_dim % 2) return fail(G4_EINVAL, "fusedPerHeadNormRope: head_dim %u", p.head_dim);
    if (p.num_heads == 0) return G4_OK;
    G4_LAUNCH(k_fused_per_head_norm_rope, dim3(p.num_heads), dim3(kWG), 0, as_stream(stream), data, weight,
                       rope_freqs, p);
    G4_CHECK_LAUNCH("fusedPerHeadNormRope");
    return G4_OK;
}

int g4_per_head_rms_norm_no_weight(float* data, g4_norm_params p, void* stream) {
    if (!data) return fail(G4_EINVAL, "perHeadRmsNormNoWeight: NULL data");
    if (p.head_dim == 0) return fail(G4_EINVAL, "perHeadRmsNormNoWeight: head_dim 0");
    if (p.num_heads == 0) return G4_OK;
    G4_LAUNCH(k_per_head_rms_norm_no_weight, dim3(p.num_heads), dim3(kWG), 0, as_stream(stream), data, p);
    G4_CHECK_LAUNCH("perHeadRmsNormNoWeight");
    return G4_OK;
}

int g4_kv_cache_store(const float* k_in, const float* v_in, uint16_t* k_cache, uint16_t* v_cache,
                      g4_kv_store_params p, void* stream) {
    if (!k_in || !v_in || !k_cache || !v_cache) return fail(G4_EINVAL, "kvCacheStore: NULL pointer");
    if (p.position >= p.max_seq_len)
        return fail(G4_EINVAL, "kvCacheStore: slot %u >= max_seq_len %u", p.position, p.max_seq_len);
    const uint64_t total = (uint64_t)p.num_kv_heads * p.head_dim;
    if (total == 0) return G4_OK;
    G4_LAUNCH(k_kv_cache_store, dim3(ceil_div_u(total, kWG)), dim3(kWG), 0, as_stream(stream), k_in, v_in,
                       k_cache, v_cache, p);
    G4_CHECK_LAUNCH("kvCacheStore");
    return G4_OK;
}

int g4_attn_score(const float* q, const uint16_t* k_cache, float* scores, g4_attn_score_params p, void* stream) {
    if (!q || !k_cache || !scores) return fail(G4_EINVAL, "attnScore: NULL pointer");
    if (p.seq_len == 0) return fail(G4_EINVAL, "attnScore: seq_len 0");
    if (p.num_kv_heads == 0 || p.num_q_heads % p.num_kv_heads)
        return fail(G4_EINVAL, "attnScore: num_q_heads %u not a multiple of num_kv_heads %u", p.num_q_heads,
                    p.num_kv_heads);
    const uint64_t total = (uint64_t)p.num_q_heads * p.seq_len;
    if (total == 0) return G4_OK;
    const unsigned group = p.num_q_heads / p.num_kv_heads;
    const uint64_t hblocks = (uint64_t)p.num_kv_heads * ((group + kScoreHeads - 1) / kScoreHeads);
    // The tile form: the head_dims it is built for, 16-byte K rows, and a grid within the launch limit.
    if ((p.head_dim == 256 || p.head_dim == 512) && !(reinterpret_cast<uintptr_t>(k_cache) & 15) && hblocks <= 65535) {
        const dim3 grid(ceil_div_u(p.seq_len, kScoreRows), (unsigned)hblocks);
        if (p.head_dim == 256)
            G4_LAUNCH(k_attn_score_tile<256>, grid, dim3(kWG), 0, as_stream(stream), q, k_cache, scores, p);
        else
            G4_LAUNCH(k_attn_score_tile<512>, grid, dim3(kWG), 0, as_stream(stream), q, k_cache, scores, p);
        G4_CHECK_LAUNCH("attnScore");
        return G4_OK;
    }
    G4_LAUNCH(k_attn_score, dim3(ceil_div_u(total, kWG)), dim3(kWG), 0, as_stream(stream), q, k_cache,
                       scores, p);
    G4_CHECK_LAUNCH("attnScore");
    return G4_OK;
}

int g4_softmax(float* scores, g4_softmax_params p, void* stream) {
    if (!scores) return fail(G4_EINVAL, "softmax: NULL scores");
    if (p.seq_len == 0) return fail(G4_EINVAL, "softmax: seq_len 0");
    if (p.num_heads == 0) return G4_OK;
    const unsigned per_thread = softmax_scores_per_thread(p.num_heads, p.seq_len);
    if (per_thread == 4)
        G4_LAUNCH(k_softmax_reg<4>, dim3(p.num_heads), dim3(kSoftThreads), 0, as_stream(stream), scores, p);
    else if (per_thread == 16)
        G4_LAUNCH(k_softmax_reg<16>, dim3(p.num_heads), dim3(kSoftThreads), 0, as_stream(stream), scores, p);
    else
        G4_LAUNCH(k_softmax, dim3(p.num_heads), dim3(kWG), 0, as_stream(stream), scores, p);
    G4_CHECK_LAUNCH("softmax");
    return G4_OK;
}

int g4_attn_output(const float* probs, const uint16_t* v_cache, float* out, g4_attn_output_params p, void* stream) {
    if (!probs || !v_cache || !out) return fail(G4_EINVAL, "attnOutput: NULL pointer");
    if (p.num_kv_heads == 0 || p.num_q_heads % p.num_kv_heads)
        return fail(G4_EINVAL, "attnOutput: num_q_heads %u not a multiple of num_kv_heads %u", p.num_q_heads,
                    p.num_kv_heads);
    const uint64_t total = (uint64_t)p.num_q_heads * p.head_dim;
    if (total == 0) return G4_OK;
    if (p.head_dim % 64 == 0 && p.seq_len < 0x40000000u && p.num_q_heads <= 65535 &&
        !(reinterpret_cast<uintptr_t>(v_cache) & 15) && attn_output_chain(total / 64, p.seq_len, device_cus())) {
        G4_LAUNCH(k_attn_output_chain, dim3(p.head_dim / 64, p.num_q_heads), dim3(64 * (kOutMul + 1)), 0,
                  as_stream(stream), probs, v_cache, out, p);
        G4_CHECK_LAUNCH("attnOutput");
        return G4_OK;
    }
    G4_LAUNCH(k_attn_output, dim3(ceil_div_u(total, kWG)), dim3(kWG), 0, as_stream(stream), probs, v_cache,
                       out, p);
    G4_CHECK_LAUNCH("attnOutput");
    return G4_OK;
}

int g4_zero(void* dev_dst, size_t bytes, void* stream) {
    if (!dev_dst) return fail(G4_EINVAL, "g4_zero: NULL pointer");
    if (bytes == 0) return G4_OK;
    if (reinterpret_cast<uintptr_t>(dev_dst) % 4) return fail(G4_EINVAL, "g4_zero: pointer not 4-byte aligned");
    const uint64_t words = bytes / 4;
    const unsigned tail = (unsigned)(bytes % 4);
    unsigned blocks = words ? ceil_div_u(words, kWG) : 1;
    if (blocks > 4096) blocks = 4096;
    G4_LAUNCH(k_zero, dim3(blocks), dim3(kWG), 0, as_stream(stream), static_cast<uint32_t*>(dev_dst), words,
                       static_cast<uint8_t*>(dev_dst) + words * 4, tail);
    G4_CHECK_LAUNCH("g4_zero");
    return G4_OK;
}

}  // extern "C"
