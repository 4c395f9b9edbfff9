// mp_batched.hip -- gfx950 kernels of the batched MoE layer (prefill chunks and
// decode at batch > 1).
//
//   dispatch_kernel      per-expert histogram, exclusive scan and the stable
//                        permutation of (token, k) pairs
//   quant_rows_kernel    Q8_K of rows (x per token) into the form the matrix
//                        cores consume: the int8 values as fp16 codes, the
//                        block scale, and the 16-value group sums as fp16 --
//                        all exact
//   grouped_q4_tile_kernel  per (expert's pairs in chunks, 128-row tiles): the
//                        expert's Q4_K rows against the activations of the
//                        chunk's pairs, on MFMA 32x32x16 f16; up and gate as
//                        one 2I-row matrix (the expert's [up | gate] layout),
//                        and Q4_K down with the pair's gate weight, scattered
//                        to the pair's row
//   grouped_q4_kernel    the same per (64-row tile, expert) on MFMA 16x16x32,
//                        for shapes of few workgroups
//   grouped_q6_tile_kernel, grouped_q6_kernel  the same for a Q6_K down matrix
//   swiglu_quant_kernel  h = silu(gate) * up, and its Q8_K
//   combine_kernel       out[t] = sum over k of the weighted rows, k in order
//
// Exact integer products on fp16 matrix cores.  A Q4_K weight is
// d*sc*q - dmin*m with q a nibble and sc, m six-bit.  The B operand holds sc*q
// (<= 945, an integer fp16 represents exactly: 11-bit significand; bf16's 8 bits
// cannot), the A operand the Q8_K integers of the activation (|q8| <= 127,
// exact).  Each 128-value half of a 256-value super-block accumulates in fp32
// exactly (below 2^24), and the halves add once: the block's integer sum
// sum_j sc_j * sum_i q_i q8_i of ggml's vec_dot_q4_K_q8_K rounded once, as its
// (float)sumi.  The min
// term sum_j m_j * bsum_j is a second, 16-deep MFMA of the six-bit mins
// against the Q8_K group sums (|bsum16| <= 2032, exact).  fp32 appears only
// where ggml has it, in ggml's order: y += (d*dx)*sumi; y -= (dmin*dx)*summ per
// super-block, so a row's value is the CPU chain's bit for bit.  Q6_K weights
// are (q - 32) * sc with an int8 sc, split into two exact products (below).
//
// Every MFMA pairs the k-th element of lane group g of A with the k-th element
// of lane group g of B, so the order of the K elements inside one instruction
// is free: each lane feeds the 8 weights its own 16-byte load decodes, and the
// activation rows are read at the same positions.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "mp_device.h"
#include "mp_format.h"
#include "mp_internal.h"

namespace mp {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lptr_t;

// ---------------------------------------------------------------------------
// dispatch: ids [P] (P = n_tok * K, pair i = t*K + k) -> counts[E], offsets[E+1],
// perm[offsets[e] + r] = i of the r-th pair routed to e in pair order.
// A workgroup places a segment of 1,024 pairs, a wave a chunk of 64.  Every
// workgroup counts all of ids with LDS atomics (order-free; the pairs before its
// segment in the high half of the word), one wave turns the counts into offsets
// with a prefix sum (lane l holds experts 4l .. 4l+3), and the pairs are ranked:
// lanes holding the same id find each other with 8 ballots (one per id bit), their
// rank inside the chunk is a popcount, and a per-expert scan over the segment's
// chunks gives each chunk's base.  Counting everything in each workgroup (P <
// 2^16 words from L2) costs less than a second launch or a hand-over, and needs
// no scratch.  One workgroup placing 4,096 pairs a round took 11, 23, 37 and 70
// us for 4,096, 8,000, 16,384 and 32,768 pairs.
constexpr int DSP_WAVES = 16, DSP_SEG = 64 * DSP_WAVES;
static_assert(MAX_E <= 256, "4 experts a lane in the offsets' prefix sum");

// inclusive prefix sum over the 64 lanes of a wave
__device__ inline int wave_incl_sum(int v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

__global__ __launch_bounds__(64 * DSP_WAVES) void dispatch_kernel(const int32_t *ids, int P, int E, int32_t *counts,
                                                                  int32_t *offsets, int32_t *perm) {
    __shared__ uint32_t s_cnt[MAX_E];       // pairs of the expert: (before the segment << 16) | all
    __shared__ int s_off[MAX_E];            // where the segment's first pair of the expert goes
    __shared__ uint16_t s_c[DSP_WAVES][MAX_E];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int seg = (int)blockIdx.x * DSP_SEG;
    for (int e = tid; e < E; e += 64 * DSP_WAVES) s_cnt[e] = 0;
    for (int i = tid; i < DSP_WAVES * MAX_E; i += 64 * DSP_WAVES) ((uint16_t *)s_c)[i] = 0;
    __syncthreads();
#pragma unroll 8
    for (int i = tid; i < P; i += 64 * DSP_WAVES) {
        const int e = ids[i];
        if (e >= 0 && e < E) atomicAdd(&s_cnt[e], i < seg ? 0x10001u : 1u);
    }
    // the segment's own pairs, a chunk a wave
    const int i = seg + tid;
    const int e = i < P ? ids[i] : -1;
    const bool valid = e >= 0 && e < E;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (e >> b) & 1;
        const uint64_t bb = __ballot(valid && bit);
        m &= bit ? bb : ~bb;
    }
    const int r = __popcll(m & ((1ull << lane) - 1ull));
    if (valid && r == 0) s_c[wave][e] = (uint16_t)__popcll(m);
    __syncthreads();
    if (wave == 0) {
        int c[4], before[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t w = 4 * lane + j < E ? s_cnt[4 * lane + j] : 0u;
            c[j] = (int)(w & 0xffffu);
            before[j] = (int)(w >> 16);
            sum += c[j];
        }
        const int incl = wave_incl_sum(sum, lane);
        int acc = incl - sum;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int x = 4 * lane + j;
            if (x < E) {
                s_off[x] = acc + before[j];
                if (seg == 0) {
                    counts[x] = c[j];
                    offsets[x] = acc;
                }
            }
            acc += c[j];
        }
        if (lane == 63 && seg == 0) offsets[E] = incl;
    }
    for (int x = tid - 64; x >= 0 && x < E; x += 64 * (DSP_WAVES - 1)) {       // beside wave 0's prefix sum
        int run = 0;
#pragma unroll
        for (int c = 0; c < DSP_WAVES; ++c) {
            const int v = s_c[c][x];
            s_c[c][x] = (uint16_t)run;
            run += v;
        }
    }
    __syncthreads();
    if (valid) perm[s_off[e] + s_c[wave][e] + r] = i;
}

// ---------------------------------------------------------------------------
// Q8_K rows for the matrix cores: one wavefront per (row, 256-value block)
template <bool MFMA>
__global__ __launch_bounds__(256) void quant_rows_kernel(const void *src, int bf16, int n_rows, int n,
                                                         uint16_t *q16, float *dx, uint16_t *bs16) {
    const int lane = threadIdx.x & 63;
    const int nb = n / QK;
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= (int64_t)n_rows * nb) return;
    const int64_t row = blk / nb;
    const int b = (int)(blk % nb);
    const size_t off = (size_t)row * n + (size_t)b * QK + 4 * lane;
    float xv[4];
    if (bf16) {
        const uint2 v = *(const uint2 *)((const uint16_t *)src + off);
        xv[0] = bits_f32(v.x << 16);
        xv[1] = bits_f32(v.x & 0xffff0000u);
        xv[2] = bits_f32(v.y << 16);
        xv[3] = bits_f32(v.y & 0xffff0000u);
    } else {
        const float4 v = *(const float4 *)((const float *)src + off);
        xv[0] = v.x; xv[1] = v.y; xv[2] = v.z; xv[3] = v.w;
    }
    q8_rows_out<MFMA>(xv, lane, off, (size_t)row, b, n, q16, dx, bs16);
}

// SiLU with the canonical exp (the oracle evaluates the same function)
__device__ inline float silu_mul(float g, float u) { return g / (1.0f + canon_expf(-g)) * u; }

// h = silu(gate) * up from the up/gate rows y2 [P][2I] (up first), then its
// Q8_K: one wavefront per (pair, 256-value block); h itself of the first n_h pairs
// to h_out if given
__global__ __launch_bounds__(256) void swiglu_quant_kernel(const float *y2, int P, int I, float *h_out, int n_h,
                                                           uint16_t *q16, float *dx, uint16_t *bs16) {
    const int lane = threadIdx.x & 63;
    const int nb = I / QK;
    const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= (int64_t)P * nb) return;
    const int64_t p = blk / nb;
    const int b = (int)(blk % nb);
    const float *yr = y2 + (size_t)p * 2 * I + (size_t)b * QK + 4 * lane;
    const float4 u = *(const float4 *)yr;
    const float4 g = *(const float4 *)(yr + I);
    const float hv[4] = {silu_mul(g.x, u.x), silu_mul(g.y, u.y), silu_mul(g.z, u.z), silu_mul(g.w, u.w)};
    const size_t off = (size_t)p * I + (size_t)b * QK + 4 * lane;
    if (h_out && p < n_h) *(float4 *)(h_out + off) = make_float4(hv[0], hv[1], hv[2], hv[3]);
    q8_rows_out<true>(hv, lane, off, (size_t)p, b, I, q16, dx, bs16);
}

// ---------------------------------------------------------------------------
// grouped expert products

__device__ inline const uint8_t *grouped_expert(const GroupedArgs &a, int e) {
    if (a.host_mask && a.host_mask[e]) return nullptr;          // computed by the host
    if (a.table) {
        const int s = a.table[e];
        if (a.slot_pool && s >= 0 && s < a.n_slots) return a.slot_pool + (size_t)s * a.slot_bytes;
    }
    if (!a.store || e >= a.n_store) return nullptr;
    return a.store + (size_t)e * a.expert_bytes;
}

// 8 small unsigned bytes (two words) -> 8 fp16 holding 1024 + v: byte v under
// the exponent byte 0x64 (1024 has a unit last place up to 2048).  Each word's
// bytes in the order 0, 2, 1, 3, in which masks alone separate them (q4_tile_b);
// the activation codes of the grouped products are stored in the same order.
__device__ inline half8_t pack_1024(uint32_t w0, uint32_t w1) {
    const uint32_t K = 0x64646464u;
    uint4 r;
    r.x = __builtin_amdgcn_perm(K, w0, 0x04020400u);
    r.y = __builtin_amdgcn_perm(K, w0, 0x04030401u);
    r.z = __builtin_amdgcn_perm(K, w1, 0x04020400u);
    r.w = __builtin_amdgcn_perm(K, w1, 0x04030401u);
    return __builtin_bit_cast(half8_t, r);
}

__device__ inline half8_t splat8(_Float16 v) { return half8_t{v, v, v, v, v, v, v, v}; }

// (1024 + q) * sc - 1024 * sc = q * sc, one rounding of an exact value
__device__ inline half8_t q4_scaled(uint32_t w0, uint32_t w1, int sc) {
    const _Float16 s = (_Float16)(float)sc;
    const _Float16 nb = (_Float16)(float)(-1024 * sc);
    return __builtin_elementwise_fma(pack_1024(w0, w1), splat8(s), splat8(nb));
}

__device__ inline float4_t mfma32(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Q4_K lane layout.  Lane (n = lane & 15: row, h = lane >> 4) of a wave loads
// the 16-byte header and qs bytes 16h .. 16h+15 (group g_0 = h >> 1) and
// 64+16h .. 64+16h+15 (group g_1 = 2 + (h >> 1)) of each super-block: elements
// 16*(h & 1) .. +15 of sub-blocks 2g_L (low nibbles) and 2g_L + 1 (high).  MFMA
// i = 4L + 2*nibble + half multiplies 8 of them; the activation values at the
// same positions sit at this offset of the 256-value block:
__device__ inline int q4_a_offset(int h, int i) {
    const int L = i >> 2, nib = (i >> 1) & 1, half = i & 1;
    const int g = (h >> 1) + 2 * L;
    return 32 * (2 * g + nib) + 16 * (h & 1) + 8 * half;
}

// Q4_K B operand of MFMA i from the lane's raw 16-byte qs load of group g_L
__device__ inline half8_t q4_b(const uint4 &q, int i, int sc) {
    const uint32_t M = 0x0F0F0F0Fu;
    uint32_t w0 = (i & 1) ? q.z : q.x, w1 = (i & 1) ? q.w : q.y;
    if ((i >> 1) & 1) { w0 >>= 4; w1 >>= 4; }
    return q4_scaled(w0 & M, w1 & M, sc);
}

struct Q4Scales {
    int sc[2][2];      // [L][nibble]
    half4_t bm;        // min operand: mins of sub-blocks 2g, 2g+1, g = g_{h & 1}, each twice
    float d, dmin;
};

__device__ inline void q4_scales(const uint4 &hdr, int h, Q4Scales &o) {
    o.d = h2f_dev((uint16_t)(hdr.x & 0xffff));
    o.dmin = h2f_dev((uint16_t)(hdr.x >> 16));
#pragma unroll
    for (int L = 0; L < 2; ++L) {
        const int g = (h >> 1) + 2 * L;
        int m0, m1;
        q4k_sm(hdr, 2 * g, o.sc[L][0], m0);
        q4k_sm(hdr, 2 * g + 1, o.sc[L][1], m1);
        if (L == (h & 1)) {
            const _Float16 x0 = (_Float16)(float)m0, x1 = (_Float16)(float)m1;
            o.bm = half4_t{x0, x0, x1, x1};
        }
    }
}

// ---- activation staging ------------------------------------------------------
// One 256-value block of the activation rows of a pass's pairs, in LDS.  The
// 16-byte chunk c of row r sits at position c ^ (r & 15), so the 16 rows one
// fragment read touches fall in distinct banks.

// R activation rows (32 for two M tiles of 16 pairs, 16 for one) and their group sums
template <int R>
struct __attribute__((aligned(16))) AStageR {
    _Float16 a[R][QK];
    _Float16 bs[R][16];
};

template <int R>
__device__ inline half8_t stage_frag(const AStageR<R> &st, int r, int off) {
    const int c = (off >> 3) ^ (r & 15);
    return *(const half8_t *)&st.a[r][8 * c];
}

// Staging by direct buffer -> LDS loads: lane l of an instruction writes
// base + 16*l.  rows[r]: activation row of pair r of the pass (r < np); rows
// are K values long.  Wave w stages rows (R/4)w .. (R/4)w + R/4 - 1 (two per
// instruction), wave 0 also the group sums (two lanes a row); rows past np are not loaded.  The
// activation codes and the group sums are raw buffers, the lane's byte offsets
// are computed once per pass of a chunk and block s's offset s*QK*2 is a
// scalar: a step's staging costs no per-lane address arithmetic (up/gate at
// 512 tokens 104.0 -> 97.8 us a launch against 64-bit pointers per load).
constexpr int BUF_WORD3 = 0x00020000;    // raw buffer, 32-bit elements (gfx9)
typedef int i32x4_t __attribute__((ext_vector_type(4)));
__device__ void buffer_load_lds(i32x4_t rsrc, lptr_t *lds, int size, int voffset, int soffset, int offset,
                                int aux) __asm("llvm.amdgcn.raw.buffer.load.lds");
__device__ i32x4_t buffer_load_v4(i32x4_t rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.v4i32");
typedef int i32x2_t __attribute__((ext_vector_type(2)));
__device__ i32x2_t buffer_load_v2(i32x4_t rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.v2i32");
__device__ short buffer_load_i16(i32x4_t rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.i16");
// a buffer resource over [p, p + bytes): base address, no stride, the size, raw
// (the words are the same in every lane: scalar registers)
__device__ inline i32x4_t raw_buffer(const void *p, uint32_t bytes) {
    const uint64_t a = (uint64_t)p;
    i32x4_t r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu));
    r.z = __builtin_amdgcn_readfirstlane((int)bytes);
    r.w = BUF_WORD3;
    // a vector memory instruction may read a scalar register five wait states after the vector
    // unit (readfirstlane) wrote it; the compiler does not count them before inline assembly
    asm("s_nop 4" : "+s"(r));
    return r;
}
template <int R>
struct StageOff {
    int a[R / 8];       // instruction j: the lane's row and swizzled chunk, bytes
    int bs;             // the lane's group-sum chunk (wave 0), bytes
};
template <int R>
__device__ inline void stage_offsets(StageOff<R> &o, const int *rows, int np, int K, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < R / 8; ++j) {
        const int r0 = (R / 4) * wave + 2 * j;
        const int r = min(r0 + (lane >> 5), np - 1);
        const int c = (lane & 31) ^ ((r0 + (lane >> 5)) & 15);
        o.a[j] = 2 * (rows[max(r, 0)] * K + 8 * c);
    }
    const int r = min(lane >> 1, np - 1);
    o.bs = 2 * (rows[max(r, 0)] * (K / 16) + 8 * (lane & 1));
}
template <int R, bool SUMS = true>
__device__ inline void stage_a_buf(AStageR<R> &st, const StageOff<R> &o, int np, i32x4_t ra, i32x4_t rbs, int s,
                                   int wave, int lane) {
#pragma unroll
    for (int j = 0; j < R / 8; ++j) {
        const int r0 = (R / 4) * wave + 2 * j;
        if (r0 >= np) break;
        buffer_load_lds(ra, (lptr_t *)&st.a[r0][0], 16, o.a[j], s * QK * 2, 0, 0);
    }
    if (SUMS && wave == 0 && lane < 2 * R) buffer_load_lds(rbs, (lptr_t *)&st.bs[0][0], 16, o.bs, s * 32, 0, 0);
}
__device__ inline uint4 buf_load16(i32x4_t r, int voff, int soff) {
    const i32x4_t v = buffer_load_v4(r, voff, soff, 0);
    return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
}

// Workgroup -> (row tile, expert).  Workgroups go to the 8 XCDs round-robin
// (workgroup L on XCD L % 8); with E a multiple of 8, every row tile of
// expert e lands on XCD e % 8, so the tiles of an expert share one L2 copy of
// its activation rows instead of fetching them into all eight.
__device__ inline void tile_expert(int L, int T, int E, int &tile, int &e) {
    if (E % 8 == 0) {
        const int j = L >> 3;
        e = (L & 7) + 8 * (j / T);
        tile = j % T;
    } else {
        e = L / T;
        tile = L % T;
    }
}

// ---------------------------------------------------------------------------
// Q6_K lane layout of the streamed kernel.  Lane (n = row, h) takes, of the
// 128-value half hh = h >> 1, the 16 positions l = 16*(h & 1) .. +15 of each
// of its four 32-value groups g: ql bytes 64hh + l (g = 0 low nibbles, g = 2
// high) and 64hh + 32 + l (g = 1, 3), qh bytes 32hh + l (two bits a group),
// so each group's 16 values share one scale, 8hh + 2g + (h & 1).  MFMA
// i = 2g + half multiplies positions l = 16*(h & 1) + 8*half .. +7 of group g;
// the activation values at those positions sit at this offset of the block:
__device__ inline int q6_a_offset(int h, int i) {
    return 128 * (h >> 1) + 32 * (i >> 1) + 16 * (h & 1) + 8 * (i & 1);
}

struct Q6Lane {
    uint4 qa, qb, qh;      // ql bytes 64hh + l, 64hh + 32 + l, qh bytes 32hh + l
    uint2 sc;              // scales 8hh .. 8hh + 7
    uint32_t d;            // the block's fp16 scale in the low half
};

// The lane's offsets into its row's blocks, and one block's pieces by buffer
// loads at the block's offset (a scalar).  A Q6_K block starts 2-byte aligned
// (210-byte blocks); the loads are unaligned.
struct Q6Off {
    int qa, qb, qh, sc, d;
};
__device__ inline Q6Off q6_lane_offsets(int row_off, int h) {
    const int hh = h >> 1, l0 = 16 * (h & 1);
    return Q6Off{row_off + 64 * hh + l0, row_off + 64 * hh + 32 + l0, row_off + 128 + 32 * hh + l0,
                 row_off + 192 + 8 * hh, row_off + 208};
}
__device__ inline void q6_lane_load(Q6Lane &w, i32x4_t rw, const Q6Off &o, int blk_off) {
    const i32x4_t a = buffer_load_v4(rw, o.qa, blk_off, 0), b = buffer_load_v4(rw, o.qb, blk_off, 0);
    const i32x4_t q = buffer_load_v4(rw, o.qh, blk_off, 0);
    const i32x2_t sc = buffer_load_v2(rw, o.sc, blk_off, 0);
    w.qa = make_uint4((uint32_t)a.x, (uint32_t)a.y, (uint32_t)a.z, (uint32_t)a.w);
    w.qb = make_uint4((uint32_t)b.x, (uint32_t)b.y, (uint32_t)b.z, (uint32_t)b.w);
    w.qh = make_uint4((uint32_t)q.x, (uint32_t)q.y, (uint32_t)q.z, (uint32_t)q.w);
    w.sc = make_uint2((uint32_t)sc.x, (uint32_t)sc.y);
    w.d = (uint16_t)buffer_load_i16(rw, o.d, blk_off, 0);
}

// The B operands of MFMA i: (q - 32) * sc in two exact halves, sc = 16*sh + sl
// (|(q - 32) * sh| <= 256, |(q - 32) * sl| <= 480); (1024 + q)*s - 1056*s is
// one rounding of an exact integer.
__device__ inline void q6_lane_b(const Q6Lane &w, int i, int h, half8_t &bh, half8_t &bl) {
    const uint32_t M = 0x0F0F0F0Fu, HM = 0x30303030u;
    const int g = i >> 1, half = i & 1;
    const uint4 &ql = (g & 1) ? w.qb : w.qa;
    uint32_t l0 = half ? ql.z : ql.x, l1 = half ? ql.w : ql.y;
    uint32_t q0 = half ? w.qh.z : w.qh.x, q1 = half ? w.qh.w : w.qh.y;
    if (g >= 2) {
        l0 >>= 4;
        l1 >>= 4;
    }
    // group g's two high bits (qh bits 2g, 2g+1) to bits 4, 5 of each byte
    if (g == 0) { q0 <<= 4; q1 <<= 4; }
    if (g == 1) { q0 <<= 2; q1 <<= 2; }
    if (g == 3) { q0 >>= 2; q1 >>= 2; }
    const half8_t q = pack_1024((l0 & M) | (q0 & HM), (l1 & M) | (q1 & HM));
    const int j = 2 * g + (h & 1);
    const int sc = (int)(int8_t)(uint8_t)((j < 4 ? w.sc.x : w.sc.y) >> (8 * (j & 3)));
    const _Float16 sh = (_Float16)(float)(sc >> 4), sl = (_Float16)(float)(sc & 15);   // arithmetic shift
    bh = __builtin_elementwise_fma(q, splat8(sh), splat8((_Float16)(float)(-1056 * (sc >> 4))));
    bl = __builtin_elementwise_fma(q, splat8(sl), splat8((_Float16)(float)(-1056 * (sc & 15))));
}

// The grouped down product for a Q6_K matrix of few workgroups or, at I = 512, few
// pairs (see plan_q6): 64 rows of one expert a workgroup, the lane's weights streamed
// from HBM into registers (block s + 1 in flight while block s is multiplied),
// the pairs in passes of MT tiles of 16 on MFMA 16x16x32.  A block's two integer sums stay
// below 2^24 (256 * 32 * 8 * 127 and 256 * 32 * 15 * 127), so each is exact and
// 16*acc_h + acc_l rounds once, as ggml's (float)sumi.  y = the pair's gate
// weight times the row value, to the pair's (t*K + k) row.
template <int NB, int MT>
__global__ __launch_bounds__(256, 4) void grouped_q6_kernel(GroupedArgs a) {
    constexpr int GK = 16 * MT;
    int e, tile;
    tile_expert(blockIdx.x, a.H / 64, a.E, tile, e);
    const int n0 = a.offsets[e], ne = a.offsets[e + 1] - n0;
    if (ne <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, h = lane >> 4;
    const int r0 = tile * 64;
    const int row = r0 + wave * 16 + n;
    constexpr int K = NB * QK;
    const uint8_t *base = grouped_expert(a, e);
    if (!base) {
        for (int i = tid; i < ne * 64; i += 256) {
            const int pos = n0 + i / 64, c = r0 + (i % 64);
            a.ypair[(size_t)a.perm[pos] * a.H + c] = 0.0f;
        }
        return;
    }
    // the expert's down matrix and the Q8_K codes of h as raw buffers
    const i32x4_t rw = raw_buffer(base + 2ull * a.I * (a.H / QK) * Q4K_BYTES, (uint32_t)(a.H * NB * Q6K_BYTES));
    const i32x4_t ra = raw_buffer(a.ha, 0xffffffffu);
    const Q6Off wo = q6_lane_offsets(row * (NB * Q6K_BYTES), h);

    __shared__ AStageR<GK> st[2];
    __shared__ int s_rows[GK];
    __shared__ __attribute__((aligned(16))) float s_dx[NB][GK];

    for (int cb = 0; cb < ne; cb += GK) {
        const int np = min(GK, ne - cb);
        if (tid < GK) s_rows[tid] = n0 + cb + min(tid, np - 1);   // h rows are in dispatch order
        __syncthreads();
        for (int i = tid; i < GK * NB; i += 256) s_dx[i % NB][i / NB] = a.hdx[(size_t)s_rows[i / NB] * NB + (i % NB)];
        StageOff<GK> so;
        stage_offsets(so, s_rows, np, K, wave, lane);
        stage_a_buf<GK, false>(st[0], so, np, ra, ra, 0, wave, lane);
        Q6Lane cw, nw;
        q6_lane_load(cw, rw, wo, 0);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        float y[MT][4];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[t][i] = 0.0f;
#pragma unroll 1
        for (int s = 0; s < NB; ++s) {
            if (s + 1 < NB) {
                q6_lane_load(nw, rw, wo, (s + 1) * Q6K_BYTES);
                stage_a_buf<GK, false>(st[(s + 1) & 1], so, np, ra, ra, s + 1, wave, lane);
            }
            const float d = h2f_dev((uint16_t)cw.d);
            const AStageR<GK> &S = st[s & 1];
            float4_t acc[MT], accl[MT];
            half8_t fa[2][MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc[t] = accl[t] = float4_t{0, 0, 0, 0};
                fa[0][t] = stage_frag(S, 16 * t + n, q6_a_offset(h, 0));
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                half8_t bh, bl;
                if (i + 1 < 8) {
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        fa[(i + 1) & 1][t] = stage_frag(S, 16 * t + n, q6_a_offset(h, i + 1 < 8 ? i + 1 : 0));
                }
                q6_lane_b(cw, i, h, bh, bl);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[t] = mfma32(fa[i & 1][t], bh, acc[t]);
                    accl[t] = mfma32(fa[i & 1][t], bl, accl[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const float4 dxv = *(const float4 *)&s_dx[s][16 * t + 4 * h];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float dx = i == 0 ? dxv.x : i == 1 ? dxv.y : i == 2 ? dxv.z : dxv.w;
                    const float sumi = 16.0f * acc[t][i] + accl[t][i];
                    y[t][i] = y[t][i] + (d * dx) * sumi;   // ggml's order: acc += (d*dx)*sumi
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            cw = nw;
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * t + 4 * h + i;
                if (r < np) {
                    const int q = a.perm[n0 + cb + r];
                    a.ypair[(size_t)q * a.H + row] = a.w[q] * y[t][i];
                }
            }
        __syncthreads();
    }
}

// the trivial dispatch of one expert over n pairs: offsets {0, n}, perm = 0..n-1,
// weights 1 (the always-on shared expert)
__global__ void iota_kernel(int n, int32_t *offsets, int32_t *perm, float *ones) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        perm[i] = i;
        ones[i] = 1.0f;
    }
    if (i == 0) {
        offsets[0] = 0;
        offsets[1] = n;
    }
}

// out[t] (+)= sum_k ypair[t*K + k], k ascending, then the shared expert's row
// yshared[t] if given; one float4 per thread
__global__ __launch_bounds__(256) void combine_kernel(const float *ypair, const float *yshared, int n_tok, int K, int H,
                                                      float *out, int accumulate) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t h4 = (size_t)H / 4;
    if (i >= (size_t)n_tok * h4) return;
    const size_t t = i / h4, c = i % h4;
    const float4 *y = (const float4 *)ypair + (size_t)t * K * h4 + c;
    float4 s = y[0];
    for (int k = 1; k < K; ++k) {
        const float4 v = y[(size_t)k * h4];
        s.x = s.x + v.x; s.y = s.y + v.y; s.z = s.z + v.z; s.w = s.w + v.w;
    }
    float4 *o = (float4 *)out + i;
    if (accumulate) {
        const float4 p = *o;
        s.x = p.x + s.x; s.y = p.y + s.y; s.z = p.z + s.z; s.w = p.w + s.w;
    }
    if (yshared) {
        const float4 v = ((const float4 *)yshared)[i];
        s.x = s.x + v.x; s.y = s.y + v.y; s.z = s.z + v.z; s.w = s.w + v.w;
    }
    *o = s;
}

// the same with the host's rows: pair i's row from hrows when hflag[i] (mapped
// host memory, read over PCIe), else from ypair; k ascending either way
__global__ __launch_bounds__(256) void combine_host_kernel(const float *ypair, const float *hrows, const uint8_t *hflag,
                                                           const float *yshared, int n_tok, int K, int H, float *out,
                                                           int accumulate) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t h4 = (size_t)H / 4;
    if (i >= (size_t)n_tok * h4) return;
    const size_t t = i / h4, c = i % h4;
    auto row = [&](int k) {
        const size_t pr = (size_t)t * K + k;
        return hflag[pr] ? ((const float4 *)hrows)[pr * h4 + c] : ((const float4 *)ypair)[pr * h4 + c];
    };
    float4 s = row(0);
    for (int k = 1; k < K; ++k) {
        const float4 v = row(k);
        s.x = s.x + v.x; s.y = s.y + v.y; s.z = s.z + v.z; s.w = s.w + v.w;
    }
    float4 *o = (float4 *)out + i;
    if (accumulate) {
        const float4 p = *o;
        s.x = p.x + s.x; s.y = p.y + s.y; s.z = p.z + s.z; s.w = p.w + s.w;
    }
    if (yshared) {
        const float4 v = ((const float4 *)yshared)[i];
        s.x = s.x + v.x; s.y = s.y + v.y; s.z = s.z + v.z; s.w = s.w + v.w;
    }
    *o = s;
}

// ---------------------------------------------------------------------------
// launchers (shapes checked by the caller)
template <typename F, typename... A>
static hipError_t launch_b(F k, dim3 grid, dim3 block, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1, A... args) {
    if (ev0) hipExtLaunchKernelGGL(k, grid, block, 0, st, ev0, ev1, 0, args...);
    else hipLaunchKernelGGL(k, grid, block, 0, st, args...);
    return hipGetLastError();
}

hipError_t launch_dispatch(const int32_t *ids, int P, int E, int32_t *counts, int32_t *offsets, int32_t *perm,
                           hipStream_t st) {
    const unsigned segs = (unsigned)max(1, (P + DSP_SEG - 1) / DSP_SEG);
    return launch_b(dispatch_kernel, dim3(segs), dim3(64 * DSP_WAVES), st, nullptr, nullptr, ids, P, E, counts, offsets,
                    perm);
}

hipError_t launch_quant_rows(const void *src, int bf16, int n_rows, int n, uint16_t *q16, float *dx, uint16_t *bs16,
                             bool mfma_order, hipStream_t st) {
    const int64_t blocks = ((int64_t)n_rows * (n / QK) + 3) / 4;
    if (blocks == 0) return hipSuccess;
    return launch_b(mfma_order ? quant_rows_kernel<true> : quant_rows_kernel<false>, dim3((unsigned)blocks), dim3(256),
                    st, nullptr, nullptr, src, bf16, n_rows, n, q16, dx, bs16);
}

hipError_t launch_swiglu_quant(const float *y2, int P, int I, float *h_out, int n_h, uint16_t *q16, float *dx,
                               uint16_t *bs16, hipStream_t st) {
    const int64_t blocks = ((int64_t)P * (I / QK) + 3) / 4;
    if (blocks == 0) return hipSuccess;
    return launch_b(swiglu_quant_kernel, dim3((unsigned)blocks), dim3(256), st, nullptr, nullptr, y2, P, I, h_out, n_h,
                    q16, dx, bs16);
}

// ---------------------------------------------------------------------------
// The Q4_K grouped product of few workgroups (see plan_q4): 64 rows of one
// expert a workgroup, its pairs in passes of MT tiles of 16 on MFMA 16x16x32.  For each
// super-block s the lane's weights are loaded once (block s + 1 in flight
// meanwhile); four waves per SIMD.
template <int NB, bool DOWN, int MT>
__global__ __launch_bounds__(256, 4) void grouped_q4_kernel(GroupedArgs a) {
    constexpr int GK = 16 * MT;           // pairs per pass
    int e, tile;
    tile_expert(blockIdx.x, (DOWN ? a.H : 2 * a.I) / 64, a.E, tile, e);
    const int n0 = a.offsets[e], ne = a.offsets[e + 1] - n0;
    if (ne <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, h = lane >> 4;
    const int r0 = tile * 64;
    const int row = r0 + wave * 16 + n;
    constexpr int K = NB * QK;
    constexpr int ROWB = NB * Q4K_BYTES;
    const int out_n = DOWN ? a.H : 2 * a.I;
    const uint8_t *base = grouped_expert(a, e);
    if (!base) {
        for (int i = tid; i < ne * 64; i += 256) {
            const int pos = n0 + i / 64, c = r0 + (i % 64);
            if (DOWN) a.ypair[(size_t)a.perm[pos] * a.H + c] = 0.0f;
            else a.y2[(size_t)pos * out_n + c] = 0.0f;
        }
        return;
    }
    const uint8_t *mat = DOWN ? base + 2ull * a.I * (a.H / QK) * Q4K_BYTES : base;
    const uint16_t *act = DOWN ? a.ha : a.xa;
    const uint16_t *abs16 = DOWN ? a.hbs : a.xbs;
    const float *adx = DOWN ? a.hdx : a.xdx;

    __shared__ AStageR<GK> st[2];
    __shared__ int s_rows[GK];
    __shared__ __attribute__((aligned(16))) float s_dx[NB][GK];   // [block][pair]: a lane's 4 rows in one read
    const int gm = (h >> 1) + 2 * (h & 1);
    // the expert's matrix, the activation codes and their group sums as raw
    // buffers; the lane's weight offsets (header, the two qs loads) fixed
    const i32x4_t rw = raw_buffer(mat, (uint32_t)((DOWN ? a.H : 2 * a.I) * ROWB));
    const i32x4_t ra = raw_buffer(act, 0xffffffffu), rbs = raw_buffer(abs16, 0xffffffffu);
    const int wo0 = row * ROWB, wo1 = wo0 + 16 + 16 * h, wo2 = wo0 + 80 + 16 * h;

    for (int cb = 0; cb < ne; cb += GK) {
        const int np = min(GK, ne - cb);
        if (tid < GK) {
            const int pos = n0 + cb + min(tid, np - 1);
            s_rows[tid] = DOWN ? pos : a.perm[pos] / a.K;
        }
        __syncthreads();
        for (int i = tid; i < GK * NB; i += 256) s_dx[i % NB][i / NB] = adx[(size_t)s_rows[i / NB] * NB + (i % NB)];
        StageOff<GK> so;
        stage_offsets(so, s_rows, np, K, wave, lane);
        stage_a_buf(st[0], so, np, ra, rbs, 0, wave, lane);
        uint4 cw[3], nw[3];
        cw[0] = buf_load16(rw, wo0, 0);
        cw[1] = buf_load16(rw, wo1, 0);
        cw[2] = buf_load16(rw, wo2, 0);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        float y[MT][4];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[t][i] = 0.0f;
#pragma unroll 1
        for (int s = 0; s < NB; ++s) {
            if (s + 1 < NB) {
                nw[0] = buf_load16(rw, wo0, (s + 1) * Q4K_BYTES);
                nw[1] = buf_load16(rw, wo1, (s + 1) * Q4K_BYTES);
                nw[2] = buf_load16(rw, wo2, (s + 1) * Q4K_BYTES);
            }
            Q4Scales sc;
            q4_scales(cw[0], h, sc);
            const AStageR<GK> &S = st[s & 1];
            if (s + 1 < NB) stage_a_buf(st[(s + 1) & 1], so, np, ra, rbs, s + 1, wave, lane);
            // each 128-value half of the super-block in its own accumulator:
            // a half's products sum to at most 128 * 63 * 15 * 127 < 2^24, so
            // it is exact in fp32, and one add gives ggml's (float)sumi (a
            // whole block's sum can pass 2^24, where a running fp32 sum rounds)
            float4_t acc[MT], acc0[MT];
            // the fragments of K chunk i+1 are read before chunk i's products
            half8_t fa[2][MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc[t] = float4_t{0, 0, 0, 0};
                fa[0][t] = stage_frag(S, 16 * t + n, q4_a_offset(h, 0));
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (i + 1 < 8) {
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        fa[(i + 1) & 1][t] = stage_frag(S, 16 * t + n, q4_a_offset(h, i + 1 < 8 ? i + 1 : 0));
                }
                const int L = i >> 2, nib = (i >> 1) & 1;
                const half8_t bi = q4_b(L ? cw[2] : cw[1], i, sc.sc[L][nib]);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    if (i == 4) {
                        acc0[t] = acc[t];
                        acc[t] = float4_t{0, 0, 0, 0};
                    }
                    acc[t] = mfma32(fa[i & 1][t], bi, acc[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc[t] = acc0[t] + acc[t];
                const float4 dxv = *(const float4 *)&s_dx[s][16 * t + 4 * h];
                const half4_t am = *(const half4_t *)&S.bs[16 * t + n][4 * gm];
                float4_t z = {0, 0, 0, 0};
                z = __builtin_amdgcn_mfma_f32_16x16x16f16(am, sc.bm, z, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // ggml's order: acc += (d*dx)*sumi; acc -= (dmin*dx)*summ
                    const float dx = i == 0 ? dxv.x : i == 1 ? dxv.y : i == 2 ? dxv.z : dxv.w;
                    y[t][i] = y[t][i] + (sc.d * dx) * acc[t][i];
                    y[t][i] = y[t][i] - (sc.dmin * dx) * z[i];
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            cw[0] = nw[0];
            cw[1] = nw[1];
            cw[2] = nw[2];
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * t + 4 * h + i;
                if (r < np) {
                    const int pos = n0 + cb + r;
                    if (DOWN) {
                        const int pp = a.perm[pos];
                        a.ypair[(size_t)pp * a.H + row] = a.w[pp] * y[t][i];
                    } else {
                        a.y2[(size_t)pos * out_n + row] = y[t][i];
                    }
                }
            }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// The Q4_K grouped product on MFMA 32x32x16 f16: a workgroup takes a chunk of up
// to 32 MT pairs of one expert and rtw tiles of 128 rows (four waves of 32).
//
// What bounds it.  The 64-row kernel above reads a row's pieces 16 bytes a lane
// with neighbouring lanes on different rows, so a load touches 64 separate 16-byte
// pieces, and each of its waves reads all the activations of the pass from LDS
// for 16 rows.  Here a wave's raw weights come into LDS lane-contiguous (9 lanes a
// row's 144 bytes; that stride puts the 16 rows an LDS read touches in distinct
// banks), no register holds a load in flight, a fragment serves 32 rows, and the
// activations are staged half a super-block ahead of the products that read
// them.  A lane decodes one nibble pair by v_and_or and v_pk_fma_f16 (1.1
// instructions a weight).  An MFMA leaves the vector unit half of its issue slots
// (measured: 32 cycles alone, 32 with 4 vector instructions, 48 with 8), so the
// vector work (decode, and 7 instructions per output and super-block in ggml's
// order) and the products add up rather than overlap: 352 us of up/gate at 4,096
// tokens x 8 of 128 experts, of which the products alone are ~115.
// MT = 1: 126 registers, four workgroups a CU, which few pairs per expert need to
// keep weights in flight; MT = 3: a decode serves up to three tiles, two a CU.
// us of up/gate (before / here), K = 8, E = 128, I = 768: 64 tokens 58.8 / 56.2,
// 197 69 / 59, 512 97 / 78, 2,048 256 / 196, 4,096 468 / 352; down 36.0 / 32.8,
// 44 / 35, 71 / 47, -, 403 / 215.
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef float float32_t __attribute__((ext_vector_type(32)));
constexpr int TL_ROWS = 128;            // rows of a workgroup
constexpr int TL_WB = 32 * Q4K_BYTES;   // one wave's raw weights of a super-block
// A direct load into LDS, 16 bytes a lane, lane-contiguous at lds (it writes no
// register).  Not by the builtin: the compiler waits for every such load in flight
// before an LDS read it cannot tell apart.  These are waited for by hand (vmcnt,
// then a barrier).
__device__ inline void dma16(uint32_t lds, int voff, i32x4_t rsrc, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "m0", "memory");
}
// A store of one word a lane, one instruction whatever the compiler makes of its
// neighbours: waits after it count the stores in flight.  (No memory clobber: it is
// in order with the loads and waits here, and nothing reads what it writes.)
__device__ inline void store_f32(float v, i32x4_t rsrc, int voff) {
    asm volatile("buffer_store_dword %0, %1, %2, 0 offen" :: "v"(v), "v"(voff), "s"(rsrc));
}
__device__ void buffer_store_f32(float v, i32x4_t rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.store.f32");
// the finished rows of one tile of 32 pairs: the pairs' gate weights gw and output rows pp in
// LDS (four of them read ahead of the stores), y to column col; rows past the chunk's pairs
// lie past the buffer's end.  16 stores
__device__ inline void store_down(const float y[16], const float *gw, const uint32_t *pp, i32x4_t ro, int h, int col) {
    float4 g[2];
    uint4 p[2];
    g[0] = *(const float4 *)&gw[4 * h];
    p[0] = *(const uint4 *)&pp[4 * h];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i + 1 < 4) {
            g[(i + 1) & 1] = *(const float4 *)&gw[8 * (i + 1) + 4 * h];
            p[(i + 1) & 1] = *(const uint4 *)&pp[8 * (i + 1) + 4 * h];
        }
        const float4 w = g[i & 1];
        const uint4 r = p[i & 1];
        store_f32(w.x * y[4 * i], ro, (int)(r.x + (uint32_t)col));
        store_f32(w.y * y[4 * i + 1], ro, (int)(r.y + (uint32_t)col));
        store_f32(w.z * y[4 * i + 2], ro, (int)(r.z + (uint32_t)col));
        store_f32(w.w * y[4 * i + 3], ro, (int)(r.w + (uint32_t)col));
    }
}
__device__ inline uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(lptr_t *)p; }
constexpr uint32_t TL_NONE = 0xe0000000u;      // an offset past every buffer: reads zeros, is not stored
constexpr int TL_QUAD = 1024 + 16;      // half a super-block of four rows of activation codes in LDS

__device__ inline void vm_lds_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The experts' pairs in chunks of up to mt tiles of 32, an expert's tiles spread
// evenly over its chunks; experts in order.  A wave finds chunk c from the
// dispatch's offsets (4 experts a lane) and a prefix sum over the lanes.
struct Chunk { int e, p0, np; };
struct ChunkScan { int off[5], cnt[4], before, total; };
__device__ inline ChunkScan chunk_scan(const int32_t *offsets, int E, int mt, int lane) {
    ChunkScan r;
#pragma unroll
    for (int j = 0; j < 5; ++j) r.off[j] = offsets[min(4 * lane + j, E)];
    int sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int tiles = (r.off[j + 1] - r.off[j] + 31) / 32;
        r.cnt[j] = (tiles + mt - 1) / mt;
        sum += r.cnt[j];
    }
    const int incl = wave_incl_sum(sum, lane);
    r.before = incl - sum;
    r.total = __builtin_amdgcn_readlane(incl, 63);
    return r;
}
__device__ inline Chunk chunk_find(const ChunkScan &s, int c, int lane) {
    int e = -1, p0 = 0, np = 0, b = s.before;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k = c - b;
        if (k >= 0 && k < s.cnt[j]) {
            const int n = s.off[j + 1] - s.off[j], tiles = (n + 31) / 32;
            const int t0 = k * tiles / s.cnt[j], t1 = (k + 1) * tiles / s.cnt[j];
            e = 4 * lane + j;
            p0 = s.off[j] + 32 * t0;
            np = min(n, 32 * t1) - 32 * t0;
        }
        b += s.cnt[j];
    }
    const int src = (int)__builtin_ctzll(__ballot(e >= 0));
    return Chunk{__builtin_amdgcn_readlane(e, src), __builtin_amdgcn_readlane(p0, src), __builtin_amdgcn_readlane(np, src)};
}

// The task'th chunk: with a shared expert its chunks first (e = -1; rows
// P .. P + n_tok - 1 of the activations and up/gate rows), then the routed ones.
__device__ inline int shared_chunks(const GroupedArgs &a, int mt) {
    return a.shared ? ((a.P / a.K + 31) / 32 + mt - 1) / mt : 0;
}
__device__ inline Chunk chunk_of(const GroupedArgs &a, const ChunkScan &scan, int c, int ns, int lane) {
    if (c >= ns) return chunk_find(scan, c - ns, lane);
    const int n = a.P / a.K, tiles = (n + 31) / 32;
    const int t0 = c * tiles / ns, t1 = (c + 1) * tiles / ns;
    return Chunk{-1, a.P + 32 * t0, min(n, 32 * t1) - 32 * t0};
}

// 4 nibbles' worth of B: words of nibbles under masks -> (1024 + q) * sc - 1024 * sc,
// high nibbles as (1024 + 16 q) * (sc / 16) - 64 * sc: one rounding of an exact integer
__device__ inline half8_t q4_tile_b(uint32_t w0, uint32_t w1, uint32_t M, uint32_t X, _Float16 s, _Float16 nb) {
    uint4 r;
    r.x = (w0 & M) | X;
    r.y = ((w0 >> 8) & M) | X;
    r.z = (w1 & M) | X;
    r.w = ((w1 >> 8) & M) | X;
    return __builtin_elementwise_fma(__builtin_bit_cast(half8_t, r), splat8(s), splat8(nb));
}

template <int NB, bool DOWN, int MT>
__global__ __launch_bounds__(256, MT == 1 ? 4 : 2) void grouped_q4_tile_kernel(GroupedArgs a, int row_tiles) {
    const int rtw = DOWN ? row_tiles : 1;
    constexpr int GK = 32 * MT;
    constexpr int K = NB * QK;
    constexpr int ROWB = NB * Q4K_BYTES;
    const int out_n = DOWN ? a.H : 2 * a.I;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> (chunk, rtw row tiles): each XCD a contiguous run of them, a chunk's
    // together
    const int nt_r = out_n / (TL_ROWS * rtw);
    const ChunkScan scan = chunk_scan(a.offsets, a.E, MT, lane);
    const int ns = shared_chunks(a, MT), total = (ns + scan.total) * nt_r;
    const int per = (total + 7) / 8, li = (int)blockIdx.x >> 3;
    const int task = ((int)blockIdx.x & 7) * per + li;
    if (li >= per || task >= total) return;
    const Chunk ch = chunk_of(a, scan, task / nt_r, ns, lane);
    const bool sh = ch.e < 0;
    const int r0 = (task % nt_r) * (TL_ROWS * rtw);
    const int np = ch.np, nt = (np + 31) / 32;
    const uint8_t *base = sh ? a.shared : grouped_expert(a, ch.e);
    if (!base) {
        for (int rt = 0; rt < rtw; ++rt)
            for (int i = tid; i < np * TL_ROWS; i += 256) {
                const int pos = ch.p0 + i / TL_ROWS, c = r0 + rt * TL_ROWS + (i % TL_ROWS);
                if (DOWN) a.ypair[(size_t)a.perm[pos] * a.H + c] = 0.0f;
                else a.y2[(size_t)pos * out_n + c] = 0.0f;
            }
        return;
    }
    const uint8_t *mat = DOWN ? base + 2ull * a.I * (a.H / QK) * Q4K_BYTES : base;
    const float *adx = DOWN ? a.hdx : a.xdx;
    const i32x4_t rw = raw_buffer(mat, (uint32_t)((DOWN ? a.H : 2 * a.I) * ROWB));
    // the activation rows; the rows past the chunk's pairs lie past the end and read as
    // zeros, which costs the products no traffic and little power (a full tile of
    // repeated rows slowed the whole of a 64-token batch by ~3 %)
    const uint32_t n_tok = (uint32_t)(a.P / a.K), n_rows = DOWN ? a.P + (sh ? n_tok : 0u) : n_tok;
    const i32x4_t ra = raw_buffer(DOWN ? a.ha : a.xa, n_rows * (2 * K));
    const i32x4_t rbs = raw_buffer(DOWN ? a.hbs : a.xbs, n_rows * (K / 8));

    // Activation codes, half a super-block at a time (the half's products read 8
    // 16-byte chunks of each 128 values): four rows of 256 bytes per direct load,
    // chunk c of row r at c ^ 4 (r & 3), four rows to 1040 bytes: the 16 rows one
    // fragment read touches fall in distinct banks.
    __shared__ __attribute__((aligned(16))) uint8_t s_a[2][GK / 4][TL_QUAD];
    __shared__ __attribute__((aligned(16))) _Float16 s_bs[GK][16];
    __shared__ __attribute__((aligned(16))) uint8_t s_w[4][TL_WB];
    __shared__ __attribute__((aligned(16))) float s_dx[NB][GK];
    __shared__ __attribute__((aligned(16))) uint32_t s_row[GK];                 // the pair's activation row, in bytes
    __shared__ __attribute__((aligned(16))) uint32_t s_pp[DOWN ? GK : 4];   // its output row, in bytes
    __shared__ __attribute__((aligned(16))) float s_gw[DOWN ? GK : 4];

    // the wave's raw weights of super-block s: its 32 rows' 144 bytes, lane-contiguous (5 loads;
    // the lane's offsets in LDS, as its activation rows are: the products need the registers)
    __shared__ int s_wo[5][64];
    const uint32_t lw = lds_addr(&s_w[wave][0]), la = lds_addr(&s_a[0][2 * wave][0]), lb = lds_addr(&s_bs[32 * wave][0]);
    auto load_w = [&](int rt, int s, bool first) {            // of row tile rt
        const int so = (r0 + TL_ROWS * rt + 32 * wave) * ROWB + s * Q4K_BYTES;
        int o[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            const int c = lane + 64 * j;
            o[j] = first ? (c / 9) * ROWB + 16 * (c % 9) : s_wo[j][lane];
            if (first && wave == 0) s_wo[j][lane] = o[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16(lw + 1024 * j, o[j], rw, so);
        if (lane < 32) dma16(lw + 4096, o[4], rw, so);
    };
    load_w(0, 0, true);
    for (int i = tid; i < GK; i += 256) {
        const int pos = ch.p0 + min(i, np - 1);
        const int row = DOWN ? pos : sh ? pos - a.P : a.perm[pos] / a.K;
        s_row[i] = i < np ? (uint32_t)row * (2 * K) : TL_NONE;
#pragma unroll
        for (int b = 0; b < NB; ++b) s_dx[b][i] = adx[(size_t)row * NB + b];
    }
    // the pairs' output rows and gate weights, fetched beside the first activations
    auto pairs = [&]() {
        for (int i = tid; i < GK; i += 256) {
            const int pos = ch.p0 + min(i, np - 1);
            const int pr = sh ? pos - a.P : a.perm[pos];
            s_pp[i] = i < np ? (uint32_t)pr * (uint32_t)(4 * a.H) : TL_NONE;        // not stored
            s_gw[i] = sh ? 1.0f : a.w[pr];
        }
    };
    __syncthreads();
    const int ac = ((lane & 15) ^ (4 * (lane >> 4)));
    const int ao = 256 * (ac >> 3) + 16 * (ac & 7);
    auto load_a = [&](auto ntc, int s, int hf) {          // half hf of super-block s
        constexpr int NT = decltype(ntc)::value;
        uint32_t o[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) o[t][j] = s_row[4 * (8 * t + 2 * wave + j) + (lane >> 4)];
        const uint32_t ob = hf ? s_row[32 * min(wave, NT - 1) + (lane >> 1)] : 0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                dma16(la + (hf * (GK / 4) + 8 * t + j) * TL_QUAD, (int)(o[t][j] + ao), ra, s * QK * 2 + 128 * hf);
        if (hf && wave < NT) dma16(lb, (int)(ob / 16 + 16 * (lane & 1)), rbs, s * 32);      // the group sums, for after the second half
    };
    const i32x4_t ro = DOWN ? raw_buffer(sh ? a.yshared : a.ypair, (sh ? n_tok : (uint32_t)a.P) * (uint32_t)(4 * a.H))
                            : raw_buffer(a.y2 + (size_t)ch.p0 * out_n, (uint32_t)np * (uint32_t)(4 * out_n));
    const int n = lane & 31, h = lane >> 5;
    const uint32_t hm = 0u - (uint32_t)h;
    // the lane's fragments of its row in a half: chunks 8h + 0..3 and 8h + 4..7
    const uint8_t *fr = &s_a[0][n >> 2][256 * (n & 3)];
    const uint8_t *f0 = fr + 16 * ((8 * h) ^ (4 * (n & 3))), *f1 = fr + 16 * ((8 * h + 4) ^ (4 * (n & 3)));
    auto frag = [&](int hf, int t, int i) {
        return *(const half8_t *)((i < 4 ? f0 : f1) + 16 * (i & 3) + (hf * (GK / 4) + 8 * t) * TL_QUAD);
    };
    // masks and the exponent in registers: one v_and_or each
    uint32_t mlo, mhi, mx;
    asm("s_mov_b32 %0, 0x000f000f" : "=s"(mlo));
    asm("s_mov_b32 %0, 0x00f000f0" : "=s"(mhi));
    asm("v_mov_b32 %0, 0x64006400" : "=v"(mx));
    float y[MT][16];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;

    // the chunk's NT tiles.  Written in the order it is to run in, fixed by the
    // scheduling barriers: a product, the read of the fragment its register is
    // needed for next, and beside them the vector work at hand (the decode of the
    // next operand, or the sums of the tile before).
    auto body = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        load_a(ntc, 0, 0);
        if (DOWN) pairs();
        vm_lds_barrier();
        load_a(ntc, 0, 1);
        // the finished rows of a row tile (up/gate has one, stored after the last wait)
        auto store = [&](int rt) {
            const int col = 4 * (r0 + TL_ROWS * rt + 32 * wave + n) + (DOWN ? 0 : 16 * h * out_n);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (DOWN) {
                    store_down(y[t], s_gw + 32 * t, s_pp + 32 * t, ro, h, col);
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        buffer_store_f32(y[t][i], ro, (32 * t + 8 * (i >> 2) + (i & 3)) * 4 * out_n + col, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;
            }
        };
        int rt = 0, s = 0;
#pragma unroll 1
        for (;;) {
            const bool last = s == NB - 1 && rt == rtw - 1;
            const int s1 = s == NB - 1 ? 0 : s + 1, rt1 = s == NB - 1 ? rt + 1 : rt;      // the next step
            // the lane's half of its row's super-block: sub-blocks 4h .. 4h + 3
            const uint8_t *wp = &s_w[wave][n * Q4K_BYTES];
            const uint4 hdr = *(const uint4 *)wp;
            uint4 q[4];
#pragma unroll
            for (int L = 0; L < 4; ++L) q[L] = *(const uint4 *)(wp + 16 + 64 * h + 16 * L);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // done with s_w
            if (!last) load_w(rt1, s1, false);
            // the rows of the tile before, behind the loads this step waits for
            const bool stored = s == 0 && rt > 0;
            if (stored) store(rt - 1);
            half8_t f[8], b[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = frag(0, 0, i);
            const uint32_t sc0 = hdr.y & 0x3f3f3f3fu, mn0 = hdr.z & 0x3f3f3f3fu;
            const uint32_t sc1 = (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u);
            const uint32_t mn1 = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
            const uint32_t scb = (sc1 & hm) | (sc0 & ~hm), mnb = (mn1 & hm) | (mn0 & ~hm);
            // B of product i of half hf: 8 values of sub-block 4h + 2hf (low nibbles, i < 4) or the next (high)
            _Float16 sf[2], sn[2];
            auto scales = [&](int hf) {
#pragma unroll
                for (int nib = 0; nib < 2; ++nib) {
                    const float sc = (float)((scb >> (8 * (2 * hf + nib))) & 0xffu);
                    sf[nib] = (_Float16)(nib ? sc * 0.0625f : sc);
                    sn[nib] = (_Float16)(sc * (nib ? -64.0f : -1024.0f));
                }
            };
            auto operand = [&](int hf, int i) {
                const uint4 &w = q[2 * hf + ((i >> 1) & 1)];
                return q4_tile_b((i & 1) ? w.z : w.x, (i & 1) ? w.w : w.y, i < 4 ? mlo : mhi, mx, sf[i >> 2], sn[i >> 2]);
            };
            float16_t a0[NT];
            scales(0);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (t == 0) b[i] = operand(0, i);
                    a0[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], b[i], i ? a0[t] : float16_t{}, 0, 0, 0);
                    if (t + 1 < NT) f[i] = frag(0, t + 1, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
            const float d = h2f_dev((uint16_t)(hdr.x & 0xffffu)), dmin = h2f_dev((uint16_t)(hdr.x >> 16));
            half8_t bm;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const _Float16 m = (_Float16)(float)((mnb >> (8 * j)) & 0xffu);
                bm[2 * j] = m;
                bm[2 * j + 1] = m;
            }
            scales(1);
            // the second half has landed (only the next weights, 5 loads, and the stores stay in
            // flight) and every wave is done with the first
            if (last) {
                vm_lds_barrier();
            } else {
                if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(5 + 16 * NT) : "memory");
                else asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                load_a(ntc, s1, 0);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = frag(1, 0, i);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                float16_t a1;
                const half8_t am = *(const half8_t *)&s_bs[32 * t + n][8 * h];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (t == 0) b[i] = operand(1, i);
                    a1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], b[i], i ? a1 : float16_t{}, 0, 0, 0);
                    if (t + 1 < NT) f[i] = frag(1, t + 1, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const float16_t z = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bm, float16_t{}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 dx = *(const float4 *)&s_dx[s][32 * t + 8 * i + 4 * h];
                    // ggml's order: acc += (d*dx)*sumi; acc -= (dmin*dx)*summ
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float x = j == 0 ? dx.x : j == 1 ? dx.y : j == 2 ? dx.z : dx.w;
                        float &v = y[t][4 * i + j];
                        v = v + (d * x) * (a0[t][4 * i + j] + a1[4 * i + j]);
                        v = v - (dmin * x) * z[4 * i + j];
                        asm volatile("" : "+v"(v));         // here, not at the end
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (last) break;
            vm_lds_barrier();               // the next weights and first half; the second half and the sums are read
            load_a(ntc, s1, 1);
            s = s1;
            rt = rt1;
        }
        store(rtw - 1);
    };
    if (MT >= 3 && nt == 3) body(std::integral_constant<int, MT < 3 ? 1 : 3>{});
    else if (MT >= 2 && nt == 2) body(std::integral_constant<int, MT < 2 ? 1 : 2>{});
    else body(std::integral_constant<int, 1>{});
}

// The same for a Q6_K down matrix (see q6_lane_b for the two exact products): the
// raw weights of a wave's 32 rows come as the 14 aligned 16-byte pieces that hold
// each row's 210-byte block, which starts at any even byte m of the first; a lane
// reads its half of the block from LDS as words and shifts them by m & 2.  Whole
// blocks' sums stay exact in one accumulator a product.  Bound by the decode (two
// operands of every weight, ~410 vector instructions a super-block of 32 rows)
// and, for few pairs, by the weights' latency.  us of down (before / here), E = 128,
// I = 768: 16 tokens x 8 48 / 39, 64 62 / 51, 512 100 / 69, 2,000 266 / 163.
constexpr int TL_W6 = 224;              // a row's pieces in LDS
template <int NB, int MT>
__global__ __launch_bounds__(256, MT == 1 ? 3 : 2) void grouped_q6_tile_kernel(GroupedArgs a, int rtw) {
    constexpr int GK = 32 * MT;
    constexpr int K = NB * QK;
    constexpr int ROWB = NB * Q6K_BYTES;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt_r = a.H / (TL_ROWS * rtw);
    const ChunkScan scan = chunk_scan(a.offsets, a.E, MT, lane);
    const int ns = shared_chunks(a, MT), total = (ns + scan.total) * nt_r;
    const int per = (total + 7) / 8, li = (int)blockIdx.x >> 3;
    const int task = ((int)blockIdx.x & 7) * per + li;
    if (li >= per || task >= total) return;
    const Chunk ch = chunk_of(a, scan, task / nt_r, ns, lane);
    const bool sh = ch.e < 0;
    const int r0 = (task % nt_r) * (TL_ROWS * rtw);
    const int np = ch.np, nt = (np + 31) / 32;
    const uint8_t *base = sh ? a.shared : grouped_expert(a, ch.e);
    if (!base) {
        for (int rt = 0; rt < rtw; ++rt)
            for (int i = tid; i < np * TL_ROWS; i += 256)
                a.ypair[(size_t)a.perm[ch.p0 + i / TL_ROWS] * a.H + r0 + rt * TL_ROWS + (i % TL_ROWS)] = 0.0f;
        return;
    }
    const i32x4_t rw = raw_buffer(base + 2ull * a.I * (a.H / QK) * Q4K_BYTES, (uint32_t)(a.H * ROWB));
    const uint32_t n_out = (uint32_t)(sh ? a.P / a.K : a.P);
    const i32x4_t ra = raw_buffer(a.ha, (uint32_t)(a.P + (sh ? a.P / a.K : 0)) * (2 * K));
    const i32x4_t ro = raw_buffer(sh ? a.yshared : a.ypair, n_out * (uint32_t)(4 * a.H));

    __shared__ __attribute__((aligned(16))) uint8_t s_a[2][GK / 4][TL_QUAD];       // as in the Q4_K kernel
    __shared__ __attribute__((aligned(16))) uint8_t s_w[4][32 * TL_W6];
    __shared__ __attribute__((aligned(16))) float s_dx[NB][GK];
    __shared__ __attribute__((aligned(16))) uint32_t s_row[GK];
    __shared__ __attribute__((aligned(16))) uint32_t s_pp[GK];
    __shared__ __attribute__((aligned(16))) float s_gw[GK];
    __shared__ uint32_t s_wo[7][64];                // piece c = 64 j + lane: row c / 14 (bytes), 16 (c % 14) above
    const uint32_t lw = lds_addr(&s_w[wave][0]), la = lds_addr(&s_a[0][2 * wave][0]);
    auto load_w = [&](int rt, int s, bool first) {              // 7 loads; 32 rows are a multiple of 16 bytes
        const int so = (r0 + TL_ROWS * rt + 32 * wave) * ROWB;
        uint32_t o[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            const int c = lane + 64 * j;
            o[j] = first ? (uint32_t)((c / 14) * ROWB) | ((uint32_t)(16 * (c % 14)) << 16) : s_wo[j][lane];
            if (first && wave == 0) s_wo[j][lane] = o[j];
        }
#pragma unroll
        for (int j = 0; j < 7; ++j)
            dma16(lw + 1024 * j, (int)((((o[j] & 0xffffu) + s * Q6K_BYTES) & ~15u) + (o[j] >> 16)), rw, so);
    };
    load_w(0, 0, true);
    for (int i = tid; i < GK; i += 256) {
        const int pos = ch.p0 + min(i, np - 1);
        s_row[i] = i < np ? (uint32_t)pos * (2 * K) : TL_NONE;      // (zeros, as in the Q4_K kernel)
#pragma unroll
        for (int b = 0; b < NB; ++b) s_dx[b][i] = a.hdx[(size_t)pos * NB + b];
    }
    auto pairs = [&]() {
        for (int i = tid; i < GK; i += 256) {
            const int pos = ch.p0 + min(i, np - 1);
            const int pr = sh ? pos - a.P : a.perm[pos];
            s_pp[i] = i < np ? (uint32_t)pr * (uint32_t)(4 * a.H) : TL_NONE;        // not stored
            s_gw[i] = sh ? 1.0f : a.w[pr];
        }
    };
    __syncthreads();
    const int ac = ((lane & 15) ^ (4 * (lane >> 4)));
    const int ao = 256 * (ac >> 3) + 16 * (ac & 7);
    auto load_a = [&](auto ntc, int s, int hf) {
        constexpr int NT = decltype(ntc)::value;
        uint32_t o[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) o[t][j] = s_row[4 * (8 * t + 2 * wave + j) + (lane >> 4)];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                dma16(la + (hf * (GK / 4) + 8 * t + j) * TL_QUAD, (int)(o[t][j] + ao), ra, s * QK * 2 + 128 * hf);
    };
    const int n = lane & 31, h = lane >> 5;
    const uint8_t *fr = &s_a[0][n >> 2][256 * (n & 3)];
    const uint8_t *f0 = fr + 16 * ((8 * h) ^ (4 * (n & 3))), *f1 = fr + 16 * ((8 * h + 4) ^ (4 * (n & 3)));
    auto frag = [&](int hf, int t, int i) {
        return *(const half8_t *)((i < 4 ? f0 : f1) + 16 * (i & 3) + (hf * (GK / 4) + 8 * t) * TL_QUAD);
    };
    float y[MT][16];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;

    auto body = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        load_a(ntc, 0, 0);
        pairs();
        vm_lds_barrier();
        load_a(ntc, 0, 1);
        auto store = [&](int rt) {                  // 16 NT stores
            const int col = 4 * (r0 + TL_ROWS * rt + 32 * wave + n);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                store_down(y[t], s_gw + 32 * t, s_pp + 32 * t, ro, h, col);
#pragma unroll
                for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;
            }
        };
        int rt = 0, s = 0;
#pragma unroll 1
        for (;;) {
            const bool last = s == NB - 1 && rt == rtw - 1;
            const int s1 = s == NB - 1 ? 0 : s + 1, rt1 = s == NB - 1 ? rt + 1 : rt;      // the next step
            // the lane's half of its row's block: ql 64 bytes, qh 32, 8 scales, and d
            const int m = (n * ROWB + s * Q6K_BYTES) & 15;
            const uint8_t *wp = &s_w[wave][n * TL_W6 + (m & ~3)];
            uint32_t ql[17], qh[9], qs[3];
            __builtin_memcpy(ql, __builtin_assume_aligned(wp + 64 * h, 4), 68);
            __builtin_memcpy(qh, __builtin_assume_aligned(wp + 128 + 32 * h, 4), 36);
            __builtin_memcpy(qs, __builtin_assume_aligned(wp + 192 + 8 * h, 4), 12);
            const float d = h2f_dev(*(const uint16_t *)(wp + 208 + (m & 2)));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // done with s_w
            if (!last) load_w(rt1, s1, false);
            const bool stored = s == 0 && rt > 0;
            if (stored) store(rt - 1);
            half8_t f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = frag(0, 0, i);
            const uint32_t sb = (uint32_t)(m & 2);
#pragma unroll
            for (int j = 0; j < 16; ++j) ql[j] = __builtin_amdgcn_alignbyte(ql[j + 1], ql[j], sb);
#pragma unroll
            for (int j = 0; j < 8; ++j) qh[j] = __builtin_amdgcn_alignbyte(qh[j + 1], qh[j], sb);
#pragma unroll
            for (int j = 0; j < 2; ++j) qs[j] = __builtin_amdgcn_alignbyte(qs[j + 1], qs[j], sb);
            // B of product i of half hf: values 8 (i & 3) .. of group g = 2 hf + (i >> 2), of scale 2 g + ((i >> 1) & 1)
            _Float16 sh[4], sl[4];
            auto scales = [&](int hf) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int sc = (int)qs[hf] << (24 - 8 * j) >> 24;
                    sh[j] = (_Float16)(short)(sc >> 4);
                    sl[j] = (_Float16)(short)(sc & 15);
                }
            };
            auto operand = [&](int hf, int i, half8_t &bh, half8_t &bl) {
                const uint32_t M = 0x0F0F0F0Fu, HM = 0x30303030u;
                const int g = 2 * hf + (i >> 2), k = i & 3;
                uint32_t v[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t lw_ = ql[8 * (g & 1) + 2 * k + j], hw = qh[2 * k + j];
                    const uint32_t lo = (g >= 2 ? lw_ >> 4 : lw_) & M;
                    const uint32_t hi = (g == 0 ? hw << 4 : g == 1 ? hw << 2 : g == 2 ? hw : hw >> 2) & HM;
                    v[j] = lo | hi;
                }
                const half8_t q = pack_1024(v[0], v[1]);
                const _Float16 s0 = sh[2 * (i >> 2) + (k >> 1)], s1_ = sl[2 * (i >> 2) + (k >> 1)];
                bh = __builtin_elementwise_fma(q, splat8(s0), splat8(s0 * (_Float16)-1056.0f));
                bl = __builtin_elementwise_fma(q, splat8(s1_), splat8(s1_ * (_Float16)-1056.0f));
            };
            float16_t ah[NT], al[NT];
            half8_t bh[8], bl[8];
            auto half = [&](auto hfc) {
                constexpr int hf = decltype(hfc)::value;
                scales(hf);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        if (t == 0) operand(hf, i, bh[i], bl[i]);
                        const bool first = hf == 0 && i == 0;
                        ah[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], bh[i], first ? float16_t{} : ah[t], 0, 0, 0);
                        al[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], bl[i], first ? float16_t{} : al[t], 0, 0, 0);
                        if (t + 1 < NT) f[i] = frag(hf, t + 1, i);
                        __builtin_amdgcn_sched_barrier(0);
                    }
            };
            half(std::integral_constant<int, 0>{});
            // the second half has landed (only the next weights, 7 loads, and the stores stay in
            // flight) and every wave is done with the first
            if (last) {
                vm_lds_barrier();
            } else {
                if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(7 + 16 * NT) : "memory");
                else asm volatile("s_waitcnt vmcnt(7) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                load_a(ntc, s1, 0);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = frag(1, 0, i);
            half(std::integral_constant<int, 1>{});
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 dx = *(const float4 *)&s_dx[s][32 * t + 8 * i + 4 * h];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float x = j == 0 ? dx.x : j == 1 ? dx.y : j == 2 ? dx.z : dx.w;
                        float &v = y[t][4 * i + j];
                        // ggml's order: acc += (d*dx)*sumi; 16 ah is exact, so the fmaf rounds once
                        v = v + (d * x) * fmaf(16.0f, ah[t][4 * i + j], al[t][4 * i + j]);
                        asm volatile("" : "+v"(v));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (last) break;
            vm_lds_barrier();               // the next weights and first half; the second half is read
            load_a(ntc, s1, 1);
            s = s1;
            rt = rt1;
        }
        store(rtw - 1);
    };
    if (MT >= 2 && nt == 2) body(std::integral_constant<int, MT < 2 ? 1 : 2>{});
    else body(std::integral_constant<int, 1>{});
}

template <int MT>
static int shared_chunks_max(const GroupedArgs &a) { return a.shared ? (a.P / a.K + 31) / 32 / MT + 1 : 0; }

template <bool DOWN, int MT>
static hipError_t launch_tile(const GroupedArgs &a, int rtw, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const int rows = DOWN ? a.H : 2 * a.I, nb = (DOWN ? a.I : a.H) / QK;
    // chunks: at most P / (32 MT) full ones and one more per expert; the rest of the grid returns at once
    const int64_t tasks = (int64_t)(a.P / (32 * MT) + a.E + shared_chunks_max<MT>(a)) * (rows / (TL_ROWS * rtw));
    const dim3 grid((unsigned)((tasks + 7) / 8 * 8)), blk(256);
    if constexpr (!DOWN) return launch_b(grouped_q4_tile_kernel<8, false, MT>, grid, blk, st, e0, e1, a, rtw);
    else if (nb == 3) return launch_b(grouped_q4_tile_kernel<3, true, MT>, grid, blk, st, e0, e1, a, rtw);
    else if (nb == 2) return launch_b(grouped_q4_tile_kernel<2, true, MT>, grid, blk, st, e0, e1, a, rtw);
    else return launch_b(grouped_q4_tile_kernel<1, true, MT>, grid, blk, st, e0, e1, a, rtw);
}

// Row tiles a workgroup takes of a down matrix in host memory: four where a row is one
// super-block, or for few pairs, but one for so few that the workgroups of an absent expert or
// two wait on PCIe's latency (ms of down, one / four: 128 experts, I = 768, 16 tokens 1.53 / 1.52, 200 2.47 /
// 2.74; 256, I = 512, 4 tokens 0.393 / 0.349; 64, I = 256, 4 tokens 0.187 / 0.151, 200 0.381 / 0.368; two layers of
// 128 experts, 16 of them absent, batch of 2, the whole call 0.324 / 0.347).
static int host_row_tiles(const GroupedArgs &a) { return a.I == QK || (a.P > 16 && a.P <= 2 * a.E) ? 4 : 1; }

// How a Q4_K product runs.  `full` estimates the chunks of one tile that the batch
// fills.
//   few  no more than 512 workgroups of 128 rows: the 64-row kernel has twice as many. A
//        pass of one tile while 16 pairs serve an expert, or the one expert of 16 tokens; of two
//        tiles to twice that (us of up/gate, there / on tiles: 64 experts, I = 256, 64 tokens 14.3 / 17.2, 128 tokens 16.0 /
//        17.4; 128, I = 256, 16-96 tokens 19.0-20.4 / 21.2-22.4, 128 tokens 23.4 / 22.4; 8 experts, I = 768, 48 pairs 10.0 / 16.0,
//        128 pairs 12.0 / 16.2, 192 pairs 18.2 / 16.6; one expert, 16 tokens 9.7 / 15.8, 32 12.1 / 15.9, 33 21.3 / 15.6)
//   wide chunks of three tiles, where they fill the chip and are mostly full themselves:
//        up/gate from 40 pairs per expert and 510 workgroups on (us, one tile / three: 128 experts, I =
//        768, 32 pairs 77.7 / 82.5, 40 90.9 / 85.8, 64 115.3 / 107.5, 250 354 / 319; 256, I = 512, 40 117.5 /
//        113.1; 64, I = 768, 64 pairs, 504 workgroups, 62.9 / 65.2), down with four row tiles from
//        600 workgroups on, or where a chunk holds an expert and these fill the 512 places of one
//        round (128 experts, I = 768, 40 pairs 55.5 / 52.4, 64 68.5 / 66.6, 96 91.3 / 107.5, 128 116.9 /
//        113.7; 64 experts, 64 pairs 40.0 / 43.6)
//   host with weights in host memory, chunks of three tiles at any number of pairs: an expert is
//        read once per chunk over PCIe, and two workgroups a CU instead of four read faster,
//        probably as fewer of the lines that two super-blocks share are fetched twice (all weights
//        pinned, 128 experts, I = 768, ms of up/gate + down, one tile / three: 64 tokens 5.86 + 3.28 /
//        5.20 + 2.42, 200 5.94 + 3.36 / 5.25 + 2.47, 700 6.00 + 2.98 / 5.34 + 2.57; 64-row kernels
//        in passes of 32 pairs, each chunk of two read once, 5.35 + 2.64)
// Down rows (short K) take several row tiles a workgroup, which share its start (us: 512
// tokens 48.7 with one, 46.8 with two; 4,096 255 with one, 215 with four of three tiles).
static GroupedPlan plan_q4(const GroupedArgs &a, bool down) {
    const int rt = (down ? a.H : 2 * a.I) / TL_ROWS, full = max(a.P / 32, min(a.E, a.P));
    const bool wide = down ? a.P >= 64 * a.E && a.P / 96 * (rt / 4) >= 600 : a.P >= 40 * a.E && a.P / 96 * rt >= 510;
    if (wide) return {TL_ROWS, 3, down ? 4 : 1};
    if (a.host) return {TL_ROWS, 3, down ? host_row_tiles(a) : 1};
    if (down && a.P >= 36 * a.E && a.P <= 64 * a.E && a.E * (rt / 4) >= 512) return {TL_ROWS, 3, 4};
    if (!a.shared) {
        if ((full * rt < 512 || (a.E * rt <= 512 && a.P < 1024)) && a.P <= 8 * a.E + 8) return {64, 1, 1};
        if (a.E * rt < 512 && a.P <= 16 * a.E + 16) return {64, 2, 1};
    }
    return {TL_ROWS, 1, down && full * rt >= 2048 ? 2 : 1};
}

template <bool DOWN, int MT>
static hipError_t launch_rows64(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const int rows = DOWN ? a.H : 2 * a.I, nb = (DOWN ? a.I : a.H) / QK;
    const dim3 grid((unsigned)(rows / 64 * a.E)), blk(256);     // (row tile, expert) from the linear id
    if constexpr (!DOWN) return launch_b(grouped_q4_kernel<8, false, MT>, grid, blk, st, e0, e1, a);
    else if (nb == 3) return launch_b(grouped_q4_kernel<3, true, MT>, grid, blk, st, e0, e1, a);
    else if (nb == 2) return launch_b(grouped_q4_kernel<2, true, MT>, grid, blk, st, e0, e1, a);
    else return launch_b(grouped_q4_kernel<1, true, MT>, grid, blk, st, e0, e1, a);
}

template <bool DOWN>
static hipError_t launch_q4(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const GroupedPlan p = plan_q4(a, DOWN);
    if (p.rows == TL_ROWS)
        return p.tiles == 3 ? launch_tile<DOWN, 3>(a, p.row_tiles, st, e0, e1) : launch_tile<DOWN, 1>(a, p.row_tiles, st, e0, e1);
    return p.tiles == 2 ? launch_rows64<DOWN, 2>(a, st, e0, e1) : launch_rows64<DOWN, 1>(a, st, e0, e1);
}

template <int MT>
static hipError_t launch_tile6(const GroupedArgs &a, int rtw, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const int nb = a.I / QK;
    const int64_t tasks = (int64_t)(a.P / (32 * MT) + a.E + shared_chunks_max<MT>(a)) * (a.H / (TL_ROWS * rtw));
    const dim3 grid((unsigned)((tasks + 7) / 8 * 8)), blk(256);
    if (nb == 3) return launch_b(grouped_q6_tile_kernel<3, MT>, grid, blk, st, e0, e1, a, rtw);
    if (nb == 2) return launch_b(grouped_q6_tile_kernel<2, MT>, grid, blk, st, e0, e1, a, rtw);
    return launch_b(grouped_q6_tile_kernel<1, MT>, grid, blk, st, e0, e1, a, rtw);
}

// How a Q6_K down product runs.
//   host with weights in host memory, chunks of two tiles, as for Q4_K (all pinned, 128
//        experts, I = 768, ms, one tile / two: 64 tokens 4.07 / 3.57, 200 4.23 / 3.67, 700 3.94 / 3.81;
//        64-row kernel in passes of 32 pairs 3.75, 3.79, 3.71)
//   few  no more than 512 workgroups of 128 rows (32 experts): the 64-row kernel, in passes of one
//        tile while 16 pairs serve an expert, of two to twice that for 8 experts (us, there /
//        on tiles: one expert, I = 768, 16 tokens 8.6 / 11.2, 32 10.2 / 11.1, 33 17.8 / 11.0; 8 experts, 32 pairs
//        8.8 / 11.3, 128 pairs 10.0 / 11.4; 16 experts, 128 pairs 12.2 / 12.8, 256 pairs 14.7 / 13.2)
//   I = 512  half a pair to 4 pairs per expert (8 of 64): the 64-row kernel, which is slower
//        at I = 256 and 768; why rows of two super-blocks differ was not found, so this line is the
//        measurement's (us, there / on tiles: 64 experts, 16 pairs 11.1 / 11.2, 128 pairs
//        20.3 / 24.4, 512 22.9 / 24.6, 768 26.4 / 24.8; 128, 128 pairs 25.8 / 31.6, 512 37.3 / 40.3, 1,024 40.8 / 41.0;
//        256, 32 pairs 16.7 / 17.6 (the whole call 44.9 / 43.1), 96 35.8 / 31.8, 128 31.8 / 35.6, 1,024 74.3 / 76.3,
//        2,048 80.9 / 79.3; I = 768, 128 experts, 512 pairs 61.4 / 50.2; I = 256 24.4 / 21.2); passes of two tiles for few
//        workgroups (16 experts, 256 pairs 11.2 / 11.9)
//   one row tile a workgroup while all run in one round, 768 workgroups: two of them leave the
//        chip idle (one expert, 512 tokens 12.9 / 18.6, and 24.7 of two tiles a chunk)
//   two tiles a chunk from 40 pairs per expert on (us, one / two: 128 experts, I = 768, 32 pairs
//        66.7 / 68.0, 48 85.8 / 75.4, 128 177 / 158; 64, I = 512, 40 pairs 37.7 / 31.2)
// Else two row tiles a workgroup, but one below two pairs per expert (us, one / two: 128
// experts, 24 tokens 43 / 48, 1,000 tokens 111 / 104).
static GroupedPlan plan_q6(const GroupedArgs &a) {
    if (a.host) return {TL_ROWS, 2, host_row_tiles(a)};
    const int full = max(a.P / 32, min(a.E, a.P)), rt = a.H / TL_ROWS;
    if (!a.shared) {
        if (a.E * rt <= 512 && a.P <= 8 * a.E + 8) return {64, 1, 1};
        if (a.E * rt <= (a.I == 512 ? 512 : 128) && a.P <= 16 * a.E + 16) return {64, 2, 1};
        if (a.I == 512 && a.E * rt > 512 && 2 * a.P >= a.E && a.P <= 4 * max(a.E, 128)) return {64, 1, 1};
    }
    if (full * rt <= 768) return {TL_ROWS, 1, 1};
    if (a.P >= 40 * a.E) return {TL_ROWS, 2, 2};
    return {TL_ROWS, 1, a.P < 2 * a.E ? 1 : 2};
}

template <int MT>
static hipError_t launch_rows64_q6(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const dim3 grid((unsigned)(a.H / 64 * a.E)), blk(256);
    if (a.I == 3 * QK) return launch_b(grouped_q6_kernel<3, MT>, grid, blk, st, e0, e1, a);
    if (a.I == 2 * QK) return launch_b(grouped_q6_kernel<2, MT>, grid, blk, st, e0, e1, a);
    return launch_b(grouped_q6_kernel<1, MT>, grid, blk, st, e0, e1, a);
}

static hipError_t launch_q6(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    const GroupedPlan p = plan_q6(a);
    if (p.rows == TL_ROWS)
        return p.tiles == 2 ? launch_tile6<2>(a, p.row_tiles, st, e0, e1) : launch_tile6<1>(a, p.row_tiles, st, e0, e1);
    return p.tiles == 2 ? launch_rows64_q6<2>(a, st, e0, e1) : launch_rows64_q6<1>(a, st, e0, e1);
}

GroupedPlan plan_gateup_grouped(const GroupedArgs &a) { return plan_q4(a, false); }
GroupedPlan plan_down_grouped(const GroupedArgs &a) { return a.down_type == TYPE_Q6K ? plan_q6(a) : plan_q4(a, true); }

hipError_t launch_gateup_grouped(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    return launch_q4<false>(a, st, e0, e1);
}

hipError_t launch_down_grouped(const GroupedArgs &a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
    return a.down_type == TYPE_Q6K ? launch_q6(a, st, e0, e1) : launch_q4<true>(a, st, e0, e1);
}

hipError_t launch_iota(int n, int32_t *offsets, int32_t *perm, float *ones, hipStream_t st) {
    return launch_b(iota_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), st, nullptr, nullptr, n, offsets, perm,
                    ones);
}

hipError_t launch_combine(const float *ypair, const float *yshared, int n_tok, int K, int H, float *out, int accumulate,
                          hipStream_t st) {
    const size_t n4 = (size_t)n_tok * H / 4;
    if (n4 == 0) return hipSuccess;
    return launch_b(combine_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), st, nullptr, nullptr, ypair, yshared,
                    n_tok, K, H, out, accumulate);
}

hipError_t launch_combine_host(const float *ypair, const float *hrows, const uint8_t *hflag, const float *yshared,
                               int n_tok, int K, int H, float *out, int accumulate, hipStream_t st) {
    const size_t n4 = (size_t)n_tok * (H / 4);
    return launch_b(combine_host_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), st, nullptr, nullptr, ypair,
                    hrows, hflag, yshared, n_tok, K, H, out, accumulate);
}

// ---------------------------------------------------------------------------
// Scratch of the allocation-free grouped entry point: the workspace of one
// call (Q8_K codes of x and h, the up/gate rows, the weighted pair rows) in
// a file-scope array.  Every device the library runs on holds its own copy
// at its own address from the code object's load until the process ends.
// In host code `scratch` names a host-side stand-in, not device memory:
// kernels are given the address static_scratch() looks up.
static __device__ __align__(256) uint8_t scratch[STATIC_SCRATCH_BYTES];

hipError_t static_scratch(void **ptr) {
    constexpr int MAX_DEV = 64;
    static std::mutex m;
    static void *addr[MAX_DEV] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= MAX_DEV) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(m);
    if (!addr[dev]) {           // once per device, with that device current
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[dev] = p;
    }
    *ptr = addr[dev];
    return hipSuccess;
}

}  // namespace mp
