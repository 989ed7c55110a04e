// rv12 prefill linear: the 12-bit decode fused into a split-float16 MFMA GEMM
// over all the prompt's tokens at once (gfx950).  Replaces the blocked
// prefill's decode_rows + fp32 GEMM
// (ramvi/engine/ramvi_engine/kernels/prefill.py:66-78, prefill_kernels.py:8-26
// and 58-110): every weight is read once per prompt in its 12-bit form, never
// written back in a wider format.
//
// y[t] (=|+=) W_dec . x'[t], t < T, with the MODE prologue (2: x' =
// silu(x[0:K]) * x[K:2K]) or the RMSNorm prologue of mode 0 (x' = lnw x,
// the token's rs = 1 / sqrt(mean x^2 + eps) applied to its outputs, as the
// decode kernels apply it).  Three launches, four with a K split:
//   1. k_prefill_stats (one wave per token): the exponents of x' and, with
//      RMS, rs (sum of squares of x 2^-32); k_prefill_parts (32 tokens x 64
//      columns per workgroup): x' 2^P_t split into parts in B-operand lane
//      order (token block; the first two parts of each step of 32 columns, then
//      the third ones; 64 lanes x 8 values, lane l: token l%16, k = 8(l/16) +
//      0..7), and x' itself in fp32, transposed (column-major over the padded
//      tokens).  Token rows past T are zeros.
//   2. k_prefill_mm: a 12-bit weight is exactly a float16 (4 exponent bits, 7
//      of mantissa), so x' goes in two float16 parts (23 bits) with two MFMAs per
//      tile where three bf16 parts (24 bits) took three.  The second part is kept
//      2^11 larger, and the first meets the weights times 2^11 (they leave half of
//      float16's exponents free): the parts hold a value 2^28 below its token's
//      largest as well as the largest (2^17 without, for 2 % less time).  The sums
//      pass from the matrix core's accumulators to fp32 ones every kPfChunk steps
//      and come out closer to 64 bits than three parts in one accumulator (8192 x
//      K over 1024 tokens, relative error, K = 512, 4096, 17408: 2.1e-7, 2.2e-7,
//      2.5e-7 against 2.4e-7, 7.0e-7, 1.5e-6).  A token whose values the float16
//      parts would not hold (see tok_exp) keeps the three bf16 parts, whatever the
//      others of its tile do, and so do all tokens of a call that asks for them
//      (parts = 3): the prompt's qkv, so that a layer leaves the same keys and
//      values in its cache, bit for bit, as earlier versions did for the same x
//      (layer 0 of a prompt; with two parts one in 10^4 bf16 entries falls on the
//      other side of its rounding, 5e-5 of the layer's keys and values).  That is
//      not for accuracy: one accumulator over K has the larger error, and the
//      Qwen3-8B layer over 2048 tokens takes about 40 us more.
//      Workgroup = 256 rows x 128 tokens, 8 waves of 64 rows x 64 tokens.  Per
//      32-column step the workgroup's 16 row blocks' Q16 tiles and the B parts
//      go from memory straight into a ring of LDS slots (buffer loads with the
//      LDS destination), one wait + barrier per step; every other instruction
//      is spread between the MFMAs.
//      Bound by issue: 51200 x 5120 over 4096 tokens, 2.15e12 useful operations
//      and twice that in MFMAs, takes 4030 us (5560 with three parts), 1.07
//      PFLOP/s of MFMAs.  Of a step's 1960 cycles the two waves of a SIMD have it
//      issue MFMAs in 1024 and other vector instructions (the unpacking, the
//      scaling, addresses: 100 a wave) in 800; LDS is active in 27 %, without bank
//      conflicts; the clock under this load is 1.78 GHz (counters of this
//      kernel).  A library's product of that shape reaches 1.17 PFLOP/s in bf16,
//      1.13 in float16.  (256-token workgroups, whose waves unpack and read less
//      per product, were 11 % faster, but leave no registers for the second sums:
//      their error stays at 5.9e-7.)
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <type_traits>

#include "rv12_device.h"
#include "rv12_internal.h"

namespace rv12 {

constexpr int kPfRowBlocks = 16;  // row blocks (of 16 rows) per workgroup
constexpr int kPfThreads = 512;
constexpr int kPfWaves = kPfThreads / 64;
// wave tile: kPfWB row blocks x kPfWT token blocks; kPfWR waves along the rows,
// kPfWC along the tokens
constexpr int kPfWB = 4, kPfWT = 4;
constexpr int kPfWR = kPfRowBlocks / kPfWB;
constexpr int kPfWC = kPfWaves / kPfWR;
constexpr int kPfTokBlocks = kPfWC * kPfWT;           // token blocks (of 16 tokens) per workgroup
constexpr int kPfTokens = kPfTokBlocks * 16;          // 128
constexpr int kPfAPerWave = kPfRowBlocks / kPfWaves;  // A tiles a wave loads per step
// LDS slot (u32x4 units): 16 A tiles of 1 KB (a 12-byte-per-lane load with the
// LDS destination writes lane l at 16 l: 768 B of each KB), then the B parts
// (64 lanes each per token block)
constexpr int kPfSlotA = kPfRowBlocks * 64;
constexpr size_t kPfLds = 160 * 1024;  // the whole CU's: one workgroup per CU
// a wave's sums of 64 rows x 64 tokens on their way past the exceptions, rows
// 68 floats apart (the four row groups of an access fall on different banks)
constexpr int kPfExcStride = 68;
static_assert((size_t)kPfWaves * 16 * kPfWB * kPfExcStride * 4 <= kPfLds, "LDS");
// float16 loop: 2 parts, a ring of five 32 KB slots
constexpr int kPfSlot2 = kPfSlotA + kPfTokBlocks * 2 * 64;
constexpr int kPfRing2 = (int)(kPfLds / (kPfSlot2 * 16));
static_assert(kPfRing2 == 5, "five slots");
constexpr int kPfB2 = kPfTokBlocks * 2 / kPfWaves;  // 1 KB chunks of B a wave loads per step
constexpr int kPfOps2 = kPfAPerWave + kPfB2;
// at the top of step s, the wave's loads of step s + 1 are followed by those
// of the kPfRing2 - 3 steps issued since
constexpr int kPfWait2 = kPfOps2 * (kPfRing2 - 3);
// Steps between the additions of the MFMA accumulators to the fp32 sums.  The
// matrix core's own additions into an accumulator lose more as it grows: all
// 128 steps of K = 4096 in one accumulator leave a relative error of 5.9e-7
// against 64 bits (7.0e-7 with three bf16 parts), chunks of 16 steps 2.3e-7,
// of 8 1.9e-7, of 4 1.7e-7; in one sweep 51200 x 5120 over 4096 tokens took 4310,
// 4115, 4170 and 4290 us.
constexpr int kPfChunk = 16;
// bf16 loop: 3 parts, four 40 KB slots
constexpr int kPfRing3 = 4;
constexpr int kPfSlot3 = kPfSlotA + kPfTokBlocks * 3 * 64;
static_assert((size_t)kPfRing3 * kPfSlot3 * 16 <= kPfLds, "LDS of one workgroup");
constexpr int kPfOps3 = kPfAPerWave + kPfTokBlocks * 3 / kPfWaves;
constexpr int kPfWait3 = kPfOps3 * (kPfRing3 - 2);  // the loads issued after step s + 1's, at the top of step s
static_assert(kPfWait3 < 64 && kPfWait2 < 64, "vmcnt holds 6 bits");
// s_waitcnt immediates (gfx9 encoding): vmcnt(n) and lgkmcnt(0), expcnt not
// waited for; vmcnt(n) alone
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }
constexpr int waitcnt_vm(int n) { return waitcnt_vm_lgkm0(n) | (15 << 8); }

// 12 or 16 bytes per lane from a descriptor straight into LDS (lane l at
// d + 16 bytes l)
typedef __attribute__((address_space(3))) void* lds_ptr;
__device__ __forceinline__ void load_lds12(__amdgpu_buffer_rsrc_t r, u32x4* d, int off, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)d, 12, off, soff, 0, 0);
}
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, u32x4* d, int off, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)d, 16, off, soff, 0, 0);
}

// x' of token row xr at columns k..k+7 (MODE 2: silu(g) * u; lnw: the RMS
// weight times x)
__device__ __forceinline__ void prefill_xprime(const float* xr, int K, int k, bool m2, const uint16_t* lnw,
                                               float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(xr + k);
    const f32x4 b = *reinterpret_cast<const f32x4*>(xr + k + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    if (lnw) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(lnw + k);
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] *= __uint_as_float(ww[i] << 16);
            v[2 * i + 1] *= __uint_as_float(ww[i] & 0xFFFF0000u);
        }
    }
    if (m2) {
        const f32x4 c = *reinterpret_cast<const f32x4*>(xr + K + k);
        const f32x4 d = *reinterpret_cast<const f32x4*>(xr + K + k + 4);
        const float u[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = silu_mul(v[e], u[e]);
    }
}

// A token's activation class, E = e << 1 | wide: e the exponent of its largest
// finite |x'| (below B = 2^e; -1000: all zeros), wide where the float16 parts
// would hold less of it than float32 sums do; such a token keeps three bf16
// parts.  The float16 parts are of
// x' 2^(15 - e): every |x'| >= 2^-28 B to 2^-23 of itself, a smaller one to 2^-51 B.
// So a token without a nonzero value below 2^-28 B is not wide.  One with such
// values must bear rows whose weights lie on them alone.  A row keeps in its tiles
// the 15 exponents that most of its weights have: at least K / 18 weights (18
// windows cover the 256 exponents), less than 2^15 apart.  With at most K / 36
// columns at or below 2^-16 B (zeros included), K / 36 of those weights are on
// larger ones, and n small values add an error of less than
// n 2^15 2^-51 / ((K / 36) 2^-16) of sum |w||x'|: below 2^-23 for n <= K / 512.
// (Base 0 is the exception: its window holds the zeros, its weights are
// below 2^-112.)  Of 1024 tokens of 12288 columns silu(g) u with normal g and u, 8
// have a value below 2^-28 B, one each, none more than 58 columns below 2^-16 B:
// none is wide.  One with half its columns 2^29 below the others is.
constexpr int kF16Exact = 28, kF16Floor = 16;  // exponents below B
__device__ __forceinline__ int tok_exp(int E) { return E >> 1; }
__device__ __forceinline__ int scale_f16(int E) { return tok_exp(E) < -500 ? 0 : 15 - tok_exp(E); }
__device__ __forceinline__ int scale_bf16(int E) {
    const int e = tok_exp(E);
    return (e >= -39 && e <= kXRangeHi) ? kXScaleExp : slow_scale_exp(e);
}

// E of the lane's token of t0 .. t0 + 63 (past T: the last one), and which of the
// wave's 64 are wide
__device__ __forceinline__ int class_of(const int* __restrict__ E, int t0, int T) {
    return E[min(t0 + (int)(threadIdx.x & 63), T - 1)];
}
__device__ __forceinline__ uint64_t wide_mask(int E) { return __ballot(E & 1); }

// 1a. k_prefill_stats: one wave per token (4 per workgroup, a grid over the
// padded tokens): the largest and smallest exponent of the nonzero x' and, with
// RMS, the sum of squares of x 2^-32, lane l over columns 8 l + 512 i, reduced
// across the wave in a fixed order; where the smallest asks for them, the counts
// of small columns in a second pass over the row; writes the token's E and rs_t.
constexpr int kPsThreads = 256;
__global__ __launch_bounds__(kPsThreads) void k_prefill_stats(const float* __restrict__ x, int T, int K, int xs,
                                                              int m2, const uint16_t* __restrict__ lnw, float eps,
                                                              int* __restrict__ E, float* __restrict__ R) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (kPsThreads / 64) + (threadIdx.x >> 6);
    uint32_t hib = 0, lob = 0xFFFFFFFFu;  // magnitudes as bits: the largest finite, the smallest nonzero less one
    float sq = 0.0f;
    const float* xr = x + (int64_t)t * xs;
    if (t < T) {
        for (int k = lane * 8; k < K; k += 512) {
            float v[8];
            prefill_xprime(xr, K, k, m2 != 0, nullptr, v);
            if (lnw) {
#pragma unroll
                for (int i = 0; i < 8; ++i) sq += (v[i] * kSsqScale) * (v[i] * kSsqScale);
                const u32x4 w = *reinterpret_cast<const u32x4*>(lnw + k);
                const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[2 * i] *= __uint_as_float(ww[i] << 16);
                    v[2 * i + 1] *= __uint_as_float(ww[i] & 0xFFFF0000u);
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t b = __float_as_uint(v[i]) & 0x7FFFFFFFu;
                hib = max(hib, b < 0x7F800000u ? b : 0u);
                lob = min(lob, b - 1);
            }
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        hib = max(hib, (uint32_t)__shfl_xor((int)hib, o));
        lob = min(lob, (uint32_t)__shfl_xor((int)lob, o));
        sq += __shfl_xor(sq, o);
    }
    const int e = exp_or_min(__uint_as_float(hib));
    // a row with small values: all the workgroup's waves count them (one wave's second
    // pass over 12288 columns would end 13 us after the others)
    constexpr int kWaves = kPsThreads / 64;
    __shared__ int top[kWaves], cnt[kWaves][2];  // the row's e, or INT_MAX without small values; counts
    const int wave = threadIdx.x >> 6;
    if (lane == 0) {
        top[wave] = hib && exp_or_min(__uint_as_float(lob + 1)) <= e - kF16Exact ? e : INT_MAX;
        cnt[wave][0] = cnt[wave][1] = 0;
    }
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) {
        const int ew = top[w];
        if (ew == INT_MAX) continue;
        const float* row = x + (int64_t)(t - wave + w) * xs;
        int tiny = 0, small = 0;
        for (int k = threadIdx.x * 8; k < K; k += kPsThreads * 8) {
            float v[8];
            prefill_xprime(row, K, k, m2 != 0, lnw, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) {  // (frexp exponents: |x'| < 2^ei)
                const int ei = exp_or_min(v[i]);
                tiny += ei > -1000 && ei <= ew - kF16Exact ? 1 : 0;
                small += v[i] == 0.0f || (ei > -1000 && ei <= ew - kF16Floor) ? 1 : 0;
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            tiny += __shfl_xor(tiny, o);
            small += __shfl_xor(small, o);
        }
        if (lane == 0) {
            atomicAdd(&cnt[w][0], tiny);
            atomicAdd(&cnt[w][1], small);
        }
    }
    __syncthreads();
    if (lane == 0) {
        const bool wide = cnt[wave][0] > K / 512 || cnt[wave][1] > K / 36;
        E[t] = e * 2 + (wide ? 1 : 0);
        if (lnw) R[t] = rms_scale(sq, K, eps);
    }
}

// 1b. k_prefill_parts: grid (32-token blocks, 64-column chunks), 256 threads,
// thread (token tok, 8-column group k8): x' (prologue applied) of token t at
// columns kc .. kc + 7 written transposed (per column, 32 consecutive tokens:
// full 128-byte lines), then its scaled parts in B-operand lane order: two of
// float16 (the second first), or three of bf16 for a wide token.  A token block's
// region holds the first two parts of its steps, then the third ones (unwritten,
// and unused, for the lanes of tokens that have two).  Tokens past T are zeros.
constexpr int kPpThreads = 256;
__global__ __launch_bounds__(kPpThreads) void k_prefill_parts(const float* __restrict__ x, int T, int K, int xs,
                                                              int m2, const uint16_t* __restrict__ lnw,
                                                              const int* __restrict__ E, u32x4* __restrict__ xb,
                                                              float* __restrict__ xt, int tp, int parts) {
    const int tok = threadIdx.x & 31, k8 = threadIdx.x >> 5;
    const int t = blockIdx.x * 32 + tok;
    const int kc = blockIdx.y * 64 + k8 * 8;
    const int nsteps = K >> 5;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (t < T && kc < K) prefill_xprime(x + (int64_t)t * xs, K, kc, m2 != 0, lnw, v);
    if (kc >= K) return;
    float* xc = xt + (int64_t)kc * tp + t;
#pragma unroll
    for (int i = 0; i < 8; ++i) xc[(int64_t)i * tp] = v[i];
    const int et = t < T ? E[t] : 0;
    const bool wide = parts == 3 || (et & 1);
    const int p = t >= T ? 0 : wide ? scale_bf16(et) : scale_f16(et);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = ldexpf(v[i], p);
    const int s = kc >> 5, l = ((kc & 31) >> 3) * 16 + (t & 15);  // step, lane of the operand
    u32x4* blk = xb + (int64_t)(t >> 4) * nsteps * 192 + l;
    u32x4 d[3];
    if (wide) split3(v, d[0], d[1], d[2]);
    else split2_f16(v, d[1], d[0]);
    blk[(int64_t)s * 128] = d[0];
    blk[(int64_t)s * 128 + 64] = d[1];
    if (wide) blk[(int64_t)nsteps * 128 + (int64_t)s * 64] = d[2];
}

// Workgroup i -> (row tile, token tile).  Workgroups are dispatched in order,
// round-robin over the 8 XCDs (each with its own L2): i runs on XCD i % 8 as
// its (i / 8)-th.  The virtual index v gives each XCD a contiguous range of
// G / 8 tiles (the remainder past 8 (G / 8) keeps v = i), and v runs over
// groups of kPfGroupRows row tiles x all token tiles, row tile fastest, so the
// ~32 workgroups an XCD holds at once cover 8 row tiles x 4 token tiles: per
// step their L2 misses are 8 A tiles (12 KB each) and 4 B sets (16 KB each at
// 128 tokens), 160 KB, where 2 row tiles x 16 token tiles (the Qwen3-8B o and
// down in launch order) would miss 280 KB.  A bijection of [0, G).
constexpr int kPfGroupRows = 8;
__device__ __forceinline__ void prefill_tile(int i, int G, int nx, int ny, int& rt, int& tt) {
    const int g8 = G / 8;
    const int v = i < g8 * 8 ? (i % 8) * g8 + i / 8 : i;
    const int per = kPfGroupRows * ny;
    const int g = v / per, r0 = g * kPfGroupRows;
    const int gr = min(kPfGroupRows, nx - r0);
    const int w = v - g * per;
    tt = w / gr;
    rt = r0 + w % gr;
}

// 2. grid (row tiles of 256 rows x token tiles of 128, in the order above),
// 512 threads.  LN (the RMS prologue: each token's rs applied to its outputs)
// is a template argument; the prologues themselves were applied in the
// pre-pass, to the parts and to the transposed x' (xt, row stride tp).
template <bool LN>
__global__ __launch_bounds__(kPfThreads) void k_prefill_mm(const uint32_t* __restrict__ tiles,
                                                           const int32_t* __restrict__ rbase,
                                                           const u32x4* __restrict__ xb, const int* __restrict__ E,
                                                           const int32_t* __restrict__ rp,
                                                           const int32_t* __restrict__ er,
                                                           const int32_t* __restrict__ ec,
                                                           const float* __restrict__ ev, const float* __restrict__ xt,
                                                           int tp, const float* __restrict__ R, float* __restrict__ y,
                                                           float* __restrict__ part, int N, int K, int T, int add,
                                                           int parts, int vec) {
    extern __shared__ u32x4 bs[];  // the ring's slots: A tiles and B parts of consecutive steps
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % kPfWR, wc = wave / kPfWR;
    const int nsteps = K >> 5;
    // K split blockIdx.y of gridDim.y: steps [s_lo, s_hi)
    const int S = gridDim.y, sp = blockIdx.y;
    const int s_lo = (int)((int64_t)sp * nsteps / S), s_hi = (int)((int64_t)(sp + 1) * nsteps / S);
    const int64_t nblk = (N + 15) / 16;
    const int nx = (int)((nblk + kPfRowBlocks - 1) / kPfRowBlocks);
    int rt, tt;
    prefill_tile(blockIdx.x, gridDim.x, nx, gridDim.x / nx, rt, tt);
    const int64_t blk0 = (int64_t)rt * kPfRowBlocks + wr * kPfWB;  // this wave's first row block
    const int tb0 = tt * kPfTokBlocks;                            // the workgroup's first token block
    const uint32_t blk_bytes = (uint32_t)nsteps * kStepBytes;
    // the classes of the tile's tokens (asked for here, answered after the first
    // loads are on their way)
    const int wl0 = class_of(E, tb0 * 16, T), wl1 = class_of(E, tb0 * 16 + 64, T);
    // the workgroup's A tiles: wave w loads row blocks 2w and 2w + 1 of the
    // workgroup through a descriptor over its valid row blocks (a row block
    // past N, or a step past the end through the 0-byte descriptor, reads
    // zeros)
    const int64_t wblk0 = (int64_t)rt * kPfRowBlocks;
    const int nvalid_wg = (int)max((int64_t)0, min((int64_t)kPfRowBlocks, nblk - wblk0));
    const char* wgbase = reinterpret_cast<const char*>(tiles) + wblk0 * (int64_t)blk_bytes;
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(wgbase, (uint32_t)nvalid_wg * blk_bytes);
    const __amdgpu_buffer_rsrc_t rnull = make_rsrc(wgbase, 0u);
    int aoff[kPfAPerWave];
#pragma unroll
    for (int i = 0; i < kPfAPerWave; ++i) aoff[i] = (int)((wave * kPfAPerWave + i) * blk_bytes) + lane * 12;
    // the B parts of the workgroup's token blocks, through a descriptor over them
    const u32x4* xbw = xb + (int64_t)tb0 * nsteps * 192;
    const __amdgpu_buffer_rsrc_t rbx = make_rsrc(xbw, (uint32_t)kPfTokBlocks * nsteps * 192 * 16);
    const __amdgpu_buffer_rsrc_t rbnull = make_rsrc(xbw, 0u);

    constexpr int kFrags = 2 * kPfWT;
    constexpr int W = 4;  // B fragments in flight (8: the same within 1 %)
    int boff[kPfB2];
#pragma unroll
    for (int j = 0; j < kPfB2; ++j) {
        const int idx = tid + j * kPfThreads;  // (token block, part, lane) of the step
        boff[j] = ((idx / 128) * nsteps * 192 + idx % 128) * 16;
    }
    // load i of step s_lo + j into the slot at `slot`; a step past the end
    // goes through the 0-byte descriptors, which write zeros, so the loop
    // has no branch around a load
    auto load_op = [&](int i, int slot, int j) {
        const int s = s_lo + j;
        const bool in = s < s_hi;
        u32x4* d = bs + slot;
        if (i < kPfAPerWave)
            load_lds12(in ? rv : rnull, d + (wave * kPfAPerWave + i) * 64, aoff[i], (in ? s : 0) * kStepBytes);
        else
            load_lds16(in ? rbx : rbnull, d + kPfSlotA + wave * 64 + (i - kPfAPerWave) * kPfThreads,
                       boff[i - kPfAPerWave], (in ? s : 0) * 128 * 16);
    };
    // steps 0 .. kPfRing2 - 2 into slots 0 .. (a tile of wide tokens alone starts
    // over: what these loads bring is in bounds and unused)
    if (parts == 2) {
#pragma unroll
        for (int j = 0; j < kPfRing2 - 1; ++j)
#pragma unroll
            for (int i = 0; i < kPfOps2; ++i) load_op(i, j * kPfSlot2, j);
    }
    // Two passes over a tile with tokens of both classes, each storing its own
    // tokens' outputs (an MFMA's output column is its own token's alone: what the other
    // class's bits give stays in columns that are not stored), so that a
    // token's result is the same beside any others.  (24576 x 4096 over 2048
    // tokens, of one class 824 and 1009 us: 862 with one wide token in one tile,
    // 1246 with one in each, 1610 with one in 20; three parts for the whole tile
    // took 1000 with any.)  Three parts: one pass.
    const uint64_t w0 = parts == 3 ? ~0ull : wide_mask(wl0), w1 = parts == 3 ? ~0ull : wide_mask(wl1);
    const uint64_t ww = wc ? w1 : w0;  // the wave's 64 tokens
    auto tile_pass = [&](auto wide_c) {
        constexpr bool wide = decltype(wide_c)::value;
        f32x4 acc[kPfWB][kPfWT];
#pragma unroll
        for (int b = 0; b < kPfWB; ++b)
#pragma unroll
            for (int c = 0; c < kPfWT; ++c) acc[b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

        if constexpr (!wide) {
            const int ra0 = wr * kPfWB * 64 + lane, rb0 = kPfSlotA + wc * kPfWT * 128 + lane;
            auto read_a = [&](int slot, int b) { return *reinterpret_cast<const u32x3*>(bs + slot + ra0 + b * 64); };
            // fragment i: part i / kPfWT of token block i % kPfWT, so that the products
            // of one accumulator are kPfWT fragments apart
            auto read_b = [&](int slot, int i) { return bs[slot + rb0 + (i % kPfWT) * 128 + (i / kPfWT) * 64]; };
            // steps 0 and 1 landed
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(kPfWait2));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            u32x4 a[2][kPfWB], up[kPfWB], fb[W];  // up: the step's weights times 2^11, for the hi parts
#pragma unroll
            for (int b = 0; b < kPfWB; ++b) {
                const u32x3 r = read_a(0, b);
                uint32_t pr[4];
                unpack_pairs_f16(r.x, r.y, r.z, pr);
                a[0][b] = u32x4{pr[0], pr[1], pr[2], pr[3]};
            }
#pragma unroll
            for (int i = 0; i < W; ++i) fb[i] = read_b(0, i);
            // Step s: wait for this wave's loads of step s + 1; barrier (every
            // wave's have landed, and every wave has used slot s - 1); then per B
            // fragment its four MFMAs, one of the loads of step s + kPfRing2 - 1 into
            // slot s - 1, the read of the fragment W ahead (the next step's at the
            // end) and a share of the next step's A reads and unpacking: memory,
            // LDS and vector instructions spread between the MFMAs, fenced so
            // that the compiler keeps them there.
            int cur = 0, nxt = kPfSlot2, fill = (kPfRing2 - 1) * kPfSlot2;
            const int nst = s_hi - s_lo;
            f32x4 sum[kPfWB][kPfWT];
#pragma unroll
            for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                for (int c = 0; c < kPfWT; ++c) sum[b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int s1 = 0; s1 < nst; s1 += kPfChunk) {
                const int s2 = min(nst, s1 + kPfChunk);
                for (int s0 = s1; s0 < s2; s0 += 2) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_s_waitcnt(waitcnt_vm(kPfWait2));
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                        u32x3 raw[kPfWB];
#pragma unroll
                        for (int i = 0; i < kFrags; ++i) {
                            if (i < kPfOps2) load_op(i, fill, s0 + u + kPfRing2 - 1);
                            if (i >= 1 && i - 1 < kPfWB) raw[i - 1] = read_a(nxt, i - 1);
                            const u32x4 bf = fb[i % W];
#pragma unroll
                            for (int b = 0; b < kPfWB; ++b)
                                acc[b][i % kPfWT] = mfma_f16(i < kPfWT ? a[u][b] : up[b], bf, acc[b][i % kPfWT]);
                            if (i < kPfWB) up[i] = f16_up11(a[u][i]);
                            fb[i % W] = i + W < kFrags ? read_b(cur, i + W) : read_b(nxt, i + W - kFrags);
                            if (i >= kFrags - kPfWB) {
                                const int b = i - (kFrags - kPfWB);
                                uint32_t pr[4];
                                unpack_pairs_f16(raw[b].x, raw[b].y, raw[b].z, pr);
                                a[u ^ 1][b] = u32x4{pr[0], pr[1], pr[2], pr[3]};
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        fill = cur;
                        cur = nxt;
                        nxt = nxt + kPfSlot2 == kPfRing2 * kPfSlot2 ? 0 : nxt + kPfSlot2;
                    }
                }
#pragma unroll
                for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                    for (int c = 0; c < kPfWT; ++c) {
                        sum[b][c] += acc[b][c];
                        acc[b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
#pragma unroll
            for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                for (int c = 0; c < kPfWT; ++c) acc[b][c] = sum[b][c];
        } else {
            // the first loads have landed, and a first pass's LDS accesses are done
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            int boff3[3], bstep3[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int ch = wave + j * kPfWaves, pt = ch % 3;  // (token block, part) of the step
                boff3[j] = ((ch / 3 * 192 + (pt < 2 ? 0 : 128)) * nsteps + (pt & 1) * 64 + lane) * 16;
                bstep3[j] = pt < 2 ? 128 * 16 : 64 * 16;
            }
            int need = 0;  // the wave's token blocks with a wide token
#pragma unroll
            for (int c = 0; c < kPfWT; ++c) need |= (ww >> (16 * c) & 0xFFFF) != 0 ? 1 << c : 0;
            auto load_step = [&](int slot, int j) {  // step s_lo + j
                const int s = s_lo + j;
                const bool in = s < s_hi;
                const __amdgpu_buffer_rsrc_t ra = in ? rv : rnull, rb = in ? rbx : rbnull;
                const int sa = (in ? s : 0) * kStepBytes, sb = in ? s : 0;
                u32x4* d = bs + slot * kPfSlot3;
#pragma unroll
                for (int i = 0; i < kPfAPerWave; ++i)
                    load_lds12(ra, d + (wave * kPfAPerWave + i) * 64, aoff[i], sa);
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    load_lds16(rb, d + kPfSlotA + wave * 64 + j * kPfThreads, boff3[j], sb * bstep3[j]);
            };
            // this wave's fragments of the step in slot `slot`: its 4 row blocks' A
            // groups and 3 parts x 4 token blocks of B, part-major so the first
            // part's MFMAs wait only for its own reads
            auto read_frags = [&](u32x3 (&fa)[kPfWB], u32x4 (&fb)[3][kPfWT], int slot) {
                const u32x4* d = bs + slot * kPfSlot3;
#pragma unroll
                for (int b = 0; b < kPfWB; ++b) fa[b] = *reinterpret_cast<const u32x3*>(d + (wr * kPfWB + b) * 64 + lane);
                const u32x4* src = d + kPfSlotA + wc * kPfWT * 192 + lane;
#pragma unroll
                for (int c = 0; c < kPfWT; ++c)
                    if (need >> c & 1)
#pragma unroll
                        for (int q = 0; q < 3; ++q) fb[q][c] = src[c * 192 + q * 64];
            };
            // steps 0-3 into slots 0-3, all landed; step 0's fragments read
#pragma unroll
            for (int i = 0; i < kPfRing3; ++i) load_step(i, i);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            u32x3 fa[2][kPfWB];
            u32x4 fb[2][3][kPfWT];
            read_frags(fa[0], fb[0], 0);
            // Step s: wait for this wave's loads of step s + 1 and its fragment reads
            // of step s; barrier; step s + 4 into slot s % 4; the fragments of step
            // s + 1 read while the 48 MFMAs of step s run (12 for each token block that
            // has a wide token).  Whole rounds of the unroll: steps past the split read
            // zeros and add nothing.
            for (int s0 = 0; s0 < s_hi - s_lo; s0 += kPfRing3) {
#pragma unroll
                for (int u = 0; u < kPfRing3; ++u) {
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(kPfWait3));
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    load_step(u, s0 + u + kPfRing3);
                    read_frags(fa[(u + 1) & 1], fb[(u + 1) & 1], (u + 1) % kPfRing3);
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    u32x4 a[kPfWB];
#pragma unroll
                    for (int b = 0; b < kPfWB; ++b) {
                        uint32_t pr[4];
                        unpack_pairs(fa[u & 1][b].x, fa[u & 1][b].y, fa[u & 1][b].z, pr);
                        a[b] = u32x4{pr[0], pr[1], pr[2], pr[3]};
                    }
#pragma unroll
                    for (int c = 0; c < kPfWT; ++c) {
                        if (!(need >> c & 1)) continue;
#pragma unroll
                        for (int q = 0; q < 3; ++q)
#pragma unroll
                            for (int b = 0; b < kPfWB; ++b) acc[b][c] = mfma(a[b], fb[u & 1][q][c], acc[b][c]);
                    }
                }
            }
        }
        // the last loads (zeros into slots nobody reads) land before the
        // workgroup's LDS can be handed on
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));

        // epilogue: lane l holds token 16 c + l%16 and rows 4(l/16) + 0..3 of each
        // tile.  v = acc 2^(sc_row - P_t) (exact), plus the row's exceptions, times
        // rs with RMS, stored or added; with a K split the split's sums go to
        // part[sp][token][row] instead (rs and the store or add are the reduce
        // pass's).  Loads that depend on nothing are issued together ahead of their
        // use, and four rows of a token are one 16-byte load or store where vec says
        // that all of them are aligned (indexes clamped into the matrix instead of
        // branches; what is read past an edge is not stored): with a load, branch and store per value
        // the pass took about 20 us of a workgroup, longer than 8 K steps.
        const int q = lane >> 4, jj = lane & 15;
        const int64_t rlo = blk0 * 16;
        __builtin_amdgcn_s_barrier();  // the ring's LDS is the exception sums' from here
        asm volatile("" ::: "memory");
        if (rlo >= N || (wide ? ww : ~ww) == 0) return;  // nothing of this pass to store
        const int32_t e_lo = rp[rlo], e_hi = rp[min(rlo + 16 * kPfWB, (int64_t)N)];
        int64_t nr[kPfWB];  // the lane's first row of each tile
        int sc[kPfWB][4];
#pragma unroll
        for (int b = 0; b < kPfWB; ++b) {
            nr[b] = rlo + b * 16 + q * 4;
            if (vec) {
                const int4 r = *reinterpret_cast<const int4*>(rbase + min(nr[b], (int64_t)N - 4));
                sc[b][0] = r.x, sc[b][1] = r.y, sc[b][2] = r.z, sc[b][3] = r.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[b][i] = rbase[min(nr[b] + i, (int64_t)N - 1)];
            }
        }
        float* xs = reinterpret_cast<float*>(bs) + wave * (16 * kPfWB * kPfExcStride);  // the wave's [64 rows][64 tokens]
        const int tbw = tb0 + wc * kPfWT;  // the wave's token blocks
        // (a) v = acc 2^(sc_row - P_t), exact
#pragma unroll
        for (int c = 0; c < kPfWT; ++c) {
            const int et = E[min((tbw + c) * 16 + jj, T - 1)];
            const int pt = wide ? scale_bf16(et) : scale_f16(et) + kF16WeightExp + 11;
#pragma unroll
            for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[b][c][i] = ldexpf(acc[b][c][i], scale_exp(sc[b][i]) - pt);
        }
        // (b) the exceptions of the wave's 64 rows (the tiles hold zeros
        // there) added in list order, lane = token: the sums go through LDS, an
        // entry's row, column and value are wave-uniform (scalar loads), x' of
        // the 64 tokens at its column is 256 contiguous bytes of the transposed
        // copy, and a row's sums stay in a register from its first entry to its
        // last.  (With a K split, the entries whose column lies in the split's
        // steps.)  One wave's LDS accesses stay in order; the fences keep the
        // compiler's in theirs.
        if (e_lo < e_hi) {
            constexpr int EB = 8;
#pragma unroll
            for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int c = 0; c < kPfWT; ++c)
                        xs[(b * 16 + q * 4 + i) * kPfExcStride + c * 16 + jj] = acc[b][c][i];
            asm volatile("" ::: "memory");
            const float* xtw = xt + (int64_t)tbw * 16 + lane;
            const int c_lo = s_lo * 32, c_hi = s_hi * 32;
            int row = 0;
            float sum = xs[lane];
            for (int32_t e0 = e_lo; e0 < e_hi; e0 += EB) {
                int r[EB];
                float g[EB], v[EB];
#pragma unroll
                for (int j = 0; j < EB; ++j) {
                    const int32_t e = min(e0 + j, e_hi - 1);
                    const int col = ec[e];
                    const bool in = e0 + j < e_hi && col >= c_lo && col < c_hi;
                    r[j] = in ? (int)(er[e] - rlo) : -1;
                    v[j] = ev[e];
                    g[j] = xtw[(int64_t)col * tp];
                }
#pragma unroll
                for (int j = 0; j < EB; ++j) {
                    if (r[j] < 0) continue;
                    if (r[j] != row) {
                        xs[row * kPfExcStride + lane] = sum;
                        row = r[j];
                        sum = xs[row * kPfExcStride + lane];
                    }
                    sum += v[j] * g[j];
                }
            }
            xs[row * kPfExcStride + lane] = sum;
            asm volatile("" ::: "memory");
#pragma unroll
            for (int b = 0; b < kPfWB; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int c = 0; c < kPfWT; ++c)
                        acc[b][c][i] = xs[(b * 16 + q * 4 + i) * kPfExcStride + c * 16 + jj];
        }
        // (c) the outputs
        int tok[kPfWT];
        float rs[kPfWT];
        f32x4 oy[kPfWB][kPfWT];
#pragma unroll
        for (int c = 0; c < kPfWT; ++c) {
            tok[c] = (tbw + c) * 16 + jj;
            const int tc = min(tok[c], T - 1);
            rs[c] = LN && S == 1 ? R[tc] : 1.0f;
            const float* yr = y + (int64_t)tc * N;
#pragma unroll
            for (int b = 0; b < kPfWB; ++b) {
                oy[b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (add && S == 1) {
                    if (vec) {
                        oy[b][c] = *reinterpret_cast<const f32x4*>(yr + min(nr[b], (int64_t)N - 4));
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) oy[b][c][i] = yr[min(nr[b] + i, (int64_t)N - 1)];
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < kPfWT; ++c) {
            float* dst = S > 1 ? part + ((int64_t)sp * tp + tok[c]) * N : y + (int64_t)tok[c] * N;
#pragma unroll
            for (int b = 0; b < kPfWB; ++b) {
                f32x4 v = acc[b][c];
                if constexpr (LN) v *= rs[c];
                if (add && S == 1) v = oy[b][c] + v;
                if (tok[c] >= T || (ww >> (16 * c + jj) & 1) != (wide ? 1 : 0)) continue;
                if (vec) {
                    if (nr[b] < N) *reinterpret_cast<f32x4*>(dst + nr[b]) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (nr[b] + i < N) dst[nr[b] + i] = v[i];
                }
            }
        }
    };
    if ((w0 & w1) != ~0ull) tile_pass(std::false_type{});
    if ((w0 | w1) != 0) tile_pass(std::true_type{});
}

int prefill_tokens_padded(int T) { return (T + kPfTokens - 1) / kPfTokens * kPfTokens; }

// 3. (K split only) y[t][n] (=|+=) rs_t * sum over the splits, in split order:
// V consecutive rows per thread (4 where N % 4 == 0), the loads of 4 splits and
// the old y in flight together
template <int V>
__global__ __launch_bounds__(256) void k_prefill_reduce(const float* __restrict__ part, const float* __restrict__ R,
                                                        float* __restrict__ y, int64_t N, int T, int tp, int S,
                                                        int add) {
    typedef float fv __attribute__((ext_vector_type(V)));
    const int64_t n = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (n >= N) return;
    for (int t = blockIdx.y; t < T; t += gridDim.y) {
        float* yp = y + (int64_t)t * N + n;
        const float* ps = part + (int64_t)t * N + n;
        const int64_t step = (int64_t)tp * N;
        const float rs = R ? R[t] : 1.0f;
        fv old = {}, v = {};
        if (add) old = *reinterpret_cast<const fv*>(yp);
        for (int sp = 0; sp < S; sp += 4) {
            fv a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = *reinterpret_cast<const fv*>(ps + min(sp + u, S - 1) * step);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (sp + u < S) v += a[u];
        }
        if (R) v *= rs;
        *reinterpret_cast<fv*>(yp) = add ? old + v : v;
    }
}

// K splits of the GEMM: those of the least modelled time.  A round of
// workgroups (one per CU) costs its steps plus 8 us of prologue and epilogue, a
// step 0.8 us and up to 0.2 more as the chip fills (its clock falls); the
// reduce pass costs 4 us + (S + 1) T N floats at 5 TB/s (1024 x 3072 over 301
// tokens: 92 us unsplit, 36 with 12 splits; 4096 x 4096 over 2048, one full
// round: 160 unsplit, 183 with 2).  No split below 8 steps.
// Three parts: a step 1.4 us and 10 us a round, 3 us + the floats for the reduce
// pass, the splits this path has always had, so that its sums keep their order.
int prefill_splits(int N, int K, int T, int parts) {
    const int64_t nx = ((int64_t)N + 16 * kPfRowBlocks - 1) / (16 * kPfRowBlocks);
    const int tp = prefill_tokens_padded(T), nsteps = K / 32;
    const int64_t G = nx * (tp / kPfTokens);
    int best = 1;
    double best_us = 0.0;
    for (int S = 1; S <= 16; ++S) {
        if (S > 1 && nsteps / S < 8) break;
        double us;
        if (parts == 3) {
            us = (double)((G * S + 255) / 256) * ((double)nsteps / S * 1.4 + 10.0);
            if (S > 1) us += 3.0 + (double)(S + 1) * tp * N * 4 / 5e6;
        } else {
            const double steps = (nsteps + S - 1) / S;
            const double last = (double)(G * S % 256) / 256;
            us = (double)(G * S / 256) * (steps * 1.0 + 8.0);
            if (last > 0) us += steps * (0.8 + 0.2 * last * last) + 8.0;
            if (S > 1) us += 4.0 + (double)(S + 1) * tp * N * 4 / 5e6;
        }
        if (S == 1 || us < best_us) {
            best = S;
            best_us = us;
        }
    }
    return best;
}

size_t prefill_ws_bytes(int N, int K, int T, int parts) {
    const size_t tp = (size_t)prefill_tokens_padded(T);
    const int S = prefill_splits(N, K, T, parts);
    // parts (room for three), E and R, transposed x', split partials
    return tp * (size_t)K * 10 + tp * 8 + (S > 1 ? (size_t)S * tp * (size_t)N * 4 : 0);
}

void launch_prefill(const rv12_matrix& w, const float* x, float* y, int T, int mode, const uint16_t* lnw, float eps,
                    int parts, void* ws, hipStream_t st) {
    const int K = w.k, N = w.n;
    const int tp = prefill_tokens_padded(T);
    u32x4* xb = reinterpret_cast<u32x4*>(ws);
    int* E = reinterpret_cast<int*>(reinterpret_cast<char*>(ws) + (size_t)tp * K * 6);
    float* R = reinterpret_cast<float*>(E + tp);
    float* xt = R + tp;
    float* part = xt + (size_t)tp * K;
    const int xs = mode == 2 ? 2 * K : K;
    const int m2 = mode == 2 ? 1 : 0;
    const int S = prefill_splits(N, K, T, parts);
    hipLaunchKernelGGL(k_prefill_stats, dim3(tp / (kPsThreads / 64)), dim3(kPsThreads), 0, st, x, T, K, xs, m2, lnw, eps,
                       E, R);
    hipLaunchKernelGGL(k_prefill_parts, dim3(tp / 32, (K + 63) / 64), dim3(kPpThreads), 0, st, x, T, K, xs, m2, lnw, E,
                       xb, xt, tp, parts);
    const int64_t nblk = ((int64_t)N + 15) / 16;
    const dim3 grid((unsigned)((nblk + kPfRowBlocks - 1) / kPfRowBlocks * (tp / kPfTokens)), (unsigned)S);
    const auto kern = lnw ? k_prefill_mm<true> : k_prefill_mm<false>;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kPfLds);
    // four rows at a time: rows of y and part start 16-byte aligned (their bases are,
    // the caller's rbase may not be)
    const int vec = N % 4 == 0 && reinterpret_cast<uintptr_t>(w.rbase) % 16 == 0;
    hipLaunchKernelGGL(kern, grid, dim3(kPfThreads), kPfLds, st, reinterpret_cast<const uint32_t*>(w.tiles), w.rbase, xb,
                       E, w.rp, w.er, w.ec, w.ev, xt, tp, R, y, part, N, K, T, mode != 0 ? 1 : 0, parts, vec);
    if (S > 1) {
        const int V = N % 4 == 0 ? 4 : 1;
        const dim3 rgrid((unsigned)((N + 256 * V - 1) / (256 * V)), (unsigned)min(T, 65535));
        hipLaunchKernelGGL((V == 4 ? k_prefill_reduce<4> : k_prefill_reduce<1>), rgrid, dim3(256), 0, st, part,
                           lnw ? R : nullptr, y, (int64_t)N, T, tp, S, mode != 0 ? 1 : 0);
    }
}

}  // namespace rv12
