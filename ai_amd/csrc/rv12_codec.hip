// rv12 codec kernels for gfx950.
//   encode   the reference 12-bit codec dict of a bf16 matrix: exponent
//            histogram, m8/e4, row-major exception list (k_hist,
//            k_encode_rows, k_exceptions)
//   to_bf16  a codec dict back to bf16 bits (k_codec_to_bf16 + k_scatter_exc)
//   pack     bf16 bits -> the Q16 layout with one exponent window per row and
//            that layout's own exception list (k_row_windows, k_pack_tiles,
//            k_exceptions)
//   compress the packed form and the reference codec's base, row pointers and
//            exception list together (k_row_windows, k_hist_sum, k_row_counts /
//            k_row_recount, k_row_pointers, k_pack_tiles, k_exceptions with both
//            lists): two reads of the weights (three of short rows), one more of
//            the rows with entries, one host read between (6144 x 4096: 79 us,
//            377 as separate calls)
//   decode   Q16 rows back to the exact bf16 / float32 values (k_decode,
//            k_decode_exc)
// The Q16 layout and the h encoding are described in rv12_device.h.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rv12_device.h"
#include "rv12_internal.h"

namespace rv12 {

// ------------------------------------------------------------------ encode
__global__ void k_zero_i32(int32_t* p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// exponent histogram of all N*K weights (atomic integer counts: exact)
__global__ __launch_bounds__(256) void k_hist(const uint16_t* __restrict__ w, int64_t count,
                                              int32_t* __restrict__ hist) {
    __shared__ int32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    int64_t stride = (int64_t)gridDim.x * blockDim.x * 8;
    for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8; i < count; i += stride) {
        if (i + 8 <= count) {
            uint4 v = *reinterpret_cast<const uint4*>(w + i);
            uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                atomicAdd(&h[(d[j] >> 7) & 0xFF], 1);
                atomicAdd(&h[(d[j] >> 23) & 0xFF], 1);
            }
        } else {
            for (int64_t j = i; j < count; ++j) atomicAdd(&h[(w[j] >> 7) & 0xFF], 1);
        }
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

// one workgroup per row: m8, e4 and the row's exception count
__global__ __launch_bounds__(256) void k_encode_rows(const uint16_t* __restrict__ w, int K, int CH, int base,
                                                     uint8_t* __restrict__ m8, uint8_t* __restrict__ e4,
                                                     int32_t* __restrict__ row_exc) {
    const int n = blockIdx.x;
    const uint16_t* row = w + (int64_t)n * K;
    const int half = CH / 2;
    int cnt = 0;
    for (int jb = threadIdx.x; jb < K / 2; jb += blockDim.x) {
        int c = jb / half, i = jb % half;
        int k0 = c * CH + i, k1 = k0 + half;
        uint32_t b0 = row[k0], b1 = row[k1];
        int c0 = (int)((b0 >> 7) & 0xFF) - base, c1 = (int)((b1 >> 7) & 0xFF) - base;
        if (c0 < 0 || c0 > 14) { c0 = 15; ++cnt; }
        if (c1 < 0 || c1 > 14) { c1 = 15; ++cnt; }
        m8[(int64_t)n * K + k0] = (uint8_t)(((b0 >> 15) << 7) | (b0 & 0x7F));
        m8[(int64_t)n * K + k1] = (uint8_t)(((b1 >> 15) << 7) | (b1 & 0x7F));
        e4[(int64_t)n * (K / 2) + jb] = (uint8_t)(c0 | (c1 << 4));
    }
    __shared__ int red[4];
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
        row_exc[n] = s;
    }
}

// One list of weights outside an exponent window: the window start of row n is
// rbase[n], or base where rbase is null; the row's entries go to rp[n] on.
struct ExcList {
    const int32_t* rbase;
    int base;
    const int32_t* rp;
    int32_t* er;
    int32_t* ec;
    float* ev;
};

// One wave per row, up to two lists at once (the codec's and the packed form's):
// a row without entries is not read; otherwise lane l takes 8 consecutive
// weights of each 512, four such chunks in flight, and a chunk without entries
// (nearly all) costs one ballot.  In a chunk with some, a wave scan of the
// lanes' counts gives their places in column order.  Bound by reading the rows
// that have entries (6144 x 4096, one entry in 6553 weights: 13 us for both
// lists, 64 for each with a thread per 16 consecutive weights).
// VEC: K % 8 == 0 and w 16-byte aligned.
constexpr int kExcWaves = 4;
template <bool VEC>
__global__ __launch_bounds__(kExcWaves * 64) void k_exceptions(const uint16_t* __restrict__ w, int N, int K, ExcList a,
                                                               ExcList b, int nlists) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * kExcWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (n >= N) return;
    int posa = a.rp[n], posb = nlists > 1 ? b.rp[n] : 0;
    const bool ina = a.rp[n + 1] != posa, inb = nlists > 1 && b.rp[n + 1] != posb;
    if (!ina && !inb) return;
    const int basea = a.rbase ? a.rbase[n] : a.base, baseb = nlists > 1 ? (b.rbase ? b.rbase[n] : b.base) : 0;
    const uint16_t* row = w + (int64_t)n * K;
    auto put = [&](const ExcList& l, int& pos, uint32_t mask, const uint32_t (&bits)[4], int k) {
        const int cnt = __popc(mask);
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        int at = pos + inc - cnt;
        pos += __shfl(inc, 63);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (!(mask >> j & 1)) continue;
            l.er[at] = n;
            l.ec[at] = k + j;
            l.ev[at] = __uint_as_float((j & 1) ? (bits[j >> 1] & 0xFFFF0000u) : (bits[j >> 1] << 16));
            ++at;
        }
    };
    constexpr int U = 4;
    for (int k0 = lane * 8; k0 - lane * 8 < K; k0 += 512 * U) {
        uint32_t d[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512;
            if constexpr (VEC) {
                const uint4 v = k < K ? *reinterpret_cast<const uint4*>(row + k) : make_uint4(0, 0, 0, 0);
                d[u][0] = v.x, d[u][1] = v.y, d[u][2] = v.z, d[u][3] = v.w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    d[u][j] = (k + 2 * j < K ? row[k + 2 * j] : 0u) | (k + 2 * j + 1 < K ? row[k + 2 * j + 1] : 0u) << 16;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512;
            uint32_t ma = 0, mb = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int e = (int)((d[u][j >> 1] >> ((j & 1) * 16 + 7)) & 0xFF);
                const bool in = k + j < K;
                ma |= (uint32_t)(in && (uint32_t)(e - basea) > 14u) << j;
                mb |= (uint32_t)(in && (uint32_t)(e - baseb) > 14u) << j;
            }
            if (ina && __ballot(ma != 0) != 0) put(a, posa, ma, d[u], k);
            if (inb && __ballot(mb != 0) != 0) put(b, posb, mb, d[u], k);
        }
    }
}

static void launch_exceptions(const uint16_t* w, int N, int K, const ExcList& a, const ExcList* b, hipStream_t st) {
    const bool vec = K % 8 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
    hipLaunchKernelGGL((vec ? k_exceptions<true> : k_exceptions<false>), dim3((unsigned)((N + kExcWaves - 1) / kExcWaves)),
                       dim3(kExcWaves * 64), 0, st, w, N, K, a, b ? *b : a, b ? 2 : 1);
}

// ------------------------------------------------------------------ to_bf16
// one thread per 8 weights of a codec dict: code 15 (an exception) -> 0 bits
__global__ __launch_bounds__(256) void k_codec_to_bf16(const uint8_t* __restrict__ m8, const uint8_t* __restrict__ e4,
                                                       int K, int CH, int base, int64_t groups,
                                                       uint16_t* __restrict__ w) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= groups) return;
    const int64_t i0 = gid * 8;  // K % 8 == 0: the 8 weights share a row and a half-chunk
    const int64_t n = i0 / K;
    const int k0 = (int)(i0 % K);
    const int half = CH / 2;
    const int c = k0 / CH, i = k0 % CH;
    const uint8_t* erow = e4 + n * (K / 2) + (int64_t)c * half + (i % half);
    const int shift = i < half ? 0 : 4;
    uint32_t b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t m = m8[i0 + j];
        const uint32_t code = (erow[j] >> shift) & 15u;
        b[j] = code == 15u ? 0u : ((m >> 7) << 15) | ((code + (uint32_t)base) << 7) | (m & 0x7Fu);
    }
    *reinterpret_cast<uint4*>(w + i0) = make_uint4(b[0] | b[1] << 16, b[2] | b[3] << 16, b[4] | b[5] << 16,
                                                   b[6] | b[7] << 16);
}

// exact exception values into a bf16 matrix
// (entries outside the matrix are skipped)
__global__ __launch_bounds__(256) void k_scatter_exc(const int32_t* __restrict__ er, const int32_t* __restrict__ ec,
                                                     const float* __restrict__ ev, int64_t E, int N, int K,
                                                     uint16_t* __restrict__ w) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= E) return;
    const int r = er[j], c = ec[j];
    if (r < 0 || r >= N || c < 0 || c >= K) return;
    w[(int64_t)r * K + c] = (uint16_t)(__float_as_uint(ev[j]) >> 16);
}

// ------------------------------------------------------------------ pack
// Every row's exponent window, chosen by the reference's rule for a whole
// matrix (wcomp.py:19-21): the first start b whose 15-wide window [b, b+14]
// holds the most weights; rbase[n] = b, row_exc[n] = the weights outside it.
// One pass over the weights, one wave per row (a grid-stride loop): counts of
// the 256 exponents in LDS, 16 copies per wave (copy lane % 16, 260 words apart,
// so that the few exponents most weights have fall on different banks and seldom
// on the same word); the copies are never cleared: a row's counts are the
// difference to the wave's running totals, whose sum over the grid is the whole
// matrix's histogram.  cs (may be null): each row's 256 inclusive prefix counts;
// part (with cs): the workgroup's share of the histogram.  Bound by the LDS
// counts beside the read of the weights (6144 x 4096: 15.6 us, 3.2 TB/s, where
// separate passes for the histogram, windows and counts, with one copy per
// workgroup, took 53, 60 and 9).
constexpr int kRowWaves = 4, kRowCopies = 16, kRowPitch = 260;
constexpr size_t kRowLds = (size_t)kRowWaves * (kRowCopies * kRowPitch + 256) * 4;
constexpr int kRowGrid = 512;  // two workgroups per CU
__global__ __launch_bounds__(kRowWaves * 64) void k_row_windows(const uint16_t* __restrict__ w, int N, int K,
                                                                int32_t* __restrict__ rbase,
                                                                int32_t* __restrict__ row_exc,
                                                                int32_t* __restrict__ cs,
                                                                int32_t* __restrict__ part) {
    extern __shared__ int32_t lds_i[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int32_t* h = lds_i + wave * (kRowCopies * kRowPitch + 256);
    int32_t* pre = h + kRowCopies * kRowPitch;  // the row's prefix counts
    for (int i = lane * 4; i < kRowCopies * kRowPitch; i += 256) *reinterpret_cast<int4*>(h + i) = make_int4(0, 0, 0, 0);
    int32_t* hc = h + (lane % kRowCopies) * kRowPitch;
    int tot[4] = {0, 0, 0, 0};  // running totals of exponents 4 lane .. 4 lane + 3
    auto count = [&](uint4 v) {
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            atomicAdd(&hc[(d[j] >> 7) & 0xFF], 1);
            atomicAdd(&hc[(d[j] >> 23) & 0xFF], 1);
        }
    };
    for (int n = blockIdx.x * kRowWaves + wave; n < N; n += gridDim.x * kRowWaves) {
        const uint16_t* row = w + (int64_t)n * K;
        constexpr int U = 4;
        int k = lane * 8;
        for (; k + 512 * (U - 1) < K; k += 512 * U) {
            uint4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const uint4*>(row + k + u * 512);
#pragma unroll
            for (int u = 0; u < U; ++u) count(v[u]);
        }
        for (; k < K; k += 512) count(*reinterpret_cast<const uint4*>(row + k));
        // (one wave's LDS accesses stay in order; the fences keep the compiler's)
        asm volatile("" ::: "memory");
        int c[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < kRowCopies; ++i) {
            const int4 q = *reinterpret_cast<const int4*>(h + i * kRowPitch + lane * 4);
            c[0] += q.x, c[1] += q.y, c[2] += q.z, c[3] += q.w;
        }
        int s[4], run = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = c[j] - tot[j];
            tot[j] = c[j];
            run += r;
            s[j] = run;
        }
        int inc = run;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        const int before = inc - run;  // weights of exponents below 4 lane
        const int4 ps = make_int4(before + s[0], before + s[1], before + s[2], before + s[3]);
        *reinterpret_cast<int4*>(pre + lane * 4) = ps;
        if (cs) *reinterpret_cast<int4*>(cs + (int64_t)n * 256 + lane * 4) = ps;
        asm volatile("" ::: "memory");
        int best = -1;  // count * 256 + 255 - b: the largest count, the first b of it (K <= 2^20)
        const int below[4] = {before, ps.x, ps.y, ps.z};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = lane * 4 + j;
            if (b <= 241) best = max(best, (pre[b + 14] - below[j]) * 256 + 255 - b);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) best = max(best, __shfl_xor(best, o));
        if (lane == 0) {
            rbase[n] = 255 - (best & 255);
            row_exc[n] = K - (best >> 8);
        }
        asm volatile("" ::: "memory");
    }
    if (part) {
        *reinterpret_cast<int4*>(pre + lane * 4) = make_int4(tot[0], tot[1], tot[2], tot[3]);
        __syncthreads();
        int sum = 0;
#pragma unroll
        for (int i = 0; i < kRowWaves; ++i)
            sum += lds_i[i * (kRowCopies * kRowPitch + 256) + kRowCopies * kRowPitch + threadIdx.x];
        part[(int64_t)blockIdx.x * 256 + threadIdx.x] = sum;
    }
}
static_assert(kRowWaves * 64 == 256 && kRowCopies * kRowPitch % 4 == 0, "one thread per exponent");

// The matrix's histogram from the parts, 4 exponents per workgroup (one
// workgroup over all of them, and over the rows' counts below, waits for one
// CU's loads: 38 us of a 6144 x 4096 matrix where these passes take about 12).
constexpr int kHistBins = 4;
__global__ __launch_bounds__(256) void k_hist_sum(const int32_t* __restrict__ part, int nparts,
                                                  int64_t* __restrict__ hist) {
    __shared__ int64_t red[256];
    const int t = threadIdx.x, bin = blockIdx.x * kHistBins + t % kHistBins;
    int64_t sum = 0;
#pragma unroll 8
    for (int i = t / kHistBins; i < nparts; i += 256 / kHistBins) sum += part[(int64_t)i * 256 + bin];
    red[t] = sum;
    __syncthreads();
    for (int d = 128; d >= kHistBins; d >>= 1) {
        if (t < d) red[t] += red[t + d];
        __syncthreads();
    }
    if (t < kHistBins) hist[bin] = red[t];
}

// The matrix's own window from its histogram, by the rows' rule (a workgroup of 256)
__device__ __forceinline__ int matrix_base(const int64_t* __restrict__ hist) {
    __shared__ int64_t h[256];
    __shared__ int64_t red[4];
    const int t = threadIdx.x;
    h[t] = hist[t];
    __syncthreads();
    int64_t key = -1;  // count * 256 + 255 - b: the largest count, the first b of it
    if (t <= 241) {
        int64_t c = 0;
        for (int j = 0; j < 15; ++j) c += h[t + j];
        key = c * 256 + 255 - t;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) key = max(key, (int64_t)__shfl_xor((long long)key, o));
    if ((t & 63) == 0) red[t >> 6] = key;
    __syncthreads();
    return 255 - (int)(max(max(red[0], red[1]), max(red[2], red[3])) & 255);
}

// The matrix's window (every workgroup finds it) and each row's weights outside
// it, from the row's prefix counts.
__global__ __launch_bounds__(256) void k_row_counts(const int64_t* __restrict__ hist, const int32_t* __restrict__ cs,
                                                    int N, int K, int32_t* __restrict__ row_exc,
                                                    int32_t* __restrict__ out) {
    const int base = matrix_base(hist);
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n < N) {
        const int32_t* r = cs + (int64_t)n * 256;
        row_exc[n] = K - (r[base + 14] - (base > 0 ? r[base - 1] : 0));
    }
    if (n == 0) out[0] = base;
}

// The same from the weights, 16 lanes per row, for rows that are shorter than their
// prefix counts would be useful (kCountColumns).
__global__ __launch_bounds__(256) void k_row_recount(const int64_t* __restrict__ hist, const uint16_t* __restrict__ w,
                                                     int N, int K, int32_t* __restrict__ row_exc,
                                                     int32_t* __restrict__ out) {
    const int base = matrix_base(hist);
    const int l = threadIdx.x & 15;
    for (int n = blockIdx.x * 16 + (threadIdx.x >> 4); n < N; n += gridDim.x * 16) {
        const uint16_t* row = w + (int64_t)n * K;
        int cnt = 0;
        for (int k = l * 8; k < K; k += 128) {
            const uint4 v = *reinterpret_cast<const uint4*>(row + k);
            const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                cnt += ((d[j] >> 7 & 0xFF) - (uint32_t)base > 14u) + ((d[j] >> 23 & 0xFF) - (uint32_t)base > 14u);
        }
#pragma unroll
        for (int o = 8; o >= 1; o >>= 1) cnt += __shfl_xor(cnt, o);
        if (l == 0) row_exc[n] = cnt;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = base;
}

// One workgroup: the row pointers of both exception lists from the rows' counts
// (16-byte aligned), out = {base (as it is), entries, packed entries}.
constexpr int kPlanThreads = 1024, kPlanRows = 4 * kPlanThreads;
__global__ __launch_bounds__(kPlanThreads) void k_row_pointers(const int32_t* __restrict__ exc,
                                                               const int32_t* __restrict__ qexc, int N,
                                                               int32_t* __restrict__ rp, int32_t* __restrict__ qrp,
                                                               int32_t* __restrict__ out) {
    __shared__ int32_t wsum[2][16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int32_t ca = 0, cb = 0;  // entries of the rows before this tile
    for (int n0 = 0; n0 < N; n0 += kPlanRows) {
        const int n = n0 + t * 4;
        int a[4] = {0, 0, 0, 0}, b[4] = {0, 0, 0, 0};
        if (n + 3 < N) {
            const int4 va = *reinterpret_cast<const int4*>(exc + n), vb = *reinterpret_cast<const int4*>(qexc + n);
            a[0] = va.x, a[1] = va.y, a[2] = va.z, a[3] = va.w;
            b[0] = vb.x, b[1] = vb.y, b[2] = vb.z, b[3] = vb.w;
        } else {
            for (int i = 0; i < 4; ++i)
                if (n + i < N) a[i] = exc[n + i], b[i] = qexc[n + i];
        }
#pragma unroll
        for (int i = 1; i < 4; ++i) a[i] += a[i - 1], b[i] += b[i - 1];
        int ia = a[3], ib = b[3];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int va = __shfl_up(ia, d), vb = __shfl_up(ib, d);
            if (lane >= d) ia += va, ib += vb;
        }
        if (lane == 63) wsum[0][wave] = ia, wsum[1][wave] = ib;
        __syncthreads();
        int oa = ca + ia - a[3], ob = cb + ib - b[3];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int va = wsum[0][i], vb = wsum[1][i];
            if (i < wave) oa += va, ob += vb;
            ca += va, cb += vb;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < N) rp[n + i + 1] = oa + a[i], qrp[n + i + 1] = ob + b[i];
    }
    if (t == 0) {
        rp[0] = qrp[0] = 0;
        out[1] = ca;
        out[2] = cb;
    }
}

// one thread per 12-byte group (row block b, step s, lane l): the 8 weights of
// row 16b + l%16 at k = 32s + 8(l/16) + 0..7 as h values of the row's window
__global__ __launch_bounds__(256) void k_pack_tiles(const uint16_t* __restrict__ w, int N, int K,
                                                    const int32_t* __restrict__ rbase, uint32_t* __restrict__ tiles,
                                                    int64_t groups) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= groups) return;
    const int nsteps = K / 32;
    const int l = (int)(gid & 63);
    const int64_t bs = gid >> 6;
    const int s = (int)(bs % nsteps);
    const int64_t b = bs / nsteps;
    const int64_t n = b * 16 + (l & 15);
    const int k0 = s * 32 + (l >> 4) * 8;
    uint32_t h[8];
    if (n < N) {
        const int base = rbase[n];
        const uint32_t off = (uint32_t)(base - scale_exp(base));  // c = code + off
        const uint4 v = *reinterpret_cast<const uint4*>(w + n * K + k0);
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t bits = (d[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu;
            const int code = (int)((bits >> 7) & 0xFF) - base;
            h[j] = (code < 0 || code > 14) ? 0u : (bits & 0x807Fu) | (((uint32_t)code + off) << 7);
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = 0u;
    }
    const uint32_t p0 = h[0] | (h[1] << 16), p1 = h[2] | (h[3] << 16), p2 = h[4] | (h[5] << 16),
                   p3 = h[6] | (h[7] << 16);
    uint32_t* o = tiles + gid * 3;
    o[0] = p0 | ((p3 & 0x000F000Fu) << 11);
    o[1] = p1 | ((p3 & 0x00F000F0u) << 7);
    o[2] = p2 | ((p3 & 0x07000700u) << 3) | ((p3 & 0x80008000u) >> 1);
}

// ------------------------------------------------------------------ decode
// one thread per 12-byte group of the row blocks covering [first, last)
__global__ __launch_bounds__(256) void k_decode(const uint32_t* __restrict__ tiles,
                                                const int32_t* __restrict__ rbase, int K, int first, int last,
                                                int64_t b0, int64_t groups, void* __restrict__ out, int out_f32) {
    int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= groups) return;
    const int nsteps = K / 32;
    const int l = (int)(gid & 63);
    const int64_t bs = gid >> 6;
    const int s = (int)(bs % nsteps);
    const int64_t b = b0 + bs / nsteps;
    const int64_t n = b * 16 + (l & 15);
    if (n < first || n >= last) return;
    const int k0 = s * 32 + (l >> 4) * 8;
    const uint32_t* t = tiles + ((b * nsteps + s) * 64 + l) * 3;
    uint32_t p[4];
    unpack_pairs(t[0], t[1], t[2], p);
    uint32_t v[8];
    const int sc = scale_exp(rbase[n]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = h_to_bf16(p[j] & 0xFFFFu, sc);
        v[2 * j + 1] = h_to_bf16(p[j] >> 16, sc);
    }
    const int64_t o = (n - first) * (int64_t)K + k0;
    if (out_f32) {
        uint4* d = reinterpret_cast<uint4*>(reinterpret_cast<uint32_t*>(out) + o);
        d[0] = make_uint4(v[0] << 16, v[1] << 16, v[2] << 16, v[3] << 16);
        d[1] = make_uint4(v[4] << 16, v[5] << 16, v[6] << 16, v[7] << 16);
    } else {
        *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(out) + o) =
            make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
    }
}

// scatter the exceptions with index in [e0, e1) whose row is in [first, last)
__global__ __launch_bounds__(256) void k_decode_exc(const int32_t* __restrict__ er, const int32_t* __restrict__ ec,
                                                    const float* __restrict__ ev, int64_t e0, int64_t e1, int K,
                                                    int first, int last, void* __restrict__ out, int out_f32) {
    int64_t j = e0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= e1) return;
    const int r = er[j];
    if (r < first || r >= last) return;
    const int64_t o = (int64_t)(r - first) * K + ec[j];
    const uint32_t bits = __float_as_uint(ev[j]);
    if (out_f32) reinterpret_cast<uint32_t*>(out)[o] = bits;
    else reinterpret_cast<uint16_t*>(out)[o] = (uint16_t)(bits >> 16);
}

// ------------------------------------------------------------------ launch
void launch_codec_to_bf16(const rv12_codec& c, uint16_t* w, hipStream_t st) {
    const int64_t groups = (int64_t)c.n * c.k / 8;
    hipLaunchKernelGGL(k_codec_to_bf16, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, c.m8, c.e4, c.k,
                       c.ch, c.base, groups, w);
    if (c.n_exc > 0)
        hipLaunchKernelGGL(k_scatter_exc, dim3((unsigned)((c.n_exc + 255) / 256)), dim3(256), 0, st, c.er, c.ec,
                           c.ev, c.n_exc, c.n, c.k, w);
}

static int row_grid(int N) { return min((N + kRowWaves - 1) / kRowWaves, kRowGrid); }
static void launch_row_windows(const uint16_t* w, int N, int K, int32_t* rbase, int32_t* row_exc, int32_t* cs,
                               int32_t* part, hipStream_t st) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_row_windows), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kRowLds);
    hipLaunchKernelGGL(k_row_windows, dim3((unsigned)row_grid(N)), dim3(kRowWaves * 64), kRowLds, st, w, N, K, rbase, row_exc, cs, part);
}

void launch_pack_plan(const uint16_t* w, int N, int K, int32_t* rbase, int32_t* row_exc, hipStream_t st) {
    launch_row_windows(w, N, K, rbase, row_exc, nullptr, nullptr, st);
}

static void launch_pack_tiles(const uint16_t* w, int N, int K, const int32_t* rbase, uint32_t* tiles, hipStream_t st) {
    const int64_t groups = (int64_t)((N + 15) / 16) * (K / 32) * 64;
    hipLaunchKernelGGL(k_pack_tiles, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, w, N, K, rbase, tiles,
                       groups);
}

void launch_pack(const uint16_t* w, int N, int K, const int32_t* rbase, const int32_t* rp, uint32_t* tiles,
                 int32_t* er, int32_t* ec, float* ev, int64_t n_exc, hipStream_t st) {
    launch_pack_tiles(w, N, K, rbase, tiles, st);
    if (n_exc > 0) launch_exceptions(w, N, K, ExcList{rbase, 0, rp, er, ec, ev}, nullptr, st);
}

// Workspace: the histogram and its parts, each row's entries in both lists, and
// from kCountColumns columns on the row prefix counts, 1 KB a row: no more there than
// the 1.5 bytes per weight of m8 / e4 that the separate calls hold beside the tiles.
// Shorter rows are counted again instead (65536 x 672: 69 MB at most beside the
// weights and 194 us, 136 MB and 184 us with prefix counts; 135 MB as separate calls).
constexpr int kCountColumns = 688;
static size_t padded4(int N) { return ((size_t)N + 3) / 4 * 4; }
size_t compress_ws_bytes(int N, int K) {
    return 256 * 8 + ((size_t)row_grid(N) * 256 + 2 * padded4(N) + (K >= kCountColumns ? (size_t)N * 256 : 0)) * 4;
}

void launch_compress_plan(const uint16_t* w, int N, int K, int32_t* rbase, int32_t* rp, int32_t* qrp, int32_t* out,
                          void* ws, hipStream_t st) {
    int64_t* hist = static_cast<int64_t*>(ws);
    int32_t* part = reinterpret_cast<int32_t*>(hist + 256);
    int32_t* exc = part + (size_t)row_grid(N) * 256;
    int32_t* qexc = exc + padded4(N);
    int32_t* cs = K >= kCountColumns ? qexc + padded4(N) : nullptr;
    launch_row_windows(w, N, K, rbase, qexc, cs, part, st);
    hipLaunchKernelGGL(k_hist_sum, dim3(256 / kHistBins), dim3(256), 0, st, part,
                       row_grid(N), hist);
    if (cs)
        hipLaunchKernelGGL(k_row_counts, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st, hist, cs, N, K, exc, out);
    else
        hipLaunchKernelGGL(k_row_recount, dim3((unsigned)min((N + 15) / 16, 2048)), dim3(256), 0, st, hist, w, N, K, exc,
                           out);
    hipLaunchKernelGGL(k_row_pointers, dim3(1), dim3(kPlanThreads), 0, st, exc, qexc, N, rp, qrp, out);
}

void launch_compress_write(const uint16_t* w, int N, int K, int base, const int32_t* rp, int32_t* er, int32_t* ec,
                           float* ev, int64_t n_exc, const int32_t* rbase, const int32_t* qrp, int32_t* qer,
                           int32_t* qec, float* qev, int64_t n_qexc, uint32_t* tiles, hipStream_t st) {
    launch_pack_tiles(w, N, K, rbase, tiles, st);
    const ExcList a = {nullptr, base, rp, er, ec, ev}, b = {rbase, 0, qrp, qer, qec, qev};
    if (n_exc > 0 && n_qexc > 0) launch_exceptions(w, N, K, a, &b, st);
    else if (n_exc > 0) launch_exceptions(w, N, K, a, nullptr, st);
    else if (n_qexc > 0) launch_exceptions(w, N, K, b, nullptr, st);
}

void launch_decode(const rv12_matrix& w, int first, int last, void* out, int out_f32, hipStream_t st,
                   int64_t e0, int64_t e1) {
    const int64_t b0 = first / 16, b1 = (last + 15) / 16;
    const int64_t groups = (b1 - b0) * (w.k / 32) * 64;
    hipLaunchKernelGGL(k_decode, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, w.tiles, w.rbase, w.k,
                       first, last, b0, groups, out, out_f32);
    if (e1 > e0)
        hipLaunchKernelGGL(k_decode_exc, dim3((unsigned)((e1 - e0 + 255) / 256)), dim3(256), 0, st, w.er, w.ec, w.ev,
                           e0, e1, w.k, first, last, out, out_f32);
}

void launch_encode_stats(const uint16_t* w, int64_t count, int32_t* hist, hipStream_t st) {
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(256), 0, st, hist, 256);
    int64_t blocks = (count / 8 + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_hist, dim3((unsigned)blocks), dim3(256), 0, st, w, count, hist);
}

void launch_encode(const uint16_t* w, int N, int K, int CH, int base, uint8_t* m8, uint8_t* e4, int32_t* row_exc,
                   hipStream_t st) {
    hipLaunchKernelGGL(k_encode_rows, dim3((unsigned)N), dim3(256), 0, st, w, K, CH, base, m8, e4, row_exc);
}

void launch_encode_exc(const uint16_t* w, int N, int K, int base, const int32_t* rp, int32_t* er, int32_t* ec,
                       float* ev, hipStream_t st) {
    launch_exceptions(w, N, K, ExcList{nullptr, base, rp, er, ec, ev}, nullptr, st);
}

}  // namespace rv12
