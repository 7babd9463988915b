// The reference's test-side attention-weights and softmax kernels for gfx950
// (get_attention_weights and softmax, attention.cu:240-343).
#include "prefill.h"

#include "tiny_llm/hip_utils.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <stdexcept>

namespace tiny_llm {
namespace detail {

namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float    f32x16 __attribute__((ext_vector_type(16)));
typedef float    f32x32 __attribute__((ext_vector_type(32)));

// Rounds x to fp32 in a register before whatever consumes it: keeps the
// compiler from folding a multiply into the fp16 conversion that follows
// (v_fma_mixlo_f16 rounds once, the reference's __float2half(a * b) twice).
__device__ __forceinline__ float materialize(float x) {
    asm volatile("" : "+v"(x));
    return x;
}

// attention_weights_kernel: W = fp16(scale * Q K^T) of one (batch, head), the
// products summed over d in order with one fp32 rounding each -- the bits of
// the reference's per-element fmaf loop (attention.cu:240-268).
//
// That order is kept by the fp32 MFMAs with a k depth of one: each is a single
// fused multiply-add per output, at twice the fp32 rate of the vector ALU (256
// flops per cycle and CU).  A holds keys, B 64 queries; the broadcast control
// gives every output block the same block of A:
//   BIG    v_mfma_f32_32x32x1_2b: a wave's tile is 64 keys x 64 queries, two
//          instructions a dimension (one for each half of the keys); 128 x
//          128 per workgroup of 4 waves
//   small  v_mfma_f32_16x16x1_4b: 16 keys x 64 queries, one instruction a
//          dimension; 64 x 64 per workgroup.  A wave's chain of dependent MFMAs
//          is a quarter as long, for launches that do not fill the chip.
// A lane then holds four consecutive keys of one query per four registers,
// which go through LDS so that every store is part of a row.  Both tiles are
// staged in LDS 64 (small: 128) dimensions at a time (fp16, rows padded by 16
// bytes: the fragment reads of 16 lanes fall on distinct banks); a workgroup
// takes 36 KB, so four share a CU and one's loads and stores run under the
// others' products (BIG with 128 dimensions a stage, two per CU: 103 us where
// this takes 85).  VIN / VOUT: rows are read / written in 16-byte pieces
// (16-byte aligned bases and row pitches), else by element.
// Bound by the matrix rate: 32 heads of 1000 x 1000 at 128 dimensions 85-93
// us (88-97 of the 157 fp32 TFLOP/s; one thread per output, each reading its
// own key row, took 11160 us), element stores (1000 x 1001) 102 us.  Launches
// of a few tiles stay at the launch floor of about 7 us, as short ones were
// (1 x 512 x 128: 17.3 before).
template <bool BIG, bool VIN, bool VOUT>
__global__ __launch_bounds__(256, 3) void attention_weights_kernel(const __half *q, const __half *k, __half *w,
                                                                   float scale, int Lq, int Lk, int D, int causal) {
    constexpr int kDims = BIG ? 64 : 128;  // dimensions per stage
    constexpr int kPitch = kDims + 8;    // halves per staged row
    constexpr int PP = kDims / 8;        // 16-byte pieces per staged row
    constexpr int TILE = BIG ? 128 : 64; // queries and keys per workgroup
    constexpr int WK = BIG ? 64 : 16;    // keys per wave (64 queries)
    constexpr int OUTP = WK + 4;         // halves per staged output row
    __shared__ __align__(16) uint16_t lds[2 * TILE * kPitch];
    static_assert(4 * 64 * OUTP <= 2 * TILE * kPitch, "the output stage fits the tiles");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Key tiles rotate with the query tile and the head: workgroups go to the 8 XCDs in
    // turn, and with a multiple of 8 key tiles one XCD would otherwise take
    // the same key tile of every row -- under the causal mask all of the
    // work, or none of it.
    const int     kt = (int)((blockIdx.x + 3 * blockIdx.y + blockIdx.z) % gridDim.x);
    const int     k0 = kt * TILE, q0 = blockIdx.y * TILE;
    const int64_t bh = blockIdx.z;
    const __half *qb = q + bh * Lq * D, *kb = k + bh * Lk * D;
    __half       *wb = w + bh * Lq * Lk;
    const int     wk = k0 + WK * (BIG ? wave >> 1 : wave), wq = q0 + (BIG ? 64 * (wave & 1) : 0); // the wave's tile
    // Nothing to add where the wave's tile is outside the matrix or wholly
    // above the diagonal; the same for a BIG tile's upper half of the keys.
    const int  lastq = min(wq + 63, Lq - 1);
    const bool live0 = wk < Lk && wq < Lq && !(causal && wk > lastq);
    const bool live1 = BIG && live0 && wk + 32 < Lk && !(causal && wk + 32 > lastq);
    const bool tile_live = !(causal && k0 > min(q0 + TILE, Lq) - 1); // uniform over the workgroup

    f32x32 acc[2]; // BIG: [half of the keys][32 x query block]; small: acc[0][4 x query block + i]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[h][i] = 0.0f;
    f32x16 acc16 = {};

    for (int d0 = 0; tile_live && d0 < D; d0 += kDims) {
        const int nd = min(kDims, D - d0);
        const int pieces = (nd + 7) >> 3; // 16-byte pieces per row of this stage
        // Rows 0 .. TILE-1 queries, then the keys; zeros past the matrix.  A
        // batch of 8 loads is in flight per thread.
        for (int p0 = 0; p0 < 2 * TILE * PP; p0 += 8 * 256) {
            uint4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int     p = p0 + u * 256 + tid, r = p / PP, x = p % PP;
                const bool    isq = r < TILE;
                const int     row = isq ? q0 + r : k0 + r - TILE;
                const __half *src = (isq ? qb : kb) + (int64_t)row * D + d0 + 8 * x;
                v[u] = make_uint4(0u, 0u, 0u, 0u);
                if (row < (isq ? Lq : Lk) && x < pieces) {
                    if constexpr (VIN) {
                        v[u] = *reinterpret_cast<const uint4 *>(src);
                    } else {
                        const uint16_t *s16 = reinterpret_cast<const uint16_t *>(src);
                        const int       n = nd - 8 * x; // halves left in the row
                        uint32_t        h[8];
#pragma unroll
                        for (int j = 0; j < 8; ++j) h[j] = s16[min(j, n - 1)];
#pragma unroll
                        for (int j = 1; j < 8; ++j) h[j] = j < n ? h[j] : 0u;
                        v[u] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int p = p0 + u * 256 + tid, r = p / PP, x = p % PP;
                *reinterpret_cast<uint4 *>(&lds[r * kPitch + 8 * x]) = v[u];
            }
        }
        __syncthreads();
        if (live0) {
            const uint16_t *qs = &lds[(wq - q0 + lane) * kPitch];
            const uint16_t *ks = &lds[(TILE + wk - k0 + (BIG ? lane : lane & 15)) * kPitch];
            // (dimensions past nd are staged as zeros: fma(0, 0, s) = s, and s is
            // never -0, a sum that starts from +0)
            f16x8 qv = *reinterpret_cast<const f16x8 *>(qs), kv = *reinterpret_cast<const f16x8 *>(ks);
            for (int x = 0; x < pieces; ++x) {
                const int   nx = min(x + 1, pieces - 1); // the next piece, read under this one's products
                const f16x8 qn = *reinterpret_cast<const f16x8 *>(qs + 8 * nx);
                const f16x8 kn = *reinterpret_cast<const f16x8 *>(ks + 8 * nx);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float a = (float)kv[j], b = (float)qv[j];
                    if constexpr (BIG) {
                        acc[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, acc[0], 1, 0, 0);
                        if (live1) acc[1] = __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, acc[1], 1, 1, 0);
                    } else {
                        acc16 = __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, acc16, 2, 0, 0);
                    }
                }
                qv = qn;
                kv = kn;
            }
        }
        __syncthreads(); // the tiles are overwritten (next stage, or the output stage)
    }

    // Output: the wave's 64 queries x WK keys through its own LDS region.
    uint16_t *st = lds + wave * 64 * OUTP;
    auto      put = [&](int qr, int kc, float s0, float s1, float s2, float s3) { // keys kc .. kc+3 of query qr
        const float s[4] = {s0, s1, s2, s3};
        f16x4       o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[i] = causal && wk + kc + i > wq + qr ? (_Float16)0.0f : (_Float16)materialize(s[i] * scale);
        *reinterpret_cast<f16x4 *>(&st[qr * OUTP + kc]) = o;
    };
    if constexpr (BIG) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    put(32 * b + (lane & 31), 32 * h + 8 * g + 4 * (lane >> 5), acc[h][16 * b + 4 * g],
                        acc[h][16 * b + 4 * g + 1], acc[h][16 * b + 4 * g + 2], acc[h][16 * b + 4 * g + 3]);
    } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
            put(16 * b + (lane & 15), 4 * (lane >> 4), acc16[4 * b], acc16[4 * b + 1], acc16[4 * b + 2], acc16[4 * b + 3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if constexpr (VOUT) { // WK / 8 lanes a row, 16 bytes each, as two 8-byte LDS reads
        constexpr int LPR = WK / 8, RPI = 64 / LPR;
        const int     kc = 8 * (lane % LPR);
#pragma unroll
        for (int u = 0; u < 64 / RPI; ++u) {
            const int r = RPI * u + lane / LPR;
            if (wq + r < Lq && wk + kc < Lk) {
                const uint2 lo = *reinterpret_cast<const uint2 *>(&st[r * OUTP + kc]);
                const uint2 hi = *reinterpret_cast<const uint2 *>(&st[r * OUTP + kc + 4]);
                *reinterpret_cast<uint4 *>(wb + (int64_t)(wq + r) * Lk + wk + kc) = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        }
    } else { // WK lanes a row
        constexpr int RPI = 64 / WK;
        uint16_t     *w16 = reinterpret_cast<uint16_t *>(wb);
        const int     kc = lane % WK;
#pragma unroll 8
        for (int u = 0; u < 64 / RPI; ++u) {
            const int r = RPI * u + lane / WK;
            if (wq + r < Lq && wk + kc < Lk) w16[(int64_t)(wq + r) * Lk + wk + kc] = st[r * OUTP + kc];
        }
    }
}

// softmax_kernel (attention.cu:288-343): y = e^(x - m) / (sum + 1e-6) of each
// row, m starting from the lowest float.  WPR waves per row (1, or 4: one
// workgroup), 8 NV values a lane held in registers, so a row is read once and
// written once; VEC: the values of a lane are 16-byte pieces (rows a multiple
// of 8 long on 16-byte aligned bases), else single elements, consecutive
// lanes on consecutive elements.  Bound by memory: 32000 rows of 1000 in 22.4
// us (5.7 TB/s), of 1001 in 37.7; three passes by 2-byte loads took 70.  One
// wave per row up to 1024 values (four rows a workgroup, no barrier), beyond
// it a workgroup, so that a lane holds at most 32 values.  Outputs beyond the L2s'
// 32 MB are stored non-temporally (nt), which leaves the caches to the inputs
// still to be read: 32000 x 1000 over four arrays in turn 25-27 -> 21-22 us.
constexpr float kLog2e = 1.4426950408889634f;

template <int WPR, int NV, bool VEC>
__global__ __launch_bounds__(256) void softmax_kernel(const __half *in, __half *out, int64_t rows, int S, bool nt) {
    constexpr int T = 64 * WPR; // lanes of a row
    __shared__ float red[8];
    const int     lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int     t = WPR == 1 ? lane : (int)threadIdx.x;
    const int64_t row = WPR == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x;
    if (row >= rows) return; // whole waves (WPR == 1: no barrier below)
    const uint16_t *x = reinterpret_cast<const uint16_t *>(in) + row * S;
    uint16_t       *y = reinterpret_cast<uint16_t *>(out) + row * S;
    auto            at = [&](int v, int j) { return VEC ? 8 * (v * T + t) + j : (8 * v + j) * T + t; };
    uint16_t        h[NV][8];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        if constexpr (VEC) {
            uint4 p = make_uint4(0u, 0u, 0u, 0u);
            if (at(v, 0) < S) p = *reinterpret_cast<const uint4 *>(x + at(v, 0));
            __builtin_memcpy(h[v], &p, 16);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) h[v][j] = at(v, j) < S ? x[at(v, j)] : (uint16_t)0;
        }
    }
    auto  val = [&](int v, int j) { return (float)__builtin_bit_cast(_Float16, h[v][j]); };
    float m = -FLT_MAX;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (at(v, j) < S) m = fmaxf(m, val(v, j));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if constexpr (WPR == 4) {
        if (lane == 0) red[wave] = m;
        __syncthreads();
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
    float e[NV][8], sum = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            e[v][j] = exp2f((val(v, j) - m) * kLog2e);
            if (at(v, j) < S) sum += e[v][j];
        }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if constexpr (WPR == 4) {
        if (lane == 0) red[4 + wave] = sum;
        __syncthreads();
        sum = (red[4] + red[5]) + (red[6] + red[7]);
    }
    const float inv = 1.0f / (sum + 1e-6f);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        uint16_t o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __builtin_bit_cast(uint16_t, (_Float16)materialize(e[v][j] * inv));
        if constexpr (VEC) {
            u32x4 p;
            __builtin_memcpy(&p, o, 16);
            u32x4 *const dst = reinterpret_cast<u32x4 *>(y + at(v, 0));
            if (at(v, 0) < S) {
                if (nt) __builtin_nontemporal_store(p, dst);
                else *dst = p;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (at(v, j) < S) y[at(v, j)] = o[j];
        }
    }
}

// Rows longer than the registers of a workgroup hold: three passes over the row.
__global__ __launch_bounds__(256) void softmax_long_kernel(const __half *in, __half *out, int S) {
    __shared__ float red[8];
    const __half *x = in + (int64_t)blockIdx.x * S;
    __half       *y = out + (int64_t)blockIdx.x * S;
    const int     tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float         m = -FLT_MAX;
    for (int i = tid; i < S; i += 256) m = fmaxf(m, __half2float(x[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.0f;
    for (int i = tid; i < S; i += 256) sum += exp2f((__half2float(x[i]) - m) * kLog2e);
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) red[4 + wave] = sum;
    __syncthreads();
    sum = (red[4] + red[5]) + (red[6] + red[7]);
    const float inv = 1.0f / (sum + 1e-6f);
    for (int i = tid; i < S; i += 256)
        y[i] = __float2half(materialize(exp2f((__half2float(x[i]) - m) * kLog2e) * inv));
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <bool VEC>
void launch_softmax_v(const __half *in, __half *out, int rows, int S, hipStream_t stream) {
    const bool nt = (int64_t)rows * S * 2 > (32LL << 20); // more than the L2s hold for the reader
    const dim3 per4((unsigned)(((int64_t)rows + 3) / 4)), per1((unsigned)rows), block(256);
    if (S <= 512) hipLaunchKernelGGL((softmax_kernel<1, 1, VEC>), per4, block, 0, stream, in, out, (int64_t)rows, S, nt);
    else if (S <= 1024) hipLaunchKernelGGL((softmax_kernel<1, 2, VEC>), per4, block, 0, stream, in, out, (int64_t)rows, S, nt);
    else if (S <= 2048) hipLaunchKernelGGL((softmax_kernel<4, 1, VEC>), per1, block, 0, stream, in, out, (int64_t)rows, S, nt);
    else if (S <= 4096) hipLaunchKernelGGL((softmax_kernel<4, 2, VEC>), per1, block, 0, stream, in, out, (int64_t)rows, S, nt);
    else if (S <= 8192) hipLaunchKernelGGL((softmax_kernel<4, 4, VEC>), per1, block, 0, stream, in, out, (int64_t)rows, S, nt);
    else hipLaunchKernelGGL(softmax_long_kernel, per1, block, 0, stream, in, out, S);
}

} // namespace

void launch_softmax(const __half *in, __half *out, int rows, int S, hipStream_t stream) {
    if (rows <= 0 || S <= 0) return;
    if (S % 8 == 0 && aligned16(in) && aligned16(out)) launch_softmax_v<true>(in, out, rows, S, stream);
    else launch_softmax_v<false>(in, out, rows, S, stream);
    HIP_CHECK(hipGetLastError());
}

void launch_attention_weights(const __half *q, const __half *k, __half *w, float scale, int B,
                              int H, int Lq, int Lk, int D, bool causal, hipStream_t stream) {
    if (B <= 0 || H <= 0 || Lq <= 0 || Lk <= 0 || D <= 0) return;
    const bool vin = D % 8 == 0 && aligned16(q) && aligned16(k);
    const bool vout = Lk % 8 == 0 && aligned16(w);
    // 128 x 128 tiles where they give every CU two workgroups, else 64 x 64
    // ones: 8 heads of 700 x 700 at 256 dimensions (288 large tiles) 33 us
    // against 75, 1 x 128 x 128 at 128 dimensions 7.4 against 13.
    const int64_t big_tiles = (int64_t)((Lk + 127) / 128) * ((Lq + 127) / 128) * B * H;
    const bool    big = Lq > 64 && big_tiles >= 2 * device_cus();
    const int     tile = big ? 128 : 64;
    const dim3    grid((unsigned)((Lk + tile - 1) / tile), (unsigned)((Lq + tile - 1) / tile), (unsigned)(B * H));
#define TL_WEIGHTS(BIG, VIN, VOUT)                                                                          \
    hipLaunchKernelGGL((attention_weights_kernel<BIG, VIN, VOUT>), grid, dim3(256), 0, stream, q, k, w, scale, \
                       Lq, Lk, D, causal ? 1 : 0)
    if (big) {
        if (vin && vout) TL_WEIGHTS(true, true, true);
        else if (vin) TL_WEIGHTS(true, true, false);
        else if (vout) TL_WEIGHTS(true, false, true);
        else TL_WEIGHTS(true, false, false);
    } else {
        if (vin && vout) TL_WEIGHTS(false, true, true);
        else if (vin) TL_WEIGHTS(false, true, false);
        else if (vout) TL_WEIGHTS(false, false, true);
        else TL_WEIGHTS(false, false, false);
    }
#undef TL_WEIGHTS
    HIP_CHECK(hipGetLastError());
}

} // namespace detail
} // namespace tiny_llm
