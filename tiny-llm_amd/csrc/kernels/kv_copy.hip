// Byte-moving kernels of the KV path: fused batched append and gather.
// Both are HBM-bound integer work; each lane moves one 16-byte piece with a
// vector load and a vector store, consecutive lanes on consecutive pieces.
#include "kv_kernels.h"

#include "tiny_llm/hip_utils.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace tiny_llm {
namespace detail {

namespace {

constexpr int kCopyThreads = 256;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int64_t row_offset(const KvView &v, int b, int t) {
    const int     row = v.seq_row ? v.seq_row[b] : b;
    const int64_t blk =
        v.block_table ? (int64_t)v.block_table[(int64_t)row * v.bt_stride + (t >> v.log2_blk)] : row;
    return blk * v.blk_stride + (int64_t)(t & ((1 << v.log2_blk) - 1)) * v.tok_stride;
}

struct AppendArgs {
    KvView         view;
    int64_t        layer_stride;
    const int32_t *wpos;
    int            first_pos;
    int            n;
    int            row_pieces; // 16-byte pieces per token row (Hkv*D/8)
    const __half  *new_k;
    const __half  *new_v;
};

// grid (ceil(row_pieces/256), n entries, num_layers): the same bytes as the
// two cudaMemcpyAsync of appendKV (kv_cache.cpp:230-233) for each entry and
// layer, written as one coalesced launch.
__global__ __launch_bounds__(kCopyThreads) void kv_append_kernel(AppendArgs a) {
    const int piece = blockIdx.x * kCopyThreads + threadIdx.x;
    if (piece >= a.row_pieces) return;
    const int     i = blockIdx.y;
    const int     l = blockIdx.z;
    const int     t = a.wpos ? a.wpos[i] : a.first_pos + i;
    const int64_t dst = row_offset(a.view, i, t) + (int64_t)l * a.layer_stride + (int64_t)piece * 8;
    const int64_t src = ((int64_t)l * a.n + i) * (int64_t)a.row_pieces * 8 + (int64_t)piece * 8;
    const uint4   k = *reinterpret_cast<const uint4 *>(a.new_k + src);
    const uint4   v = *reinterpret_cast<const uint4 *>(a.new_v + src);
    *reinterpret_cast<uint4 *>(const_cast<__half *>(a.view.k_base) + dst) = k;
    *reinterpret_cast<uint4 *>(const_cast<__half *>(a.view.v_base) + dst) = v;
}

// Token ranges of one append launch: range r writes rows tok0[r] ..
// tok0[r+1]-1 of new_k/new_v (counted from src_tok) to cache row row[r] at
// positions pos0[r], pos0[r]+1, ...  The table travels in the kernel
// arguments, so the launch needs no metadata copy.
constexpr int kAppendRanges = 64;
constexpr int kAppendTokens = 32768; // tokens per launch (grid y)
struct RangeArgs {
    KvView        view;
    int           n;
    int           row_pieces;
    int64_t       src_tok;
    const __half *new_k;
    const __half *new_v;
    int32_t       row[kAppendRanges];
    int32_t       pos0[kAppendRanges];
    int32_t       tok0[kAppendRanges + 1];
};

// grid (ceil(row_pieces/256), tokens of the launch): one token row per block
// row, the bytes of appendKV (kv_cache.cpp:226-233) for every range.
__global__ __launch_bounds__(kCopyThreads) void kv_append_ranges_kernel(RangeArgs a) {
    const int piece = blockIdx.x * kCopyThreads + threadIdx.x;
    if (piece >= a.row_pieces) return;
    const int t = blockIdx.y;
    int       r = 0; // the range holding token t (uniform over the block)
    while (r + 1 < a.n && a.tok0[r + 1] <= t) ++r;
    const int     pos = a.pos0[r] + (t - a.tok0[r]);
    const int64_t blk =
        a.view.block_table
            ? (int64_t)a.view.block_table[(int64_t)a.row[r] * a.view.bt_stride + (pos >> a.view.log2_blk)]
            : (int64_t)a.row[r];
    const int64_t dst = blk * a.view.blk_stride +
                        (int64_t)(pos & ((1 << a.view.log2_blk) - 1)) * a.view.tok_stride + (int64_t)piece * 8;
    const int64_t src = (a.src_tok + t) * (int64_t)a.row_pieces * 8 + (int64_t)piece * 8;
    const uint4   k = *reinterpret_cast<const uint4 *>(a.new_k + src);
    const uint4   v = *reinterpret_cast<const uint4 *>(a.new_v + src);
    *reinterpret_cast<uint4 *>(const_cast<__half *>(a.view.k_base) + dst) = k;
    *reinterpret_cast<uint4 *>(const_cast<__half *>(a.view.v_base) + dst) = v;
}

constexpr int kGatherPieces = 2; // 16-byte pieces per thread
struct GatherArgs {
    KvView         view; // seq_row: the cache rows
    const int32_t *lens; // attended lengths
    int            Hkv;
    int            D;
    int            s_max;
    int            n;      // entries
    const __half  *src[2]; // what grid z counts: n entries of each output, K then V
    __half        *out[2];
};

// The first gather of a prepared step: lengths and rows in its arguments, up to
// kGatherInline entries, so that it needs no metadata copy.  The 3 KB cost a
// launch 0.4 us, so the kernel leaves them in device memory for the step's further
// layers, which keep the small arguments (K of 3 sequences of 300 tokens: 6.8 us a
// layer, 7.3 with the arrays in every launch).
constexpr int kGatherInline = kGatherStore / 2;
struct GatherStepArgs : GatherArgs {
    int32_t *store; // [n lengths | n rows], or null
    int32_t  len[kGatherInline];
    int32_t  row[kGatherInline];
};

// grid (token blocks, Hkv, outputs * n): out[b][g][t][:] from the cache.  Two
// pieces per thread, both loads before the stores (one or four: 83 / 76 us where
// this took 73; kv head fastest in the grid: level to 4% slower).  STREAM:
// non-temporal stores, for outputs that the L2s (32 MB) cannot hold for their
// reader: they no longer evict what is still to be read.  (Non-temporal loads
// too: 68 us where this takes 53.)  Bound by memory: 16 ragged sequences of up
// to 4096 tokens from 16-token blocks, 8 heads of 128, prepare + gather over
// three caches in turn 81.0 -> 65.8 us (6.1 TB/s read and written), over one 80.7
// -> 52.8; 3 sequences of 300 tokens, where the metadata copy and the second
// launch were most of it, 17.9 -> 10.7.
// Args by value: through a reference they would be copied to scratch memory.
template <bool STREAM, class Args>
__device__ __forceinline__ void gather_body(Args a) {
    const int z = (int)blockIdx.z, which = z >= a.n, b = z - which * a.n;
    const int g = (int)blockIdx.y, blk = (int)blockIdx.x;
    const int ppt = a.D >> 3; // pieces per token
    int       len, row;
    if constexpr (std::is_same_v<Args, GatherStepArgs>) {
        len = a.len[b];
        row = a.row[b];
    } else {
        len = a.lens[b];
        row = a.view.seq_row[b];
    }
    const __half *const src = (which ? a.src[1] : a.src[0]) + (int64_t)g * a.view.head_stride;
    __half *const       out = (which ? a.out[1] : a.out[0]) + ((int64_t)b * a.Hkv + g) * a.s_max * a.D;
    uint4 val[kGatherPieces];
#pragma unroll
    for (int u = 0; u < kGatherPieces; ++u) {
        const int piece = (blk * kGatherPieces + u) * kCopyThreads + (int)threadIdx.x;
        const int t = piece / ppt, e = piece - t * ppt;
        val[u] = make_uint4(0u, 0u, 0u, 0u);
        if (t < len && t < a.s_max) {
            const int64_t pb = a.view.block_table
                                   ? (int64_t)a.view.block_table[(int64_t)row * a.view.bt_stride + (t >> a.view.log2_blk)]
                                   : row;
            val[u] = *reinterpret_cast<const uint4 *>(
                src + pb * a.view.blk_stride + (int64_t)(t & ((1 << a.view.log2_blk) - 1)) * a.view.tok_stride + e * 8);
        }
    }
#pragma unroll
    for (int u = 0; u < kGatherPieces; ++u) {
        const int piece = (blk * kGatherPieces + u) * kCopyThreads + (int)threadIdx.x;
        if (piece >= a.s_max * ppt) continue;
        u32x4 *const dst = reinterpret_cast<u32x4 *>(out + (int64_t)piece * 8);
        if constexpr (STREAM) __builtin_nontemporal_store(__builtin_bit_cast(u32x4, val[u]), dst);
        else *dst = __builtin_bit_cast(u32x4, val[u]);
    }
}

template <bool STREAM>
__global__ __launch_bounds__(kCopyThreads) void kv_gather_kernel(GatherArgs a) {
    gather_body<STREAM>(a);
}

template <bool STREAM>
__global__ __launch_bounds__(kCopyThreads) void kv_gather_step_kernel(GatherStepArgs a) {
    gather_body<STREAM>(a);
    if (a.store && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)
        for (int i = (int)threadIdx.x; i < a.n; i += kCopyThreads) {
            a.store[i] = a.len[i];
            a.store[a.n + i] = a.row[i];
        }
}

struct TableArgs {
    int32_t *table;
    int32_t  n;
    int32_t  idx[kTableBatch];
    int32_t  val[kTableBatch];
};

__global__ __launch_bounds__(256) void table_update_kernel(TableArgs a) {
    const int i = (int)threadIdx.x;
    if (i < a.n) a.table[a.idx[i]] = a.val[i];
}

} // namespace

void launch_table_update(int32_t *table, const std::pair<int32_t, int32_t> *upd, size_t n,
                         hipStream_t stream) {
    static_assert(kTableBatch <= 256, "one thread per pair");
    for (size_t first = 0; first < n; first += kTableBatch) {
        TableArgs a;
        a.table = table;
        a.n = (int32_t)std::min<size_t>(kTableBatch, n - first);
        for (int i = 0; i < a.n; ++i) {
            a.idx[i] = upd[first + (size_t)i].first;
            a.val[i] = upd[first + (size_t)i].second;
        }
        hipLaunchKernelGGL(table_update_kernel, dim3(1), dim3(256), 0, stream, a);
        HIP_CHECK(hipGetLastError());
    }
}

void launch_kv_append(const KvView &view, int64_t layer_stride, const int32_t *wpos, int first_pos,
                      int n, int num_layers, int row_elems, const __half *new_k,
                      const __half *new_v, hipStream_t stream) {
    if (n <= 0 || num_layers <= 0) return;
    AppendArgs a;
    a.view = view;
    a.layer_stride = layer_stride;
    a.wpos = wpos;
    a.first_pos = first_pos;
    a.n = n;
    a.row_pieces = row_elems / 8;
    a.new_k = new_k;
    a.new_v = new_v;
    dim3 grid((unsigned)((a.row_pieces + kCopyThreads - 1) / kCopyThreads), (unsigned)n,
              (unsigned)num_layers);
    profile_begin(KernelId::KvAppend, stream);
    hipLaunchKernelGGL(kv_append_kernel, grid, dim3(kCopyThreads), 0, stream, a);
    HIP_CHECK(hipGetLastError());
    profile_end(KernelId::KvAppend, stream);
}

void launch_kv_append_ranges(const KvView &view, const int32_t *rows, const int32_t *pos0,
                             const int32_t *counts, int n, int row_elems, const __half *new_k,
                             const __half *new_v, hipStream_t stream) {
    RangeArgs a;
    a.view = view;
    a.row_pieces = row_elems / 8;
    a.new_k = new_k;
    a.new_v = new_v;
    a.n = 0;
    a.tok0[0] = 0;
    int64_t done = 0; // tokens of earlier launches
    auto flush = [&]() {
        if (a.n == 0) return;
        dim3 grid((unsigned)((a.row_pieces + kCopyThreads - 1) / kCopyThreads), (unsigned)a.tok0[a.n]);
        a.src_tok = done;
        profile_begin(KernelId::KvAppend, stream);
        hipLaunchKernelGGL(kv_append_ranges_kernel, grid, dim3(kCopyThreads), 0, stream, a);
        HIP_CHECK(hipGetLastError());
        profile_end(KernelId::KvAppend, stream);
        done += a.tok0[a.n];
        a.n = 0;
        a.tok0[0] = 0;
    };
    for (int i = 0; i < n; ++i) {
        int off = 0; // a range longer than a launch holds continues in the next
        while (off < counts[i]) {
            if (a.n == kAppendRanges || a.tok0[a.n] == kAppendTokens) flush();
            const int take = std::min(counts[i] - off, kAppendTokens - a.tok0[a.n]);
            a.row[a.n] = rows[i];
            a.pos0[a.n] = pos0[i] + off;
            a.tok0[a.n + 1] = a.tok0[a.n] + take;
            ++a.n;
            off += take;
        }
    }
    flush();
}

bool gather_inline(int n) { return n <= kGatherInline; }

void launch_kv_gather(const KvView &view, const GatherMeta &meta, int n, int Hkv, int D, int s_max, __half *k_out,
                      __half *v_out, hipStream_t stream) {
    if (n <= 0 || s_max <= 0 || (!k_out && !v_out)) return;
    GatherStepArgs    a;
    const GatherArgs &small = a;
    const bool        inl = !meta.lens;
    a.view = view;
    a.view.seq_row = meta.rows;
    a.lens = meta.lens;
    a.Hkv = Hkv;
    a.D = D;
    a.s_max = s_max;
    a.n = n;
    if (inl) {
        std::memcpy(a.len, meta.host_lens, sizeof(int32_t) * (size_t)n);
        std::memcpy(a.row, meta.host_rows, sizeof(int32_t) * (size_t)n);
        a.store = meta.store;
    }
    const int64_t pieces = (int64_t)s_max * (D / 8), per = (int64_t)kCopyThreads * kGatherPieces;
    const int64_t blocks = (pieces + per - 1) / per;
    const int64_t bytes = pieces * 16 * Hkv * n * ((k_out != nullptr) + (v_out != nullptr));
    auto          go = [&](int outputs) {
        const dim3 grid((unsigned)blocks, (unsigned)Hkv, (unsigned)(outputs * n));
        profile_begin(KernelId::KvGather, stream);
        const bool big = bytes > (32LL << 20);
        const dim3 block(kCopyThreads);
        if (inl && big) hipLaunchKernelGGL((kv_gather_step_kernel<true>), grid, block, 0, stream, a);
        else if (inl) hipLaunchKernelGGL((kv_gather_step_kernel<false>), grid, block, 0, stream, a);
        else if (big) hipLaunchKernelGGL((kv_gather_kernel<true>), grid, block, 0, stream, small);
        else hipLaunchKernelGGL((kv_gather_kernel<false>), grid, block, 0, stream, small);
        HIP_CHECK(hipGetLastError());
        profile_end(KernelId::KvGather, stream);
    };
    if (k_out && v_out && n <= 65535 / 2) { // one launch for both
        a.src[0] = view.k_base;
        a.src[1] = view.v_base;
        a.out[0] = k_out;
        a.out[1] = v_out;
        go(2);
        return;
    }
    for (int which = 0; which < 2; ++which) {
        a.src[0] = a.src[1] = which ? view.v_base : view.k_base;
        a.out[0] = a.out[1] = which ? v_out : k_out;
        if (a.out[0]) go(1);
    }
}

} // namespace detail
} // namespace tiny_llm
