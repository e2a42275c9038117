// Row selection for the fused head: which token rows a caller wants (a mask, or labels with an ignored value), their
// hidden states and targets packed together, and results and gradients spread out again.  What boolean indexing needs a
// scan of several launches, a host synchronisation per indexed tensor and a sort for (its backward) is one launch each
// here (the selection from more than 65536 positions takes three) and one synchronisation in all (the count, which the sizes
// of the packed tensors depend on).
//
// Bound by launch latency at a few thousand tokens and by their bytes beyond that.
// An SFT step on 2052 positions, 1396 of them kept (H = 2048): 63 -> 27 launches, the selection 5.2, gather 6.6 and gradient
// scatter 5.1 us, the step 1549 -> 1187 us.
#include "common.hpp"

#include <type_traits>

namespace trlk {
namespace {

constexpr int kScan = 1024, kScanWaves = kScan / kWave;  // positions per workgroup of the selection

// keep(r, c) = p[r * stride + c] != skip, positions numbered e = r * cols + c.
template <typename T>
struct Keep {
    const T* p;
    int64_t stride;
    int cols;
    T skip;
    __device__ __forceinline__ bool operator()(int e) const {
        const int r = e / cols;
        return p[int64_t(r) * stride + (e - r * cols)] != skip;
    }
};

// idx[j] = the j-th kept position, pos[e] = its number or -1, *count = how many.  Workgroup b needs the number of kept
// positions before its own 1024.  Up to kOneLaunch positions it counts them itself (at most 8 bytes per position out of the
// L2, eight loads in flight per lane) instead of waiting for the others; that reads n^2 / 2048 positions in all, so beyond
// that (BASE) pos[1024 b] holds the number already, from the two kernels below.  One launch against three, int64 labels: 49152
// positions 13.8 us against about 15 (three launches), 65536 17.3, 81920 20.8 against 16.0, 131072 31 against 15.7, 1048576
// 523 against 15.3 us.
constexpr int kOneLaunch = 65536;
template <typename T, bool BASE>
__global__ __launch_bounds__(kScan) void select_rows_kernel(Keep<T> kept, int n, int32_t* idx, int32_t* pos, int64_t* count) {
    __shared__ int before_wave[kScanWaves], in_wave[kScanWaves];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int first = blockIdx.x * kScan, e = first + tid;
    const bool mine = e < n && kept(e);
    int before = 0;
    if constexpr (BASE) {
        before = tid == 0 ? pos[first] : 0;  // (read before the barrier below, overwritten after it, by this workgroup alone)
    } else {
        int k = tid;
        for (; k + 7 * kScan < first; k += 8 * kScan) {
            bool q[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) q[i] = kept(k + i * kScan);
#pragma unroll
            for (int i = 0; i < 8; ++i) before += q[i];
        }
        for (; k < first; k += kScan) before += kept(k);
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) before += __shfl_xor(before, o);
    const uint64_t vote = __ballot(mine);
    if (lane == 0) {
        before_wave[wave] = before;
        in_wave[wave] = __popcll(vote);
    }
    __syncthreads();
    int at = __popcll(vote & ((uint64_t(1) << lane) - 1)), total = 0;
#pragma unroll
    for (int w = 0; w < kScanWaves; ++w) {
        total += before_wave[w] + in_wave[w];
        at += before_wave[w] + (w < wave ? in_wave[w] : 0);
    }
    if (e < n) {
        pos[e] = mine ? at : -1;
        if (mine) idx[at] = e;
    }
    if (tid == 0 && int(blockIdx.x) == int(gridDim.x) - 1) *count = total;
}

// pos[1024 b] = kept positions among the 1024 from there on
template <typename T>
__global__ __launch_bounds__(kScan) void count_rows_kernel(Keep<T> kept, int n, int32_t* pos) {
    __shared__ int in_wave[kScanWaves];
    const int tid = threadIdx.x, e = blockIdx.x * kScan + tid;
    const uint64_t vote = __ballot(e < n && kept(e));
    if ((tid & (kWave - 1)) == 0) in_wave[tid / kWave] = __popcll(vote);
    __syncthreads();
    if (tid == 0) {
        int s = 0;
#pragma unroll
        for (int w = 0; w < kScanWaves; ++w) s += in_wave[w];
        pos[blockIdx.x * kScan] = s;
    }
}

// pos[1024 b] -> the sum of those before it, for b < blocks: one workgroup, 1024 of them at a time
__global__ __launch_bounds__(kScan) void count_prefix_kernel(int blocks, int32_t* pos) {
    __shared__ int in_wave[kScanWaves];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    int carry = 0;
    for (int b0 = 0; b0 < blocks; b0 += kScan) {
        const int b = b0 + tid;
        const int own = b < blocks ? pos[int64_t(b) * kScan] : 0;
        int upto = own;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int other = __shfl_up(upto, o);
            if (lane >= o) upto += other;
        }
        if (lane == kWave - 1) in_wave[wave] = upto;
        __syncthreads();
        int before = carry;
#pragma unroll
        for (int w = 0; w < kScanWaves; ++w) {
            before += w < wave ? in_wave[w] : 0;
            carry += in_wave[w];
        }
        if (b < blocks) pos[int64_t(b) * kScan] = before + upto - own;
        __syncthreads();  // (in_wave is written again)
    }
}

// One wave per row, 16 bytes per lane (VEC) or 2 where rows, strides or pointers are not whole 16-byte pieces.
constexpr int kRowsPerBlock = 4;
template <bool VEC>
using Piece = std::conditional_t<VEC, u32x4, uint16_t>;

// out[j] = row idx[j] of src (position e = b * cols + t at b * seq_stride + t * row_stride, strides in pieces) and its target.
template <bool VEC>
__global__ __launch_bounds__(kRowsPerBlock * kWave) void gather_rows_kernel(const Piece<VEC>* src, int64_t seq_stride,
                                                                            int64_t row_stride, int cols, const int32_t* idx,
                                                                            int n, int pieces, Piece<VEC>* out,
                                                                            const int64_t* targets, int64_t target_stride,
                                                                            int64_t* out_targets) {
    const int j = blockIdx.x * kRowsPerBlock + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (j >= n) return;
    const int e = idx[j], b = e / cols, t = e - b * cols;
    const Piece<VEC>* row = src + int64_t(b) * seq_stride + int64_t(t) * row_stride;
    Piece<VEC>* o = out + int64_t(j) * pieces;
    for (int c = lane; c < pieces; c += kWave) o[c] = row[c];
    if (lane == 0) out_targets[j] = targets[int64_t(b) * target_stride + t];
}

// The inverse: row (b, s) of out [n_seq, out_cols] = src[pos[b * cols + s]], zero where that is -1 or s >= cols.
template <bool VEC>
__global__ __launch_bounds__(kRowsPerBlock * kWave) void scatter_rows_kernel(const Piece<VEC>* src, const int32_t* pos, int cols,
                                                                             int out_cols, int out_rows, int pieces,
                                                                             Piece<VEC>* out) {
    const int r = blockIdx.x * kRowsPerBlock + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (r >= out_rows) return;
    const int b = r / out_cols, s = r - b * out_cols;
    const int from = s < cols ? pos[int64_t(b) * cols + s] : -1;
    Piece<VEC>* o = out + int64_t(r) * pieces;
    if (from >= 0) {
        const Piece<VEC>* row = src + int64_t(from) * pieces;
        for (int c = lane; c < pieces; c += kWave) o[c] = row[c];
    } else {
        const Piece<VEC> zero{};
        for (int c = lane; c < pieces; c += kWave) o[c] = zero;
    }
}

// Two packed fp32 vectors back into place, zeros elsewhere.
__global__ __launch_bounds__(256) void scatter_values_kernel(const float* a, const float* b, const int32_t* pos, int n,
                                                             float* out_a, float* out_b) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int from = pos[e];
    out_a[e] = from >= 0 ? a[from] : 0.f;
    if (out_b != nullptr) out_b[e] = from >= 0 ? b[from] : 0.f;
}

// ---- mean logits of whole sequences without logits: mean over t and v of hidden[b, t] . weight[v] =
// (sum_t hidden[b, t] . wsum) / (T V) with wsum = sum_v weight[v].  Bound by the read of the weight (525 MB and 2048 hidden
// rows: 86 us, 6.1 TB/s, of 96 us for all three launches; 90 of 113 with one set of eight rows in flight, four rows to a wave of
// the dot products and the partial sums read one by one; all three after a flush of the caches, with their gaps: 173 -> 108;
// 32000 x 4096 150 -> 89; 50257 x 1024 67 -> 40); converting it to fp32 first and summing that copy moved five times the bytes,
// 470 us.
//
// A mean logit is small against the terms it is made of, and a chain of 250 fp32 additions per column (what 128256 rows in
// 512 partial sums make) left it four times as far from 64 bits as the torch product (5e-7 against 1.3e-7 of its value on
// [2, 512] positions).  So sums are exact or in fp64 on the chip and rounded to fp32 once on their way to memory: in 2^-24 of
// the size that such a sum of random terms has, 0.7 to 1.3 where the torch product is 2.7 to 3.6 away (32000 to 202048 rows).
//
// Column sums: workgroup (x, y) sums rows y, y + gridDim.y, ... of 2048 columns, 8 columns per lane, eight rows in flight
// while the eight before them are summed (1024 row sets with half as much work each: 108 -> 142 us): those are added up in
// pairs in fp32 (their 16-bit values leave 13 bits and more to spare), then to the fp64 sum; the partial sums of the gridDim.y
// row sets are added in order by the second kernel.
constexpr int kColBlock = 256, kColParts = 512;
template <int DT>
__global__ __launch_bounds__(kColBlock) void column_sum_kernel(const uint16_t* w, int64_t ld, int rows, int cols8, float* parts) {
    const int c = blockIdx.x * kColBlock + threadIdx.x, step = gridDim.y;
    if (c >= cols8) return;
    const u32x4* p = reinterpret_cast<const u32x4*>(w) + c;
    const int64_t ld8 = ld / 8;
    double acc[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
    int r = blockIdx.y;
    u32x4 q[8], next[8];
    auto fetch = [&](int from, u32x4(&to)[8]) {
#pragma unroll
        for (int k = 0; k < 8; ++k) to[k] = __builtin_nontemporal_load(p + int64_t(from + k * step) * ld8);
    };
    auto add_rows = [&] {
        float x[8][8];
#pragma unroll
        for (int k = 0; k < 8; ++k) Elem<DT>::unpack(q[k], x[k]);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            acc[i] += double(((x[0][i] + x[1][i]) + (x[2][i] + x[3][i])) + ((x[4][i] + x[5][i]) + (x[6][i] + x[7][i])));
    };
    if (r + 7 * step < rows) {
        fetch(r, q);
        for (r += 8 * step; r + 7 * step < rows; r += 8 * step) {
            fetch(r, next);
            add_rows();
#pragma unroll
            for (int k = 0; k < 8; ++k) q[k] = next[k];
        }
        add_rows();
    }
    for (; r < rows; r += step) {
        float x[8];
        Elem<DT>::unpack(p[int64_t(r) * ld8], x);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += double(x[i]);
    }
    float* o = parts + (int64_t(blockIdx.y) * cols8 + c) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = float(acc[i]);
}
// One workgroup per 64 columns: its 16 waves add every 16th partial, then each other.
__global__ __launch_bounds__(1024) void column_sum_finish_kernel(const float* parts, int n_parts, int cols, float* out) {
    __shared__ double sum[16][kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, c = blockIdx.x * kWave + lane;
    double s = 0.;
    if (c < cols)
#pragma unroll 8
        for (int p = wave; p < n_parts; p += 16) s += double(parts[int64_t(p) * cols + c]);
    sum[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && c < cols) {
        double t = 0.;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += sum[k][lane];
        out[c] = float(t);
    }
}
// out[b][chunk] = scale * sum over the chunk's rows of hidden[b, t] . wsum, one wave per row.
constexpr int kDotRows = 16;  // rows per workgroup
template <int DT>
__global__ __launch_bounds__(kDotRows * kWave) void row_dot_kernel(const uint16_t* hidden, int64_t seq_stride, int64_t row_stride, int T,
                                                      int cols8, const float* wsum, double scale, float* out) {
    __shared__ double part[kDotRows];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int t = blockIdx.x * kDotRows + wave;
    double s = 0.;
    if (t < T) {
        const u32x4* row = reinterpret_cast<const u32x4*>(hidden + int64_t(blockIdx.y) * seq_stride + int64_t(t) * row_stride);
#pragma unroll 4
        for (int c = lane; c < cols8; c += kWave) {
            float x[8];
            Elem<DT>::unpack(row[c], x);
#pragma unroll
            for (int i = 0; i < 8; ++i) s = fma(double(x[i]), double(wsum[c * 8 + i]), s);
        }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) part[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double sum = 0.;
#pragma unroll
        for (int w = 0; w < kDotRows; ++w) sum += part[w];
        out[int64_t(blockIdx.y) * gridDim.x + blockIdx.x] = float(scale * sum);
    }
}

bool whole_pieces(const void* a, const void* b, int64_t bytes) {
    return reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0 && bytes % 16 == 0;
}

}  // namespace
}  // namespace trlk

using namespace trlk;

extern "C" int trlk_select_rows(const void* d_keep, int keep_type, int64_t n_rows, int64_t n_cols, int64_t row_stride,
                                int64_t skip, int32_t* d_out_index, int32_t* d_out_position, int64_t* d_out_count,
                                trlk_stream_t stream) {
    clear_error();
    // (the kernels count positions in 32 bits, up to a workgroup's share beyond the last one)
    TRLK_REQUIRE(n_rows >= 1 && n_cols >= 1 && n_rows <= ((int64_t(1) << 31) - 1 - kScan) / n_cols, TRLK_ERR_BAD_SHAPE,
                 "select_rows: bad shape %lld x %lld", (long long)n_rows, (long long)n_cols);
    TRLK_REQUIRE(n_rows == 1 || row_stride >= 0, TRLK_ERR_BAD_STRIDE, "select_rows: row_stride %lld", (long long)row_stride);
    TRLK_REQUIRE(d_keep && d_out_index && d_out_position && d_out_count, TRLK_ERR_NULL_POINTER, "select_rows: null pointer");
    const int n = int(n_rows * n_cols), cols = int(n_cols);
    const dim3 grid(unsigned((n + kScan - 1) / kScan));
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto tag) {
        typedef decltype(tag) T;
        const Keep<T> kept{static_cast<const T*>(d_keep), row_stride, cols, T(skip)};
        if (n <= kOneLaunch) {
            hipLaunchKernelGGL((select_rows_kernel<T, false>), grid, dim3(kScan), 0, s, kept, n, d_out_index, d_out_position,
                               d_out_count);
            return;
        }
        hipLaunchKernelGGL(count_rows_kernel<T>, grid, dim3(kScan), 0, s, kept, n, d_out_position);
        hipLaunchKernelGGL(count_prefix_kernel, dim3(1), dim3(kScan), 0, s, int(grid.x), d_out_position);
        hipLaunchKernelGGL((select_rows_kernel<T, true>), grid, dim3(kScan), 0, s, kept, n, d_out_index, d_out_position,
                           d_out_count);
    };
    switch (keep_type) {
        case TRLK_KEEP_U8: go(uint8_t{}); break;
        case TRLK_KEEP_I32: go(int32_t{}); break;
        case TRLK_KEEP_I64: go(int64_t{}); break;
        case TRLK_KEEP_F32: go(float{}); break;
        default: return fail(TRLK_ERR_BAD_DTYPE, "select_rows: unknown element type %d", keep_type);
    }
    return launch_status("select_rows");
}

extern "C" int trlk_gather_rows(const void* d_src, int64_t row_bytes, int64_t seq_stride_bytes, int64_t row_stride_bytes,
                                int64_t n_cols, const int32_t* d_index, int64_t n, void* d_out, const int64_t* d_targets,
                                int64_t target_stride, int64_t* d_out_targets, trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(n >= 0 && n < (int64_t(1) << 31) - kRowsPerBlock && n_cols >= 1 && n_cols < (int64_t(1) << 31) && row_bytes >= 2 &&
                     row_bytes < (int64_t(1) << 31),
                 TRLK_ERR_BAD_SHAPE, "gather_rows: bad sizes n=%lld cols=%lld row bytes=%lld", (long long)n, (long long)n_cols,
                 (long long)row_bytes);
    TRLK_REQUIRE((row_bytes | seq_stride_bytes | row_stride_bytes) % 2 == 0, TRLK_ERR_BAD_STRIDE,
                 "gather_rows: rows and strides must be whole 2-byte elements");
    if (n == 0) return TRLK_OK;
    TRLK_REQUIRE(d_src && d_index && d_out && d_targets && d_out_targets, TRLK_ERR_NULL_POINTER, "gather_rows: null pointer");
    const dim3 grid(unsigned((n + kRowsPerBlock - 1) / kRowsPerBlock)), block(kRowsPerBlock * kWave);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto vec) {
        constexpr bool V = decltype(vec)::value;
        constexpr int64_t size = sizeof(Piece<V>);
        hipLaunchKernelGGL(gather_rows_kernel<V>, grid, block, 0, s, static_cast<const Piece<V>*>(d_src), seq_stride_bytes / size,
                           row_stride_bytes / size, int(n_cols), d_index, int(n), int(row_bytes / size),
                           static_cast<Piece<V>*>(d_out), d_targets, target_stride, d_out_targets);
    };
    if (whole_pieces(d_src, d_out, row_bytes | seq_stride_bytes | row_stride_bytes))
        go(std::true_type{});
    else
        go(std::false_type{});
    return launch_status("gather_rows");
}

extern "C" int trlk_scatter_rows(const void* d_src, int64_t row_bytes, const int32_t* d_position, int64_t n_seq, int64_t n_cols,
                                 int64_t out_cols, void* d_out, trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(n_seq >= 1 && n_cols >= 1 && out_cols >= n_cols && n_seq <= ((int64_t(1) << 31) - 1 - kRowsPerBlock) / out_cols &&
                     row_bytes >= 2 && row_bytes < (int64_t(1) << 31) && row_bytes % 2 == 0,
                 TRLK_ERR_BAD_SHAPE, "scatter_rows: bad sizes n_seq=%lld cols=%lld of %lld row bytes=%lld", (long long)n_seq,
                 (long long)n_cols, (long long)out_cols, (long long)row_bytes);
    TRLK_REQUIRE(d_position && d_out, TRLK_ERR_NULL_POINTER, "scatter_rows: null pointer");  // (src: no row may be kept)
    const int out_rows = int(n_seq * out_cols);
    const dim3 grid(unsigned((out_rows + kRowsPerBlock - 1) / kRowsPerBlock)), block(kRowsPerBlock * kWave);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto vec) {
        constexpr bool V = decltype(vec)::value;
        hipLaunchKernelGGL(scatter_rows_kernel<V>, grid, block, 0, s, static_cast<const Piece<V>*>(d_src), d_position, int(n_cols),
                           int(out_cols), out_rows, int(row_bytes / int64_t(sizeof(Piece<V>))), static_cast<Piece<V>*>(d_out));
    };
    if (whole_pieces(d_src, d_out, row_bytes))
        go(std::true_type{});
    else
        go(std::false_type{});
    return launch_status("scatter_rows");
}

extern "C" int trlk_scatter_values(const float* d_a, const float* d_b, const int32_t* d_position, int64_t n, float* d_out_a,
                                   float* d_out_b, trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(n >= 1 && n < (int64_t(1) << 31) - 256, TRLK_ERR_BAD_SHAPE, "scatter_values: bad size %lld", (long long)n);
    TRLK_REQUIRE(d_position && d_out_a, TRLK_ERR_NULL_POINTER, "scatter_values: null pointer");  // (a, b: no row may be kept)
    hipLaunchKernelGGL(scatter_values_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), d_a,
                       d_b, d_position, int(n), d_out_a, d_out_b);
    return launch_status("scatter_values");
}

extern "C" size_t trlk_mean_logits_workspace_bytes(int64_t hidden_size) {
    return hidden_size > 0 ? size_t(kColParts + 1) * size_t(hidden_size) * sizeof(float) : 0;
}

extern "C" int64_t trlk_mean_logits_chunks(int64_t rows_per_seq) { return (rows_per_seq + kDotRows - 1) / kDotRows; }

extern "C" int trlk_mean_logits(const void* d_hidden, const void* d_weight, int dtype, int64_t n_seq, int64_t rows_per_seq,
                                int64_t vocab, int64_t hidden_size, int64_t seq_stride, int64_t row_stride,
                                int64_t weight_stride, float* d_out, void* d_workspace, size_t workspace_bytes,
                                trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(dtype == TRLK_BF16 || dtype == TRLK_F16, TRLK_ERR_BAD_DTYPE, "mean_logits: bf16 or fp16 operands (dtype code %d)",
                 dtype);
    TRLK_REQUIRE(n_seq >= 1 && n_seq < 65536 && rows_per_seq >= 1 && rows_per_seq < (int64_t(1) << 31) - kDotRows && vocab >= 1 &&
                     vocab < (int64_t(1) << 31) - 8 * kColParts && hidden_size >= 1 && hidden_size < (int64_t(1) << 31) - 2048,
                 TRLK_ERR_BAD_SHAPE, "mean_logits: bad sizes n_seq=%lld rows=%lld vocab=%lld hidden=%lld", (long long)n_seq,
                 (long long)rows_per_seq, (long long)vocab, (long long)hidden_size);
    TRLK_REQUIRE(hidden_size % 8 == 0 && (seq_stride | row_stride | weight_stride) % 8 == 0 && weight_stride >= hidden_size,
                 TRLK_ERR_BAD_STRIDE, "mean_logits: the hidden size and all strides must be multiples of 8 elements");
    TRLK_REQUIRE(d_hidden && d_weight && d_out && d_workspace, TRLK_ERR_NULL_POINTER, "mean_logits: null pointer");
    TRLK_REQUIRE(reinterpret_cast<uintptr_t>(d_hidden) % 16 == 0 && reinterpret_cast<uintptr_t>(d_weight) % 16 == 0,
                 TRLK_ERR_BAD_STRIDE, "mean_logits: operands must be 16-byte aligned");
    TRLK_REQUIRE(workspace_bytes >= trlk_mean_logits_workspace_bytes(hidden_size), TRLK_ERR_WORKSPACE,
                 "mean_logits: workspace of %zu bytes needed, %zu given", trlk_mean_logits_workspace_bytes(hidden_size), workspace_bytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int cols8 = int(hidden_size / 8), n_parts = int(vocab < kColParts ? vocab : kColParts);
    float* parts = static_cast<float*>(d_workspace);
    float* wsum = parts + int64_t(n_parts) * hidden_size;
    const double scale = 1.0 / (double(rows_per_seq) * double(vocab));
    auto go = [&](auto tag) {
        constexpr int DT = decltype(tag)::value;
        hipLaunchKernelGGL(column_sum_kernel<DT>, dim3(unsigned((cols8 + kColBlock - 1) / kColBlock), unsigned(n_parts)),
                           dim3(kColBlock), 0, s, static_cast<const uint16_t*>(d_weight), weight_stride, int(vocab), cols8, parts);
        hipLaunchKernelGGL(column_sum_finish_kernel, dim3(unsigned((hidden_size + kWave - 1) / kWave)), dim3(1024), 0, s, parts,
                           n_parts, int(hidden_size), wsum);
        hipLaunchKernelGGL(row_dot_kernel<DT>, dim3(unsigned(trlk_mean_logits_chunks(rows_per_seq)), unsigned(n_seq)), dim3(kDotRows * kWave), 0,
                           s, static_cast<const uint16_t*>(d_hidden), seq_stride, row_stride, int(rows_per_seq), cols8, wsum, scale,
                           d_out);
    };
    if (dtype == TRLK_BF16)
        go(std::integral_constant<int, TRLK_BF16>{});
    else
        go(std::integral_constant<int, TRLK_F16>{});
    return launch_status("mean_logits");
}
