// K5 / K6: lm_head fused with the log-prob / entropy reduction (forward) and its backward.
//
// All contractions run on the matrix cores (v_mfma_f32_16x16x32_{bf16,f16}, in the forward 32x32x16, fp32 accumulate) as
// "NT" tiles: C[256 x 256] += A[256 x K] * B[256 x K]^T with both operands
// row-major and K contiguous, which is the layout the MFMA A/B fragments want (a lane holds 8
// consecutive k of one row), so fragments come straight out of LDS with 16-byte reads and nothing
// is ever transposed on the fly.  512 threads = 8 waves, 2 along M x 4 along N; a wave owns 128 x 64 of
// the tile = 8 x 4 (4 x 2) MFMA blocks = 128 accumulator registers per lane.  Tiles go from memory
// straight into two LDS stages (global_load_lds_dwordx4) when K is a multiple of the k step,
// through registers otherwise.
//
// Forward (K5): the tile is computed TRANSPOSED -- M = vocabulary rows of W, N = tokens -- so that
// a lane of the accumulator layout holds 16 vocabulary entries of ONE token per block.  The online
// log-sum-exp state of a token therefore lives in the lane's own registers and the per-tile
// epilogue needs no cross-lane traffic; a workgroup keeps 256 tokens and walks over its share of
// the vocabulary tiles, the logits exist only as accumulators.
//
// Backward (K6), per vocabulary chunk: (1) dz = dL/dlogits as scaled fp16 [chunk, tokens] (vocabulary-major, each
// token's column in that token's own power-of-two scale) -- from a recompute of the chunk's logits (equal to the forward's
// to the last bit),
// or, when the forward was asked to stash its softmax numerators, from one elementwise sweep over that stash;
// (2) dHidden += dz * W_chunk: the tile loop with dz as a K-MAJOR operand (its k rows go to LDS as they lie in
// memory and the MFMA fragments come out through the LDS transpose loads, ds_read_b64_tr_b16) against W_chunk, which with few
// tokens is read k-major too and otherwise comes as a transposed copy;
// (3) dW_chunk = dz^T * hidden as an NT product against hidden^T, whose columns carry the inverse of the tokens'
// scales; all on fp16 operands (bf16 inputs are converted while they are transposed).  Both are computed transposed too
// (M = columns of the output), so that a lane of the accumulator layout holds 4 consecutive columns of one output row.  The contraction of (2)/(3)
// is over a different axis than the recompute, and with H in the thousands the output tile of a fused kernel cannot
// stay in registers, so dz goes through a chunk-sized workspace (never the whole [N, V] matrix).
#include "common.hpp"

#include <type_traits>

namespace trlk {
namespace {

constexpr int BM = 256, BN = 256, BK = 64;  // a workgroup's tile, the k step
constexpr int WGM = 2, WGN = 4;               // waves along M and N
constexpr int kHeadThreads = WGM * WGN * 64;
#define TRLK_HEAD_KERNEL __global__ __launch_bounds__(kHeadThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
constexpr int WM = BM / WGM, WN = BN / WGN;  // per-wave tile
constexpr int MI = WM / 16, NI = WN / 16;    // MFMA blocks of it
constexpr int MB = WM / 32, NB = WN / 32;    // ... in the forward
constexpr int kLdsRow = BK + 8;  // register-staged loop: elements per LDS row (16 bytes of padding keep 16-byte reads conflict-free)
constexpr int kCpr = BK / 8;                        // 16-byte chunks per tile row
constexpr int kRowStep = kHeadThreads / kCpr;       // rows staged per pass of the workgroup
constexpr int kLoadsA = BM / kRowStep, kLoadsB = BN / kRowStep;
constexpr int kTileABytes = BM * kLdsRow * 2, kTileBBytes = BN * kLdsRow * 2;
constexpr int kStageBytes = kTileABytes + kTileBBytes;
constexpr int kRowBytes = BK * 2;                    // direct-to-LDS loop: a dense LDS row
constexpr int kDenseA = BM * kRowBytes, kDenseStage = (BM + BN) * kRowBytes;
constexpr int kDzLdsRow = BN * 2 + 16;     // bytes per vocabulary row of the dz tile staged in LDS by the backward
constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int kHeadLdsBytes = cmax(cmax(2 * kStageBytes, 2 * kDenseStage), BM * kDzLdsRow);
static_assert(2 * WGM * BN * 4 * 4 <= kHeadLdsBytes && BN <= kHeadThreads, "merge scratch");
static_assert(BM % kRowStep == 0 && BN % kRowStep == 0, "tile shape");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The 16x16x32 shape reads and writes half as many accumulators per multiply-add as 32x32x16 does.  The part is limited by
// power under matrix load, so that shows as speed: a bare loop of MFMAs on random bf16 operands runs at 2020-2060 TFLOP/s
// (2.05-2.12 GHz) against 1830-1880 TFLOP/s (1.87-1.90 GHz), on zeros both at 2450-2490 TFLOP/s (2.4 GHz).
// The forward uses 32x32x16.  Its loop has registers for two sets of fragments there (nothing of the softmax state is
// spilled) and takes, against the same loop as the products', 272 for 286 us with 1396 tokens, H = 2048, V = 50257 and
// 302 for 330 us with 879 tokens, H = 1024, V = 151665; 8345 for 8240 us with 9664 tokens, H = 3584, V = 151936, where
// power decides, is the other side.  The logits come out the same, to the last bit, in both shapes (180000 compared, bf16
// and fp16, sums that cancel and sums that do not): the backward's recompute may use the other one, and the rounding of z
// still cancels against that in log_z.  But the layout of 16x16x32 spreads a token's exponentials over twice as many lanes,
// which changes the order of THEIR sum and the last bits of log_z; with the forward's loop as it is, what a run has stored of
// its old or its reference policy stays what it computes again.
template <int DT>
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (DT == TRLK_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
}

// The same value, but nothing computed from it is kept across loop iterations: what the compiler hoists out of the
// forward's tile loop it spills, and a reload waits for every tile transfer in flight.
__device__ __forceinline__ int fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// A value that is the same in every lane, in a scalar register.
__device__ __forceinline__ float uniform(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

template <int DT>
__device__ __forceinline__ f32x16 mfma_fwd(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (DT == TRLK_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
}

// Where a wave sits in the tile.  A SIMD runs waves w and w + 4: they differ in their columns (N) by half the tile, so
// that a tile of at most 128 columns leaves every SIMD one wave with work, not two of them both.
__device__ __forceinline__ int wave_m(int wave) { return (wave >> 1) & 1; }
__device__ __forceinline__ int wave_n(int wave) { return (wave & 1) | ((wave >> 2) << 1); }

// One operand of the NT product: `rows` x K, row-major with leading dimension ld (elements).  The right operand may
// instead be given "k-major" (BKM below): K x `rows`, row-major with leading dimension ld -- the transpose of what the
// product wants, read through the LDS transpose loads; its columns must be readable (and zero) up to the next
// multiple of the tile size.
struct Operand {
    const uint16_t* p;
    int64_t ld;
    int rows;
};
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Direct-to-LDS variant of the tile loop (K % BK == 0): `global_load_lds_dwordx4` moves 16 bytes per
// lane from memory straight into LDS, 1 KiB contiguous per wave instruction = 8 tile rows of 64 k, with no register
// staging and no ds_write.  Rows are dense (no padding is possible inside a wave's 1 KiB), so bank conflicts are avoided
// by an XOR swizzle of the 16-byte chunk index: the chunk at physical position pc of row r holds logical chunk
//   pc ^ swz(r),  swz(r) = (r & 7) ^ ((r >> 3) & 1),
// which makes the 16 rows that one ds_read_b128 phase touches cover all 64 banks once.  The lane
// fetches that logical chunk from memory (a permutation inside one row, still coalesced) and the
// fragment reads apply the same XOR.
//
// The loop keeps two 64 KiB stages in LDS; a stage is refilled as soon as the barrier that ends its last use has passed,
// one step before it is needed again.
__device__ __forceinline__ int tile_swizzle(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Loader side of the direct-to-LDS loop: per-lane source offsets of the wave's tile blocks and the
// transfer of one stage.
// BKM: the right operand is k-major.  Its stage is then 64 k rows of 512 bytes (256 columns); one transfer fills two
// k rows; the 16-byte unit at physical position pu of k row r holds logical unit pu ^ ((r & 3) << 1) ^ (r & 8), which
// spreads the eight k rows that two neighbouring groups of 16 lanes read with a transpose load over all banks.
// LEFT: the left operand travels this way too (otherwise LeftKm moves it).
template <bool BKM = false, bool LEFT = true>
struct DirectLoader {
    static constexpr int kWaves = kHeadThreads / 64, kRowsPerBlk = 1024 / kRowBytes;
    static constexpr int kBlkA = LEFT ? BM / kRowsPerBlk / kWaves : 0, kBlkB = BN / kRowsPerBlk / kWaves;  // per wave and stage
    static constexpr int kStageLoads = kBlkA + kBlkB;
    static_assert(BM % (kRowsPerBlk * kWaves) == 0 && BN % (kRowsPerBlk * kWaves) == 0 && BN == 256, "blocks per wave");
    const char *abase, *bbase;
    char* smem;
    int wave;
    int64_t bkstep;  // bytes between two k of the right operand
    uint32_t ao[LEFT ? kBlkA : 1], bo[kBlkB];

    __device__ __forceinline__ DirectLoader(const Operand A, int m0, const Operand B, int n0, char* lds) : smem(lds) {
        const int lane = fresh(threadIdx.x & 63);
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: LDS targets stay scalar
        const int rr = lane / kCpr, pc = lane % kCpr;  // row inside a block, chunk position
        abase = reinterpret_cast<const char*>(A.p + int64_t(m0) * A.ld);
        bbase = reinterpret_cast<const char*>(BKM ? B.p + n0 : B.p + int64_t(n0) * B.ld);
        bkstep = BKM ? B.ld * 2 : 2;
        const uint32_t lda = uint32_t(A.ld * 2), ldb = uint32_t(B.ld * 2);  // (a tile spans less than 4 GiB)
#pragma unroll
        for (int j = 0; j < kBlkA; ++j) {
            const int row = (wave + kWaves * j) * kRowsPerBlk + rr;
            const int kc = pc ^ tile_swizzle(row);  // the logical chunk this lane fetches
            const int r = m0 + row < A.rows ? row : A.rows - 1 - m0;
            ao[j] = uint32_t(r) * lda + uint32_t(kc * 16);
        }
#pragma unroll
        for (int j = 0; j < kBlkB; ++j) {
            if constexpr (BKM) {
                const int krow = (wave + kWaves * j) * 2 + (lane >> 5);
                const int lu = (lane & 31) ^ ((krow & 3) << 1) ^ (krow & 8);  // the logical 16-byte unit this lane fetches
                bo[j] = uint32_t(krow) * ldb + uint32_t(lu * 16);
                continue;
            }
            const int row = (wave + kWaves * j) * kRowsPerBlk + rr;
            const int kc = pc ^ tile_swizzle(row);
            const int r = n0 + row < B.rows ? row : B.rows - 1 - n0;
            bo[j] = uint32_t(r) * ldb + uint32_t(kc * 16);
        }
    }
    // One 1 KiB transfer: 16 bytes per lane from `src` to LDS offset `lds` + 16 * lane.  Issued as
    // inline assembly on purpose: the compiler books a global_load_lds as an access of both memory
    // and LDS, after which every wait on a fragment read becomes lgkmcnt(0) (it stalls on the
    // reads just issued); the loop keeps its own vmcnt bookkeeping for these transfers anyway.
    // (m0 is a reserved register; naming it as clobbered is what tells the compiler not to keep a value there)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    // The source is a uniform 64-bit base (scalar registers) plus the lane's 32-bit byte offset: one vector register
    // per transfer instead of an address pair, and the k step is added on the scalar side.
    static __device__ __forceinline__ void transfer(const char* base, uint32_t lane_off, uint32_t lds) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(lane_off),
                     "s"(reinterpret_cast<uint64_t>(base))
                     : "memory", "m0");
    }
#pragma clang diagnostic pop
    __device__ __forceinline__ uint32_t lds_base(int buf) const {
        return uint32_t(reinterpret_cast<uintptr_t>(smem)) + uint32_t(buf * kDenseStage);
    }
    // transfer j of a stage (A blocks first, then B blocks)
    __device__ __forceinline__ void issue_one(int buf, int k0, int j) const {
        if (j < kBlkA)
            transfer(abase + int64_t(k0) * 2, ao[j], lds_base(buf) + (wave + kWaves * j) * 1024);
        else
            transfer(bbase + int64_t(k0) * bkstep, bo[j - kBlkA], lds_base(buf) + kDenseA + (wave + kWaves * (j - kBlkA)) * 1024);
    }
    __device__ __forceinline__ void issue(int buf, int k0) const {
#pragma unroll
        for (int j = 0; j < kStageLoads; ++j) issue_one(buf, k0, j);
    }
    // the first two stages of a product; both must be free (all reads of the LDS done)
    __device__ __forceinline__ void prologue(int K) const {
        issue(0, 0);
        if (K > BK) issue(1, BK);
    }
    __device__ __forceinline__ void first_stage_landed(int nk) const {
        if (nk >= 2)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStageLoads) : "memory");
        else
            __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
};

// The left operand of the dHidden product straight from the weight: k-major (A.p is [krows, A.rows], K = krows rounded up to
// the k step) and, with CONVERT, bf16 that becomes fp16 times a power of two.  A stage is 64 k rows of 256 columns, laid out
// like a k-major right operand's; it goes through registers, because the conversion is done on the way: a lane holds 4 vectors
// of 8 columns, of k rows 16 apart, loaded one step before they are converted and written to the LDS.  k rows beyond the last
// are read as the last (the other operand is zero there), columns beyond the last as the last 8 (nobody stores them).
// The conversion is what this costs beside the plain loop: 1392 tokens, H = 2048, V = 128256, backward of a bf16 problem 1562 us,
// of an fp16 problem (nothing to convert) 1555; behind every MFMA of the refill instead of behind two of three 1577.
// An entry whose scaled value fp16 does not hold counts as fp16's largest (see direct_scale).
template <bool CONVERT>
struct LeftKm {
    static constexpr int kVecs = 4;
    const char* base;
    char* lds;
    uint32_t row_bytes, col;  // (a tile spans less than 4 GiB)
    int row0, krows;
    float scale, top;  // top: the largest magnitude converted so far, times the scale
    __device__ __forceinline__ LeftKm(const Operand A, int m0, int krows_, float scale_, char* smem)
        : krows(krows_), scale(scale_), top(0.f) {
        // FP16_OVFL: what overflows fp16 becomes its largest value (infinities stay), for the rest of the wave's life.  A bit of
        // the mode register, where a clamp would be two instructions more per pair of columns in the tile loop.
        if constexpr (CONVERT) asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1" ::: "memory");
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        base = reinterpret_cast<const char*>(A.p + m0);
        row_bytes = uint32_t(A.ld * 2);
        row0 = wave * 2 + (lane >> 5);
        const int unit = (lane & 31) ^ ((row0 & 3) << 1) ^ (row0 & 8);  // the logical 16-byte unit of this lane, as in DirectLoader
        col = uint32_t(min(unit * 8, A.rows - m0 - 8)) * 2u;
        lds = smem + wave * 1024 + lane * 16;
    }
    __device__ __forceinline__ void load(int k0, int j, u32x4& w) const {
        const int row = min(row0 + 16 * j, krows - 1 - k0);
        w = *reinterpret_cast<const u32x4*>(base + int64_t(k0) * row_bytes + (uint32_t(row) * row_bytes + col));
    }
    // two neighbouring columns; exact wherever fp16 holds the scaled value (below its range one rounding to nearest)
    __device__ __forceinline__ void convert(uint32_t& w) {
        if constexpr (CONVERT) {
            const float lo = __uint_as_float(w << 16) * scale, hi = __uint_as_float(w & 0xffff0000u) * scale;
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(lo), "v"(hi));
            w = Elem<TRLK_F16>::pack2(lo, hi);
        }
    }
    __device__ __forceinline__ void store(int buf, int j, u32x4 w) const {
        *reinterpret_cast<u32x4*>(lds + buf * kDenseStage + j * 8192) = w;
    }
    // the first two stages into the LDS, the third (or, where there is none, the last) into `w`
    __device__ __forceinline__ void prologue(int nk, u32x4 (&w)[kVecs]) {
        u32x4 first[2][kVecs];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < kVecs; ++j) load(min(s, nk - 1) * BK, j, first[s][j]);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < kVecs; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint32_t x = first[s][j][i];
                    convert(x);
                    first[s][j][i] = x;
                }
                store(s, j, first[s][j]);
            }
#pragma unroll
        for (int j = 0; j < kVecs; ++j) load(min(2, nk - 1) * BK, j, w[j]);
    }
};
struct NoLeftKm {};

// What a wave whose rows or columns all lie beyond the operands does in place of the tile loop: it moves its share of the
// tiles (exactly the transfers, waits and barriers of the loop) and spends nothing on matrix work.
template <bool BKM, bool LEFT, typename Left = NoLeftKm>
__device__ __forceinline__ void move_tiles_only(const DirectLoader<BKM, LEFT>& loader, int K, bool prefetched, Left left = {}) {
    const int nk = K / BK;
    u32x4 w[4];
    if (!prefetched) loader.prologue(K);
    if constexpr (LEFT) {
        loader.first_stage_landed(nk);
    } else {
        left.prologue(nk, w);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (kt + 2 < nk) {
            loader.issue(kt & 1, (kt + 2) * BK);
            if constexpr (!LEFT) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uint32_t x = w[j][i];
                        left.convert(x);
                        w[j][i] = x;
                    }
                    left.store(kt & 1, j, w[j]);
                    left.load(min(kt + 3, nk - 1) * BK, j, w[j]);
                }
            }
        }
    }
}

// `left`: a LeftKm, where the left operand is k-major.
template <int DT, bool BKM = false, typename Left = NoLeftKm>
__device__ __forceinline__ void gemm_tile_nt_direct(const Operand A, int m0, const Operand B, int n0, int K,
                                                    f32x4 (&acc)[MI][NI], char* smem, Left&& left = {}) {
    constexpr bool AKM = !std::is_same_v<std::decay_t<Left>, NoLeftKm>;
    const DirectLoader<BKM, !AKM> loader(A, m0, B, n0, smem);
    constexpr int kStageLoads = DirectLoader<BKM, !AKM>::kStageLoads;
    const int lane = threadIdx.x & 63, wave = loader.wave;
    const int wm = wave_m(wave), wn = wave_n(wave);

    // --- fragment side (blocks start at multiples of 16 rows, so the swizzle depends on the lane only).  A fragment is
    // 16 rows x 32 k: lane l holds the 8 k from 8 (l / 16) on of row l % 16.
    const int g = lane >> 4, l15 = lane & 15;
    const int koff[2] = {(g ^ tile_swizzle(l15)) * 16, ((4 + g) ^ tile_swizzle(l15)) * 16};
    const int fa_row = (wm * WM + l15) * kRowBytes, fb_row = (wn * WN + l15) * kRowBytes;
    // k-major right operand: a fragment is two transpose loads of 8 bytes.  The lanes work in groups of 16: lane t of a
    // group points at the 8 bytes that hold columns 4 (t % 4) .. + 3 of k row t / 4 (of the group's 4 k rows), and
    // receives column t of those 4 k rows.  Group g takes the block's 16 columns at k 8 g .. + 3 (second load: + 4 .. + 7).
    int fb_km[NI];
    if constexpr (BKM) {
        const int f = ((l15 >> 2) << 1) ^ ((g & 1) << 3);  // the unit swizzle of this lane's k rows
#pragma unroll
        for (int j = 0; j < NI; ++j)
            fb_km[j] = (8 * g + (l15 >> 2)) * (BN * 2) + (((wn * WN + j * 16) / 8 + ((l15 & 3) >> 1)) ^ f) * 16 + (l15 & 1) * 8;
    }
    int fa_km[MI];  // the same for a k-major left operand
    if constexpr (AKM) {
        const int f = ((l15 >> 2) << 1) ^ ((g & 1) << 3);
#pragma unroll
        for (int i = 0; i < MI; ++i)
            fa_km[i] = (8 * g + (l15 >> 2)) * (BM * 2) + (((wm * WM + i * 16) / 8 + ((l15 & 3) >> 1)) ^ f) * 16 + (l15 & 1) * 8;
    }
    // (absolute LDS addresses of the stage that is read next, changed over once a step)
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(smem));
    uint32_t at_a[MI], at_b[NI];
    if constexpr (AKM)
#pragma unroll
        for (int i = 0; i < MI; ++i) at_a[i] = lds0 + fa_km[i];
    if constexpr (BKM)
#pragma unroll
        for (int j = 0; j < NI; ++j) at_b[j] = lds0 + kDenseA + fb_km[j];
    auto other_stage = [&] {
        static_assert(kDenseStage == 65536, "one address bit tells the stages apart");
        if constexpr (AKM)
#pragma unroll
            for (int i = 0; i < MI; ++i) at_a[i] ^= kDenseStage;
        if constexpr (BKM)
#pragma unroll
            for (int j = 0; j < NI; ++j) at_b[j] ^= kDenseStage;
    };
    auto read_tr = [&](uint32_t base, int ks) -> u32x4 {
        static_assert(BM == BN, "k rows of both operands have one length");
        const uint32_t at = base + uint32_t(ks * 32 * (BN * 2));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(at));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(at + 4 * (BN * 2)));
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(u32x4, both);
    };
    auto read_a = [&](const char* sa, int i, int ks) -> u32x4 {
        if constexpr (AKM)
            return read_tr(at_a[i], ks);
        else
            return *reinterpret_cast<const u32x4*>(sa + fa_row + i * 16 * kRowBytes + koff[ks]);
    };
    auto read_b = [&](const char* sb, int j, int ks) -> u32x4 {
        if constexpr (BKM)
            return read_tr(at_b[j], ks);
        else
            return *reinterpret_cast<const u32x4*>(sb + fb_row + j * 16 * kRowBytes + koff[ks]);
    };

    const int nk = K / BK;
    u32x4 lw[4];  // the left operand's stage kt + 2 at the start of step kt
    loader.prologue(K);
    if constexpr (AKM) {
        left.prologue(nk, lw);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    } else {
        loader.first_stage_landed(nk);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Software pipeline over slices of 32 k, two per step.  A slice runs over the wave's blocks twice, first with the
    // column blocks 0, 1, then with 2, 3.  Every fragment register is loaded again, for the next slice, right behind its
    // last use: a row fragment in the second half, a pair of column fragments at the end of its half -- 14 to 16 MFMAs
    // before the next use, with one set of fragment registers (48; a second set would not fit beside the epilogues).
    // The compiler's own scheduler sinks every ds_read next to its first use (one exposed LDS latency per MFMA pair), so
    // the issue order is pinned explicitly: MFMA, then at most two fragment reads and one tile transfer.
    //
    // The barrier that frees a stage sits inside the step's second slice, kBarAt row blocks into its first half: by then
    // the last fragments of the stage, read at the end of the first slice, have arrived.  The stage's refill follows
    // it, one transfer every other MFMA, and has until the same place of the next step to land.
    //
    // Bound by power (clock 1.5-1.7 GHz) and the arrival of the tiles.  Forward and backward, of which the two products are
    // two thirds, against products on 32x32x16 MFMAs with two sets of fragments and the tile order of that time: 9664
    // tokens, H = 3584, V = 151936 27.7 -> 26.4 ms; 1396 tokens, H = 2048, V = 50257 1115 -> 1020 us; 459 tokens, H = 3584,
    // V = 151936 2554 -> 2300 us.
    constexpr int kBarAt = 4;
    static_assert(NI == 4 && 2 * kStageLoads <= 2 * (MI - kBarAt) + 2 * MI, "the refill fits behind the barrier");
    u32x4 a[MI], b[NI];
    {
        const char* sa = smem;
        const char* sb = smem + kDenseA;
        b[0] = read_b(sb, 0, 0);
        b[1] = read_b(sb, 1, 0);
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i] = read_a(sa, i, 0);
        b[2] = read_b(sb, 2, 0);
        b[3] = read_b(sb, 3, 0);
    }
    auto step = [&](int kt, auto refill_tag, auto next_tag) {
        constexpr bool REFILL = decltype(refill_tag)::value, NEXT = decltype(next_tag)::value;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            // the next slice: this stage's second, or the next stage's first
            const char* na = smem + ((kt + ks) & 1) * kDenseStage;
            const char* nb = na + kDenseA;
            const bool load = ks == 0 || NEXT;
            int issued = 0, slot = 0;
            if (ks == 1) other_stage();
#pragma unroll
            for (int half = 0; half < 2; ++half) {
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    if (ks == 1 && half == 0 && i == kBarAt) {
                        // Every fragment read of this stage has returned and the next stage has landed.  A bare s_barrier:
                        // __syncthreads() carries release / acquire fences; nothing may move across it.
                        // (with a left operand in registers the wait is one that the compiler counts: it need not wait for them again)
                        if constexpr (AKM)
                            __builtin_amdgcn_s_waitcnt(0);
                        else
                            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                        __builtin_amdgcn_s_barrier();
                        __builtin_amdgcn_sched_barrier(0);
                        asm volatile("" ::: "memory");
                    }
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj) {
                        const int j = half * 2 + jj;
                        acc[i][j] = mfma<DT>(a[i], b[j], acc[i][j]);
                        __builtin_amdgcn_sched_barrier(0);  // (a load moved above the MFMA would need registers of its own)
                        if (load) {
                            if (half == 1 && jj == 1) a[i] = read_a(na, i, ks ^ 1);
                            if (i == MI - 1) b[j] = read_b(nb, j, ks ^ 1);
                        }
                        if (REFILL && ks == 1 && (half == 1 || i >= kBarAt)) {
                            if ((AKM ? slot % 3 == 2 : (slot & 1)) && issued < kStageLoads) {
                                loader.issue_one(kt & 1, (kt + 2) * BK, issued);
                                ++issued;
                            }
                            // a pair of columns behind two of three MFMAs (its six instructions keep the vector unit as busy as
                            // three MFMAs of the SIMD's two waves do the matrix unit); a vector that is whole makes room
                            // for the next stage's
                            if constexpr (AKM) {
                                if (slot % 3 != 2) {
                                    const int pair = slot - slot / 3;
                                    uint32_t x = lw[pair >> 2][pair & 3];
                                    left.convert(x);
                                    lw[pair >> 2][pair & 3] = x;
                                    if ((pair & 3) == 3) {
                                        left.store(kt & 1, pair >> 2, lw[pair >> 2]);
                                        left.load(min(kt + 3, nk - 1) * BK, pair >> 2, lw[pair >> 2]);
                                    }
                                }
                            }
                            ++slot;
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    };
    constexpr std::true_type T{};
    constexpr std::false_type F{};
    int kt = 0;
    for (; kt + 2 < nk; ++kt) step(kt, T, T);
    if (kt + 1 < nk) step(kt++, F, T);
    step(kt, F, F);
    // every LDS read of this tile completed before the last barrier: the caller may reuse the LDS right away
}

// The register-staged tile, sum_k A[m0 + .., k] * B[n0 + .., k].  Rows beyond the operand's end are clamped to
// its last row (callers ignore those outputs); k beyond K reads as zero (K % 8 == 0).
// `compute(sa, sb)` multiplies one stage (rows of kLdsRow elements).
template <typename Compute>
__device__ __forceinline__ void staged_tile(const Operand A, int m0, const Operand B, int n0, int K, char* smem, Compute compute) {
    const int tid = threadIdx.x;
    const int kc = tid % kCpr, r0 = tid / kCpr;  // this thread stages rows r0 + kRowStep*j, 16-byte chunk kc

    // uniform tile base + 32-bit per-lane byte offsets (a tile spans < 4 GiB)
    const char* abase = reinterpret_cast<const char*>(A.p + int64_t(m0) * A.ld);
    const char* bbase = reinterpret_cast<const char*>(B.p + int64_t(n0) * B.ld);
    uint32_t ao[kLoadsA], bo[kLoadsB];
#pragma unroll
    for (int j = 0; j < kLoadsA; ++j) {
        int ra = r0 + kRowStep * j;
        ra = m0 + ra < A.rows ? ra : A.rows - 1 - m0;  // clamp to the operand's last row
        ao[j] = uint32_t((int64_t(ra) * A.ld + kc * 8) * 2);
    }
#pragma unroll
    for (int j = 0; j < kLoadsB; ++j) {
        int rb = r0 + kRowStep * j;
        rb = n0 + rb < B.rows ? rb : B.rows - 1 - n0;
        bo[j] = uint32_t((int64_t(rb) * B.ld + kc * 8) * 2);
    }
    const int st_off = (r0 * kLdsRow + kc * 8) * 2;        // + j * kRowStep rows

    const u32x4 zero = {0u, 0u, 0u, 0u};
    // full k steps load unconditionally; only the last, partial step (K % BK != 0) masks its chunks
    auto load_stage = [&](u32x4(&ra)[kLoadsA], u32x4(&rb)[kLoadsB], int k0) {
        const char* ap = abase + int64_t(k0) * 2;
        const char* bp = bbase + int64_t(k0) * 2;
        if (k0 + BK <= K) {
#pragma unroll
            for (int j = 0; j < kLoadsA; ++j) ra[j] = *reinterpret_cast<const u32x4*>(ap + ao[j]);
#pragma unroll
            for (int j = 0; j < kLoadsB; ++j) rb[j] = *reinterpret_cast<const u32x4*>(bp + bo[j]);
        } else {
            const bool in = k0 + kc * 8 < K;
#pragma unroll
            for (int j = 0; j < kLoadsA; ++j) ra[j] = in ? *reinterpret_cast<const u32x4*>(ap + ao[j]) : zero;
#pragma unroll
            for (int j = 0; j < kLoadsB; ++j) rb[j] = in ? *reinterpret_cast<const u32x4*>(bp + bo[j]) : zero;
        }
    };
    auto store_stage = [&](const u32x4(&ra)[kLoadsA], const u32x4(&rb)[kLoadsB], int buf) {
        char* sa = smem + buf * kStageBytes;
        char* sb = sa + kTileABytes;
#pragma unroll
        for (int j = 0; j < kLoadsA; ++j) *reinterpret_cast<u32x4*>(sa + st_off + j * kRowStep * kLdsRow * 2) = ra[j];
#pragma unroll
        for (int j = 0; j < kLoadsB; ++j) *reinterpret_cast<u32x4*>(sb + st_off + j * kRowStep * kLdsRow * 2) = rb[j];
    };
    // Registers hold the tile of step kt+1 while step kt computes out of LDS; it is written to the
    // other LDS buffer at the end of the step (one barrier per step).
    const int nk = (K + BK - 1) / BK;
    u32x4 ra[kLoadsA], rb[kLoadsB];
    load_stage(ra, rb, 0);
    store_stage(ra, rb, 0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const bool more = kt + 1 < nk;
        if (more) load_stage(ra, rb, (kt + 1) * BK);
        compute(smem + (kt & 1) * kStageBytes, smem + (kt & 1) * kStageBytes + kTileABytes);
        if (more) store_stage(ra, rb, (kt + 1) & 1);
        __syncthreads();
    }
}

template <int DT>
__device__ __forceinline__ void gemm_tile_nt_staged(const Operand A, int m0, const Operand B, int n0, int K,
                                                    f32x4 (&acc)[MI][NI], char* smem) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave_m(wave), wn = wave_n(wave);
    const int fa_off = ((wm * WM + (lane & 15)) * kLdsRow + (lane >> 4) * 8) * 2;  // + i * 16 rows, + ks * 32
    const int fb_off = ((wn * WN + (lane & 15)) * kLdsRow + (lane >> 4) * 8) * 2;

#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    staged_tile(A, m0, B, n0, K, smem, [&](const char* sa, const char* sb) {
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            u32x4 fa[MI], fb[NI];
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[i] = *reinterpret_cast<const u32x4*>(sa + fa_off + (i * 16 * kLdsRow + ks * 32) * 2);
#pragma unroll
            for (int j = 0; j < NI; ++j) fb[j] = *reinterpret_cast<const u32x4*>(sb + fb_off + (j * 16 * kLdsRow + ks * 32) * 2);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) acc[i][j] = mfma<DT>(fa[i], fb[j], acc[i][j]);
        }
    });
}

// The forward's tile loop: 32x32x16 MFMAs (a fragment is 32 rows x 16 k).  The caller has run DirectLoader::prologue.
template <int DT>
__device__ __forceinline__ void fwd_tile_direct(const Operand A, int m0, const Operand B, int n0, int K, f32x16 (&acc)[MB][NB],
                                                char* smem) {
    const DirectLoader<> loader(A, m0, B, n0, smem);
    const int lane = threadIdx.x & 63, wave = loader.wave;
    const int wm = wave_m(wave), wn = wave_n(wave);

    // --- fragment side (tile rows of a wave start at multiples of 32, so the swizzle depends on the lane only)
    const int swz = tile_swizzle(lane & 31);
    const int hl = lane >> 5;
    const int fa_row = (wm * WM + (lane & 31)) * kRowBytes, fb_row = (wn * WN + (lane & 31)) * kRowBytes;
    constexpr int KS = BK / 16;
    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) koff[ks] = ((ks * 2 + hl) ^ swz) * 16;
    auto read_a = [&](const char* sa, int mb, int ks) -> u32x4 {
        return *reinterpret_cast<const u32x4*>(sa + fa_row + mb * 32 * kRowBytes + koff[ks]);
    };

#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.f;

    // Software pipeline.  Fragment loads run one 16-wide k slice ahead of the MFMAs that consume them,
    // across the barrier too: the last slice of a stage is already in registers when the workgroup
    // synchronises, so its MFMAs cover the refill of the freed stage and the first fragment reads of
    // the next one.
    constexpr int kStageLoads = DirectLoader<>::kStageLoads;
    auto load_frags = [&](int buf, int ks, u32x4(&fa)[MB], u32x4(&fb)[NB]) {
        const char* sa = smem + buf * kDenseStage;
        const char* sb = sa + kDenseA;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) fa[mb] = read_a(sa, mb, ks);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            fb[nb] = *reinterpret_cast<const u32x4*>(sb + fb_row + nb * 32 * kRowBytes + koff[ks]);
    };
    u32x4 fa[2][MB], fb[2][NB];
    static_assert(KS % 2 == 0 && MB * NB > MB + NB, "pipeline shape");
    constexpr std::true_type T{};
    constexpr std::false_type F{};
    const int nk = K / BK;
    loader.first_stage_landed(nk);
    constexpr int kLoadsPost = (kStageLoads + 1) / 2, kLoadsPre = kStageLoads - kLoadsPost;
    load_frags(0, 0, fa[0], fb[0]);
    // Exact issue order, pinned instruction by instruction (sched_barrier(0) between the groups):
    // MFMA i of the slice, then at most one fragment read of the next slice and at most one tile
    // transfer.  Fragments are read in the order the mb-major MFMA sequence needs them (fa0, fb*,
    // fa1, ...), so every read has most of a slice between its issue and its first use.  The refill
    // of a stage is split: the first half of its transfers goes behind the barrier that frees it, the
    // second half into the first slice of the following step.
    constexpr int M = MB * NB, R = MB + NB;
    auto slice = [&](u32x4(&ca)[MB], u32x4(&cb)[NB], auto read_tag, int rbuf, int rks, u32x4(&na)[MB], u32x4(&nb_)[NB],
                     auto nload_tag, int lbuf, int lk0, int lfirst) {
        constexpr bool READ = decltype(read_tag)::value;
        constexpr int NL = decltype(nload_tag)::value;
        const char* sa = smem + rbuf * kDenseStage;
        const char* sb = sa + kDenseA;
        int issued = 0;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const int mb = i / NB, nb = i % NB;
            acc[mb][nb] = mfma_fwd<DT>(ca[mb], cb[nb], acc[mb][nb]);
            if (READ && i < R) {
                // read order: fa[0], fb[0..NB-1], fa[1..MB-1]
                if (i == 0)
                    na[0] = read_a(sa, 0, rks);
                else if (i <= NB)
                    nb_[i - 1] = *reinterpret_cast<const u32x4*>(sb + fb_row + (i - 1) * 32 * kRowBytes + koff[rks]);
                else
                    na[i - NB] = read_a(sa, i - NB, rks);
            }
            if (NL > 0 && (i + 1) * NL / M > i * NL / M) {
                loader.issue_one(lbuf, lk0, lfirst + issued);
                ++issued;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    typedef std::integral_constant<int, kLoadsPost> post_t;
    typedef std::integral_constant<int, kLoadsPre> pre_t;
    typedef std::integral_constant<int, 0> zero_t;
    // POST / PRE: this step issues the first half of the refill of the stage it frees / the second
    // half of the refill the previous step started.  NEXT: another step follows.
    auto step = [&](int kt, auto post_tag, auto pre_tag, auto next_tag) {
        constexpr bool POST = decltype(post_tag)::value, PRE = decltype(pre_tag)::value, NEXT = decltype(next_tag)::value;
        const int cur = kt & 1, nxt = cur ^ 1;
#pragma unroll
        for (int ks = 0; ks + 1 < KS; ++ks) {
            if (PRE && ks == 0)
                slice(fa[ks & 1], fb[ks & 1], T, cur, ks + 1, fa[(ks + 1) & 1], fb[(ks + 1) & 1], pre_t{}, nxt,
                      (kt + 1) * BK, kLoadsPost);
            else
                slice(fa[ks & 1], fb[ks & 1], T, cur, ks + 1, fa[(ks + 1) & 1], fb[(ks + 1) & 1], zero_t{}, 0, 0, 0);
        }
        // every fragment read of this stage has returned and the next stage has landed
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        // A bare s_barrier: __syncthreads() carries release/acquire fences, for which the compiler
        // adds waits of its own.  The waits above are the ones this exchange needs; nothing may move across the barrier.
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        constexpr int L = (KS - 1) & 1;
        if constexpr (NEXT && POST)
            slice(fa[L], fb[L], T, nxt, 0, fa[0], fb[0], post_t{}, cur, (kt + 2) * BK, 0);
        else if constexpr (NEXT)
            slice(fa[L], fb[L], T, nxt, 0, fa[0], fb[0], zero_t{}, 0, 0, 0);
        else
            slice(fa[L], fb[L], F, 0, 0, fa[0], fb[0], zero_t{}, 0, 0, 0);
    };
    static_assert(((KS - 1) & 1) == 1, "the last slice of a stage sits in fragment buffer 1, the next stage's first in 0");
    int kt = 0;
    if (nk > 2) {
        step(kt++, T, F, T);
        for (; kt + 2 < nk; ++kt) step(kt, T, T, T);
        step(kt++, F, T, T);  // kt = nk - 2: completes the last refill
    } else if (nk == 2) {
        step(kt++, F, F, T);
    }
    // No step is left.  Without this loop, and with six other ways to write these lines, one or two registers of the kernel with
    // a stash are spilled: 0.5 to 1 % more time (1396 tokens, H = 2048, V = 50257 259 -> 262 us; 9664 tokens, H = 3584, V = 151936
    // 8415 -> 8441 us).
    for (; kt + 1 < nk; ++kt) step(kt, F, F, T);
    step(kt, F, F, F);
    // every LDS read of this tile completed before the last barrier: the caller may reuse the LDS right away
}

template <int DT>
__device__ __forceinline__ void fwd_tile_staged(const Operand A, int m0, const Operand B, int n0, int K, f32x16 (&acc)[MB][NB],
                                                char* smem) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fa_off = ((wave_m(wave) * WM + (lane & 31)) * kLdsRow + (lane >> 5) * 8) * 2;  // + mb * 32 rows, + ks * 16
    const int fb_off = ((wave_n(wave) * WN + (lane & 31)) * kLdsRow + (lane >> 5) * 8) * 2;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.f;
    staged_tile(A, m0, B, n0, K, smem, [&](const char* sa, const char* sb) {
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            u32x4 fa[MB], fb[NB];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                fa[mb] = *reinterpret_cast<const u32x4*>(sa + fa_off + (mb * 32 * kLdsRow + ks * 16) * 2);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                fb[nb] = *reinterpret_cast<const u32x4*>(sb + fb_off + (nb * 32 * kLdsRow + ks * 16) * 2);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mfma_fwd<DT>(fa[mb], fb[nb], acc[mb][nb]);
        }
    });
}

template <int DT, bool BKM = false, typename Left = NoLeftKm>
__device__ __forceinline__ void gemm_tile_nt(const Operand A, int m0, const Operand B, int n0, int K,
                                             f32x4 (&acc)[MI][NI], char* smem, Left&& left = {}) {
    if constexpr (BKM) {  // (callers of this form pad K to whole steps)
        gemm_tile_nt_direct<DT, true>(A, m0, B, n0, K, acc, smem, left);
    } else {
        if ((K & (BK - 1)) == 0)
            gemm_tile_nt_direct<DT>(A, m0, B, n0, K, acc, smem);
        else
            gemm_tile_nt_staged<DT>(A, m0, B, n0, K, acc, smem);
    }
}

// Row (M index) inside the workgroup tile of accumulator element r of block i, for this lane.
__device__ __forceinline__ int acc_row(int wm, int i, int r, int lane) { return wm * WM + i * 16 + (lane >> 4) * 4 + r; }
// Column (N index) inside the workgroup tile of block j, for this lane.
__device__ __forceinline__ int acc_col(int wn, int j, int lane) { return wn * WN + j * 16 + (lane & 15); }
// The same in the forward: element r of block mb, block nb.
__device__ __forceinline__ int fwd_row(int wm, int mb, int r, int lane) {
    return wm * WM + mb * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
}
__device__ __forceinline__ int fwd_col(int wn, int nb, int lane) { return wn * WN + nb * 32 + (lane & 31); }

// Workgroup id -> (tile along axis `a`, tile along axis `b`) such that the workgroups that run
// together on one XCD (ids congruent mod 8, dispatched round-robin) form patches of about 4 x 8 tiles: they share
// operand slabs through that XCD's L2.  No workgroup of the grid but a few at the end is empty: the hardware deals
// workgroups to the CUs in order, and with empty ones interleaved at a fixed stride the real ones end up on a fraction of
// the CUs (measured: a third more time for 65 instead of 64 a tiles with a grid padded to whole bands).
//
// From 32 a tiles on an XCD owns the `a` tiles congruent to its number mod 8, in bands of 4; inside a band it walks b
// with the band's a tiles innermost.  The last band holds only as many a tiles per XCD as n_a needs.  The n_a % 8 a tiles
// that are left when every XCD has the same number are not given to that many XCDs whole (one XCD in eight would then
// carry an a tile more than the others and the launch would wait for it): their n_b tiles each are dealt out
// in equal runs over all eight XCDs, a innermost.
//
// Fewer a tiles (token counts below 8192) are put into even bands of at most 8; inside a band b is walked with the band's a
// tiles innermost, and each XCD takes one eighth of that sequence: 4 to 8 a tiles beside 4 to 8 b tiles at a time.  Under
// the rule for many a tiles an XCD has ONE a tile beside 32 b tiles when there are 8 to 15, and fetches 33 slabs where
// 12 would do: 2300 tokens, H = 2048, V = 128256 forward 1140 -> 1107 us, with backward 3720 -> 3690 us; 3000 tokens, H =
// 3072, V = 50257 866 -> 834 and 2713 -> 2664 us; 1000 tokens, H = 2048, V = 128256 (there the slices of dHidden) 1948 -> 1918 us.
// The same for the last few of many a tiles loses (79 a tiles: forward 3653 -> 3735 us).
// The caller skips ta >= n_a or tb >= n_b.
__device__ __forceinline__ void xcd_patch(int w, int n_a, int n_b, int& ta, int& tb) {
    const int xcd = w & 7, q = w >> 3;
    const int groups = n_a >= 32 ? n_a >> 3 : 0;   // a tiles every XCD owns whole
    const int bands = groups >> 2;                 // full bands of 4 of them
    const int full = bands * 4 * n_b;              // workgroups of this XCD in the full bands
    const int m = groups & 3;                      // whole a tiles per XCD in the last band
    if (q < full) {
        const int rem = q % (4 * n_b);
        tb = rem >> 2;
        ta = ((q / (4 * n_b)) * 4 + (rem & 3)) * 8 + xcd;
        return;
    }
    if (q < full + m * n_b) {
        const int qq = q - full;
        tb = qq / m;
        ta = (bands * 4 + qq % m) * 8 + xcd;
        return;
    }
    // the a tiles that are left, from n_a - left on, dealt out in runs
    const int left = n_a - groups * 8, share = (left * n_b + 7) >> 3, i = q - full - m * n_b, t = xcd * share + i;
    if (i >= share || t >= left * n_b) {
        ta = n_a;
        tb = n_b;
        return;
    }
    const int n_bands = (left + 7) >> 3, narrow = left / n_bands, wide = left % n_bands;  // `wide` bands of narrow + 1, then narrow
    const int in_wide = wide * (narrow + 1) * n_b;
    const int width = t < in_wide ? narrow + 1 : narrow, u = t < in_wide ? t : t - in_wide;
    const int band = u / (width * n_b), v = u - band * (width * n_b);
    tb = v / width;
    ta = groups * 8 + (t < in_wide ? 0 : wide * (narrow + 1)) + band * width + (v - tb * width);
}
inline int xcd_patch_grid(int n_a, int n_b) {
    const int groups = n_a >= 32 ? n_a / 8 : 0, left = n_a - groups * 8;
    return 8 * (groups * n_b + (left * n_b + 7) / 8);
}

// What a forward keeps for the backward when it is given a stash: for every logit its softmax numerator
//   e[v][n] = exp2(z[v][n] * log2(e) - ref) * 2^15   as fp16,   0 < e <= 2^15,
// where `ref` is the integer reference exponent that the lane which owned the logit held when it summed the tile
// (the running maximum of its part of the row, rounded up).  One reference covers the 64 rows of a 128-row block
// whose row quad (v / 4) has the same parity, for one token.  The backward's sweep turns a numerator into the
// probability with one multiplication: p = e * exp2(ref - 15 - log_z * log2(e)).  fp16 keeps 11 significant bits of
// every numerator down to 2^-29 of the running maximum and flushes below 2^-39 of it: the same accuracy d logits
// has after it is rounded to fp16 for the products, at half the bytes of the raw fp32 products.
//   quads  [vpad / 4][ld] x 8 bytes: the 4 rows of a quad for one token (rows are the vocabulary, vpad = V rounded up
//          to the tile; the accumulator layout gives a lane 4 consecutive rows of one token)
//   refs   [vpad / 128][2][ld] fp32: reference exponent of (128-row block, parity of the row quad, token)
//   zt     [ld] fp32: the target's logit z (a soft-capped head needs it for the chain factor of the one-hot term)
struct StashView {
    char* base;
    int64_t ld;    // tokens per row (>= N rounded up to the tile, or any with stash_cols)
    int64_t vpad;  // vocabulary rows the forward covered
    __host__ __device__ static int64_t rows8(int64_t vpad) { return vpad / 4 + vpad / 128 + 1; }  // rows of ld x 8 bytes
    __host__ __device__ uint2* quads() const { return reinterpret_cast<uint2*>(base); }
    __host__ __device__ float* refs() const { return reinterpret_cast<float*>(base + (vpad / 4) * ld * 8); }
    __host__ __device__ float* zt() const { return reinterpret_cast<float*>(base + (vpad / 4 + vpad / 128) * ld * 8); }
};

struct HeadArgs {
    const uint16_t* hidden;  // [N, H]
    const uint16_t* weight;  // [V, H]
    const int64_t* targets;  // [N]
    const float* bias;       // [V] added to hidden . weight[v] before scaling, or null
    int N, V, H;
    int64_t ldh, ldw;
    float logit_scale, inv_t, softcap;  // softcap <= 0: none
    // forward
    int v_splits, tiles_per_split;
    float* partial;  // [N, v_splits, 4]: (reference exponent, S, U, exact max of z)
    float* tgt;      // [N] logit of the target token (NaN until found)
    // backward (dz pass)
    const float* log_z;  // [N]
    const float* g;      // [N] upstream d loss / d logp
    int c0, c1;          // vocabulary rows of this chunk
    StashView stash;     // forward (written) and backward (read): the softmax numerators, or base == null
    const int32_t* stash_cols;  // backward: stash column of token n (tokens were compacted since the forward), or null
    uint16_t* dzT;       // [chunk rows padded, ldzt] (columns = tokens), fp16, column n scaled by pow2_scale(|g[n]| * zs)
    int64_t ldzt;
    const uint32_t* g_max;
    int sdz_token_blocks, sdz_tiles;  // stash sweep: token blocks per row group, tiles of the launch  // backward: bit pattern of max |g| over the tokens
};

// ---- scaled fp16 copies of the backward's operands -----------------------------------------------------------------
// The two backward products run on fp16 operands whatever the dtype of the problem: d logits rounded to bf16 would
// carry 8 significant bits into both gradients (relative error 3e-3), fp16 carries 11 (4e-4) at the same matrix-core
// rate.  fp16 has 5 exponent bits, so every operand is multiplied by a power of two that puts its largest magnitude
// into [2^13, 2^14) (exact, undone in the products' epilogue): d logits per token (|dz[:, n]| <= |g[n]| * logit_scale
// / T, so token n's column carries s_n = pow2_scale(|g[n]| * logit_scale / T) and a token whose upstream gradient is
// a million times smaller than the largest keeps its own relative accuracy in dHidden, whose row n the epilogue
// divides by s_n), W^T and hidden^T of a bf16 problem by their largest magnitude (of W's a sample decides; bf16 -> fp16 is then exact down to
// 2^-31 of that maximum).  The dW product sums over the tokens, so it needs the columns of d logits in ONE scale: row
// n of hidden^T's source is multiplied by s_all / s_n on its way (s_all = the scale of the largest |g|, so the factor
// is a power of two <= 1), which leaves dz^T[v, n] * hidden^T[h, n] in the scale s_all * s_hidden for every n.  A token
// whose gradient is 2^-25 of the largest starts to lose bits of its hidden row there -- where its whole contribution
// to dW is below the rounding of the fp32 sum.
__device__ __forceinline__ float pow2_scale(float m) {
    if (!(m > 0.f) || !(m < INFINITY)) return 1.f;
    int e;
    (void)frexpf(m, &e);  // m = f * 2^e with f in [0.5, 1)
    int k = 14 - e;
    k = k > 100 ? 100 : (k < -100 ? -100 : k);
    return ldexpf(1.f, k);
}
__device__ __forceinline__ float slot_scale(const uint32_t* slot, float mult) {
    return slot != nullptr ? pow2_scale(__uint_as_float(*slot) * mult) : 1.f;
}
// The weight's scale comes from a SAMPLE of it (one of every kSampleRows rows, see sample_row), so that no pass over the whole weight is needed
// before the one that converts it; that pass finds the true maximum on its way.  slots[0] is the sample's largest magnitude,
// slots[1] that of the entries that exceed it (0 if none does).  The sample's scale leaves a factor of 4 to fp16's largest
// value; only when the chunk reaches beyond it, or the sample holds nothing but zeros, is the chunk converted again
// with the scale of its own maximum.
constexpr int kSampleRows = 32;
// The row that stands for rows 32 i to 32 i + 31 of V: not the same one of every 32, so that a period in the weight (large entries in
// every other row) does not hide from the sample.
__device__ __forceinline__ int sample_row(int i, int V) {
    static_assert(kSampleRows == 32, "5 bits of the product");
    return min(i * kSampleRows + int((uint32_t(i) * 2654435761u) >> 27), V - 1);
}
struct WeightScale {
    float scale;
    bool again;  // the chunk has to be converted (again) with `scale`
};
__device__ __forceinline__ WeightScale weight_scale(const uint32_t* sample, const uint32_t* beyond) {
    const float m = __uint_as_float(*sample), top = __uint_as_float(max(*sample, *beyond)), s = pow2_scale(m);
    if (top == 0.f || (m > 0.f && top * s <= 65504.f)) return {s, false};
    return {pow2_scale(top), true};
}

// The scale in which the dHidden product converts a weight that it reads itself: the sample's, whatever the other entries are.
// What exceeds fp16 there (|w| * scale > kF16Max, four to eight times the sample's maximum) counts as kF16Max in the product; the
// rest of it is added by the pass that sums the product's slices, from the rows in which beyond_rows_kernel finds such
// entries.  So one large entry neither makes the product be done again nor takes bits from the others.  (At most 2^60, also
// for a sample of nothing but zeros.  w * scale has to be finite in fp32: an entry of 2^113 times the sample's maximum, and of 2^68
// beside such a sample, counts as infinite.)
constexpr float kF16Max = 65504.f;
__device__ __forceinline__ float direct_scale(const uint32_t* sample) {
    const float m = __uint_as_float(*sample);
    return m > 0.f ? fminf(pow2_scale(m), 0x1p60f) : 0x1p60f;
}

// tanh for soft-capping: sign(x) (1 - t) / (1 + t) with t = exp(-2 |x|) from the hardware's exp2 and reciprocal (a
// relative error of a few 1e-7), and the odd series x - x^3/3 + 2 x^5/15 below 0.05, where 1 - t cancels.  A third of
// the instructions of the library routine, in an epilogue that runs it once per logit.
__device__ __forceinline__ float head_tanh(float x) {
    const float ax = fabsf(x), x2 = x * x;
    const float t = fast_exp2(ax * (-2.f * kLog2e));
    const float big = (1.f - t) * __builtin_amdgcn_rcpf(1.f + t);
    const float small = ax * fmaf(x2, fmaf(x2, 2.f / 15.f, -1.f / 3.f), 1.f);
    return copysignf(ax < 0.05f ? small : big, x);
}

constexpr float kStashExp = 15.f;  // the numerators are summed and stashed times 2^15 (fp16's range above 1)

// GENERAL: soft-capping or a non-positive scale (z is computed per logit).  Otherwise z = (y + bias) * zs with one
// positive scale: the maximum is taken on the raw accumulators, the scale is folded into the exponent's multiplier and
// sum(e * z) is accumulated as zs * sum(e * y) -- the kernel of the usual head then carries no code of the other.
// STAGED: the hidden size is not a multiple of the direct-to-LDS loop's k step (a kernel of its own, so that the
// usual one does not carry the register-staged loop's code and loop-invariant registers through its tile loop).
template <int DT, bool STASH, bool GENERAL, bool STAGED>
TRLK_HEAD_KERNEL void fused_head_fwd_kernel(HeadArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int n_tb = (a.N + BN - 1) / BN;
    int tb, vs;
    xcd_patch(blockIdx.x, n_tb, a.v_splits, tb, vs);
    if (tb >= n_tb || vs >= a.v_splits) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave_m(wave), wn = wave_n(wave);
    const int n0 = tb * BN;
    const int n_vt = (a.V + BM - 1) / BM;
    const int vt0 = vs * a.tiles_per_split;
    const int vt1 = vt0 + a.tiles_per_split < n_vt ? vt0 + a.tiles_per_split : n_vt;

    // per-lane online state of the NB tokens this lane owns (base-2, integer reference exponent)
    float ref[NB], S[NB], U[NB], zmax[NB];
    int tg[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        ref[nb] = -INFINITY;
        zmax[nb] = -INFINITY;
        S[nb] = 0.f;
        U[nb] = 0.f;
        const int tok = n0 + fwd_col(wn, nb, tid & 63);
        const int64_t t = tok < a.N ? a.targets[tok] : -1;
        tg[nb] = t >= 0 && t < a.V ? int(t) : -1;
    }
    const Operand W{a.weight, a.ldw, a.V}, Hd{a.hidden, a.ldh, a.N};

    if constexpr (!STAGED)
        if (vt0 < vt1) DirectLoader<>(W, vt0 * BM, Hd, n0, smem).prologue(a.H);
    const float zs = uniform(a.logit_scale * a.inv_t), zs2 = uniform(zs * kLog2e);
    const bool idle = !STAGED && n0 + wn * WN >= a.N;  // all of this wave's tokens lie beyond the last one
    if (idle) {
#pragma unroll 1
        for (int vt = vt0; vt < vt1; ++vt) {
            move_tiles_only(DirectLoader<>(W, vt * BM, Hd, n0, smem), a.H, true);
            if (vt + 1 < vt1) DirectLoader<>(W, (vt + 1) * BM, Hd, n0, smem).prologue(a.H);
        }
    }
    for (int vt = vt0; vt < vt1 && !idle; ++vt) {
        const int m0 = vt * BM;
        f32x16 acc[MB][NB];
        if constexpr (STAGED) {
            fwd_tile_staged<DT>(W, m0, Hd, n0, a.H, acc, smem);
        } else {
            fwd_tile_direct<DT>(W, m0, Hd, n0, a.H, acc, smem);
            // What of the state did not fit beside the accumulators and fragments comes back from scratch here: behind the
            // transfers below each reload would wait for them to land.
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                asm volatile("" : "+v"(ref[nb]), "+v"(S[nb]), "+v"(U[nb]), "+v"(zmax[nb]), "+v"(tg[nb]));
            // the next tile's first stages travel while this tile's logits are reduced (registers only)
            if (vt + 1 < vt1) DirectLoader<>(W, m0 + BM, Hd, n0, smem).prologue(a.H);
        }
        const int lane = fresh(tid & 63), half = lane >> 5;
        // Stash: for one accumulator quad (4 consecutive vocabulary rows of one token per lane) the 32 lanes of a
        // half-wave hold 32 consecutive tokens = 256 contiguous bytes per store.  The buffer is padded to whole tiles.
        // Addresses are a uniform pointer that walks down the quads (scalar registers, one addition per store) plus
        // the lane's byte offset (one vector register; the entry point bounds ld so that it fits 32 bits).
        char* stash_blk = nullptr;
        float* ref_blk = nullptr;
        uint32_t stash_lane = 0, ref_lane = 0;
        if constexpr (STASH) {
            const int col = n0 + wn * WN;
            stash_blk = reinterpret_cast<char*>(a.stash.quads() + int64_t(m0 / 4 + wm * (WM / 4)) * a.stash.ld + col);
            ref_blk = a.stash.refs() + int64_t(m0 / 128 + wm) * 2 * a.stash.ld + col;
            ref_lane = uint32_t(half) * uint32_t(a.stash.ld) + uint32_t(lane & 31);
            stash_lane = ref_lane * 8u;
        }
        const bool partial_tile = m0 + BM > a.V;
        constexpr bool plain = !GENERAL;
        // Before the reduction, only where needed (a bias, the general form of z, or the vocabulary's last tile, whose
        // rows beyond the vocabulary count as -inf): the accumulators become y + bias (usual head) or z itself
        // (general form).  A lane's 16 accumulators of a block are 4 quads of consecutive vocabulary rows, so the bias
        // comes as one 16-byte load per quad, all of a block row's loads issued before the first is used.
        if (GENERAL || a.bias != nullptr || partial_tile) {
            const float inv_cap = a.softcap > 0.f ? 1.f / a.softcap : 0.f;
            typedef float f32x4_dword_aligned __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                f32x4 bq[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int v0 = m0 + fwd_row(wm, mb, q * 4, lane);
                    bq[q] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (a.bias != nullptr) {
                        if (v0 + 3 < a.V) {
                            bq[q] = *reinterpret_cast<const f32x4_dword_aligned*>(a.bias + v0);
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (v0 + i < a.V) bq[q][i] = a.bias[v0 + i];
                        }
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int v0 = m0 + fwd_row(wm, mb, q * 4, lane);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const bool beyond = partial_tile && v0 + i >= a.V;
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) {
                            float y = acc[mb][nb][q * 4 + i] + bq[q][i];
                            if constexpr (GENERAL) {
                                y *= a.logit_scale;
                                if (a.softcap > 0.f) y = head_tanh(y * inv_cap) * a.softcap;
                                y *= a.inv_t;
                            }
                            acc[mb][nb][q * 4 + i] = beyond ? -INFINITY : y;
                        }
                    }
                }
            }
        }
        // (With a stash the numerators are stored as they are produced.  Packed into registers and stored in one run
        // at the end of the epilogue they cost more: 28.6 against 27.8 ms for the benchmark's forward.)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float bm = -INFINITY;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) bm = fmaxf(bm, acc[mb][nb][r]);
            if constexpr (plain) bm *= zs;
            // target logit: rarely inside this wave's 128 vocabulary rows.  It is selected into one register
            // and stored once: a conditional store per accumulator held the wave for about 20 us, and a
            // workgroup that falls behind the others no longer finds the tiles they share in the L2.
            const int rel = tg[nb] - (m0 + wm * WM);
            if (tg[nb] >= 0 && rel >= 0 && rel < WM) {
                const int want = rel - half * 4;  // fwd_row() without this lane's half-wave offset
                float tv = 0.f;
                bool mine = false;
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const bool m = (mb * 32 + (r >> 2) * 8 + (r & 3)) == want;
                        tv = m ? acc[mb][nb][r] : tv;
                        mine |= m;
                    }
                if (mine) a.tgt[n0 + fwd_col(wn, nb, lane)] = plain ? tv * zs : tv;
            }
            zmax[nb] = fmaxf(zmax[nb], bm);
            const float need = ceilf(bm * kLog2e);
            if (need > ref[nb]) {
                const float sc = fast_exp2(ref[nb] - need);
                S[nb] *= sc;
                U[nb] *= sc;
                ref[nb] = need;
            }
            const float rr = ref[nb] == -INFINITY ? 0.f : ref[nb];
            // numerators times 2^15 (exact; S and U carry the factor until they are written out), with or without a
            // stash: the outputs must not depend on stashing
            int64_t stash_off = nb * 32 * 8;  // byte offset of this token block's column of quads (uniform)
            if constexpr (STASH) ref_blk[nb * 32 + ref_lane] = rr;
            const float rsub = rr - kStashExp;
            float s = 0.f, u = 0.f;
            auto sum_tile = [&](auto guard_tag) {
                constexpr bool kGuard = decltype(guard_tag)::value;  // -inf among the logits (0 * -inf in sum(e * y))
                const float mul = plain ? zs2 : kLog2e;  // general path: the accumulators hold z itself by now
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float e[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float y = acc[mb][nb][q * 4 + i];
                            e[i] = fast_exp2(fmaf(y, mul, -rsub));
                            s += e[i];
                            u = (kGuard && y == -INFINITY) ? u : fmaf(e[i], y, u);
                        }
                        if constexpr (STASH) {
                            uint2 w;
                            w.x = Elem<TRLK_F16>::pack2(e[0], e[1]);
                            w.y = Elem<TRLK_F16>::pack2(e[2], e[3]);
                            *reinterpret_cast<uint2*>(stash_blk + stash_off + stash_lane) = w;
                            stash_off += a.stash.ld * 16;  // two quads down: the other parity is the other half-wave's
                            // (one running offset, not 16 precomputed ones; an offset, because a pointer that
                            // passed through here would no longer be known to point to global memory)
                            asm volatile("" : "+s"(stash_off));
                        }
                    }
            };
            if (GENERAL || partial_tile)
                sum_tile(std::true_type{});
            else
                sum_tile(std::false_type{});
            if constexpr (plain) u *= zs;
            S[nb] += s;
            U[nb] += u;
        }
    }

    // merge the partial states of every token (2 lane halves x WGM M-waves) through LDS
    const int lane = tid & 63;
    constexpr int kParts = 2 * WGM;
    float* sm = reinterpret_cast<float*>(smem);  // [kParts][BN tokens][4]
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int col = fwd_col(wn, nb, lane);
        const int part = wm * 2 + (lane >> 5);
        // (copies of their own: joined to a 16-byte store's registers, the state would be kept as vectors through the whole
        // tile loop, and spilled)
        float r, z;
        asm volatile("v_mov_b32 %0, %2\n\tv_mov_b32 %1, %3" : "=&v"(r), "=v"(z) : "v"(ref[nb]), "v"(zmax[nb]));
        *reinterpret_cast<f32x4*>(sm + (part * BN + col) * 4) = f32x4{r, S[nb] * 0x1p-15f, U[nb] * 0x1p-15f, z};
    }
    __syncthreads();
    if (tid < BN && n0 + tid < a.N) {
        float R = -INFINITY;
        float zm = -INFINITY;
        for (int p = 0; p < kParts; ++p) {
            R = fmaxf(R, sm[(p * BN + tid) * 4]);
            zm = fmaxf(zm, sm[(p * BN + tid) * 4 + 3]);
        }
        float s = 0.f, u = 0.f;
        for (int p = 0; p < kParts; ++p) {
            const float* src = sm + (p * BN + tid) * 4;
            const float sc = (src[0] == -INFINITY) ? 0.f : fast_exp2(src[0] - R);
            s += src[1] * sc;
            u += src[2] * sc;
        }
        float* out = a.partial + (int64_t(n0 + tid) * a.v_splits + vs) * 4;
        out[0] = R;
        out[1] = s;
        out[2] = u;
        out[3] = zm;
    }
}

__global__ void head_fill_kernel(float* p, int64_t n, float v) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Merges the vocabulary splits of every token: logp, entropy, log_z.  One wave per token, lane s on splits s, s + 64, ...:
// bound by the latency of a couple of dependent loads (a token's partials are one contiguous piece of memory), where a
// thread per token walked the splits one after the other with the grid nearly empty: 459 tokens x 119 splits 40 -> 4.7 us.
constexpr int kMergeTokens = 4;  // tokens per workgroup
__global__ __launch_bounds__(kMergeTokens * kWave) void head_merge_kernel(
    const float* partial, const float* tgt, const int64_t* targets, int N, int V, int v_splits, float* logp, float* entropy,
    float* log_z, float* target_is_max, int32_t* error_flag, float* stash_zt) {
    const int n = blockIdx.x * kMergeTokens + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (n >= N) return;
    const f32x4* p = reinterpret_cast<const f32x4*>(partial) + int64_t(n) * v_splits;
    float R = -INFINITY, S = 0.f, U = 0.f, zm = -INFINITY;
    for (int s = lane; s < v_splits; s += kWave) {
        const f32x4 q = p[s];
        zm = fmaxf(zm, q[3]);
        const float r = fmaxf(R, q[0]);
        const float keep = R == -INFINITY ? 0.f : fast_exp2(R - r), add = q[0] == -INFINITY ? 0.f : fast_exp2(q[0] - r);
        S = S * keep + q[1] * add;  // (the references are integers: the factors are powers of two)
        U = U * keep + q[2] * add;
        R = r;
    }
    const float r = wave_max(R), sc = R == -INFINITY ? 0.f : fast_exp2(R - r);
    R = r;
    S = wave_sum(S * sc);
    U = wave_sum(U * sc);
    zm = wave_max(zm);
    if (lane != 0) return;
    constexpr float kLn2Hi = 0.693145751953125f, kLn2Lo = 1.42860677e-06f;
    const float lz = fmaf(R, kLn2Hi, fmaf(R, kLn2Lo, logf(S)));
    const int64_t t = targets[n];
    float lp;
    if (t < 0 || t >= V) {
        lp = NAN;
        if (error_flag) atomicOr(error_flag, TRLK_FLAG_INDEX_OUT_OF_RANGE);
    } else {
        lp = tgt[n] - lz;
    }
    logp[n] = lp;
    if (stash_zt) stash_zt[n] = tgt[n];
    entropy[n] = lz - U / S;
    log_z[n] = lz;
    // 1 if the target holds the row maximum, i.e. argmax(logits) == target up to ties
    if (target_is_max) target_is_max[n] = (t >= 0 && t < V && tgt[n] >= zm) ? 1.f : 0.f;
}

// dz pass of the backward: one 256 (vocabulary) x 256 (tokens) tile per workgroup.
template <int DT>
TRLK_HEAD_KERNEL void fused_head_dz_kernel(HeadArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int n_tb = (a.N + BN - 1) / BN;
    const int n_vt = (a.c1 - a.c0 + BM - 1) / BM;
    int tb, vt;
    xcd_patch(blockIdx.x, n_tb, n_vt, tb, vt);
    if (tb >= n_tb || vt >= n_vt) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave_m(wave), wn = wave_n(wave);
    const int n0 = tb * BN, m0 = a.c0 + vt * BM;
    const Operand W{a.weight, a.ldw, a.V}, Hd{a.hidden, a.ldh, a.N};
    f32x4 acc[MI][NI];
    gemm_tile_nt<DT>(W, m0, Hd, n0, a.H, acc, smem);

    // Common case (no soft-capping, tile inside the chunk): dz = -(g * chain) * exp2(y * zs2 - lzc)
    // with one scale folded into the exponent; the target's one-hot term is patched afterwards.
    const float zs = a.logit_scale * a.inv_t, zs2 = zs * kLog2e;
    const bool plain = a.softcap <= 0.f && m0 + BM <= a.c1 && a.bias == nullptr;
    typedef Elem<TRLK_F16> EO;  // storage of dz
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int tok = n0 + acc_col(wn, j, lane);
        const bool tok_ok = tok < a.N;
        const float g = tok_ok ? a.g[tok] * pow2_scale(fabsf(a.g[tok]) * zs) : 0.f;  // g carries the token's scale
        const float lzc = tok_ok ? a.log_z[tok] * kLog2e : INFINITY;  // rows beyond N: exp2(-inf) = 0
        const int64_t tg = tok_ok ? a.targets[tok] : -1;
        const int64_t rel = tg - (m0 + wm * WM);  // target row relative to this wave's rows
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            f32x4 d;
            if (plain) {
                const float ngc = -g * zs;
#pragma unroll
                for (int r = 0; r < 4; ++r) d[r] = ngc * fast_exp2(fmaf(acc[i][j][r], zs2, -lzc));
                if (rel >= i * 16 && rel < i * 16 + 16) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (acc_row(0, i, r, lane) == int(rel)) d[r] -= ngc;
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int v = m0 + acc_row(wm, i, r, lane);
                    float y = acc[i][j][r];
                    if (a.bias != nullptr && v < a.c1) y += a.bias[v];
                    y *= a.logit_scale;
                    float chain = a.inv_t * a.logit_scale;
                    if (a.softcap > 0.f) {
                        const float th = head_tanh(y / a.softcap);
                        y = th * a.softcap;
                        chain *= 1.f - th * th;
                    }
                    const float z = y * a.inv_t;
                    const float p = fast_exp2(fmaf(z, kLog2e, -lzc));
                    float dzv = -g * p;
                    if (v == tg) dzv += g;
                    d[r] = (v < a.c1 && tok_ok) ? dzv * chain : 0.f;
                }
            }
            acc[i][j] = d;
        }
    }
    // dz^T [chunk row][token]: the lanes of a block hold consecutive tokens of one vocabulary row.
    // Neighbouring lanes swap one value each, so that the even lane owns two tokens of row r and
    // the odd lane two tokens of row r + 1; the 4-byte pieces are staged as a [vocabulary][token]
    // tile in LDS and leave as 512-byte runs.
    constexpr int kChunksPerRow = BN / 8;  // 16-byte pieces per row of the staged tile
    const int odd = lane & 1;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int tcol = (acc_col(wn, j, lane) & ~1) * 2;  // byte offset of the token pair inside a staged row
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const float mine0 = acc[i][j][r], mine1 = acc[i][j][r + 1];
                const float give = odd ? mine0 : mine1;
                const float got = __builtin_bit_cast(
                    float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, give), 0xB1 /* quad_perm 1,0,3,2 */, 0xf, 0xf, true));
                const uint32_t w = odd ? EO::pack2(got, mine1) : EO::pack2(mine0, got);
                const int vrow = acc_row(wm, i, r, lane) + odd;
                *reinterpret_cast<uint32_t*>(smem + vrow * kDzLdsRow + tcol) = w;
            }
    }
    __syncthreads();
#pragma unroll 4
    for (int c = tid; c < BM * kChunksPerRow; c += kHeadThreads) {
        const int vrow = c / kChunksPerRow, tc = c % kChunksPerRow;  // chunk-local row (padding rows are written as 0)
        *reinterpret_cast<u32x4*>(a.dzT + int64_t(vt * BM + vrow) * a.ldzt + n0 + tc * 8) =
            *reinterpret_cast<const u32x4*>(smem + vrow * kDzLdsRow + tc * 16);
    }
}

// dz pass of the backward from the forward's stashed softmax numerators instead of a recompute: an
// elementwise sweep (memory bound: 2 bytes read, 2 bytes written per logit, one multiplication each).
// One workgroup = 128 vocabulary rows x 256 tokens.  A lane owns two pairs of tokens, a wave 32 rows = 8 row quads
// whose 16 loads (16 bytes each: 2 tokens x 4 rows) are all issued before the first result is used.
// dz^T (vocabulary-major, like the stash) is written in place, each token's column in that token's own scale.
// Rows beyond the chunk and tokens beyond N are written as zeros.
constexpr int kSdzRows = 128, kSdzTokens = 256, kSdzQuads = kSdzRows / 4 / 4;  // quads per wave
// COLS: the tokens were compacted since the forward, a.stash_cols maps them to their stash columns.
// CAPPED: soft-capped head (the chain factor needs the logit: a logarithm per numerator); a kernel of its own, so that
// the usual sweep is straight-line code.
template <bool COLS, bool CAPPED>
__global__ __launch_bounds__(256) void head_dz_from_stash_kernel(HeadArgs a) {
    typedef Elem<TRLK_F16> E;  // the numerators and dz are fp16
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // consecutive tiles take consecutive token blocks of one row group: the stash rows they read and the
    // dz^T rows they write are then neighbours in memory.  Consecutive workgroups go to the eight XCDs in turn:
    // each XCD walks one contiguous eighth of the tiles.
    const int per_xcd = int(gridDim.x) >> 3;  // (the grid is a multiple of 8)
    const int tile = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
    if (tile >= a.sdz_tiles) return;
    const int n0 = (tile % a.sdz_token_blocks) * kSdzTokens, r0 = (tile / a.sdz_token_blocks) * kSdzRows;  // r0: chunk-local row
    const int rows = a.c1 - a.c0;
    const float zs = a.logit_scale * a.inv_t;
    const int64_t ld = a.stash.ld;
    // A lane owns two pairs of neighbouring tokens, 128 apart: every load instruction of the wave then reads 1 KiB of
    // one stash row without gaps (16 bytes = 2 tokens x 4 rows per lane), every store 256 contiguous bytes of a dz row.
    const int tl[4] = {lane * 2, lane * 2 + 1, 128 + lane * 2, 128 + lane * 2 + 1};
    float ngc[4], lzc[4];  // -g * zs in the token's own scale; log_z in base 2
    int tg[4], col[4];     // chunk-local target row (or -1); stash column
    bool live[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int tok = n0 + tl[j];
        const bool ok = tok < a.N;
        col[j] = ok ? (COLS ? a.stash_cols[tok] : tok) : -1;
        const float g = ok ? a.g[tok] : 0.f;
        live[j] = g != 0.f;
        ngc[j] = -g * pow2_scale(fabsf(g) * zs) * zs;
        lzc[j] = ok ? a.log_z[tok] * kLog2e : INFINITY;
        const int64_t t = ok ? a.targets[tok] - a.c0 : -1;
        tg[j] = (t >= 0 && t < rows) ? int(t) : -1;
    }
    // (tokens beyond N of the last block are inside the padded row)
    const bool pair0 = !COLS || (col[0] >= 0 && col[1] == col[0] + 1), pair1 = !COLS || (col[2] >= 0 && col[3] == col[2] + 1);
    const int c0 = COLS ? col[0] : n0 + tl[0], c2 = COLS ? col[2] : n0 + tl[2];
    // the numerators of the wave's 8 quads
    const int row_w = r0 + wave * (kSdzRows / 4);                         // chunk-local first row of the wave
    const uint2* qrow = a.stash.quads() + int64_t((a.c0 + row_w) / 4) * ld;  // (chunks and tiles start on whole 128-row blocks)
    uint2 eb[kSdzQuads][4];
#pragma unroll
    for (int qi = 0; qi < kSdzQuads; ++qi) {
        const uint2* src = qrow + int64_t(qi) * ld;
        typedef uint32_t u32x4_8 __attribute__((ext_vector_type(4), aligned(8)));
        if (pair0) {
            const u32x4_8 lo = __builtin_nontemporal_load(reinterpret_cast<const u32x4_8*>(src + c0));
            eb[qi][0] = make_uint2(lo.x, lo.y);
            eb[qi][1] = make_uint2(lo.z, lo.w);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) eb[qi][j] = col[j] >= 0 ? src[col[j]] : make_uint2(0u, 0u);
        }
        if (pair1) {
            const u32x4_8 hi = __builtin_nontemporal_load(reinterpret_cast<const u32x4_8*>(src + c2));
            eb[qi][2] = make_uint2(hi.x, hi.y);
            eb[qi][3] = make_uint2(hi.z, hi.w);
        } else {
#pragma unroll
            for (int j = 2; j < 4; ++j) eb[qi][j] = col[j] >= 0 ? src[col[j]] : make_uint2(0u, 0u);
        }
    }
    // reference exponents of the two quad parities -> the factor that turns a numerator into -g * zs * p
    const float* refs = a.stash.refs() + int64_t((a.c0 + row_w) / 128) * 2 * ld;
    float rf[2][4], pf[2][4];  // p = e * pf
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int cj = COLS ? col[j] : n0 + tl[j];
            rf[h][j] = (COLS && cj < 0) ? 0.f : refs[int64_t(h) * ld + cj];
            pf[h][j] = fast_exp2(rf[h][j] - kStashExp - lzc[j]);
        }
    constexpr bool capped = CAPPED;
    float zt[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (capped) {
#pragma unroll
        for (int j = 0; j < 4; ++j) zt[j] = col[j] >= 0 ? a.stash.zt()[col[j]] : 0.f;
    }
    const float th_mul = capped ? 1.f / (a.inv_t * a.softcap) : 0.f;  // tanh(.) of a soft-capped logit = z * T / cap
#pragma unroll
    for (int qi = 0; qi < kSdzQuads; ++qi) {
        const int h = qi & 1;  // (the wave's first quad is even)
        float e[4][4];         // [token][row of the quad]
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            E::unpack2(eb[qi][j].x, &e[j][0]);
            E::unpack2(eb[qi][j].y, &e[j][2]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = row_w + qi * 4 + i;
            float d[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float p = e[j][i] * pf[h][j];
                float dv;
                if constexpr (!capped) {
                    dv = ngc[j] * p;
                    if (tg[j] == row) dv -= ngc[j];
                } else {
                    // z from the numerator (a flushed one has p = 0 and, unless it is the target, no gradient)
                    const bool is_t = tg[j] == row;
                    const float z = is_t ? zt[j] : (__log2f(e[j][i]) - kStashExp + rf[h][j]) * kLn2;
                    const float th = z * th_mul;
                    dv = ngc[j] * (is_t ? p - 1.f : p) * (1.f - th * th);
                    if (!is_t && e[j][i] == 0.f) dv = 0.f;
                }
                d[j] = (row < rows && live[j]) ? dv : 0.f;
            }
            // (non-temporal: 2 GB per chunk that no cache holds until the products read it)
            uint32_t* out = reinterpret_cast<uint32_t*>(a.dzT + int64_t(row) * a.ldzt + n0);
            __builtin_nontemporal_store(E::pack2(d[0], d[1]), out + lane);
            __builtin_nontemporal_store(E::pack2(d[2], d[3]), out + 64 + lane);
        }
    }
}

// Plain NT product with an output epilogue: C[M, N] (+)= A[M, K] * B[N, K]^T.
//   MODE 0: store to `out_lp` in the storage dtype.
//   MODE 1: fp32 accumulate into `out_f32` (first = overwrite).
//   MODE 2: like 1 but the sum is rounded into `out_lp` instead of being written back (last chunk).
//   The accumulators are multiplied by 1 / (scale of A * scale of B) first: the scales are powers of two derived from
//   the maxima in `max_a` (times `mult_a`) and `max_b` (null = 1), and, when `g_rows` is given, row m of A carries its
//   own scale pow2_scale(|g_rows[m]| * mult_a) instead of the common one.
// The tile is computed transposed (B is the tile loop's left operand): a lane then holds 4 consecutive columns of one row.
struct GemmArgs {
    Operand A, B;
    int M, N, K;
    float* out_f32;
    int64_t ld_f32;
    uint16_t* out_lp;
    int64_t ld_lp;
    int first;
    const uint32_t* max_a;
    const uint32_t* max_b;
    const uint32_t* beyond_b;  // B is the weight: max_b and this are the two slots of weight_scale()
    // B is the weight itself, [b_krows, N] as it lies in memory, not a transposed copy (bf16: converted on its way, see
    // direct_scale; *beyond_out becomes 1 where fp16 does not hold all of it).
    int b_krows;
    uint32_t* beyond_out;
    const float* g_rows;
    float mult_a;
    // K-major A, epilogue 1: the contraction cut into `slices` pieces of `kslice` (a multiple of the k step), each
    // with its own fp32 sum at out_f32 + slice * M * ld_f32.  The slices are further columns of the tile grid, so that an
    // XCD works on few of them: its tiles of one slice share their slabs of both operands.
    int slices, kslice;
};

// DT: dtype of the operands (the matrix-core instruction), ODT: storage dtype of `out_lp`.
// AKM: A is given k-major ([K, M], leading dimension A.ld).  BW: B is the weight in its own layout and dtype (ODT).
template <int DT, int MODE, int ODT, bool AKM = false, bool BW = false>
__device__ __forceinline__ void gemm_nt_body(const GemmArgs& a, int block, char* smem) {
    typedef Elem<ODT> E;
    const int n_mt = (a.M + BN - 1) / BN, n_nt = (a.N + BM - 1) / BM;
    Operand A = a.A, B = a.B;
    int K = a.K, b_krows = a.b_krows;
    float* out_f32 = a.out_f32;
    constexpr bool kSlices = AKM && MODE == 1;
    const int n_cols = kSlices ? n_nt * a.slices : n_nt;
    int tm, tn;
    xcd_patch(block, n_mt, n_cols, tm, tn);
    if (tm >= n_mt || tn >= n_cols) return;
    if constexpr (kSlices) {
        const int slice = tn / n_nt, k0 = slice * a.kslice;
        tn -= slice * n_nt;
        A.p += int64_t(k0) * A.ld;
        B.p += BW ? int64_t(k0) * B.ld : int64_t(k0);
        b_krows -= k0;
        K = min(a.kslice, K - k0);
        out_f32 += int64_t(slice) * a.M * a.ld_f32;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave_m(wave), wn = wave_n(wave);
    const int r0 = tm * BN, c0 = tn * BM;  // the tile's first row and column of the output
    f32x4 acc[MI][NI];
    const bool idle = r0 + wn * WN >= a.M || c0 + wm * WM >= a.N;  // all of this wave's rows or columns lie beyond the output
    float inv_b;
    if constexpr (BW) {
        constexpr bool kConvert = ODT == TRLK_BF16;
        const float scale = uniform(kConvert ? direct_scale(a.max_b) : 1.f);
        typedef LeftKm<kConvert> Left;
        Left left(B, c0, b_krows, scale, smem);
        if (idle)
            move_tiles_only<true, false, Left&>(DirectLoader<true, false>(B, c0, A, r0, smem), K, false, left);
        else
            gemm_tile_nt<DT, true>(B, c0, A, r0, K, acc, smem, left);
        if (kConvert && __any(left.top > kF16Max) && lane == 0)
            __hip_atomic_store(a.beyond_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (idle) return;  // (no barrier follows)
        inv_b = 1.f / scale;
    } else {
        if (idle && (AKM || (K & (BK - 1)) == 0))
            return move_tiles_only(DirectLoader<AKM>(B, c0, A, r0, smem), K, false);
        gemm_tile_nt<DT, AKM>(B, c0, A, r0, K, acc, smem);
        if (idle) return;  // (no barrier follows)
        inv_b = 1.f / (a.beyond_b != nullptr ? weight_scale(a.max_b, a.beyond_b).scale : slot_scale(a.max_b, 1.f));
    }
    const float inv_common = inv_b / slot_scale(a.max_a, a.mult_a);
    const int g = lane >> 4;
    // The wave's 128 columns inside the output (nearly every tile), rows aligned for vector accesses: a row's 8 running
    // sums of 16 bytes are loaded before the first is used, its results stored in one run.  (Written per element with a
    // bounds test each, the compiler lost count of the loads in flight and waited for EVERYTHING outstanding before each
    // accumulate, i.e. for the previous store's acknowledgement: 128 store round trips per tile.)
    const bool f32_ok = MODE == 0 || ((reinterpret_cast<uintptr_t>(out_f32) & 15) == 0 && (a.ld_f32 & 3) == 0);
    const bool lp_ok = MODE == 1 || ((reinterpret_cast<uintptr_t>(a.out_lp) & 15) == 0 && (a.ld_lp & 7) == 0);
    const bool fast = c0 + (wm + 1) * WM <= a.N && f32_ok && lp_ok;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int row = r0 + acc_col(wn, j, lane);
        if (row >= a.M) continue;
        const float inv = a.g_rows != nullptr ? inv_b / pow2_scale(fabsf(a.g_rows[row]) * a.mult_a) : inv_common;
        if (fast) {
            f32x4 v[MI];
            if constexpr (MODE != 0) {
                float* out = out_f32 + int64_t(row) * a.ld_f32 + (c0 + acc_row(wm, 0, 0, lane));
                f32x4 prev[MI];
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    prev[i] = a.first ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(out + i * 16);
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[i][r] = fmaf(acc[i][j][r], inv, prev[i][r]);
                if constexpr (MODE == 1) {
#pragma unroll
                    for (int i = 0; i < MI; ++i) *reinterpret_cast<f32x4*>(out + i * 16) = v[i];
                }
            } else {
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[i][r] = acc[i][j][r] * inv;
            }
            if constexpr (MODE != 1) {
                // 16-bit outputs: of two neighbouring blocks the lane groups 0, 2 take the first and 1, 3 the second, 8
                // consecutive columns (16 bytes) per lane, 64 contiguous bytes per row and store
                typename E::type* out = a.out_lp + int64_t(row) * a.ld_lp + (c0 + wm * WM + (g & 1) * 16 + (g >> 1) * 8);
#pragma unroll
                for (int i = 0; i < MI; i += 2) {
                    const auto lo = __builtin_amdgcn_permlane16_swap(E::pack2(v[i][0], v[i][1]), E::pack2(v[i + 1][0], v[i + 1][1]),
                                                                     false, false);
                    const auto hi = __builtin_amdgcn_permlane16_swap(E::pack2(v[i][2], v[i][3]), E::pack2(v[i + 1][2], v[i + 1][3]),
                                                                     false, false);
                    *reinterpret_cast<u32x4*>(out + i * 16) = u32x4{lo[0], hi[0], lo[1], hi[1]};
                }
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int col = c0 + acc_row(wm, i, r, lane);
                if (col >= a.N) continue;
                const float prev = (MODE != 0 && !a.first) ? out_f32[int64_t(row) * a.ld_f32 + col] : 0.f;
                const float v = fmaf(acc[i][j][r], inv, prev);
                if (MODE == 1)
                    out_f32[int64_t(row) * a.ld_f32 + col] = v;
                else
                    E::store1(a.out_lp + int64_t(row) * a.ld_lp + col, v);
            }
    }
}

// Two independent products in one launch: workgroups [0, grid_a) take `a` (epilogue MODE_A; its left operand is
// k-major), the rest take `b` (epilogue 0).  When the tile count of one product is not a multiple of the CU count, the other product's
// tiles fill the CUs its last round leaves idle.  grid_a is a multiple of 8 (the XCD mapping of `b` is kept).
template <int MODE_A, int ODT, bool BW>
TRLK_HEAD_KERNEL void gemm_nt_pair_kernel(GemmArgs a, int grid_a, GemmArgs b) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    if (int(blockIdx.x) < grid_a)
        gemm_nt_body<TRLK_F16, MODE_A, ODT, true, BW>(a, blockIdx.x, smem);
    else
        gemm_nt_body<TRLK_F16, 0, ODT>(b, int(blockIdx.x) - grid_a, smem);
}

__device__ __forceinline__ uint32_t max_bits(uint32_t m, u32x4 q) {  // of the 8 bf16 in q, as fp32 bit patterns
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max(m, max((q[i] << 16) & 0x7fff0000u, q[i] & 0x7fff0000u));
    return m;
}

// The rows of a weight in which entries exceed fp16 in the scale of direct_scale, a bit each: returns at once where the product
// met none.  Bound by the read of the weight where it did.  One workgroup per CU, which makes a launch with nothing to do cheap.
constexpr int kBeyondThreads = 1024, kBeyondBlocks = 256;
__global__ __launch_bounds__(kBeyondThreads) void beyond_rows_kernel(const uint16_t* w, int64_t ld, int rows, int cols8,
                                                                     const uint32_t* sample, const uint32_t* any,
                                                                     uint32_t* row_bits) {
    if (*any == 0u) return;
    const float scale = direct_scale(sample);
    const int lane = threadIdx.x & (kWave - 1), step = int(gridDim.x) * (kBeyondThreads / kWave);
    for (int row = blockIdx.x * (kBeyondThreads / kWave) + threadIdx.x / kWave; row < rows; row += step) {
        const u32x4* p = reinterpret_cast<const u32x4*>(w + int64_t(row) * ld);
        uint32_t m = 0;
#pragma unroll 4
        for (int c = lane; c < cols8; c += kWave) m = max_bits(m, p[c]);
        if (__any(__uint_as_float(m) * scale > kF16Max) && lane == 0) atomicOr(row_bits + (row >> 5), 1u << (row & 31));
    }
}

// What the dHidden product left out of a weight that it converted itself: sum over v of dz[v, n] * (w[v, h] -+ kF16Max / scale) over
// the entries that exceed fp16, in fp32 and in the order of the rows.
struct BeyondArgs {
    const uint32_t* any;       // null: the product left nothing out
    const uint32_t* row_bits;  // see beyond_rows_kernel
    const uint32_t* sample;
    const uint16_t *weight, *dzt;
    int64_t ldw, ldzt;
    const float* g;
    float zs;
    int n_words, H;
};
constexpr int kSumThreads = 256;
// Adds it for the 8 outputs from i on (token i / H); every lane of the workgroup takes part.  8192 rows at a time: their numbers
// are put in a list in LDS, eight of them are in flight (sixteen take no less time, and their registers leave the launch with no such
// rows four waves per SIMD: 7.4 for 7.0 us).  Whole backward, weight of deviation 0.02 -> one entry of 50 -> 300 rows times 100 (a
// sample of 1/32 of the rows misses all of 300 once in 1e4 weights): 1396 tokens, H = 2048, V = 50257 715 -> 690 -> 837 us; 1392
// tokens, V = 128256 1578 -> 1640 -> 1727; 459 tokens, H = 3584, V = 151936 1241 -> 1415 -> 1520; 64 tokens, H = 1024, V = 32000 100 ->
// 112 -> 163.  With the whole product done again in another scale, one entry: 1029, 2590, 1967 and 124 us.
__device__ __forceinline__ void add_beyond(const BeyondArgs& b, int64_t i, bool live, float (&x)[8]) {
    constexpr int kInFlight = 8;
    __shared__ uint16_t list[32 * kSumThreads];
    __shared__ int counts[kSumThreads / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const float most = kF16Max / direct_scale(b.sample);
    const int n = live ? int(i / b.H) : 0, h = live ? int(i - int64_t(n) * b.H) : 0;
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int w0 = 0; w0 < b.n_words; w0 += kSumThreads) {
        uint32_t bits = w0 + tid < b.n_words ? b.row_bits[w0 + tid] : 0u;
        const int mine = __popc(bits);
        int at = mine;  // inclusive sum over the wave's lanes
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int below = __shfl_up(at, o);
            if (lane >= o) at += below;
        }
        if (lane == kWave - 1) counts[wave] = at;
        __syncthreads();
        at -= mine;
        int total = 0;
#pragma unroll
        for (int k = 0; k < kSumThreads / kWave; ++k) {
            if (k < wave) at += counts[k];
            total += counts[k];
        }
        for (; bits != 0u; bits &= bits - 1u) list[at++] = uint16_t(tid * 32 + __ffs(bits) - 1);
        __syncthreads();
        for (int k0 = 0; k0 < total; k0 += kInFlight) {
            int at[kInFlight];
            uint16_t dz[kInFlight];
            u32x4 row[kInFlight];
#pragma unroll
            for (int k = 0; k < kInFlight; ++k) at[k] = list[min(k0 + k, total - 1)];  // (beyond the last one: the last one, times 0)
#pragma unroll
            for (int k = 0; k < kInFlight; ++k) {
                dz[k] = b.dzt[int64_t(w0 * 32 + at[k]) * b.ldzt + n];
                row[k] = *reinterpret_cast<const u32x4*>(b.weight + int64_t(w0 * 32 + at[k]) * b.ldw + h);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < kInFlight; ++k) {
                const float d = k0 + k < total ? Elem<TRLK_F16>::to_float(dz[k]) : 0.f;
                float w[8];
                Elem<TRLK_BF16>::unpack(row[k], w);
#pragma unroll
                for (int q = 0; q < 8; ++q)  // (0 for an entry that fp16 holds)
                    sum[q] = fmaf(d, w[q] - __builtin_amdgcn_fmed3f(w[q], -most, most), sum[q]);
            }
        }
        __syncthreads();  // (the next rows overwrite the list)
    }
    const float inv = live ? 1.f / pow2_scale(fabsf(b.g[n]) * b.zs) : 0.f;  // (token n's d logits are in its own scale)
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = fmaf(sum[q], inv, x[q]);
}

// dHidden from the sums of the slices of its contraction, in slice order: out[i] = sum_s parts[s][i], 8 values per lane
// (n is a multiple of 8), and what the product left out.
template <int ODT>
__global__ __launch_bounds__(kSumThreads) void sum_slices_kernel(const float* parts, int slices, int64_t n, uint16_t* out,
                                                                 BeyondArgs beyond) {
    const int64_t i = (int64_t(blockIdx.x) * kSumThreads + threadIdx.x) * 8;
    const bool live = i < n;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (live)
        for (int s = 0; s < slices; ++s) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(parts + s * n + i);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(parts + s * n + i + 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                x[k] += lo[k];
                x[4 + k] += hi[k];
            }
        }
    if constexpr (ODT == TRLK_BF16)
        if (beyond.any != nullptr && *beyond.any != 0u) add_beyond(beyond, i, live, x);
    if (live) *reinterpret_cast<u32x4*>(out + i) = Elem<ODT>::pack(x);
}

// A single product (epilogue 1: fp32 output, overwritten or accumulated into).
template <int DT>
TRLK_HEAD_KERNEL void gemm_nt_kernel(GemmArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    gemm_nt_body<DT, 1, DT>(a, blockIdx.x, smem);
}

// fp32 [R, C] (row stride ld) -> bf16 [R, 6 * cpad] (row stride ldo, cpad = C rounded up to 8, padding zero): the three
// bf16 pieces x = p0 + p1 + p2 (p0 = bf16(x), p1 = bf16(x - p0), p2 = bf16(x - p0 - p1); 24 significant bits in all,
// with the exponent range of fp32) laid out along the contraction axis so that an NT product of an "A side" and a
// "B side" matrix sums the six piece products that matter, smallest first:
//   slot        0      1      2      3      4      5
//   A side      p2     p1     p0     p1     p0     p0
//   B side      p0     p1     p2     p0     p1     p0      (p1*p2, p2*p1, p2*p2 are below fp32 rounding: dropped)
__global__ __launch_bounds__(256) void split_bf16x3_kernel(const float* in, int64_t ld, int64_t R, int C, int cpad, int side,
                                                           uint16_t* out, int64_t ldo) {
    typedef Elem<TRLK_BF16> E;
    const int64_t r = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (r >= R || c >= cpad) return;
    float p[3] = {0.f, 0.f, 0.f};
    if (c < C) {
        const float x = in[r * ld + c];
        uint16_t h;
        E::store1(&h, x);
        p[0] = E::to_float(h);
        const float r1 = x - p[0];
        E::store1(&h, r1);
        p[1] = E::to_float(h);
        E::store1(&h, r1 - p[1]);
        p[2] = E::to_float(h);
    }
    const int a_map[6] = {2, 1, 0, 1, 0, 0}, b_map[6] = {0, 1, 2, 0, 1, 0};
    uint16_t* o = out + r * ldo + c;
#pragma unroll
    for (int sl = 0; sl < 6; ++sl) E::store1(o + int64_t(sl) * cpad, p[side == 0 ? a_map[sl] : b_map[sl]]);
}

// Largest magnitudes of the backward's operands in one launch: out[0] of the fp32 vector g [n_g], out[1] of hidden, out[2]
// of a sample of the weight's rows (bf16 matrices of C8 * 8 columns; no workgroups are launched for them in an
// fp16 problem), as the bit patterns of those floats (non-negative floats order like unsigned integers; the caller clears
// `out`).
//
// Bound by the read of hidden and of the sample.  Workgroups of 1024 lanes, at most two per CU for a matrix, eight 16-byte
// loads in flight per lane, one atomic per workgroup and only when it would raise the maximum: atomics on one address
// retire about one per 15 ns, so one per wave of 4096 small workgroups took 250 us whatever the size of the matrix.
constexpr int kMaxThreads = 1024, kMaxBlocks = 512;
struct MaxAbsArgs {
    const float* g;
    int64_t n_g;
    const uint16_t *hidden, *weight;
    int64_t ld_hidden, ld_weight;
    int n_hidden, n_weight, C8;         // rows (of the weight those in the sample); 16-byte vectors per row
    int vocab;
    int blocks_g, blocks_h, blocks_w;   // workgroups of each
    uint32_t* out;
};
__global__ __launch_bounds__(kMaxThreads) void head_maxabs_kernel(MaxAbsArgs a) {
    __shared__ uint32_t part[kMaxThreads / kWave];
    int block = blockIdx.x, slot;
    uint32_t m = 0;
    if (block >= a.blocks_w + a.blocks_h) {
        slot = 0;
        block -= a.blocks_w + a.blocks_h;
        for (int64_t i = int64_t(block) * kMaxThreads + threadIdx.x; i < a.n_g; i += int64_t(a.blocks_g) * kMaxThreads)
            m = max(m, __float_as_uint(a.g[i]) & 0x7fffffffu);
    } else {
        const bool is_w = block < a.blocks_w;
        slot = is_w ? 2 : 1;
        const int blocks = is_w ? a.blocks_w : a.blocks_h;
        block -= is_w ? 0 : a.blocks_w;
        const uint16_t* in = is_w ? a.weight : a.hidden;
        const int64_t ld = is_w ? a.ld_weight : a.ld_hidden;
        const int R = is_w ? a.n_weight : a.n_hidden;
        const int64_t n = int64_t(R) * a.C8, step = int64_t(blocks) * kMaxThreads;
        auto at = [&](int64_t v) {
            const int64_t r = v / a.C8, row = is_w ? sample_row(int(r), a.vocab) : r;
            return *reinterpret_cast<const u32x4*>(in + row * ld + (v - r * a.C8) * 8);
        };
        int64_t v = int64_t(block) * kMaxThreads + threadIdx.x;
        for (; v + 7 * step < n; v += 8 * step) {
            u32x4 q[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) q[k] = at(v + k * step);
#pragma unroll
            for (int k = 0; k < 8; ++k) m = max_bits(m, q[k]);
        }
        for (; v < n; v += step) m = max_bits(m, at(v));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), off, 64)));
    if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < kMaxThreads / kWave; ++w) m = max(m, part[w]);
        // (a stale value only costs an atomic that changes nothing)
        if (m > __hip_atomic_load(a.out + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(a.out + slot, m);
    }
}

// One 64 x 64 tile of [R, C] (ld) -> [C, ldo] with columns >= R zero-filled up to `fill`, through LDS.
// TO_F16: the input is bf16 and the output fp16, multiplied by the power of two `sc`.
// ROW_G: input row r is also multiplied by s_all / pow2_scale(|row_g[r]| * zs) (0 where row_g[r] is 0), s_all from
// `g_max`: what brings the columns of hidden^T into the scales of the d logits' columns (see above).
// Returns the largest magnitude (bit pattern) of what this lane read when TRACK is set.
constexpr int kTransposeStride = 136;
template <bool TO_F16, bool ROW_G, bool TRACK>
__device__ __forceinline__ uint32_t transpose16_tile(uint16_t* tile, int c0, int r0, const uint16_t* in, int64_t ld, int R, int C,
                                                     uint16_t* out, int64_t ldo, int64_t fill, float sc, const float* row_g,
                                                     const uint32_t* g_max, float zs) {
    // C, ld, ldo and fill are multiples of 8 and both matrices 16-byte aligned (the callers' operands are): a lane
    // moves 8 elements at a time.  Tile rows are skewed by 8 elements per group of 8 rows, which spreads the
    // 2-byte column reads of the second phase over all banks.
    constexpr int kStride = kTransposeStride;
    const int tid = threadIdx.x, hi = tid >> 3, lo = tid & 7;
    uint32_t m = 0;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int row = hi + 32 * p, cc = lo * 8;
        u32x4 q = {0u, 0u, 0u, 0u};
        if (r0 + row < R && c0 + cc < C) q = *reinterpret_cast<const u32x4*>(in + int64_t(r0 + row) * ld + c0 + cc);
        if (TRACK) m = max_bits(m, q);
        if (TO_F16 || ROW_G) {
            float f = sc;
            if (ROW_G) {
                const float gr = r0 + row < R ? fabsf(row_g[r0 + row]) : 0.f;
                f = gr > 0.f ? sc * (slot_scale(g_max, zs) / pow2_scale(gr * zs)) : 0.f;
            }
            float x[8];
            if (TO_F16)
                Elem<TRLK_BF16>::unpack(q, x);
            else
                Elem<TRLK_F16>::unpack(q, x);
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] *= f;
            q = Elem<TRLK_F16>::pack(x);
        }
        *reinterpret_cast<u32x4*>(tile + row * kStride + cc + 8 * (row >> 3)) = q;
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int c = hi + 32 * p, r8 = lo;  // output row c0 + c, its columns r0 + 8 r8 .. + 7
        if (c0 + c < C && r0 + r8 * 8 < fill) {
            const uint16_t* src = tile + (r8 * 8) * kStride + c + 8 * r8;
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = uint32_t(src[(2 * i) * kStride]) | (uint32_t(src[(2 * i + 1) * kStride]) << 16);
            const u32x4 q = {w[0], w[1], w[2], w[3]};
            *reinterpret_cast<u32x4*>(out + int64_t(c0 + c) * ldo + r0 + r8 * 8) = q;
        }
    }
    return m;
}
// hidden^T, its columns in the scales of the d logits' columns.
template <bool TO_F16>
__global__ __launch_bounds__(256) void transpose_hidden_kernel(const uint16_t* in, int64_t ld, int R, int C, uint16_t* out,
                                                               int64_t ldo, int64_t fill, const uint32_t* in_max,
                                                               const float* row_g, const uint32_t* g_max, float zs) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kTransposeStride];
    transpose16_tile<TO_F16, true, false>(tile, blockIdx.x * 64, blockIdx.y * 64, in, ld, R, C, out, ldo, fill,
                                          TO_F16 ? slot_scale(in_max, 1.f) : 1.f, row_g, g_max, zs);
}
// W_chunk^T of an fp16 problem, as it is.
__global__ __launch_bounds__(256) void transpose_weight_f16_kernel(const uint16_t* in, int64_t ld, int R, int C, uint16_t* out,
                                                                   int64_t ldo, int64_t fill) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kTransposeStride];
    transpose16_tile<false, false, false>(tile, blockIdx.x * 64, blockIdx.y * 64, in, ld, R, C, out, ldo, fill, 1.f, nullptr,
                                          nullptr, 1.f);
}
// W_chunk^T of a bf16 problem in the sample's scale.  The largest magnitude of what it converts is found on the way: a wave
// whose entries all stay below the sample's maximum (nearly every one) spends one comparison on it, the others one atomic.
// The separate pass over the whole weight that used to precede this one took 36 / 93 / 214 us for weights of 206 / 525 / 1089 MB
// (50257 x 2048, 128256 x 2048, 151936 x 3584); the launch that reads the sample takes 9 / 10 / 15 us with few tokens (28 with
// the 69 MB of 9664 hidden states of 3584, which it reads too), a second launch with nothing to do 5 us.
__global__ __launch_bounds__(256) void transpose_weight_kernel(const uint16_t* in, int64_t ld, int R, int C, uint16_t* out,
                                                               int64_t ldo, int64_t fill, const uint32_t* sample, uint32_t* beyond) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kTransposeStride];
    uint32_t m = transpose16_tile<true, false, true>(tile, blockIdx.x * 64, blockIdx.y * 64, in, ld, R, C, out, ldo, fill,
                                                     slot_scale(sample, 1.f), nullptr, nullptr, 1.f);
    const uint32_t known = max(*sample, __hip_atomic_load(beyond, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (__any(m > known)) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), off, 64)));
        if ((threadIdx.x & (kWave - 1)) == 0) atomicMax(beyond, m);
    }
}
// The same again in the scale of the chunk's own maximum, where the sample's does not do: returns at once everywhere else (few
// workgroups that step through the tiles, so that a launch with nothing to do takes 5 us).  One entry of 50 in a weight of
// deviation 0.02, which makes the chunk that holds it convert again: whole backward 1336-1375 -> 1396 us (3300 tokens, H = 2048, V =
// 50257, one chunk), 3255 -> 3258 (V = 128256, one of two chunks), 5255 -> 5390 (2600 tokens, H = 3584, V = 151936, one of two).
constexpr int kAgainBlocks = 1024;
__global__ __launch_bounds__(256) void transpose_weight_again_kernel(const uint16_t* in, int64_t ld, int R, int C, uint16_t* out,
                                                                     int64_t ldo, int64_t fill, const uint32_t* sample,
                                                                     const uint32_t* beyond, int tiles_c, int tiles) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * kTransposeStride];
    const WeightScale w = weight_scale(sample, beyond);
    if (!w.again) return;
    for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
        transpose16_tile<true, false, false>(tile, t % tiles_c * 64, t / tiles_c * 64, in, ld, R, C, out, ldo, fill, w.scale,
                                             nullptr, nullptr, 1.f);
        __syncthreads();  // (the next tile overwrites the LDS)
    }
}

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// d bias[v] = sum over tokens of dz[token, v]: row sums of the transposed dz copy (padding columns are zero).
__global__ __launch_bounds__(256) void dz_row_sum_kernel(const uint16_t* dzT, int64_t ld, int n_cols8, float* out,
                                                         const float* g, int n_tokens, float zs) {
    typedef Elem<TRLK_F16> E;
    const uint16_t* row = dzT + int64_t(blockIdx.x) * ld;
    float acc = 0.f;
    for (int c = threadIdx.x; c < n_cols8; c += 256) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(row + c * 8);
        float x[8];
        E::unpack(w, x);
#pragma unroll
        for (int q = 0; q < 8; ++q) {  // column n is in token n's scale
            const int n = c * 8 + q;
            if (n < n_tokens) acc += x[q] / pow2_scale(fabsf(g[n]) * zs);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Row strides of the workspace matrices carry 128 extra bytes: their padded extents are multiples
// of large powers of two (tokens, chunk), and with such a stride the 256 rows of a tile step all
// fall into the same memory channels.
constexpr int64_t kLdSkew = 64;
struct BwdLayout {
    int64_t vpad, npad, cpad;    // padded extents (zero-filled)
    int64_t ld_v, ld_n, ld_c;    // row strides of [*, vpad], [*, npad], [*, cpad] matrices
    size_t off_wt, off_ht, off_dzt, off_dh, off_max, total;
    int64_t n_chunks, n_maxima;
    bool direct;         // the dHidden product reads the weight itself: no transposed copy
    int64_t dh_k;        // length of the dHidden product's contraction over a whole chunk
    int slices, kslice;  // of that contraction
    // Slices that a contraction of length k reaches: `slices` of a whole chunk, fewer of a shorter last one.  What is launched and
    // what is summed both come from here; a slice that is summed and not launched would add what the workspace held before.
    int reached(int64_t k) const { return int((k + kslice - 1) / kslice); }
};
// Slices of the contraction of the dHidden product.  Its tiles (token blocks x hidden tiles) contract over the whole
// chunk, tens of times longer than the dW tiles of the same launch, and they are few when there are few tokens: 48 tiles of
// 788 k steps beside 1576 tiles of 24 for 1396 tokens, H = 2048 and one chunk of 50257 rows, so the launch lasts as long as
// one of them.  The fewest slices (each costs a write and a read of [N, H] in fp32) that make the tiles' chain shorter than
// an even share of the whole launch.  Measured there (whole backward): 1 / 2 / 3 / 6 / 16
// slices 1331 / 854 / 765 / 776 / 858 us, the rule takes 3; 240 tokens, H = 3584, V = 151936: 1 / 3 / 8 / 16 slices 4496 /
// 2208 / 1478 / 1519 us, the rule takes 7; 2500 tokens: 1 slice, 5.67 ms (3: 5.64, 8: 5.77).
int dh_slices(int64_t n_tb, int64_t n_ht, int64_t kpad, int64_t npad) {
    constexpr int64_t kEpilogue = 4, kCuCount = 256;  // a tile's start and epilogue in k steps
    const int64_t steps = kpad / BK, tiles = n_tb * n_ht;
    int best = 1;
    int64_t best_chain = INT64_MAX;
    for (int64_t s = 1; s <= 32 && steps / s >= 16; ++s) {
        const int64_t chain = (tiles * s + kCuCount - 1) / kCuCount * ((steps + s - 1) / s + kEpilogue);
        const int64_t share = (tiles * (steps + s * kEpilogue) + kpad / BM * n_ht * (npad / BK + kEpilogue)) / kCuCount;
        if (chain < best_chain) {
            best_chain = chain;
            best = int(s);
        }
        if (chain * 10 <= share * 9) break;
    }
    return best;
}
// Up to this many tokens the dHidden product takes the weight as it lies in memory (LeftKm) and not a transposed fp16 copy.  The
// copy costs the same for every token count (525 MB read, 525 written: 193 us of a backward for V = 128256, H = 2048; 390 us for
// 151936 x 3584), the conversion in the tile loop 5 to 10 % of the product.  Whole backward with the copy -> without, in us:
// 100 tokens, H = 3584, V = 151936 1341 -> 859; 459 the same 1712 -> 1263; 300, H = 1024, V = 128256 506 -> 388; 900, H = 2560,
// V = 151665 1784 -> 1557; 1396, H = 2048, V = 50257 710 -> 648; 1392, V = 128256 1662 -> 1562; 2300, H = 4096, V = 50264
// 1800 -> 1760; from there on it loses: 2600, H = 3584, V = 151936 5298 -> 5340, 3300, H = 2048, V = 128256 3305 -> 3325, 7000,
// V = 50264 2653 -> 2735.  Only with the whole vocabulary in one chunk: there is one product to add left-out entries to
// (direct_scale).  A bf16 problem's sums are left in fp32 for that even where one slice would do (tiles of dHidden enough for the whole
// chip): 2304 tokens, H = 4096, V = 50257 1740 -> 1762 us, 1792 tokens, H = 5120, V = 128256 4378 -> 4400.
constexpr int64_t kDirectTokens = 2304;
BwdLayout bwd_layout(int64_t N, int64_t V, int64_t H, int64_t chunk) {
    BwdLayout l;
    l.vpad = round_up(V, BK);
    l.npad = round_up(N, BN);
    l.cpad = round_up(chunk < V ? chunk : V, BM);
    l.ld_v = l.vpad + kLdSkew;
    l.ld_n = l.npad + kLdSkew;
    l.ld_c = l.cpad + kLdSkew;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += (bytes + 255) / 256 * 256;
        return at;
    };
    l.direct = l.cpad >= V && N <= kDirectTokens;
    l.off_wt = take(l.direct ? 0 : size_t(H) * l.ld_c * 2);
    l.off_ht = take(size_t(H) * l.ld_n * 2);
    l.off_dzt = take(size_t(l.cpad) * l.ld_n * 2);
    const int want = dh_slices(l.npad / BN, (H + BN - 1) / BN, l.cpad, l.npad);
    l.dh_k = l.direct ? l.vpad : l.cpad;  // (a transposed copy is padded to whole tiles, the weight is read in whole k steps)
    l.kslice = int(round_up((l.dh_k + want - 1) / want, BK));
    l.slices = l.reached(l.dh_k);
    l.off_dh = take(size_t(l.slices) * N * H * 4);
    l.n_chunks = (V + l.cpad - 1) / l.cpad;
    // largest magnitudes: g, hidden, sample of W, what exceeds it in each chunk -- or whether fp16 does not hold all of W, and
    // a bit for each row of it
    l.n_maxima = 3 + l.n_chunks + (l.direct ? (V + 31) / 32 : 0);
    l.off_max = take(size_t(l.n_maxima) * 4);
    l.total = o;
    return l;
}

// Vocabulary splits of the forward.  A workgroup keeps one token block and walks over its share of the vocabulary tiles,
// one workgroup per CU at a time, so a launch takes (rounds of 256 workgroups) x (tiles per share) tile times; the number
// of splits is the one that makes this smallest, the fewest on a tie.  Any number is allowed, not only powers of two with
// at least four tiles each: 6 token blocks x 197 (501) vocabulary tiles run 42 splits of 5 (12) tiles in one round, where
// 32 (64) splits took 1 round of 7 (2 rounds of 8) tiles, 384 -> 290 us (896 -> 713 us), both
// with H = 2048 and the stash.  Long launches are bound by power and gain nothing: 38 token blocks x 594 tiles run 3 rounds
// of 30 where they ran 5 of 19, 8.6 ms either way.
constexpr int kCus = 256, kMinFwdSplits = 8, kMaxFwdSplits = 256;
int max_fwd_splits(int64_t n_tokens) {  // bounds the workspace, which is sized before the vocabulary is known
    const int64_t n_tb = (n_tokens + BN - 1) / BN, most = 2048 / n_tb;
    return int(most < kMinFwdSplits ? kMinFwdSplits : (most > kMaxFwdSplits ? kMaxFwdSplits : most));
}
int fwd_splits(int64_t n_tokens, int n_vt, int64_t H) {
    const int64_t n_tb = (n_tokens + BN - 1) / BN;
    // in k steps of the tile loop: a tile's own steps plus its reduction, and a workgroup's start and final merge
    const double tile = double(H) / BK + 3., start = 4.;
    const int most = max_fwd_splits(n_tokens) < n_vt ? max_fwd_splits(n_tokens) : n_vt;
    int best = 1;
    double best_cost = 1e300;
    // (fewer than 8 splits would leave an XCD's 32 workgroups with fewer than 8 vocabulary tiles to share)
    for (int sp = most < kMinFwdSplits ? most : kMinFwdSplits; sp <= most; ++sp) {
        const int tps = (n_vt + sp - 1) / sp;
        if (sp > kMinFwdSplits && (n_vt + tps - 1) / tps != sp) continue;  // some splits would be empty
        const int64_t per_xcd = (n_tb * sp + 7) / 8, rounds = (per_xcd + kCus / 8 - 1) / (kCus / 8);
        const double cost = double(rounds) * (tps * tile + start);
        if (cost < best_cost * 0.99) {
            best_cost = cost;
            best = sp;
        }
    }
    return best;
}

int check_head(const char* what, const void* hidden, const void* weight, const int64_t* targets, int dtype, int64_t N,
               int64_t V, int64_t H, int64_t ldh, int64_t ldw, float temperature) {
    TRLK_REQUIRE(dtype == TRLK_BF16 || dtype == TRLK_F16, TRLK_ERR_BAD_DTYPE,
                 "%s: the fused head takes bf16 or fp16 operands (dtype code %d)", what, dtype);
    TRLK_REQUIRE(N >= 0 && V >= 1 && H >= 1, TRLK_ERR_BAD_SHAPE, "%s: bad sizes N=%lld V=%lld H=%lld", what, (long long)N,
                 (long long)V, (long long)H);
    TRLK_REQUIRE(N < (int64_t(1) << 31) - BN && V < (int64_t(1) << 31) - BM, TRLK_ERR_BAD_SHAPE, "%s: N or V too large",
                 what);
    TRLK_REQUIRE(H % 8 == 0 && ldh % 8 == 0 && ldw % 8 == 0 && ldh >= H && ldw >= H, TRLK_ERR_BAD_STRIDE,
                 "%s: H and the row strides must be multiples of 8 elements (H=%lld ldh=%lld ldw=%lld)", what,
                 (long long)H, (long long)ldh, (long long)ldw);
    TRLK_REQUIRE(temperature > 0.f && temperature < INFINITY, TRLK_ERR_BAD_VALUE, "%s: temperature must be positive", what);
    if (N > 0) {
        TRLK_REQUIRE(hidden && weight && targets, TRLK_ERR_NULL_POINTER, "%s: null operand pointer", what);
        TRLK_REQUIRE(reinterpret_cast<uintptr_t>(hidden) % 16 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0,
                     TRLK_ERR_BAD_STRIDE, "%s: operands must be 16-byte aligned", what);
    }
    return TRLK_OK;
}

template <typename Kern>
int reserve_head_lds(Kern kern, const char* what);

template <typename Kern>
int launch_head_pair(Kern kern, int grid_a, const GemmArgs& a, int grid_b, const GemmArgs& b, hipStream_t s,
                     const char* what) {
    if (int rc = reserve_head_lds(kern, what)) return rc;
    hipLaunchKernelGGL(kern, dim3(grid_a + grid_b), dim3(kHeadThreads), kHeadLdsBytes, s, a, grid_a, b);
    return launch_status(what);
}

template <typename Kern, typename Args>
int launch_head(Kern kern, int grid, const Args& a, hipStream_t s, const char* what) {
    if (int rc = reserve_head_lds(kern, what)) return rc;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kHeadThreads), kHeadLdsBytes, s, a);
    return launch_status(what);
}

template <typename Kern>
int reserve_head_lds(Kern kern, const char* what) {
    // dynamic LDS above 64 KiB has to be allowed per kernel and device once
    struct Done {
        const void* kern;
        int device;
    };
    static thread_local Done configured[32] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) device = 0;
    const void* key = reinterpret_cast<const void*>(kern);
    for (const Done& c : configured)
        if (c.kern == key && c.device == device) return TRLK_OK;
    const hipError_t e = hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, kHeadLdsBytes);
    if (e != hipSuccess) return fail(int(e), "%s: cannot reserve %d bytes of LDS: %s", what, kHeadLdsBytes, hipGetErrorString(e));
    for (Done& c : configured)
        if (c.kern == nullptr) {
            c.kern = key;
            c.device = device;
            break;
        }
    return TRLK_OK;
}

}  // namespace
}  // namespace trlk

using namespace trlk;

extern "C" size_t trlk_fused_head_fwd_workspace_bytes(int64_t n_tokens) {
    return n_tokens > 0 ? size_t(n_tokens) * (max_fwd_splits(n_tokens) * 4 + 1) * sizeof(float) : 0;
}

extern "C" size_t trlk_fused_head_stash_bytes(int64_t n_tokens, int64_t vocab, int64_t* out_ld) {
    if (n_tokens <= 0 || vocab <= 0) return 0;
    const int64_t ld = round_up(n_tokens, BN);
    if (out_ld) *out_ld = ld;
    return size_t(StashView::rows8(round_up(vocab, BM))) * size_t(ld) * 8;
}

extern "C" size_t trlk_fused_head_bwd_workspace_bytes(int64_t n_tokens, int64_t vocab, int64_t hidden_size,
                                                      int64_t chunk_size) {
    if (n_tokens <= 0 || vocab <= 0 || hidden_size <= 0 || chunk_size <= 0) return 0;
    return bwd_layout(n_tokens, vocab, hidden_size, chunk_size).total;
}

extern "C" int trlk_fused_head_fwd(const void* d_hidden, const void* d_weight, const int64_t* d_targets, int dtype,
                                   int64_t n_tokens, int64_t vocab, int64_t hidden_size, int64_t hidden_stride,
                                   int64_t weight_stride, float temperature, float final_logit_softcapping,
                                   float logit_scale, const float* d_bias, float* d_out_logp, float* d_out_entropy,
                                   float* d_out_log_z, float* d_out_target_is_max, void* d_out_stash,
                                   int64_t stash_ld, int32_t* d_error_flag, void* d_workspace, size_t workspace_bytes,
                                   trlk_stream_t stream) {
    clear_error();
    if (int rc = check_head("fused_head_fwd", d_hidden, d_weight, d_targets, dtype, n_tokens, vocab, hidden_size,
                            hidden_stride, weight_stride, temperature))
        return rc;
    if (n_tokens == 0) return TRLK_OK;
    TRLK_REQUIRE(d_out_logp && d_out_entropy && d_out_log_z, TRLK_ERR_NULL_POINTER, "fused_head_fwd: null output pointer");
    TRLK_REQUIRE(d_workspace && workspace_bytes >= trlk_fused_head_fwd_workspace_bytes(n_tokens), TRLK_ERR_WORKSPACE,
                 "fused_head_fwd: workspace of %zu bytes needed, %zu given", trlk_fused_head_fwd_workspace_bytes(n_tokens),
                 workspace_bytes);
    TRLK_REQUIRE(d_out_stash == nullptr || (stash_ld >= round_up(n_tokens, BN) && stash_ld % 4 == 0 &&
                                            stash_ld < (int64_t(1) << 31) / 16 &&
                                            reinterpret_cast<uintptr_t>(d_out_stash) % 16 == 0),
                 TRLK_ERR_BAD_STRIDE, "fused_head_fwd: the stash needs a 16-byte aligned buffer with a row stride >= %lld (got %lld)",
                 (long long)round_up(n_tokens, BN), (long long)stash_ld);
    hipStream_t s = static_cast<hipStream_t>(stream);
    HeadArgs a{};
    a.hidden = static_cast<const uint16_t*>(d_hidden);
    a.weight = static_cast<const uint16_t*>(d_weight);
    a.targets = d_targets;
    a.bias = d_bias;
    a.stash = StashView{static_cast<char*>(d_out_stash), stash_ld, round_up(vocab, BM)};
    a.N = int(n_tokens);
    a.V = int(vocab);
    a.H = int(hidden_size);
    a.ldh = hidden_stride;
    a.ldw = weight_stride;
    a.logit_scale = logit_scale;
    a.inv_t = 1.f / temperature;
    a.softcap = final_logit_softcapping > 0.f ? final_logit_softcapping : 0.f;
    const int n_vt = int((vocab + BM - 1) / BM);
    const int splits = fwd_splits(n_tokens, n_vt, hidden_size);
    a.v_splits = splits;
    a.tiles_per_split = (n_vt + splits - 1) / splits;
    a.partial = static_cast<float*>(d_workspace);
    a.tgt = a.partial + size_t(n_tokens) * splits * 4;
    hipLaunchKernelGGL(head_fill_kernel, dim3(unsigned((n_tokens + 255) / 256)), dim3(256), 0, s, a.tgt, n_tokens, NAN);
    if (int rc = launch_status("fused_head_fwd (fill)")) return rc;
    const int n_tb = int((n_tokens + BN - 1) / BN);
    const int grid = xcd_patch_grid(n_tb, splits);
    const char* what = "fused_head_fwd";
    int rc;
    const bool general = a.softcap > 0.f || !(a.logit_scale * a.inv_t > 0.f);
    const bool staged = hidden_size % BK != 0;
    auto launch_fwd = [&](auto stash_tag, auto general_tag) {
        constexpr bool kS = decltype(stash_tag)::value, kG = decltype(general_tag)::value;
        if (staged)
            return dtype == TRLK_BF16 ? launch_head(fused_head_fwd_kernel<TRLK_BF16, kS, kG, true>, grid, a, s, what)
                                      : launch_head(fused_head_fwd_kernel<TRLK_F16, kS, kG, true>, grid, a, s, what);
        return dtype == TRLK_BF16 ? launch_head(fused_head_fwd_kernel<TRLK_BF16, kS, kG, false>, grid, a, s, what)
                                  : launch_head(fused_head_fwd_kernel<TRLK_F16, kS, kG, false>, grid, a, s, what);
    };
    if (d_out_stash != nullptr)
        rc = general ? launch_fwd(std::true_type{}, std::true_type{}) : launch_fwd(std::true_type{}, std::false_type{});
    else
        rc = general ? launch_fwd(std::false_type{}, std::true_type{}) : launch_fwd(std::false_type{}, std::false_type{});
    if (rc) return rc;
    hipLaunchKernelGGL(head_merge_kernel, dim3(unsigned((n_tokens + kMergeTokens - 1) / kMergeTokens)),
                       dim3(kMergeTokens * kWave), 0, s, a.partial, a.tgt,
                       d_targets, int(n_tokens), int(vocab), splits, d_out_logp, d_out_entropy, d_out_log_z,
                       d_out_target_is_max, d_error_flag, d_out_stash != nullptr ? a.stash.zt() : nullptr);
    return launch_status("fused_head_fwd (merge)");
}

extern "C" int trlk_fused_head_bwd(const void* d_hidden, const void* d_weight, const int64_t* d_targets, int dtype,
                                   int64_t n_tokens, int64_t vocab, int64_t hidden_size, int64_t hidden_stride,
                                   int64_t weight_stride, float temperature, float final_logit_softcapping,
                                   float logit_scale, const float* d_bias, const float* d_log_z, const float* d_g_logp,
                                   int64_t chunk_size, const void* d_stash, int64_t stash_ld, const int32_t* d_stash_cols,
                                   void* d_out_dhidden, void* d_out_dweight, float* d_out_dbias, void* d_workspace,
                                   size_t workspace_bytes, trlk_stream_t stream) {
    clear_error();
    if (int rc = check_head("fused_head_bwd", d_hidden, d_weight, d_targets, dtype, n_tokens, vocab, hidden_size,
                            hidden_stride, weight_stride, temperature))
        return rc;
    TRLK_REQUIRE(chunk_size >= 1, TRLK_ERR_BAD_VALUE, "fused_head_bwd: chunk_size must be >= 1");
    TRLK_REQUIRE(d_out_dhidden && d_out_dweight, TRLK_ERR_NULL_POINTER, "fused_head_bwd: null output pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n_tokens == 0) {  // no tokens: both gradients are zero
        hipLaunchKernelGGL(head_fill_kernel, dim3(unsigned((vocab * hidden_size / 2 + 255) / 256)), dim3(256), 0, s,
                           static_cast<float*>(d_out_dweight), vocab * hidden_size / 2, 0.f);
        if (d_out_dbias)
            hipLaunchKernelGGL(head_fill_kernel, dim3(unsigned((vocab + 255) / 256)), dim3(256), 0, s, d_out_dbias, vocab, 0.f);
        return launch_status("fused_head_bwd (zero dW)");
    }
    TRLK_REQUIRE(d_log_z && d_g_logp, TRLK_ERR_NULL_POINTER, "fused_head_bwd: log_z / g_logp pointer is null");
    TRLK_REQUIRE(d_stash == nullptr || chunk_size <= int64_t(65535) * kSdzRows || vocab <= int64_t(65535) * kSdzRows,
                 TRLK_ERR_BAD_SHAPE, "fused_head_bwd: chunk of %lld rows is too large for the stash path",
                 (long long)chunk_size);
    TRLK_REQUIRE(d_stash_cols == nullptr || d_stash != nullptr, TRLK_ERR_NULL_POINTER,
                 "fused_head_bwd: stash columns given without a stash");
    TRLK_REQUIRE(d_stash == nullptr || ((d_stash_cols != nullptr || stash_ld >= round_up(n_tokens, BN)) && stash_ld % 4 == 0 &&
                                        reinterpret_cast<uintptr_t>(d_stash) % 16 == 0),
                 TRLK_ERR_BAD_STRIDE, "fused_head_bwd: the stash needs a 16-byte aligned buffer with a row stride >= %lld (got %lld)",
                 (long long)round_up(n_tokens, BN), (long long)stash_ld);
    const int64_t chunk = round_up(chunk_size < vocab ? chunk_size : vocab, BM);
    const BwdLayout l = bwd_layout(n_tokens, vocab, hidden_size, chunk);
    TRLK_REQUIRE(d_workspace && workspace_bytes >= l.total, TRLK_ERR_WORKSPACE,
                 "fused_head_bwd: workspace of %zu bytes needed, %zu given", l.total, workspace_bytes);
    char* ws = static_cast<char*>(d_workspace);
    uint16_t* wt = reinterpret_cast<uint16_t*>(ws + l.off_wt);    // [H, cpad], row stride ld_c (one chunk at a time)
    uint16_t* ht = reinterpret_cast<uint16_t*>(ws + l.off_ht);    // [H, npad], row stride ld_n
    uint16_t* dzt = reinterpret_cast<uint16_t*>(ws + l.off_dzt);  // [cpad, npad], row stride ld_n
    float* dh = reinterpret_cast<float*>(ws + l.off_dh);          // [slices][N, H]
    uint32_t* maxima = reinterpret_cast<uint32_t*>(ws + l.off_max);  // [0] g, [1] hidden, [2] sample of W, the rest: see bwd_layout
    const int H = int(hidden_size), N = int(n_tokens), V = int(vocab);
    const bool from_bf16 = dtype == TRLK_BF16;  // the products' operands are fp16: bf16 inputs are converted on the way
    const uint32_t* max_g = maxima;
    const uint32_t* max_h = from_bf16 ? maxima + 1 : nullptr;
    hipLaunchKernelGGL(head_fill_kernel, dim3(unsigned((l.n_maxima + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<float*>(maxima), l.n_maxima, 0.f);
    MaxAbsArgs ma{};
    ma.g = d_g_logp;
    ma.n_g = n_tokens;
    ma.blocks_g = int(N < 32 * kMaxThreads ? (N + kMaxThreads - 1) / kMaxThreads : 32);
    ma.out = maxima;
    if (from_bf16) {
        const auto blocks = [&](int64_t rows) {
            const int64_t b = (rows * (H / 8) + 8 * kMaxThreads - 1) / (8 * kMaxThreads);
            return int(b < kMaxBlocks ? b : kMaxBlocks);
        };
        ma.hidden = static_cast<const uint16_t*>(d_hidden);
        ma.weight = static_cast<const uint16_t*>(d_weight);
        ma.ld_hidden = hidden_stride;
        ma.ld_weight = weight_stride;
        ma.vocab = V;
        ma.n_hidden = N;
        ma.n_weight = (V + kSampleRows - 1) / kSampleRows;
        ma.C8 = H / 8;
        ma.blocks_h = blocks(N);
        ma.blocks_w = blocks(ma.n_weight);
    }
    hipLaunchKernelGGL(head_maxabs_kernel, dim3(unsigned(ma.blocks_w + ma.blocks_h + ma.blocks_g)), dim3(kMaxThreads), 0, s, ma);
    if (from_bf16) {
        hipLaunchKernelGGL(transpose_hidden_kernel<true>, dim3((H + 63) / 64, unsigned((l.npad + 63) / 64)), dim3(256), 0, s,
                           static_cast<const uint16_t*>(d_hidden), hidden_stride, N, H, ht, l.ld_n, l.npad, max_h, d_g_logp,
                           max_g, logit_scale / temperature);
    } else {
        hipLaunchKernelGGL(transpose_hidden_kernel<false>, dim3((H + 63) / 64, unsigned((l.npad + 63) / 64)), dim3(256), 0, s,
                           static_cast<const uint16_t*>(d_hidden), hidden_stride, N, H, ht, l.ld_n, l.npad, max_h, d_g_logp,
                           max_g, logit_scale / temperature);
    }
    if (int rc = launch_status("fused_head_bwd (hidden^T)")) return rc;

    HeadArgs a{};
    a.hidden = static_cast<const uint16_t*>(d_hidden);
    a.weight = static_cast<const uint16_t*>(d_weight);
    a.targets = d_targets;
    a.bias = d_bias;
    a.N = N;
    a.V = V;
    a.H = H;
    a.ldh = hidden_stride;
    a.ldw = weight_stride;
    a.logit_scale = logit_scale;
    a.inv_t = 1.f / temperature;
    a.softcap = final_logit_softcapping > 0.f ? final_logit_softcapping : 0.f;
    a.log_z = d_log_z;
    a.g = d_g_logp;
    a.stash = StashView{static_cast<char*>(const_cast<void*>(d_stash)), stash_ld, round_up(vocab, BM)};
    a.stash_cols = d_stash_cols;
    a.dzT = dzt;
    a.ldzt = l.ld_n;
    a.g_max = max_g;
    const float zs = logit_scale / temperature;  // |dz[n, v]| <= |g[n]| * zs
    const int n_tb = int((n_tokens + BN - 1) / BN);
    const int n_ht = (H + BN - 1) / BN;
    const bool converts = l.direct && from_bf16;   // the dHidden product may leave something out (see direct_scale)
    const bool sums = l.slices > 1 || converts;  // dHidden is left in fp32 and rounded by a pass of its own
    for (int64_t c0 = 0; c0 < vocab; c0 += chunk) {
        const int64_t c1 = c0 + chunk < vocab ? c0 + chunk : vocab;
        const int rows = int(c1 - c0);
        const int kpad = int(round_up(rows, BM));  // dz / dz^T are zero beyond the chunk's rows
        a.c0 = int(c0);
        a.c1 = int(c1);
        const int n_vt = (rows + BM - 1) / BM;
        int rc;
        if (d_stash != nullptr) {
            a.sdz_token_blocks = int(l.npad / kSdzTokens);
            a.sdz_tiles = a.sdz_token_blocks * int(kpad / kSdzRows);
            const dim3 grid(unsigned((a.sdz_tiles + 7) / 8 * 8));
            const bool capped = a.softcap > 0.f;
            if (d_stash_cols && capped)
                hipLaunchKernelGGL((head_dz_from_stash_kernel<true, true>), grid, dim3(256), 0, s, a);
            else if (d_stash_cols)
                hipLaunchKernelGGL((head_dz_from_stash_kernel<true, false>), grid, dim3(256), 0, s, a);
            else if (capped)
                hipLaunchKernelGGL((head_dz_from_stash_kernel<false, true>), grid, dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((head_dz_from_stash_kernel<false, false>), grid, dim3(256), 0, s, a);
            rc = launch_status("fused_head_bwd (dz from the stash)");
        } else {
            rc = dtype == TRLK_BF16
                     ? launch_head(fused_head_dz_kernel<TRLK_BF16>, xcd_patch_grid(n_tb, n_vt), a, s, "fused_head_bwd (dz)")
                     : launch_head(fused_head_dz_kernel<TRLK_F16>, xcd_patch_grid(n_tb, n_vt), a, s, "fused_head_bwd (dz)");
        }
        if (rc) return rc;
        if (d_out_dbias) {
            hipLaunchKernelGGL(dz_row_sum_kernel, dim3(rows), dim3(256), 0, s, dzt, l.ld_n, int(l.npad / 8), d_out_dbias + c0,
                               d_g_logp, N, zs);
            if (int rc2 = launch_status("fused_head_bwd (dBias)")) return rc2;
        }
        const bool first = c0 == 0, last = c1 == vocab;
        // W_chunk^T [H, kpad] (columns beyond the chunk's rows are zero): the chunk's own transposed copy keeps the
        // row stride of this operand as short as that of the other three
        const uint16_t* w_chunk = static_cast<const uint16_t*>(d_weight) + c0 * weight_stride;
        const uint32_t* max_w = from_bf16 ? maxima + 2 : nullptr;
        uint32_t* beyond_w = from_bf16 ? maxima + 3 + c0 / chunk : nullptr;
        const dim3 tgrid((H + 63) / 64, unsigned((kpad + 63) / 64));
        if (l.direct) {
        } else if (from_bf16) {
            hipLaunchKernelGGL(transpose_weight_kernel, tgrid, dim3(256), 0, s, w_chunk, weight_stride, rows, H, wt, l.ld_c,
                               int64_t(kpad), max_w, beyond_w);
            const int tiles = int(tgrid.x * tgrid.y);
            hipLaunchKernelGGL(transpose_weight_again_kernel, dim3(tiles < kAgainBlocks ? tiles : kAgainBlocks), dim3(256), 0, s,
                               w_chunk, weight_stride, rows, H, wt, l.ld_c, int64_t(kpad), max_w, beyond_w, int(tgrid.x), tiles);
        } else {
            hipLaunchKernelGGL(transpose_weight_f16_kernel, tgrid, dim3(256), 0, s, w_chunk, weight_stride, rows, H, wt, l.ld_c,
                               int64_t(kpad));
        }
        if (int rc2 = launch_status("fused_head_bwd (W^T)")) return rc2;
        // dHidden[N, H] += dz[N, chunk] * (W_chunk^T[H, chunk])^T
        GemmArgs gh{};
        gh.A = Operand{dzt, l.ld_n, N};  // k-major: [chunk rows, tokens]
        gh.B = Operand{wt, l.ld_c, H};
        gh.M = N;
        gh.N = H;
        gh.K = kpad;
        gh.out_f32 = dh;
        gh.ld_f32 = H;
        gh.out_lp = static_cast<uint16_t*>(d_out_dhidden);
        gh.ld_lp = H;
        gh.first = first;
        gh.max_a = nullptr;  // the rows of dz carry their own scales
        gh.g_rows = d_g_logp;
        gh.mult_a = zs;
        gh.max_b = max_w;
        gh.beyond_b = beyond_w;
        if (l.direct) {
            gh.B = Operand{w_chunk, weight_stride, H};
            gh.K = int(l.dh_k);
            gh.b_krows = rows;
            gh.beyond_out = beyond_w;
        }
        gh.slices = l.reached(gh.K);
        gh.kslice = l.kslice;
        const int ghgrid = xcd_patch_grid(n_tb, n_ht * gh.slices);
        // dW[chunk, H] = dz^T[chunk, N] * (hidden^T[H, N])^T
        GemmArgs gw{};
        gw.A = Operand{dzt, l.ld_n, kpad};
        gw.B = Operand{ht, l.ld_n, H};
        gw.M = rows;
        gw.N = H;
        gw.K = int(round_up(N, BK));  // (dz is zero from there to npad)
        gw.out_lp = static_cast<uint16_t*>(d_out_dweight) + c0 * hidden_size;
        gw.ld_lp = hidden_size;
        gw.first = 1;
        gw.max_a = max_g;
        gw.g_rows = nullptr;
        gw.mult_a = zs;
        gw.max_b = max_h;
        // both products of the chunk in one launch (dHidden's workgroups first)
        const int gwgrid = xcd_patch_grid(n_vt, n_ht);
        const char* what = "fused_head_bwd (dHidden, dW)";
        auto launch_pair = [&](auto mode_tag, auto bw_tag) {
            constexpr int kMode = decltype(mode_tag)::value;
            constexpr bool kBW = decltype(bw_tag)::value;
            return from_bf16 ? launch_head_pair(gemm_nt_pair_kernel<kMode, TRLK_BF16, kBW>, ghgrid, gh, gwgrid, gw, s, what)
                             : launch_head_pair(gemm_nt_pair_kernel<kMode, TRLK_F16, kBW>, ghgrid, gh, gwgrid, gw, s, what);
        };
        typedef std::integral_constant<int, 1> accumulate_t;
        typedef std::integral_constant<int, 2> round_t;
        if (last && !sums)
            rc = l.direct ? launch_pair(round_t{}, std::true_type{}) : launch_pair(round_t{}, std::false_type{});
        else
            rc = l.direct ? launch_pair(accumulate_t{}, std::true_type{}) : launch_pair(accumulate_t{}, std::false_type{});
        if (rc) return rc;
    }
    if (sums) {
        BeyondArgs beyond{};
        if (converts) {
            beyond = BeyondArgs{maxima + 3, maxima + 4, maxima + 2, a.weight, dzt, weight_stride, l.ld_n, d_g_logp, zs, int((vocab + 31) / 32), H};
            hipLaunchKernelGGL(beyond_rows_kernel, dim3(kBeyondBlocks), dim3(kBeyondThreads), 0, s, a.weight, weight_stride, V, H / 8,
                               maxima + 2, maxima + 3, maxima + 4);
        }
        const int64_t n = int64_t(N) * H;
        const dim3 grid(unsigned((n / 8 + kSumThreads - 1) / kSumThreads)), block(kSumThreads);
        uint16_t* out = static_cast<uint16_t*>(d_out_dhidden);
        if (from_bf16)
            hipLaunchKernelGGL(sum_slices_kernel<TRLK_BF16>, grid, block, 0, s, dh, l.slices, n, out, beyond);
        else
            hipLaunchKernelGGL(sum_slices_kernel<TRLK_F16>, grid, block, 0, s, dh, l.slices, n, out, beyond);
        return launch_status("fused_head_bwd (dHidden)");
    }
    return TRLK_OK;
}

extern "C" int trlk_split_bf16x3(const float* d_in, int64_t rows, int64_t cols, int64_t ld_in, int side, void* d_out,
                                 int64_t ld_out, trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(rows >= 0 && cols >= 1 && cols < (int64_t(1) << 28), TRLK_ERR_BAD_SHAPE, "split_bf16x3: bad shape %lld x %lld",
                 (long long)rows, (long long)cols);
    TRLK_REQUIRE(side == 0 || side == 1, TRLK_ERR_BAD_VALUE, "split_bf16x3: side must be 0 (A) or 1 (B), got %d", side);
    const int64_t cpad = round_up(cols, 8);
    TRLK_REQUIRE(ld_in >= cols && ld_out >= 6 * cpad && ld_out % 8 == 0, TRLK_ERR_BAD_STRIDE,
                 "split_bf16x3: row strides too short (in %lld for %lld columns, out %lld for %lld)", (long long)ld_in,
                 (long long)cols, (long long)ld_out, (long long)(6 * cpad));
    if (rows == 0) return TRLK_OK;
    TRLK_REQUIRE(d_in && d_out, TRLK_ERR_NULL_POINTER, "split_bf16x3: null pointer");
    TRLK_REQUIRE(rows < 65536 * int64_t(32768), TRLK_ERR_BAD_SHAPE, "split_bf16x3: too many rows");
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int64_t r0 = 0; r0 < rows; r0 += 65535) {  // grid.y limit
        const int64_t nr = rows - r0 < 65535 ? rows - r0 : 65535;
        hipLaunchKernelGGL(split_bf16x3_kernel, dim3(unsigned((cpad + 255) / 256), unsigned(nr)), dim3(256), 0, s,
                           d_in + r0 * ld_in, ld_in, nr, int(cols), int(cpad), side,
                           static_cast<uint16_t*>(d_out) + r0 * ld_out, ld_out);
    }
    return launch_status("split_bf16x3");
}

extern "C" int trlk_gemm_nt(const void* d_a, int64_t lda, const void* d_b, int64_t ldb, int dtype, int64_t m, int64_t n,
                            int64_t k, float* d_out, int64_t ldo, int accumulate, trlk_stream_t stream) {
    clear_error();
    TRLK_REQUIRE(dtype == TRLK_BF16 || dtype == TRLK_F16, TRLK_ERR_BAD_DTYPE, "gemm_nt: bf16 or fp16 operands (dtype code %d)",
                 dtype);
    TRLK_REQUIRE(m >= 0 && n >= 0 && k >= 8 && m < (int64_t(1) << 31) - BM && n < (int64_t(1) << 31) - BN &&
                     k < (int64_t(1) << 31) - BK,
                 TRLK_ERR_BAD_SHAPE, "gemm_nt: bad sizes m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
    TRLK_REQUIRE(k % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && lda >= k && ldb >= k && ldo >= n, TRLK_ERR_BAD_STRIDE,
                 "gemm_nt: k and the operands' row strides must be multiples of 8 elements (k=%lld lda=%lld ldb=%lld ldo=%lld)",
                 (long long)k, (long long)lda, (long long)ldb, (long long)ldo);
    // tile-relative operand offsets are 32-bit
    TRLK_REQUIRE(lda * 2 * BM < (int64_t(1) << 32) && ldb * 2 * BN < (int64_t(1) << 32), TRLK_ERR_BAD_STRIDE,
                 "gemm_nt: row strides too long (lda=%lld ldb=%lld)", (long long)lda, (long long)ldb);
    if (m == 0 || n == 0) return TRLK_OK;
    TRLK_REQUIRE(d_a && d_b && d_out, TRLK_ERR_NULL_POINTER, "gemm_nt: null pointer");
    TRLK_REQUIRE(reinterpret_cast<uintptr_t>(d_a) % 16 == 0 && reinterpret_cast<uintptr_t>(d_b) % 16 == 0, TRLK_ERR_BAD_STRIDE,
                 "gemm_nt: operands must be 16-byte aligned");
    GemmArgs g{};
    g.A = Operand{static_cast<const uint16_t*>(d_a), lda, int(m)};
    g.B = Operand{static_cast<const uint16_t*>(d_b), ldb, int(n)};
    g.M = int(m);
    g.N = int(n);
    g.K = int(k);
    g.out_f32 = d_out;
    g.ld_f32 = ldo;
    g.first = accumulate ? 0 : 1;
    g.mult_a = 1.f;
    const int grid = xcd_patch_grid(int((m + BM - 1) / BM), int((n + BN - 1) / BN));
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dtype == TRLK_BF16 ? launch_head(gemm_nt_kernel<TRLK_BF16>, grid, g, s, "gemm_nt")
                              : launch_head(gemm_nt_kernel<TRLK_F16>, grid, g, s, "gemm_nt");
}
