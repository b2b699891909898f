// W8A8 int8 x int8 -> int32 GEMM with the reference's fused f32 epilogue, gfx950.
//
// Semantics (crates/omni-kernel/src/int8_matmul.rs:145-373):
//   acc[m][n] = sum_k x[m][k] * w[n][k]                       exact int32
//   out[m][n] = f32(acc - x_sum[m] * w_zero[n]) * x_scale[m] * w_scale[n]
// left to right in f32 (store, :145-159), optionally + bias[n], stored as f32
// (the reference's output) or rounded once to f16.
//
// Two lowerings, as the reference has two (int8_dot and int8_dot_tile64):
//  * the int8 MFMA path (v_mfma_i32_32x32x32_i8). Both operands are
//    K-contiguous ("NT"), the layout the instruction wants for A and B alike:
//    each lane feeds 16 consecutive k bytes of one row of X and one row of W.
//    K tiles are staged through LDS with an XOR swizzle of the 16-byte chunk
//    index so both the global->LDS writes and the fragment reads are
//    bank-conflict free, and the epilogue runs on the accumulators in
//    registers, so no int32 accumulator array ever reaches HBM (the
//    reference's tile64 lowering round-trips one, int8_matmul.rs:423-439).
//    Three kernels cover the shapes: w8a8_ring_kernel (persistent, 256 x BN
//    tiles, a 3-4 stage LDS-DMA ring), w8a8_dma_kernel (512 x BN tiles, two
//    waves per SIMD) and w8a8_mfma_kernel (register-staged copies; any
//    K % 16 == 0). launch_w8a8_mfma picks one with a cost model.
//  * w8a8_scalar_kernel — v_dot4_i32_i8 per thread, the analog of the
//    reference's scalar int8_dot; it serves widths that are not a multiple of
//    16 and the OMNI_CONVROT_TENSOROPS=0 / OMNI_INT8_FORCE_SCALAR=1 override.
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace omni {

#ifdef OMNI_PHASE_TIMELINE
// Tile-phase timeline, in the library built with OMNI_PHASE_TIMELINE only
// (make -C omni-rs_amd timeline; bench.py --phase-timeline reads it): thread
// 0 of each ring-kernel workgroup b records, for its units r < 8, at
// g_phase[b * 64 + 8 r + k] the 100 MHz real-time counter at the K loop's
// start (k = 0, after the first barrier), the K loop's end (1), the
// epilogue's start (2, after the next unit's first copies) and end (3), the
// shader-clock counter at the K loop's start and end (4, 5), and at [b * 64 +
// 62, 63] the real-time counter at the workgroup's start and its first unit
// index. Vector stores from one lane, a few per unit.
__device__ unsigned long long g_phase[1024 * 64];
#define OMNI_PHASE(slot, value) \
    do {                        \
        if (phase && tid == 0) phase[(slot)] = (value); \
    } while (0)
#else
#define OMNI_PHASE(slot, value) \
    do {                        \
    } while (0)
#endif

namespace {

// crates/omni-kernel/src/int8_matmul.rs:156-158. Contraction is off so that
// (centered * row_scale) * w_scale and the bias add round as separate f32 ops.
__device__ __forceinline__ float w8a8_epilogue(int acc, int sum, int zero, float row_scale,
                                               float w_scale, float bias, bool has_bias) {
#pragma clang fp contract(off)
    int centered = acc - sum * zero;
    float t = (float)centered * row_scale;
    float v = t * w_scale;
    if (has_bias) v = v + bias;
    return v;
}

// v sign-extended from its low 24 bits (v itself when -2^23 <= v < 2^23):
// a product of two such values compiles to v_mul_i32_i24 (full rate).
__device__ __forceinline__ int sext24(int v) { return (int)((unsigned)v << 8) >> 8; }

// The same epilogue on a centred accumulator with the bias always added
// (a missing bias is -0.0, which leaves every value bit for bit unchanged).
__device__ __forceinline__ float w8a8_scale(int centered, float row_scale, float w_scale, float bias) {
#pragma clang fp contract(off)
    float t = (float)centered * row_scale;
    float v = t * w_scale;
    return v + bias;
}

// Nontemporal stores through a buffer resource (base, 4 GiB range): a
// per-lane byte offset in a vector register plus a wave-uniform byte offset
// in a scalar register, so a wave walking rows advances only the scalar part.
// Cache-policy bit 1 is the nontemporal hint on gfx940 and later.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t out_rsrc(void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)0xffffffff, 0x00020000);
}
__device__ __forceinline__ void buf_store_nt(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)voff, (int)soff, 2);
}
__device__ __forceinline__ void buf_store_nt(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, _Float16 v) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, (int)voff, (int)soff, 2);
}

// Output stores of the MFMA kernels: the output is written once and read by
// the next operator, not by this kernel, so it is stored nontemporally.
template <typename T>
__device__ __forceinline__ void stream_store(T* p, T v) {
    __builtin_nontemporal_store(v, p);
}

__device__ __forceinline__ void store_out(void* out, int64_t idx, float v, bool out_f16) {
    if (out_f16)
        static_cast<_Float16*>(out)[idx] = (_Float16)v;  // v_cvt_f16_f32: round to nearest even
    else
        static_cast<float*>(out)[idx] = v;
}

// ---------------------------------------------------------------------------
// Scalar lowering: one thread = one row x 4 consecutive columns, v_dot4 over K.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void w8a8_scalar_row(const W8A8Args& a, int64_t row, int64_t col0) {
    const int64_t words = a.width / 4;
    const u32* xr = reinterpret_cast<const u32*>(a.x + row * a.width);
    int acc[4] = {0, 0, 0, 0};
    const u32* wr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t c = col0 + j < a.columns ? col0 + j : a.columns - 1;
        wr[j] = reinterpret_cast<const u32*>(a.w + c * a.width);
    }
    for (int64_t k = 0; k < words; ++k) {
        const int xw = (int)xr[k];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_sdot4(xw, (int)wr[j][k], acc[j], false);
    }
    const float rs = a.x_scale[row];
    const int sum = a.x_sum ? a.x_sum[row] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t c = col0 + j;
        if (c >= a.columns) break;
        const int64_t idx = row * a.columns + c;
        if (a.acc_dump) a.acc_dump[idx] = acc[j];
        const int zero = a.w_zero ? a.w_zero[c] : 0;
        const float b = a.bias ? a.bias[c] : 0.0f;
        store_out(a.out, idx, w8a8_epilogue(acc[j], sum, zero, rs, a.w_scale[c], b, a.bias != nullptr),
                  a.out_f16);
    }
}

__global__ __launch_bounds__(256) void w8a8_scalar_kernel(W8A8Args a) {
    const int64_t col0 = ((int64_t)blockIdx.x * 64 + threadIdx.x) * 4;
    if (col0 >= a.columns) return;
    for (int64_t row = (int64_t)blockIdx.y * 4 + threadIdx.y; row < a.rows; row += (int64_t)gridDim.y * 4)
        w8a8_scalar_row(a, row, col0);
}


// ---------------------------------------------------------------------------
// MFMA lowering.
// ---------------------------------------------------------------------------

// Physical 16-byte chunk slot of logical chunk c in tile row r. gfx950 LDS
// has 64 four-byte banks and serves ds_read_b128 / ds_write_b128 16 lanes at
// a time, i.e. one 256-byte window: 256 / (16 * kChunks) consecutive rows
// share a window, so the XOR key is the row's window index. A fragment read
// (16 consecutive rows, one logical chunk) and a tile-row write (consecutive
// chunks of consecutive rows) then touch 16 distinct 16-byte bank groups.
template <int kChunks>
__device__ __forceinline__ int swz(int r, int c) {
    constexpr int kRowsPerWindow = 16 / kChunks;
    return c ^ ((r / kRowsPerWindow) & (kChunks - 1));
}

// Persistent int8-MFMA GEMM: 256 x BN output tiles (BN = 256, 192 or 128),
// 4 waves in a 2 x 2 grid, each wave a 128 x BN/2 block of 32x32 int32
// accumulators held in AGPRs; K tiles of 64 bytes.
//
// Every address is one per-thread base plus compile-time offsets: rows past
// M (or N) are clamped to the last row, so loads need no predicates (their
// accumulators are never stored); only a K tail (K % 64 != 0) zero-fills,
// in a separate instantiation.
//
// Pipeline, per output tile:
//  * K tiles t+1 .. t+PF are in flight in PF register sets while tile t is
//    multiplied out of LDS (double-buffered LDS, one barrier per K tile);
//  * after the last K tile, the workgroup's next output tile has its first PF
//    K tiles issued before this tile's epilogue runs, so the epilogue's stores
//    overlap the next tile's loads. The epilogue's per-row and per-column
//    values are staged in LDS with the first K tile, so reading them never
//    waits on the prefetch (vector loads complete in order).
template <int BN, int PF, bool KTAIL, bool OUT16, bool DUMP>
__global__ __launch_bounds__(256, 1) void w8a8_mfma_kernel(W8A8Args a) {
    constexpr int BM = 256, BK = 64;
    constexpr int WM = 128, WN = BN / 2;
    constexpr int FM = WM / 32, FN = WN / 32;
    constexpr int kALd = BM / 64;  // 16-byte loads per thread per K tile (A)
    constexpr int kBLd = BN / 64;  // (W)
    constexpr int kABuf = BM * BK, kBBuf = BN * BK;
    static_assert(BN % 64 == 0 && WN % 32 == 0, "tile shape");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* sA = smem;                       // [2][BM][BK]
    uint8_t* sB = smem + 2 * kABuf;           // [2][BN][BK]
    float* sRowScale = reinterpret_cast<float*>(smem + 2 * (kABuf + kBBuf));  // [BM]
    int* sRowSum = reinterpret_cast<int*>(sRowScale + BM);                    // [BM]
    float* sColScale = reinterpret_cast<float*>(sRowSum + BM);                // [BN]
    int* sColZero = reinterpret_cast<int*>(sColScale + BN);                   // [BN]
    float* sColBias = reinterpret_cast<float*>(sColZero + BN);                // [BN]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int tiles_m = (int)((a.rows + BM - 1) / BM);
    const int tiles_n = (int)((a.columns + BN - 1) / BN);
    const int total = tiles_m * tiles_n;
    const int K = (int)a.width;
    const int ktiles = (K + BK - 1) / BK;
    const bool has_bias = a.bias != nullptr;
    const bool has_zero = a.w_zero != nullptr;
    constexpr int kGroupM = 4;

    // Global->LDS copy slot of this thread: tile row ld_row + 64*i, chunk ld_c.
    const int ld_row = tid >> 2, ld_c = tid & 3;
    // Swizzled LDS offset of that slot (the XOR key (row / 4) % 4 does not
    // depend on i, since 64*i is a multiple of 16 rows).
    const int st_off = ld_row * BK + ((ld_c ^ ((ld_row >> 2) & 3)) << 4);
    // Fragment read bases for k steps 0 and 1 (32 bytes each): lane feeds row
    // (lane & 31), 16-byte half (lane >> 5).
    const int fr = lane & 31, fh = lane >> 5, fq = (fr >> 2) & 3;
    const int fragA0 = (wm * WM + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragA1 = (wm * WM + fr) * BK + (((2 + fh) ^ fq) << 4);
    const int fragB0 = (wn * WN + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragB1 = (wn * WN + fr) * BK + (((2 + fh) ^ fq) << 4);

    int L = xcd_remap(blockIdx.x, gridDim.x);
    if (L >= total) return;

    int64_t m0 = 0, n0 = 0;
    const uint8_t* gA;  // this thread's A row for slot 0, chunk ld_c, k = 0
    const uint8_t* gB;
    int offA[kALd], offB[kBLd];  // byte offsets of slots i > 0 from gA / gB
    auto setup_tile = [&](int l) {
        const int group_size = kGroupM * tiles_n;
        const int first_m = (l / group_size) * kGroupM;
        const int gm = min(tiles_m - first_m, kGroupM);
        // Integer division runs on the VALU; pin the (uniform) results to SGPRs.
        m0 = (int64_t)__builtin_amdgcn_readfirstlane(first_m + (l % group_size) % gm) * BM;
        n0 = (int64_t)__builtin_amdgcn_readfirstlane((l % group_size) / gm) * BN;
        const int64_t last_r = a.rows - 1, last_c = a.columns - 1;
        const int64_t r0 = min(m0 + ld_row, last_r);
        const int64_t c0 = min(n0 + ld_row, last_c);
        gA = a.x + r0 * K + ld_c * 16;
        gB = a.w + c0 * K + ld_c * 16;
#pragma unroll
        for (int i = 0; i < kALd; ++i) offA[i] = (int)((min(m0 + ld_row + 64 * i, last_r) - r0) * K);
#pragma unroll
        for (int i = 0; i < kBLd; ++i) offB[i] = (int)((min(n0 + ld_row + 64 * i, last_c) - c0) * K);
    };

    uint4 ra[PF][kALd];
    uint4 rb[PF][kBLd];
    auto load_tile = [&](int kt, uint4 (&xa)[kALd], uint4 (&xb)[kBLd]) {
        const int k0 = kt * BK;
        const bool in_k = !KTAIL || k0 + ld_c * 16 < K;
#pragma unroll
        for (int i = 0; i < kALd; ++i)
            xa[i] = in_k ? *reinterpret_cast<const uint4*>(gA + offA[i] + k0) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < kBLd; ++i)
            xb[i] = in_k ? *reinterpret_cast<const uint4*>(gB + offB[i] + k0) : make_uint4(0, 0, 0, 0);
    };
    auto store_tile = [&](int buf, const uint4 (&xa)[kALd], const uint4 (&xb)[kBLd]) {
        uint8_t* dA = sA + buf * kABuf + st_off;
        uint8_t* dB = sB + buf * kBBuf + st_off;
#pragma unroll
        for (int i = 0; i < kALd; ++i) *reinterpret_cast<uint4*>(dA + i * 64 * BK) = xa[i];
#pragma unroll
        for (int i = 0; i < kBLd; ++i) *reinterpret_cast<uint4*>(dB + i * 64 * BK) = xb[i];
    };
    // Epilogue values of a tile: thread tid holds row tid's and column tid's.
    float p_rs = 0.0f, p_cs = 0.0f, p_cb = 0.0f;
    int p_rsum = 0, p_cz = 0;
    auto load_params = [&]() {
        const int64_t row = min(m0 + tid, (int64_t)a.rows - 1);
        p_rs = a.x_scale[row];
        p_rsum = has_zero ? a.x_sum[row] : 0;
        if (tid < BN) {
            const int64_t col = min(n0 + tid, (int64_t)a.columns - 1);
            p_cs = a.w_scale[col];
            p_cz = has_zero ? a.w_zero[col] : 0;
            p_cb = has_bias ? a.bias[col] : 0.0f;
        }
    };
    auto store_params = [&]() {
        sRowScale[tid] = p_rs;
        sRowSum[tid] = p_rsum;
        if (tid < BN) {
            sColScale[tid] = p_cs;
            sColZero[tid] = p_cz;
            sColBias[tid] = p_cb;
        }
    };
    // Every prefetch is issued unconditionally, clamped to the last K tile,
    // so that all paths through the K loop carry the same sequence of loads:
    // vector loads complete in order, and the compiler can then wait for just
    // the oldest register set instead of all outstanding loads.
    auto issue_tile_start = [&]() {
        load_params();
#pragma unroll
        for (int u = 0; u < PF; ++u) load_tile(min(u, ktiles - 1), ra[u], rb[u]);
    };

    setup_tile(L);
    issue_tile_start();

    while (true) {
        v16i acc[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = v16i{};

        __syncthreads();  // the previous tile's epilogue is done with LDS
        store_params();
        store_tile(0, ra[0], rb[0]);
        __syncthreads();
        load_tile(min(PF, ktiles - 1), ra[0], rb[0]);

        for (int t0 = 0; t0 < ktiles; t0 += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int kt = t0 + u;
                const int buf = kt & 1;
                if (kt < ktiles) {
                    const uint8_t* tA = sA + buf * kABuf;
                    const uint8_t* tB = sB + buf * kBBuf;
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        v4i fa[FM], fb[FN];
                        const uint8_t* pa = tA + (ks ? fragA1 : fragA0);
                        const uint8_t* pb = tB + (ks ? fragB1 : fragB0);
#pragma unroll
                        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const v4i*>(pa + i * 32 * BK);
#pragma unroll
                        for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const v4i*>(pb + j * 32 * BK);
#pragma unroll
                        for (int i = 0; i < FM; ++i)
#pragma unroll
                            for (int j = 0; j < FN; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
                    }
                }
                // Tile kt+1 lives in register set (u+1) % PF; stage it, then
                // reuse the set for tile kt+1+PF.
                const int next = (u + 1) % PF;  // a constant once u is unrolled
                if (kt + 1 < ktiles) store_tile(buf ^ 1, ra[next], rb[next]);
                __syncthreads();
                load_tile(min(kt + 1 + PF, ktiles - 1), ra[next], rb[next]);
            }
        }

        // Issue the next tile's first K tiles, then run this tile's epilogue.
        const int64_t em0 = m0, en0 = n0;
        const int Ln = L + gridDim.x;
        const bool more = Ln < total;
        if (more) {
            setup_tile(Ln);
            issue_tile_start();
        }

        // 32x32 accumulator layout: lane holds column (lane & 31) and rows
        // 8*(r/4) + 4*(lane/32) + (r%4) of each 32x32 block. Offsets are
        // 32-bit, relative to the tile's first element (the host guarantees
        // 256 * columns < 2^31).
        const int N = (int)a.columns;
        const int64_t tile_base = em0 * a.columns + en0;
        // Keep the epilogue's lane-dependent index math inside the tile loop:
        // hoisted out of it, its values would stay live across the K loop.
        int efr = fr, efh = fh;
        asm volatile("" : "+v"(efr), "+v"(efh));
        const bool full = em0 + BM <= a.rows && en0 + BN <= a.columns;
        const int rows_left = (int)min((int64_t)BM, a.rows - em0);
        const int cols_left = (int)min((int64_t)BN, a.columns - en0);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int lr0 = wm * WM + i * 32 + 4 * efh;
                const int lc = wn * WN + j * 32 + efr;
                const float ws = sColScale[lc];
                const int zero = sColZero[lc];
                const float bias = sColBias[lc];
                const int base = lr0 * N + lc;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 s4 = *reinterpret_cast<const float4*>(sRowScale + lr0 + 8 * q);
                    const int4 z4 = *reinterpret_cast<const int4*>(sRowSum + lr0 + 8 * q);
                    const float rs[4] = {s4.x, s4.y, s4.z, s4.w};
                    const int rsum[4] = {z4.x, z4.y, z4.z, z4.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 4 * q + e;
                        const int dr = 8 * q + e;
                        const int off = base + dr * N;
                        const int v = acc[i][j][r];
                        const float o = w8a8_epilogue(v, rsum[e], zero, rs[e], ws, bias, has_bias);
                        if (full || (lr0 + dr < rows_left && lc < cols_left)) {
                            if constexpr (DUMP) a.acc_dump[tile_base + off] = v;
                            if constexpr (OUT16)
                                static_cast<_Float16*>(a.out)[tile_base + off] = (_Float16)o;
                            else
                                static_cast<float*>(a.out)[tile_base + off] = o;
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!more) break;
        L = Ln;
    }
}

// LDS-DMA GEMM (K % 64 == 0): one 128*WAVES_M x BN output tile per workgroup
// of 2*WAVES_M waves (512 x BN with 8 waves, two per SIMD, is the one the
// launcher uses: one wave's MFMAs cover the other's copies). K tiles are copied global -> LDS by global_load_lds_dwordx4:
// no staging registers and no LDS write instructions. A wave's copy
// instruction fills a contiguous 1 KiB block (16 tile rows of 64 bytes, lane
// l at byte 16*l), so the bank swizzle is applied on the global side: lane l
// reads logical chunk (l % 4) ^ ((l / 16) % 4) of row l / 4 of the block. The
// S stage buffers are distinct LDS arrays and the K loop is unrolled by S
// (S divides the K-tile count) so every copy and read names its array
// statically; the wait for K tile kt is vmcnt(copies issued after it),
// leaving S-2 later tiles in flight, then one barrier per K tile.
template <int BN, int WAVES_M>
struct DmaCfg {
    static constexpr int BM = 128 * WAVES_M, BK = 64;
    static constexpr int kWaves = 2 * WAVES_M;
    static constexpr int kStageBytes = (BM + BN) * BK;
    // 1 KiB copies (16 rows) per K tile: A's are spread over all waves; W's
    // over the first 4 waves (BN / 64 each).
    static constexpr int kACopies = BM / 16 / kWaves;
    static constexpr int kBCopies = BN / 64;
    static_assert(BM % (16 * kWaves) == 0, "A copies divide among waves");
};

template <int BN, int WAVES_M, int S, bool OUT16, bool DUMP>
__global__ __launch_bounds__(128 * WAVES_M, 512 / (128 * WAVES_M)) void w8a8_dma_kernel(W8A8Args a) {
    using C = DmaCfg<BN, WAVES_M>;
    constexpr int BM = C::BM, BK = C::BK;
    constexpr int WM = 128, WN = BN / 2;
    constexpr int FM = WM / 32, FN = WN / 32;
    static_assert(S >= 2 && S <= 3, "2 or 3 stages");
    static_assert(S == 2 || WAVES_M == 2, "uneven copy counts per wave need S == 2 (vmcnt(0))");
    __shared__ __attribute__((aligned(1024))) uint8_t st0[C::kStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t st1[C::kStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t st2[S > 2 ? C::kStageBytes : 1024];
    __shared__ __attribute__((aligned(16))) float sRowScale[BM];
    __shared__ __attribute__((aligned(16))) int sRowSum[BM];
    __shared__ float sColScale[BN];
    __shared__ int sColZero[BN];
    __shared__ float sColBias[BN];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;  // 2 waves across the columns
    const int tiles_m = (int)((a.rows + BM - 1) / BM);
    const int tiles_n = (int)((a.columns + BN - 1) / BN);
    const int K = (int)a.width;
    const int ktiles = K / BK;
    const bool has_bias = a.bias != nullptr;
    const bool has_zero = a.w_zero != nullptr;
    constexpr int kGroupM = 4;

    const int l = xcd_remap(blockIdx.x, tiles_m * tiles_n);
    const int group_size = kGroupM * tiles_n;
    const int first_m = (l / group_size) * kGroupM;
    const int gm = min(tiles_m - first_m, kGroupM);
    const int64_t m0 = (int64_t)__builtin_amdgcn_readfirstlane(first_m + (l % group_size) % gm) * BM;
    const int64_t n0 = (int64_t)__builtin_amdgcn_readfirstlane((l % group_size) / gm) * BN;

    // Copy sources: wave w copies A rows [16*kACopies*w, ...) as kACopies
    // blocks of 16 rows; waves 0..3 copy W rows [BN/4 * w, ...) as kBCopies
    // blocks. Rows past the matrix are clamped (their accumulators are never
    // stored).
    const int cp_row = lane >> 2;
    const int cp_chunk = (lane & 3) ^ ((lane >> 4) & 3);
    const uint8_t* srcA[C::kACopies];
    const uint8_t* srcB[C::kBCopies];
#pragma unroll
    for (int i = 0; i < C::kACopies; ++i) {
        const int64_t r = min(m0 + (wave * C::kACopies + i) * 16 + cp_row, a.rows - 1);
        srcA[i] = a.x + r * K + cp_chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < C::kBCopies; ++i) {
        const int64_t r = min(n0 + (wave & 3) * (BN / 4) + i * 16 + cp_row, a.columns - 1);
        srcB[i] = a.w + r * K + cp_chunk * 16;
    }
    // Copy K tile kt (clamped to the last, so that every K tile issues the
    // same number of copies) into stage buffer dst.
    auto copy_tile = [&](int kt, uint8_t* dst) {
        const int k0 = min(kt, ktiles - 1) * BK;
#pragma unroll
        for (int i = 0; i < C::kACopies; ++i)
            lds_copy16(srcA[i] + k0, dst + ((wave * C::kACopies + i) * 16) * BK);
        if (wave < 4) {
#pragma unroll
            for (int i = 0; i < C::kBCopies; ++i)
                lds_copy16(srcB[i] + k0, dst + BM * BK + (wave * (BN / 4) + i * 16) * BK);
        }
    };

    // Epilogue values, staged in LDS before the K loop (their loads are the
    // first vector-memory operations, so the K loop's waits cover them).
    {
        const int64_t row = min(m0 + tid, (int64_t)a.rows - 1);
        sRowScale[tid] = a.x_scale[row];
        sRowSum[tid] = has_zero ? a.x_sum[row] : 0;
        if (tid < BN) {
            const int64_t col = min(n0 + tid, (int64_t)a.columns - 1);
            sColScale[tid] = a.w_scale[col];
            sColZero[tid] = has_zero ? a.w_zero[col] : 0;
            sColBias[tid] = has_bias ? a.bias[col] : 0.0f;
        }
    }

    __syncthreads();  // params visible to all waves (before any copy is in flight)
    copy_tile(0, st0);
    if constexpr (S > 2) copy_tile(1, st1);

    // Fragment read bases (the same swizzled layout as the register-staged kernel).
    const int fr = lane & 31, fh = lane >> 5, fq = (fr >> 2) & 3;
    const int fragA0 = (wm * WM + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragA1 = (wm * WM + fr) * BK + (((2 + fh) ^ fq) << 4);
    const int fragB0 = BM * BK + (wn * WN + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragB1 = BM * BK + (wn * WN + fr) * BK + (((2 + fh) ^ fq) << 4);

    v16i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v16i{};

    auto stage = [&](int b) -> uint8_t* { return b == 0 ? st0 : b == 1 ? st1 : st2; };
    for (int t0 = 0; t0 < ktiles; t0 += S) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int kt = t0 + u;
            // K tiles kt .. kt+S-2 are in flight; wait for kt's copies and for
            // this wave's reads of the previous stage, then for every wave.
            s_waitcnt_vm<(S - 2) * (C::kACopies + C::kBCopies), true>();
            lds_barrier();  // all copies of kt landed; stage (u - 1) % S is free
            copy_tile(kt + S - 1, stage((u + S - 1) % S));
            const uint8_t* tb = stage(u);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                v4i fa[FM], fb[FN];
                const uint8_t* pa = tb + (ks ? fragA1 : fragA0);
                const uint8_t* pb = tb + (ks ? fragB1 : fragB0);
#pragma unroll
                for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const v4i*>(pa + i * 32 * BK);
#pragma unroll
                for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const v4i*>(pb + j * 32 * BK);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
        }
    }

    // 32x32 accumulator layout: lane holds column (lane & 31) and rows
    // 8*(r/4) + 4*(lane/32) + (r%4) of each 32x32 block. Offsets are 32-bit,
    // relative to the tile's first element (host: 256 * columns < 2^31).
    const int N = (int)a.columns;
    const int64_t tile_base = m0 * a.columns + n0;
    const bool full = m0 + BM <= a.rows && n0 + BN <= a.columns;
    const int rows_left = (int)min((int64_t)BM, a.rows - m0);
    const int cols_left = (int)min((int64_t)BN, a.columns - n0);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int lr0 = wm * WM + i * 32 + 4 * fh;
            const int lc = wn * WN + j * 32 + fr;
            const float ws = sColScale[lc];
            const int zero = sColZero[lc];
            const float bias = sColBias[lc];
            const int base = lr0 * N + lc;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 s4 = *reinterpret_cast<const float4*>(sRowScale + lr0 + 8 * q);
                const int4 z4 = *reinterpret_cast<const int4*>(sRowSum + lr0 + 8 * q);
                const float rs[4] = {s4.x, s4.y, s4.z, s4.w};
                const int rsum[4] = {z4.x, z4.y, z4.z, z4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int dr = 8 * q + e;
                    const int off = base + dr * N;
                    const int v = acc[i][j][4 * q + e];
                    const float o = w8a8_epilogue(v, rsum[e], zero, rs[e], ws, bias, has_bias);
                    if (full || (lr0 + dr < rows_left && lc < cols_left)) {
                        if constexpr (DUMP) a.acc_dump[tile_base + off] = v;
                        if constexpr (OUT16)
                            stream_store(static_cast<_Float16*>(a.out) + tile_base + off, (_Float16)o);
                        else
                            stream_store(static_cast<float*>(a.out) + tile_base + off, o);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The clamped copies of the last K tiles may still be landing in LDS;
    // drain them before the workgroup's LDS is released.
    s_waitcnt_vm<0>();
}

// Persistent LDS-DMA ring GEMM (K % 64 == 0, S divides the K-tile count).
// One workgroup of 4 waves per CU walks 256 x BN output tiles; each wave owns
// a 128 x BN/2 block of 32x32 int32 accumulators (AGPRs). K tiles of 64 bytes
// reach LDS through global_load_lds_dwordx4 into an S-stage ring (distinct
// LDS arrays so each copy and read names its stage statically). Per K tile
// the schedule is
//   MFMAs (tile kt, k step 0)    | fragment reads (tile kt, k step 1)
//   wait for tile kt+1's copies, barrier (stage kt % S is now fully read)
//   MFMAs (tile kt, k step 1)    | copy tile kt+S into stage kt % S,
//                                | fragment reads (tile kt+1, k step 0)
// so S-1 tiles are in flight across the barrier: a copy is issued about S-1
// K tiles before its data is read.
// with one read and one copy issued after each MFMA, so every LDS read has
// most of an MFMA group to land, no copy burst holds up an MFMA, and the only
// barrier sits between two MFMA groups. (With one wave per SIMD a copy that
// waits for the CU's texture unit blocks its wave's next MFMA: measured on
// MI355X, copies issued in a burst and MFMAs do not overlap at all.) The
// next output tile's first copies are issued before this tile's epilogue,
// whose per-row and per-column values sit in a parity-double-buffered LDS
// block. Epilogue stores of partial tiles are
// unconditional too: rows and columns past the matrix were loaded clamped to
// the last row and column, so their values equal the last row's (column's)
// and are stored there, a duplicate write of the same value.
//
// PAIR = true refills the ring two K tiles at a time. Each copy instruction
// reads 16 rows x 64 bytes, half of each 128-byte cache line; issued one by
// one, K tile kt+1's copy of a row comes a full K tile after kt's, by which
// time the CU has streamed ~56 KB of other lines through its L1 and the line
// is fetched from L2 a second time. The pair schedule issues copy j of tiles
// 2p and 2p+1 back to back, so the second half-line read hits the line the
// first just brought in: L2->L1 traffic halves (measured on MI355X: the K
// loop's copies cost 12 % instead of 27 % of a 4096x12288x3072 GEMM). With
// S = 5 slots, pair (t, t+1) goes into slots t%5 and (t+1)%5 once both are
// free: the first half of its copies after the barrier of tile t-4, the rest
// in the first half of tile t-3, so tile t is issued at least 2.5 K tiles
// before it is read. The K loop is unrolled over 2S tiles (slot and pair
// parity compile-time) with a uniform exit, so any K % 64 == 0 is taken.
//
// SK (split K, `splits` > 1): the work units are (tile, split) pairs, split s
// covering K tiles [s * kts, min(ktiles, (s + 1) * kts)) with kts =
// ceil(ktiles / splits) (the host keeps every split non-empty); a unit
// stores its raw int32 sums to partial[s][rows][columns] and
// w8a8_split_reduce_kernel adds the splits (int32 wrapping sums are exact in
// any order) and applies the epilogue, so the output is bit-identical to the
// unsplit kernel's. Units of one split are consecutive.
//
// NW = 8: eight waves (two per SIMD) share the ring, 4 x 2 of them over the
// tile, each owning half as many accumulators, so one wave's MFMAs can issue
// while the other waits on LDS or the barrier.
template <int BN, int S, bool OUT16, bool DUMP, bool PAIR = false, bool SK = false, int NW = 4>
__global__ __launch_bounds__(64 * NW, 1) void w8a8_ring_kernel(W8A8Args a, int splits) {
    constexpr int BM = 256, BK = 64;
    constexpr int WMW = NW / 2, WNW = 2;      // waves along M and N
    constexpr int WM = BM / WMW, WN = BN / WNW;
    constexpr int FM = WM / 32, FN = WN / 32;
    constexpr int kRows = BM + BN;            // tile rows per stage (A then W)
    constexpr int kStage = kRows * BK;
    constexpr int kCpw = kRows / 16 / NW;     // 1 KiB copies per wave per K tile
    static_assert(NW == 4 || NW == 8, "four or eight waves");
    static_assert(kRows % (16 * NW) == 0 && WN % 32 == 0 && WM % 32 == 0, "tile shape");
    static_assert(FM + FN <= FM * FN && kCpw <= FM * FN, "one read and one copy per MFMA slot");
    static_assert(S >= 3 && S <= 5, "3 to 5 stages");
    static_assert(!PAIR || S == 5, "the pair schedule is laid out for 5 slots");
    // Pair schedule: copy units (copy j of both tiles of a pair) issued after
    // the barrier of the refill tile (kPU of them) and in the next tile's
    // first half (the rest), spread evenly over the MFMAs.
    constexpr int kPU = (kCpw + 1) / 2, kPU2 = kCpw - kPU;
    constexpr int kPStep1 = FM * FN / kPU, kPStep2 = kPU2 ? FM * FN / kPU2 : 1;
    static_assert(!PAIR || (kPStep1 >= 1 && kPStep2 >= 1), "pair units per MFMA group");
    __shared__ __attribute__((aligned(1024))) uint8_t st0[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t st1[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t st2[kStage];
    __shared__ __attribute__((aligned(1024))) uint8_t st3[S > 3 ? kStage : 1024];
    __shared__ __attribute__((aligned(1024))) uint8_t st4[S > 4 ? kStage : 1024];
    __shared__ __attribute__((aligned(16))) float sRowScale[2][BM];
    __shared__ __attribute__((aligned(16))) int sRowSum[2][BM];
    __shared__ float sColScale[2][BN];
    __shared__ int sColZero[2][BN];
    __shared__ float sColBias[2][BN];
    // Nonzero when a row sum or zero point of the tile lies outside
    // [-2^23, 2^23) (the epilogue then multiplies them in 32 bits), and when
    // some zero point of the tile is not 0 (else it drops the sum * zero term).
    __shared__ int sWide[2];
    __shared__ int sZero[2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: an SGPR
    const int wm = wave / WNW, wn = wave % WNW;
    const int tiles_m = (int)((a.rows + BM - 1) / BM);
    const int tiles_n = (int)((a.columns + BN - 1) / BN);
    const int total = tiles_m * tiles_n;
    const int units = SK ? total * splits : total;
    const int K = (int)a.width;
    const int ktiles_all = K / BK;
    const int kts = SK ? (ktiles_all + splits - 1) / splits : ktiles_all;
    // K tiles [kbase, kbase + ktiles) of the unit being copied; its split.
    int kbase = 0, ktiles = ktiles_all, split = 0;
    const bool has_bias = a.bias != nullptr;
    const bool has_zero = a.w_zero != nullptr;
    constexpr int kGroupM = 4;

    auto stage = [&](int s) -> uint8_t* {
        return s == 0 ? st0 : s == 1 ? st1 : s == 2 ? st2 : s == 3 ? st3 : st4;
    };

    // Copy c (0 .. kRows/16) fills stage rows 16c .. 16c+15; this wave owns
    // copies wave*kCpw + j. Lane l reads logical chunk (l%4) ^ ((l/16)%4) of
    // row l/4, landing at physical chunk l%4 (the fragment reads' swizzle).
    // Copies are inline-assembly LDS-DMA (lds_copy16_saddr): the compiler
    // sees no LDS write in flight and adds no vmcnt(0) drain of its own
    // before the ring's LDS reads and writes; the explicit waits below order
    // every copy. Each reads a wave-uniform base (x or W plus the K tile
    // offset) plus a 32-bit per-lane byte offset (the host keeps rows * K and
    // columns * K below 2^32).
    const int cp_row = lane >> 2;
    const int cp_chunk = (lane & 3) ^ ((lane >> 4) & 3);
    // Stage row block (16 rows) of this wave's copy j (wave-uniform).
    auto copy_block = [&](int j) { return wave * kCpw + j; };
    unsigned voff[kCpw];
    const unsigned stage_lds[5] = {lds_addr(st0), lds_addr(st1), lds_addr(st2), S > 3 ? lds_addr(st3) : 0u,
                                   S > 4 ? lds_addr(st4) : 0u};
    int64_t m0 = 0, n0 = 0;
    float p_rs = 0.0f, p_cs = 0.0f, p_cb = 0.0f;
    int p_rsum = 0, p_cz = 0;
    auto tile_origin = [&](int u, int64_t& tm0, int64_t& tn0) {
        const int l = SK ? u % total : u;
        const int group_size = kGroupM * tiles_n;
        const int first_m = (l / group_size) * kGroupM;
        const int gm = min(tiles_m - first_m, kGroupM);
        tm0 = (int64_t)__builtin_amdgcn_readfirstlane(first_m + (l % group_size) % gm) * BM;
        tn0 = (int64_t)__builtin_amdgcn_readfirstlane((l % group_size) / gm) * BN;
    };
    auto unit_k = [&](int u) {
        if constexpr (SK) {
            split = __builtin_amdgcn_readfirstlane(u / total);
            kbase = split * kts;
            ktiles = min(kts, ktiles_all - kbase);
        }
    };
    // Copy sources of the tile at (m0, n0). Which matrix a copy reads and its
    // first row are wave-uniform (scalar selects, no branches).
    auto setup_copies = [&]() {
#pragma unroll
        for (int j = 0; j < kCpw; ++j) {
            const int c16 = copy_block(j) * 16;  // first stage row of copy j
            const bool is_a = c16 < BM;
            const int64_t first = is_a ? m0 + c16 : n0 + (c16 - BM);
            const int64_t last = is_a ? a.rows - 1 : a.columns - 1;
            const int64_t row = min(first + cp_row, last);
            voff[j] = (unsigned)(row * K) + cp_chunk * 16;
        }
    };
    // Epilogue values of the tile at (pm0, pn0) into registers: thread tid
    // holds row tid's and column tid's.
    // A missing bias is stored as -0.0: v + (-0.0) == v for every v the
    // epilogue makes (it is never a signalling NaN), so the add is
    // unconditional and the result is bit-identical to skipping it.
    auto load_params = [&](int64_t pm0, int64_t pn0) {
        if (tid < BM) {
            const int64_t row = min(pm0 + tid, a.rows - 1);
            p_rs = a.x_scale[row];
            p_rsum = has_zero ? a.x_sum[row] : 0;
        }
        if (tid < BN) {
            const int64_t col = min(pn0 + tid, a.columns - 1);
            p_cs = a.w_scale[col];
            p_cz = has_zero ? a.w_zero[col] : 0;
            p_cb = has_bias ? a.bias[col] : -0.0f;
        }
    };
    auto fits24 = [](int v) { return (unsigned)v + (1u << 23) < (1u << 24); };
    auto store_params = [&](int p) {
        if (tid < BM) {
            sRowScale[p][tid] = p_rs;
            sRowSum[p][tid] = p_rsum;
        }
        if (tid < BN) {
            sColScale[p][tid] = p_cs;
            sColZero[p][tid] = p_cz;
            sColBias[p][tid] = p_cb;
        }
        if (!fits24(p_rsum) || (tid < BN && !fits24(p_cz))) sWide[p] = 1;
        if (tid < BN && p_cz != 0) sZero[p] = 1;
    };
    auto copy_one = [&](int kt, int s, int j) {
        const int k0 = (kbase + min(kt, ktiles - 1)) * BK;
        const bool is_a = copy_block(j) * 16 < BM;  // wave-uniform
        const uint8_t* base = (is_a ? a.x : a.w) + k0;
        lds_copy16_saddr(voff[j], base, stage_lds[s] + copy_block(j) * 1024);
    };
    auto copy_tile = [&](int kt, int s) {
#pragma unroll
        for (int j = 0; j < kCpw; ++j) copy_one(kt, s, j);
    };

    // Fragment read offsets within a stage, k steps 0 and 1.
    const int fr = lane & 31, fh = lane >> 5, fq = (fr >> 2) & 3;
    const int fragA0 = (wm * WM + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragA1 = (wm * WM + fr) * BK + (((2 + fh) ^ fq) << 4);
    const int fragB0 = BM * BK + (wn * WN + fr) * BK + (((0 + fh) ^ fq) << 4);
    const int fragB1 = BM * BK + (wn * WN + fr) * BK + (((2 + fh) ^ fq) << 4);
    v4i fa0[FM], fb0[FN], fa1[FM], fb1[FN];
    // Fragment idx < FM is A fragment idx, else B fragment idx - FM.
    auto read_frag = [&](int s, int ks, int idx, v4i (&fa)[FM], v4i (&fb)[FN]) {
        if (idx < FM)
            fa[idx] = *reinterpret_cast<const v4i*>(stage(s) + (ks ? fragA1 : fragA0) + idx * 32 * BK);
        else
            fb[idx - FM] = *reinterpret_cast<const v4i*>(stage(s) + (ks ? fragB1 : fragB0) + (idx - FM) * 32 * BK);
    };
    auto read_frags = [&](int s, int ks, v4i (&fa)[FM], v4i (&fb)[FN]) {
        const uint8_t* pa = stage(s) + (ks ? fragA1 : fragA0);
        const uint8_t* pb = stage(s) + (ks ? fragB1 : fragB0);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const v4i*>(pa + i * 32 * BK);
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const v4i*>(pb + j * 32 * BK);
    };

    // Copy unit j of the pair (t, t+1): copy j of both tiles, back to back.
    auto copy_unit = [&](int t, int st, int j) {
        copy_one(t, st, j);
        copy_one(t + 1, (st + 1) % S, j);
    };
    // The ring's first fill: S tiles, or (pairs) tiles 0..3, slot 4 empty.
    auto prologue = [&]() {
        if constexpr (PAIR) {
#pragma unroll
            for (int j = 0; j < kCpw; ++j) copy_unit(0, 0, j);
#pragma unroll
            for (int j = 0; j < kCpw; ++j) copy_unit(2, 2, j);
        } else {
#pragma unroll
            for (int u = 0; u < S; ++u) copy_tile(u, u);
        }
    };

    int L = xcd_remap(blockIdx.x, gridDim.x);
    if (L >= units) return;
#ifdef OMNI_PHASE_TIMELINE
    unsigned long long* phase = blockIdx.x < 1024 ? g_phase + blockIdx.x * 64 : nullptr;
    int unit_no = 0;
#endif
    OMNI_PHASE(62, __builtin_amdgcn_s_memrealtime());
    OMNI_PHASE(63, (unsigned long long)L);
    if (tid == 0) sWide[0] = sWide[1] = sZero[0] = sZero[1] = 0;
    __syncthreads();
    tile_origin(L, m0, n0);
    unit_k(L);
    setup_copies();
    load_params(m0, n0);
    store_params(0);
    prologue();
    int parity = 0;

    while (true) {
        const int Ln = L + gridDim.x;
        const bool more = Ln < units;
        int64_t nm0 = 0, nn0 = 0;
        if (more) {
            // The next tile's epilogue values, loaded a whole tile early.
            tile_origin(Ln, nm0, nn0);
            load_params(nm0, nn0);
        }
        v16i acc[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = v16i{};

        // Tile 0's copies (and the parameter stores) visible to every wave.
        // Pairs: tile 0's last copy is followed by tile 1's and pair (2, 3).
        s_waitcnt_vm<PAIR ? 2 * kCpw + 1 : (S - 1) * kCpw, true>();
        lds_barrier();
        // Every wave is past the previous tile's epilogue: its flag may be
        // cleared for the tile after this one (store_params(parity ^ 1)
        // comes after this K loop's barriers).
        if (tid == 0) sWide[parity ^ 1] = sZero[parity ^ 1] = 0;
#ifdef OMNI_PHASE_TIMELINE
        if (unit_no >= 8) phase = nullptr;
        OMNI_PHASE(8 * unit_no + 0, __builtin_amdgcn_s_memrealtime());
        OMNI_PHASE(8 * unit_no + 4, __builtin_amdgcn_s_memtime());
#endif
        read_frags(0, 0, fa0, fb0);

        if constexpr (PAIR) {
            for (int t0 = 0; t0 < ktiles; t0 += 2 * S) {
#pragma unroll
                for (int v = 0; v < 2 * S; ++v) {
                    const int kt = t0 + v;
                    if (v > 0 && kt >= ktiles) break;  // uniform
                    const int u = v % S;               // t0 is a multiple of 2S
                    // k step 0 | fragment reads of k step 1; odd tiles also
                    // issue the second part of pair (kt+3, kt+4).
#pragma unroll
                    for (int q = 0; q < FM * FN; ++q) {
                        const int i = q / FN, j = q % FN;
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa0[i], fb0[j], acc[i][j], 0, 0, 0);
                        if (q < FM + FN) read_frag(u, 1, q, fa1, fb1);
                        if ((v % 2) == 1 && q % kPStep2 == 0 && q / kPStep2 < kPU2)
                            copy_unit(kt + S - 2, (u + S - 2) % S, kPU + q / kPStep2);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    // Tile kt+1 landed. Even kt: it ends pair (kt, kt+1),
                    // followed by all of pair (kt+2, kt+3). Odd kt: it
                    // starts pair (kt+1, kt+2), followed by that pair's last
                    // copy and all of pair (kt+3, kt+4).
                    if ((v % 2) == 0)
                        s_waitcnt_vm<2 * kCpw, true>();
                    else
                        s_waitcnt_vm<2 * kCpw + 1, true>();
                    lds_barrier();  // slot u is read
                    // k step 1 | fragment reads of tile kt+1, k step 0; even
                    // tiles also issue the first part of pair (kt+4, kt+5)
                    // into slots (kt-1)%S (free since the last barrier but
                    // one) and u.
#pragma unroll
                    for (int q = 0; q < FM * FN; ++q) {
                        const int i = q / FN, j = q % FN;
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa1[i], fb1[j], acc[i][j], 0, 0, 0);
                        if ((v % 2) == 0 && q % kPStep1 == 0 && q / kPStep1 < kPU)
                            copy_unit(kt + S - 1, (u + S - 1) % S, q / kPStep1);
                        if (q < FM + FN) read_frag((u + 1) % S, 0, q, fa0, fb0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        } else
        for (int t0 = 0; t0 < ktiles; t0 += S) {
#pragma unroll
            for (int u = 0; u < S; ++u) {
                const int kt = t0 + u;
                // k step 0 of tile kt: after each of the first FM+FN MFMAs,
                // one fragment read of k step 1. The scheduling barriers pin
                // that order: a vector-memory or LDS instruction that cannot
                // issue stalls the wave's next MFMA, so each one is placed
                // behind an MFMA rather than in a burst.
#pragma unroll
                for (int q = 0; q < FM * FN; ++q) {
                    const int i = q / FN, j = q % FN;
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa0[i], fb0[j], acc[i][j], 0, 0, 0);
                    if (q < FM + FN) read_frag(u, 1, q, fa1, fb1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                s_waitcnt_vm<(S - 2) * kCpw, true>();
                lds_barrier();  // tile kt+1 landed everywhere; stage u is read
                // k step 1: after each MFMA, one copy of tile kt+S into stage
                // u and one fragment read of tile kt+1, k step 0.
#pragma unroll
                for (int q = 0; q < FM * FN; ++q) {
                    const int i = q / FN, j = q % FN;
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa1[i], fb1[j], acc[i][j], 0, 0, 0);
                    if (q < kCpw) copy_one(kt + S, u, q);
                    if (q < FM + FN) read_frag((u + 1) % S, 0, q, fa0, fb0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }

        const int64_t em0 = m0, en0 = n0;
        const int esplit = split;
#ifdef OMNI_PHASE_TIMELINE
        OMNI_PHASE(8 * unit_no + 1, __builtin_amdgcn_s_memrealtime());
        OMNI_PHASE(8 * unit_no + 5, __builtin_amdgcn_s_memtime());
#endif
        // Every wave is done reading the ring before the next tile's copies
        // (the clamped copies still in flight land first: one wave's loads
        // complete in issue order, and each wave writes its own LDS chunks).
        s_waitcnt_vm<PAIR ? 2 * kCpw : (S - 1) * kCpw, true>();
        lds_barrier();
        if (more) {
            m0 = nm0;
            n0 = nn0;
            unit_k(Ln);
            setup_copies();
            store_params(parity ^ 1);
            prologue();
        }
#ifdef OMNI_PHASE_TIMELINE
        OMNI_PHASE(8 * unit_no + 2, __builtin_amdgcn_s_memrealtime());
#endif

        // Epilogue. 32x32 accumulator layout: lane holds column (lane & 31)
        // and rows 8*(r/4) + 4*(lane/32) + (r%4) of each 32x32 block.
        // acc - sum * zero is exact in 24-bit multiplies (full rate) when
        // every row sum and zero point of the tile lies in [-2^23, 2^23),
        // otherwise it is formed with 32-bit multiplies (quarter rate), and
        // it is acc itself when every zero point of the tile is 0. Full tiles
        // store through a wave-uniform row base (scalar registers) plus one
        // per-lane byte offset computed once, and take the bias add only when
        // there is a bias: per element a convert, two multiplies and a store.
        // Partial tiles (and the accumulator dump) take the general path:
        // clamped rows and columns, byte offsets from the tile's first
        // element (the host guarantees 256 * columns * 4 < 2^32), a missing
        // bias added as -0.0 (which leaves every value bit for bit as it was).
        const int N = (int)a.columns;
        constexpr int kES = OUT16 ? 2 : 4;
        const int64_t tile_base = em0 * a.columns + en0;
        int efr = fr, efh = fh;
        asm volatile("" : "+v"(efr), "+v"(efh));
        if constexpr (SK) {
            // Raw sums of this split (plain stores: the reduction reads them
            // back right after), in-bounds rows and columns only.
            int32_t* pt = a.partial + (int64_t)esplit * a.rows * a.columns + tile_base;
            const int rows_last = (int)min((int64_t)BM, a.rows - em0) - 1;
            const int cols_last = (int)min((int64_t)BN, a.columns - en0) - 1;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int lc = wn * WN + j * 32 + efr;
                    const int lr0 = wm * WM + i * 32 + 4 * efh;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int lr = lr0 + 8 * (r >> 2) + (r & 3);
                        if (lc <= cols_last && lr <= rows_last) pt[(unsigned)(lr * N + lc)] = acc[i][j][r];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#ifdef OMNI_PHASE_TIMELINE
            OMNI_PHASE(8 * unit_no + 3, __builtin_amdgcn_s_memrealtime());
            ++unit_no;
#endif
            if (!more) break;
            L = Ln;
            parity ^= 1;
            continue;
        }
        const bool full = em0 + BM <= a.rows && en0 + BN <= a.columns;
        const bool wide = __builtin_amdgcn_readfirstlane(sWide[parity]) != 0;
        const bool zeros = has_zero && __builtin_amdgcn_readfirstlane(sZero[parity]) != 0;
        const int rows_last = (int)min((int64_t)BM, a.rows - em0) - 1;
        const int cols_last = (int)min((int64_t)BN, a.columns - en0) - 1;
        const float* pRowScale = sRowScale[parity];
        const int* pRowSum = sRowSum[parity];
        const float* pColScale = sColScale[parity];
        const int* pColZero = sColZero[parity];
        const float* pColBias = sColBias[parity];
        char* out_tile = static_cast<char*>(a.out) + tile_base * kES;
        int32_t* dump = DUMP ? a.acc_dump + tile_base : nullptr;
        auto store_elem = [&](char* p, float o) {
            if constexpr (OUT16)
                stream_store(reinterpret_cast<_Float16*>(p), (_Float16)o);
            else
                stream_store(reinterpret_cast<float*>(p), o);
        };
        // General path: partial tiles and the accumulator dump.
        auto epilogue = [&](auto clamp_tag, auto wide_tag) {
            constexpr bool CLAMP = decltype(clamp_tag)::value;
            constexpr bool WIDE = decltype(wide_tag)::value;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int lr0 = wm * WM + i * 32 + 4 * efh;
                    int lc = wn * WN + j * 32 + efr;
                    if constexpr (CLAMP) lc = min(lc, cols_last);
                    const float ws = pColScale[lc];
                    const int zero = pColZero[lc];
                    const int zero24 = sext24(zero);
                    const float bias = pColBias[lc];
                    unsigned boff = (unsigned)(lr0 * N + lc) * kES;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 s4 = *reinterpret_cast<const float4*>(pRowScale + lr0 + 8 * q);
                        const int4 z4 = *reinterpret_cast<const int4*>(pRowSum + lr0 + 8 * q);
                        const float rs[4] = {s4.x, s4.y, s4.z, s4.w};
                        const int rsum[4] = {z4.x, z4.y, z4.z, z4.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            unsigned off;
                            if constexpr (CLAMP)
                                off = (unsigned)(min(lr0 + 8 * q + e, rows_last) * N + lc) * kES;
                            else
                                off = boff + (unsigned)((8 * q + e) * N) * kES;
                            const int v = acc[i][j][4 * q + e];
                            // Wrapping int32 arithmetic, as the reference's
                            // i32 ops; the 24-bit multiply keeps the low 32
                            // bits of the exact product.
                            const unsigned prod = WIDE ? (unsigned)rsum[e] * (unsigned)zero
                                                       : (unsigned)sext24(rsum[e]) * (unsigned)zero24;
                            const int centered = (int)((unsigned)v - prod);
                            const float o = w8a8_scale(centered, rs[e], ws, bias);
                            if constexpr (DUMP) dump[off / kES] = v;
                            store_elem(out_tile + off, o);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        // Full tiles: ZMODE 0 = no zero-point term, 1 = 24-bit, 2 = 32-bit.
        auto epilogue_full = [&](auto zmode_tag, auto bias_tag) {
            constexpr int ZMODE = decltype(zmode_tag)::value;
            constexpr bool BIAS = decltype(bias_tag)::value;
            const unsigned lane_off = (unsigned)((4 * efh) * N + wn * WN + efr) * kES;
            const __amdgpu_buffer_rsrc_t rsrc = out_rsrc(out_tile);
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int lc = wn * WN + j * 32 + efr;
                    const int lr0 = wm * WM + i * 32 + 4 * efh;
                    const float ws = pColScale[lc];
                    const int zero = ZMODE ? pColZero[lc] : 0;
                    const int zero24 = sext24(zero);
                    const float bias = BIAS ? pColBias[lc] : 0.0f;
                    // Scalar byte offset of row wm*WM + i*32 + 8q + e of the
                    // block (the lane's 4*(lane/32) rows are in lane_off),
                    // advanced by scalar adds; the empty asm keeps the chain
                    // sequential so 192 offsets are not precomputed and spilled.
                    unsigned soff = (unsigned)((wm * WM + i * 32) * N + j * 32) * kES;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 s4 = *reinterpret_cast<const float4*>(pRowScale + lr0 + 8 * q);
                        const float rs[4] = {s4.x, s4.y, s4.z, s4.w};
                        int rsum[4] = {0, 0, 0, 0};
                        if constexpr (ZMODE != 0) {
                            const int4 z4 = *reinterpret_cast<const int4*>(pRowSum + lr0 + 8 * q);
                            rsum[0] = z4.x; rsum[1] = z4.y; rsum[2] = z4.z; rsum[3] = z4.w;
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const unsigned so = soff;
                            soff += (unsigned)(e == 3 ? 5 * N : N) * kES;
                            asm volatile("" : "+s"(soff));
                            const int v = acc[i][j][4 * q + e];
                            int centered = v;
                            if constexpr (ZMODE == 1)
                                centered = (int)((unsigned)v - (unsigned)sext24(rsum[e]) * (unsigned)zero24);
                            else if constexpr (ZMODE == 2)
                                centered = (int)((unsigned)v - (unsigned)rsum[e] * (unsigned)zero);
                            float o;
                            {
#pragma clang fp contract(off)
                                const float t = (float)centered * rs[e];
                                o = t * ws;
                                if constexpr (BIAS) o = o + bias;
                            }
                            if constexpr (OUT16)
                                buf_store_nt(rsrc, lane_off, so, (_Float16)o);
                            else
                                buf_store_nt(rsrc, lane_off, so, o);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        auto full_epilogue = [&](auto zmode_tag) {
            if (has_bias)
                epilogue_full(zmode_tag, std::true_type{});
            else
                epilogue_full(zmode_tag, std::false_type{});
        };
        if (DUMP || !full) {
            if (wide)
                epilogue(std::true_type{}, std::true_type{});
            else
                epilogue(std::true_type{}, std::false_type{});
        } else if (!zeros) {
            full_epilogue(std::integral_constant<int, 0>{});
        } else if (!wide) {
            full_epilogue(std::integral_constant<int, 1>{});
        } else {
            full_epilogue(std::integral_constant<int, 2>{});
        }
#ifdef OMNI_PHASE_TIMELINE
        OMNI_PHASE(8 * unit_no + 3, __builtin_amdgcn_s_memrealtime());
        ++unit_no;
#endif
        if (!more) break;
        L = Ln;
        parity ^= 1;
    }
    // Copies of clamped K tiles may still be landing; drain before exit.
    s_waitcnt_vm<0>();
}

// OMNI_W8A8_TILE=<n> pins one tile configuration (tuning and test aid;
// 0 or unset = the shape heuristic).
int w8a8_tile_override() { return knob(Knob::W8A8Tile, 0); }

template <int BN, int PF, bool KTAIL, bool OUT16, bool DUMP>
hipError_t launch_cfg(const W8A8Args& a, hipStream_t stream) {
    auto kernel = w8a8_mfma_kernel<BN, PF, KTAIL, OUT16, DUMP>;
    const size_t smem = 2 * (size_t)(256 + BN) * 64 + (size_t)(2 * 256 + 3 * BN) * 4;
    // Dynamic LDS above 64 KiB needs an opt-in; setting it is idempotent.
    static std::atomic<bool> configured{false};
    if (!configured.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return e;
        configured.store(true, std::memory_order_release);
    }
    const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + BN - 1) / BN);
    // One persistent workgroup per CU (the kernel's occupancy is one), each
    // looping over tiles.
    const int64_t grid = tiles < num_cus() ? tiles : num_cus();
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), smem, stream, a);
    return hipGetLastError();
}

template <int BN, int WAVES_M, int S, bool OUT16, bool DUMP>
hipError_t launch_dma_cfg(const W8A8Args& a, hipStream_t stream) {
    constexpr int BM = 128 * WAVES_M;
    const int64_t tiles = ((a.rows + BM - 1) / BM) * ((a.columns + BN - 1) / BN);
    hipLaunchKernelGGL((w8a8_dma_kernel<BN, WAVES_M, S, OUT16, DUMP>), dim3((unsigned)tiles),
                       dim3(128 * WAVES_M), 0, stream, a);
    return hipGetLastError();
}

// The DMA kernel's K loop takes whole groups of S K tiles of 64 bytes.
bool dma_fits(const W8A8Args& a, int S) {
    return a.width % 64 == 0 && a.width >= 64 * S && (a.width / 64) % S == 0;
}

template <int BN, int PF>
hipError_t launch_bn(const W8A8Args& a, hipStream_t stream);

// The ring kernels' per-lane copy offsets are 32-bit byte offsets into x
// and W.
bool ring_offsets_fit(const W8A8Args& a) {
    const int64_t lim = int64_t(1) << 32;
    return a.rows * a.width < lim && a.columns * a.width < lim;
}

template <int BN, int S, bool OUT16, bool DUMP, bool PAIR = false, int NW = 4>
hipError_t launch_ring_cfg(const W8A8Args& a, hipStream_t stream) {
    const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + BN - 1) / BN);
    // Persistent: one workgroup per CU (the kernel's occupancy is one).
    const int64_t grid = tiles < num_cus() ? tiles : num_cus();
    hipLaunchKernelGGL((w8a8_ring_kernel<BN, S, OUT16, DUMP, PAIR, false, NW>), dim3((unsigned)grid),
                       dim3(64 * NW), 0, stream, a, 1);
    return hipGetLastError();
}

// Split-K reduction: acc = the splits' int32 sums added (wrapping, exact in
// any order), then the ring's epilogue, four consecutive elements per lane:
// out = f32(acc - x_sum * w_zero) * x_scale * w_scale (+ bias), as f32 or
// rounded once to f16; the accumulators to acc_dump when asked.
// S > 0 builds the kernel for exactly S splits. With columns % 4 == 0 (the
// four elements then lie in one row) every load, the partial sums and the
// epilogue's row and column parameters, goes out before the first add: the
// parameters are read unconditionally (from another in-range array where a
// pointer is null) and selected afterwards, as a load in a branch would be
// waited for in that branch. The arithmetic is the same either way.
template <bool OUT16, bool DUMP, int S = 0>
__global__ __launch_bounds__(256) void w8a8_split_reduce_kernel(W8A8Args a, int splits) {
    const int64_t n = a.rows * a.columns;
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    unsigned v[4] = {0u, 0u, 0u, 0u};
    int e_end = 4;
    const bool has_zero = a.w_zero != nullptr;
    int64_t row = i / a.columns, col = i - row * a.columns;
    float o[4];
    if (a.columns % 4 == 0) {
        const bool has_bias = a.bias != nullptr;
        const int32_t* xs_p = has_zero ? a.x_sum : reinterpret_cast<const int32_t*>(a.x_scale);
        const int32_t* wz_p = has_zero ? a.w_zero : reinterpret_cast<const int32_t*>(a.w_scale);
        const float* bi_p = has_bias ? a.bias : a.w_scale;
        const float rs = a.x_scale[row];
        const unsigned xs = (unsigned)xs_p[row];
        float ws[4], bi[4];
        unsigned wz[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            ws[e] = a.w_scale[col + e];
            wz[e] = (unsigned)wz_p[col + e];
            bi[e] = bi_p[col + e];
        }
        if constexpr (S > 0) {
            int4 t[S];
#pragma unroll
            for (int p = 0; p < S; ++p) t[p] = *reinterpret_cast<const int4*>(a.partial + p * n + i);
#pragma unroll
            for (int p = 0; p < S; ++p) {
                v[0] += (unsigned)t[p].x;
                v[1] += (unsigned)t[p].y;
                v[2] += (unsigned)t[p].z;
                v[3] += (unsigned)t[p].w;
            }
        } else {
            for (int p = 0; p < splits; ++p) {
                const int4 t = *reinterpret_cast<const int4*>(a.partial + p * n + i);
                v[0] += (unsigned)t.x;
                v[1] += (unsigned)t.y;
                v[2] += (unsigned)t.z;
                v[3] += (unsigned)t.w;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned prod = has_zero ? xs * wz[e] : 0u;
            const int centered = (int)(v[e] - prod);
            o[e] = w8a8_scale(centered, rs, ws[e], has_bias ? bi[e] : -0.0f);
        }
    } else {
        e_end = (int)min((int64_t)4, n - i);
        for (int e = 0; e < e_end; ++e)
            for (int p = 0; p < splits; ++p) v[e] += (unsigned)a.partial[p * n + i + e];
        for (int e = 0; e < e_end; ++e) {
            if (e > 0 && ++col == a.columns) col = 0, ++row;
            const unsigned prod = has_zero ? (unsigned)a.x_sum[row] * (unsigned)a.w_zero[col] : 0u;
            const int centered = (int)(v[e] - prod);
            o[e] = w8a8_scale(centered, a.x_scale[row], a.w_scale[col], a.bias ? a.bias[col] : -0.0f);
        }
    }
    // Whole 16-byte (8-byte) stores when aligned: four 4-byte nontemporal
    // stores into one line were written back to HBM separately.
    const uintptr_t oaddr = reinterpret_cast<uintptr_t>(a.out) + (uintptr_t)i * (OUT16 ? 2 : 4);
    const bool vec = e_end == 4 && oaddr % (OUT16 ? 8 : 16) == 0 &&
                     (!DUMP || reinterpret_cast<uintptr_t>(a.acc_dump + i) % 16 == 0);
    if (vec) {
        if constexpr (DUMP)
            *reinterpret_cast<int4*>(a.acc_dump + i) = make_int4((int)v[0], (int)v[1], (int)v[2], (int)v[3]);
        if constexpr (OUT16) {
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            stream_store(reinterpret_cast<h4*>(static_cast<_Float16*>(a.out) + i),
                         h4{(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]});
        } else {
            typedef float f4 __attribute__((ext_vector_type(4)));
            stream_store(reinterpret_cast<f4*>(static_cast<float*>(a.out) + i), f4{o[0], o[1], o[2], o[3]});
        }
        return;
    }
    for (int e = 0; e < e_end; ++e) {
        if constexpr (DUMP) a.acc_dump[i + e] = (int)v[e];
        if constexpr (OUT16)
            stream_store(static_cast<_Float16*>(a.out) + i + e, (_Float16)o[e]);
        else
            stream_store(static_cast<float*>(a.out) + i + e, o[e]);
    }
}

// Largest split count <= want that leaves every split of ktiles K tiles
// non-empty, keeps unit indices in int and whose partial sums fit in
// a.partial_elems.
int fit_splits(const W8A8Args& a, int64_t tiles, int ktiles, int want) {
    int s = want < ktiles ? want : ktiles;
    while (s > 1) {
        const int kts = (ktiles + s - 1) / s;
        if ((s - 1) * kts < ktiles && tiles * s <= INT32_MAX && a.partial &&
            s * a.rows * a.columns <= a.partial_elems)
            break;
        --s;
    }
    return s < 1 ? 1 : s;
}

template <int BN, bool OUT16, bool DUMP>
hipError_t launch_pair_split(const W8A8Args& a, int splits, hipStream_t stream) {
    const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + BN - 1) / BN);
    const int64_t units = tiles * splits;
    const int64_t grid = units < num_cus() ? units : num_cus();
    hipLaunchKernelGGL((w8a8_ring_kernel<BN, 5, OUT16, DUMP, true, true>), dim3((unsigned)grid), dim3(256), 0,
                       stream, a, splits);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t quads = (a.rows * a.columns + 3) / 4;
    const dim3 rgrid((unsigned)((quads + 255) / 256)), rblock(256);
    switch (splits) {
        case 2: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 2>), rgrid, rblock, 0, stream, a, splits); break;
        case 3: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 3>), rgrid, rblock, 0, stream, a, splits); break;
        case 4: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 4>), rgrid, rblock, 0, stream, a, splits); break;
        case 5: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 5>), rgrid, rblock, 0, stream, a, splits); break;
        case 6: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 6>), rgrid, rblock, 0, stream, a, splits); break;
        case 8: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP, 8>), rgrid, rblock, 0, stream, a, splits); break;
        default: hipLaunchKernelGGL((w8a8_split_reduce_kernel<OUT16, DUMP>), rgrid, rblock, 0, stream, a, splits);
    }
    return hipGetLastError();
}

// The pair-refill ring takes any K % 64 == 0; splits > 1 splits K when the
// partial sums fit (else it splits less).
template <int BN>
hipError_t launch_pair(const W8A8Args& a, hipStream_t stream, int splits = 1) {
    if (a.width % 64 != 0 || a.width == 0 || !ring_offsets_fit(a)) return launch_bn<BN == 128 ? 128 : 192, 2>(a, stream);
    if (splits > 1) {
        const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + BN - 1) / BN);
        splits = fit_splits(a, tiles, (int)(a.width / 64), splits);
    }
    if (splits > 1) {
        if (a.acc_dump) {
            if (a.out_f16) return launch_pair_split<BN, true, true>(a, splits, stream);
            return launch_pair_split<BN, false, true>(a, splits, stream);
        }
        if (a.out_f16) return launch_pair_split<BN, true, false>(a, splits, stream);
        return launch_pair_split<BN, false, false>(a, splits, stream);
    }
    if (a.acc_dump) {
        if (a.out_f16) return launch_ring_cfg<BN, 5, true, true, true>(a, stream);
        return launch_ring_cfg<BN, 5, false, true, true>(a, stream);
    }
    if (a.out_f16) return launch_ring_cfg<BN, 5, true, false, true>(a, stream);
    return launch_ring_cfg<BN, 5, false, false, true>(a, stream);
}

// The ring kernel's K loop takes whole groups of S K tiles of 64 bytes.
bool ring_fits(const W8A8Args& a, int S) {
    return a.width % 64 == 0 && a.width >= 64 * S && (a.width / 64) % S == 0 && ring_offsets_fit(a);
}

template <int BN, int S>
hipError_t launch_ring(const W8A8Args& a, hipStream_t stream) {
    if (!ring_fits(a, S)) return launch_bn<BN == 128 ? 128 : 192, 2>(a, stream);
    if (a.acc_dump) {
        if (a.out_f16) return launch_ring_cfg<BN, S, true, true>(a, stream);
        return launch_ring_cfg<BN, S, false, true>(a, stream);
    }
    if (a.out_f16) return launch_ring_cfg<BN, S, true, false>(a, stream);
    return launch_ring_cfg<BN, S, false, false>(a, stream);
}

// The eight-wave 256 x 256 ring (4 slots, single refill): K tiles % 4 == 0.
hipError_t launch_ring8_256(const W8A8Args& a, hipStream_t stream) {
    if (!ring_fits(a, 4)) return launch_bn<192, 2>(a, stream);
    if (a.acc_dump) {
        if (a.out_f16) return launch_ring_cfg<256, 4, true, true, false, 8>(a, stream);
        return launch_ring_cfg<256, 4, false, true, false, 8>(a, stream);
    }
    if (a.out_f16) return launch_ring_cfg<256, 4, true, false, false, 8>(a, stream);
    return launch_ring_cfg<256, 4, false, false, false, 8>(a, stream);
}

template <int BN, int S, int WAVES_M = 2>
hipError_t launch_dma(const W8A8Args& a, hipStream_t stream) {
    if (!dma_fits(a, S)) return launch_bn<BN == 128 ? 128 : 192, 2>(a, stream);
    if (a.acc_dump) {
        if (a.out_f16) return launch_dma_cfg<BN, WAVES_M, S, true, true>(a, stream);
        return launch_dma_cfg<BN, WAVES_M, S, false, true>(a, stream);
    }
    if (a.out_f16) return launch_dma_cfg<BN, WAVES_M, S, true, false>(a, stream);
    return launch_dma_cfg<BN, WAVES_M, S, false, false>(a, stream);
}

template <int BN, int PF, bool OUT16, bool DUMP>
hipError_t launch_out(const W8A8Args& a, hipStream_t stream) {
    if (a.width % 64 != 0) return launch_cfg<BN, PF, true, OUT16, DUMP>(a, stream);
    return launch_cfg<BN, PF, false, OUT16, DUMP>(a, stream);
}

template <int BN, int PF>
hipError_t launch_bn(const W8A8Args& a, hipStream_t stream) {
    if (a.acc_dump) {
        if (a.out_f16) return launch_out<BN, PF, true, true>(a, stream);
        return launch_out<BN, PF, false, true>(a, stream);
    }
    if (a.out_f16) return launch_out<BN, PF, true, false>(a, stream);
    return launch_out<BN, PF, false, false>(a, stream);
}

// OMNI_W8A8_SPLITS=<n> forces n-way split K on the pair ring (test aid);
// 0 or unset = the shape rule below.
int w8a8_split_override() { return knob(Knob::W8A8Splits, 0); }

// A pinned tile or split keeps the call off the streaming kernels (rows.hip),
// which have neither.
bool w8a8_pinned() { return w8a8_tile_override() != 0 || w8a8_split_override() > 1; }

// The split of K, where plan_w8a8 takes one: 256 x 128 tiles fill at most half
// of the CUs and K >= 4608, or at most an eighth of them and K >= 4096: K split up to 6 ways, at most one
// unit per CU, on the 256 x 128 pair ring. The partial sums cost one int32
// write and read per element and split, so shorter K, or more tiles, do not
// pay (MI355X, the reference's shapes: 256 x 4096 x 12288 69 -> 29 us, 256 x
// 3072 x 12288 69 -> 27 us, 512 x 4096 x 12288 69 -> 40 us; 512 x 4096 x 4096
// 26.2 unsplit against 26.6 at best split, 256 x 12288 x 4096 27.8 against
// 32.5; between K = 4608 and 8192, rows x K -> N: 503 x 7488 -> 5312 50 -> 35,
// 160 x 6848 -> 7168 42 -> 26, 301 x 5248 -> 7104 34.1 -> 32.7).
int w8a8_auto_splits(int64_t rows, int64_t columns, int64_t width, int64_t cus) {
    const int ov = w8a8_split_override();
    if (ov > 1) return ov;
    if (width % 64 != 0 || width < 4096) return 1;
    const int64_t tiles = ((rows + 255) / 256) * ((columns + 127) / 128);
    if (width >= 4608 ? 2 * tiles > cus : 8 * tiles > cus) return 1;
    const int64_t want = cus / tiles;
    return (int)(want > 6 ? 6 : want);
}

}  // namespace

hipError_t launch_w8a8_scalar(const W8A8Args& a, hipStream_t stream) {
    if (a.rows == 0 || a.columns == 0) return hipSuccess;
    dim3 block(64, 4);
    const int64_t row_blocks = (a.rows + 3) / 4;
    dim3 grid((unsigned)((a.columns + 255) / 256), (unsigned)(row_blocks < 65535 ? row_blocks : 65535));
    hipLaunchKernelGGL(w8a8_scalar_kernel, grid, block, 0, stream, a);
    return hipGetLastError();
}

namespace {

// What runs a W8A8 call: the streaming kernels (id: their column blocks), split
// K on the 256 x 128 pair ring (splits > 1), or a kernel as OMNI_W8A8_TILE
// numbers them, unsplit.
struct W8A8Plan {
    bool stream;
    int id, splits;
};

// Cost model, fitted to MI355X timings of every candidate on ten shapes
// (prefill GEMMs of 2048 and 4096 rows and the reference's 256-row benchmark
// shapes; codes of N(0,1) rows and uniform weights rotated past the MALL, f32
// out): a kernel runs its tiles in rounds of one tile per CU, a round costs
// BM * BN * (c * K + e) (c: per output element and K byte; e: the per-tile
// prologue and epilogue), and a partial last round with fill f costs
// (0.7 + 0.3 f) of a full one (the chip is power-limited on this path, so a
// partly idle round runs at a higher clock). It picks the fastest candidate,
// or one within 1 %, on all ten operands rotated; the other kernels
// (register-staged, two-waves-per-SIMD DMA, single-refill rings at 256 x 192
// and 256 x 128) lost on every one and stay reachable through OMNI_W8A8_TILE.
//
// Where the tiles leave CUs idle, the others compete by fitted times in us:
//  * whole: the cost model's (in fs) plus 2.5, 1.2 times it for the
//    register-staged kernels;
//  * split K (split_us): 1200 timings of 5 to 2000 rows, K 8192 ... 14336;
//    within 15 % (a few of 65 to 256 rows 29 %). From K = 8192 on (and where
//    the tiles fill at most an eighth of the CUs) it runs without regard to
//    whole; at K = 4608 ... 8191 where it is under 0.8 of it, since both fits
//    are that uncertain there;
//  * the streaming kernels (w8a8_rows_us): up to 64 rows unless split K over K
//    >= 8192 is under 1.03 of theirs or, from 49 rows on, over 16384 columns
//    and K > 4096, the weight rows are not whole 128-byte lines (56 rows of
//    10048 x 16832 80 us against 69, of 4288 x 17100 37.8 against 35.3; 9472 x
//    16896 57 against 62); more rows where they are under split K and 0.95 of
//    whole.
// Against the choice without the streaming kernels and splits from 8192 on
// only, 5500 drawn calls (K 1024 ... 14336, N 1024 ... 18944) take 0.46 of the
// time at 17 to 64 rows, 0.62 at 65 to 256, 0.82 at 257 to 1024 and 0.97 above;
// 1 % of them are slower by more than 3 %, the worst by 16 %. Streaming all up
// to 64 rows, and comparing tiles with a split fitted to fewer rows, was slower
// on 5 % of 49 to 64 rows, by up to half (54 of 12736 x 8512 64 us against 42),
// and above 1024 rows by up to 1.7 times (2049 of 4672 x 1728 62 against 36).
double split_us(const W8A8Args& a, int64_t tiles, int splits) {
    const double K = (double)a.width, rows = (double)a.rows, columns = (double)a.columns;
    return 7.76 + 4.52e-3 * K / splits + 1.41e-6 * splits * rows * columns + 7e-8 * K * columns +
           5.9e-6 * (double)tiles * K + 0.0154 * (rows < 256.0 ? rows : 256.0);
}

// room: the workspace holds a split's sums (the size query asks as if it did).
W8A8Plan plan_w8a8(const W8A8Args& a, bool room) {
    const int64_t cus = num_cus();
    const double K = (double)a.width;
    auto cost = [&](double c, double e, int64_t bm, int64_t bn) {
        const int64_t tiles = ((a.rows + bm - 1) / bm) * ((a.columns + bn - 1) / bn);
        const int64_t full = tiles / cus, rem = tiles % cus;
        const double rounds = (double)full + (rem ? 0.7 + 0.3 * (double)rem / (double)cus : 0.0);
        return (double)(bm * bn) * (c * K + e) * rounds;
    };
    const bool streams = !w8a8_pinned() && w8a8_rows_fits(a);
    int nb = 0;
    const double stream_us = streams ? w8a8_rows_us(a.rows, a.columns, a.width, &nb) : 1e30;
    const W8A8Plan stream{true, nb, 1};
    if (a.width % 64 != 0 || !ring_offsets_fit(a)) {
        // Register-staged kernels: any K % 16 == 0.
        const double c128 = cost(308.0, 250000.0, 256, 128), c192 = cost(280.5, 227212.0, 256, 192);
        if (streams && (a.rows <= 64 || stream_us / 0.95 < 1.2e-9 * (c128 < c192 ? c128 : c192))) return stream;
        return {false, c128 < c192 ? 4 : 3, 1};
    }
    const int64_t kt = a.width / 64;
    const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + 127) / 128);
    const int sp = room ? w8a8_auto_splits(a.rows, a.columns, a.width, cus) : 1;
    const double splitting_us = sp > 1 ? split_us(a, tiles, sp) : 1e30;
    const W8A8Plan split{false, 17, sp};
    W8A8Plan whole{false, 16, 1};
    double best = cost(243.7, 117070.0, 256, 192);
    auto consider = [&](bool ok, double t, int id) {
        if (ok && t < best) best = t, whole.id = id;
    };
    consider(true, cost(281.8, 123726.0, 256, 128), 17);
    const bool s4 = kt >= 4 && kt % 4 == 0, s3 = kt >= 3 && kt % 3 == 0;
    // The eight-wave 256 x 256 ring replaces the four-wave one (11), at 0.94
    // of its fit: measured 0.80-0.92 of its time on seven shapes (4352 x
    // 12288 -> 3072: 160 against 179 us; 2048 x 4096 -> 14336: 126 against
    // 139), a factor that keeps 4096 x 3072 -> 12288 and 4096 x 12288 -> 3072
    // on the 256 x 192 pair ring, which stays faster there.
    consider(s4, cost(240.7, 163216.0, 256, 256), 19);
    consider(!s4 && s3, cost(250.7, 210425.0, 256, 256), 14);
    const double whole_us = 1e-9 * best + 2.5;
    if (streams && a.rows <= 64) {
        if (a.rows > 16 && a.width >= 8192 && 0.97 * splitting_us < stream_us) return split;
        const bool ragged = a.rows > 48 && a.columns > 64 * cus && a.width % 128 != 0 && a.width > 4096;
        return ragged ? whole : stream;
    }
    if (stream_us < splitting_us && stream_us / 0.95 < whole_us) return stream;
    if (sp > 1 && (w8a8_split_override() > 1 || a.width >= 8192 || 8 * tiles <= cus || splitting_us < 0.8 * whole_us))
        return split;
    return whole;
}

}  // namespace

int64_t w8a8_partial_elems(int64_t rows, int64_t columns, int64_t width) {
    if (rows <= 0 || columns <= 0 || width % 64 != 0) return 0;
    W8A8Args a{};
    a.rows = rows;
    a.columns = columns;
    a.width = width;
    if (!ring_offsets_fit(a)) return 0;
    const int sp = w8a8_tile_override() != 0 ? w8a8_auto_splits(rows, columns, width, num_cus())
                                             : plan_w8a8(a, true).splits;
    return sp > 1 ? (int64_t)sp * rows * columns : 0;
}

hipError_t launch_w8a8_mfma(const W8A8Args& a, hipStream_t stream) {
    if (a.rows == 0 || a.columns == 0) return hipSuccess;
    switch (w8a8_tile_override()) {
        case 3: return launch_bn<192, 2>(a, stream);
        case 4: return launch_bn<128, 2>(a, stream);
        case 9: return launch_dma<192, 2, 4>(a, stream);
        case 10: return launch_dma<128, 2, 4>(a, stream);
        case 11: return launch_ring<256, 4>(a, stream);
        case 12: return launch_ring<192, 4>(a, stream);
        case 13: return launch_ring<128, 4>(a, stream);
        case 14: return launch_ring<256, 3>(a, stream);
        case 15: return launch_ring<192, 3>(a, stream);
        case 16: return launch_pair<192>(a, stream);
        case 17: return launch_pair<128>(a, stream, w8a8_split_override());
        case 19: return launch_ring8_256(a, stream);
        case 30:  // the streaming kernels in blocks of 32 columns, 31: of 64
        case 31:
            if (w8a8_rows_fits(a)) return launch_w8a8_rows(a, w8a8_tile_override() == 30 ? 2 : 4, stream);
            break;
        default: break;
    }
    // Whether the workspace holds the sums of the split K that would run.
    const int64_t tiles = ((a.rows + 255) / 256) * ((a.columns + 127) / 128);
    const int sp = w8a8_auto_splits(a.rows, a.columns, a.width, num_cus());
    const W8A8Plan plan = plan_w8a8(a, sp > 1 && fit_splits(a, tiles, (int)(a.width / 64), sp) > 1);
    if (plan.stream) return launch_w8a8_rows(a, plan.id, stream);
    switch (plan.id) {
        case 19: return launch_ring8_256(a, stream);
        case 14: return launch_ring<256, 3>(a, stream);
        case 17: return launch_pair<128>(a, stream, plan.splits);
        case 4: return launch_bn<128, 2>(a, stream);
        case 3: return launch_bn<192, 2>(a, stream);
        default: return launch_pair<192>(a, stream);
    }
}

}  // namespace omni

#ifdef OMNI_PHASE_TIMELINE
// Copies the tile-phase timeline (1024 workgroups x 64 entries) to dst;
// returns a hipError_t code. Not part of the operator ABI.
extern "C" int omni_phase_timeline_read(void* dst, size_t bytes) {
    const size_t cap = sizeof(omni::g_phase);
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(omni::g_phase), bytes < cap ? bytes : cap, 0,
                                    hipMemcpyDeviceToHost);
}
// Clears it (a synchronous copy of zeros; call outside any graph capture).
extern "C" int omni_phase_timeline_clear() {
    static unsigned long long zeros[1024 * 64];
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(omni::g_phase), zeros, sizeof(zeros), 0, hipMemcpyHostToDevice);
}
#endif
