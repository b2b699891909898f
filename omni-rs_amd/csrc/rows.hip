// Linears of a few rows on gfx950 (W8A8, and int8, int4 or f16 weights under
// f16 activations), bound by the stream of their weights; the matrix cores
// need a fraction of its time. Up to 64 rows one workgroup sees them all; more
// (W8A8 on small matrices, where 256-row tiles would leave most CUs idle) are
// cut into tiles of 48 or 64.
//
// A workgroup of KW waves walks blocks of 16 NB columns (units), each wave a
// KW-th of K, in tiles of TB bytes of K. Everything a tile needs, 16 NB
// weight rows and the activations' rows, is copied by LDS-DMA into a ring of
// S slots that belongs to one wave alone: the K loop has no barrier and
// holds nothing in flight in registers, and the ring runs on across units
// (the next unit's weights are on their way while this one's sums are
// added). A copy reads whole 256-byte (TB = 128: 128-byte) pieces of weight
// rows: loading v_mfma fragments straight into registers, 16 rows x 64 bytes
// per instruction, took 10-25 % longer for the bare read of the same bytes
// (MI355X, 4096 x 28672: 21.7 against 18.8 us; 4096 x 4096: 4.6 against 4.05).
// The 16-byte chunks of a row are XOR-swizzled by the row's 256-byte window,
// on the global side, so the 16 lanes of a fragment read touch 16 distinct
// 16-byte bank groups. At the end of a unit the KW partial tiles are added
// through LDS and the epilogue applied: one launch, no workspace.
//
// Measured on MI355X, the GEMM alone, weights rotated past the MALL, against
// the 256-row ring kernels (w8a8_gemm.hip) that took these calls: 8 rows,
// K x N = 4096 x 4096 6.1 against 14.3 us, 4096 x 6144 7.8 against 27.7,
// 4096 x 28672 23.4 against 40.3, 14336 x 4096 13.3 against 26.3 (the bare
// read: 4.0, 5.4, 18.5, 10.4); 48 rows of 4096 x 6144 11.0 against 28.2;
// 8 rows of 4304 x 1152 (K % 64 != 0) 5.6 against 48. In tiles: 128 rows of
// 4096 x 4096 11.9 against 20.4 us, 256 rows 15.5 against 23.7 (split K), of
// 3072 x 3072 13.5 against 33.6; a tile's K loop is bound by the copies into
// LDS, 64 KiB per wave-tile step in 1.06 us per CU.
#include <type_traits>

#include "common.hpp"
#include "dequant.hpp"
#include "kernels.hpp"

namespace omni {

namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// The weights' kind: int8 under int8 activation codes (exact int32 sums),
// int8, packed int4 (groups of 128) and f16 under f16 activations.
enum : int { kW8A8, kW8A16, kW4A16, kF16 };

// Activation bytes per weight byte.
constexpr int x_bytes(int wk) { return wk == kW8A16 ? 2 : wk == kW4A16 ? 4 : 1; }

constexpr int kInt4Group = 128;

struct RowsArgs {
    const uint8_t* x;   // [rows][width], codes or f16
    const uint8_t* w;   // [columns][row_bytes]
    int64_t rows, columns;
    int row_bytes;      // of a weight row
    void* out;
    // The f16 epilogue: scale (W8A16) and bias per column, either may be null;
    // int4's group scales, bf16 [columns][width / 128].
    const _Float16* scale16;
    const _Float16* bias16;
    const uint16_t* gscale;
    // The W8A8 epilogue, as in W8A8Args.
    const float* x_scale;
    const int32_t* x_sum;
    const float* w_scale;
    const int32_t* w_zero;
    const float* bias;
    int32_t* acc_dump;
    bool out_f16;
};

// lds_copy16_saddr as a nontemporal load: the weights are read once (4096 x
// 4096, the bare read: 4.05 against 4.45 us).
__device__ __forceinline__ void lds_copy16_nt(unsigned voff, const void* base, unsigned lds_byte) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile(OMNI_LDS_COPY("global_load_lds_dwordx4") " nt" ::"v"(voff), "s"(base), "s"(lds_byte) : "memory", "m0");
#endif
}

// Waits until at most the youngest `tiles` tiles (C copies each, fewer than
// S) are in flight, and for this wave's LDS reads. Loads return in order;
// other vector-memory operations under way only make the wait longer.
template <int C, int S>
__device__ __forceinline__ void wait_tiles(int tiles) {
    static_assert(S <= 3, "two tiles behind the awaited one");
    if (tiles <= 0)
        s_waitcnt_vm<0, true>();
    else if (S < 3 || tiles == 1)
        s_waitcnt_vm<C, true>();
    else
        s_waitcnt_vm<2 * C, true>();
    asm volatile("" ::: "memory");  // no LDS read moves above the wait
}

// Units per workgroup, at most (their epilogue values are kept in LDS).
constexpr int stream_units(int nb, bool mt) { return mt ? 8 : 32 / nb; }

// XC activation copies per tile hold XC * XR rows: 16 MB, or for MB = 1 a
// smaller power of two (the other rows of the block repeat them; they are
// never stored).
template <int WK, int MB, int NB, int XC, int S, int KW, int TB, bool MT>
__global__ __launch_bounds__(64 * KW, KW / 4) void rows_stream_kernel(RowsArgs a) {
    using Acc = std::conditional_t<WK == kW8A8, v4i, v4f>;
    using Sum = std::conditional_t<WK == kW8A8, int, float>;
    constexpr int XTB = TB * x_bytes(WK);        // activation bytes per row and tile
    constexpr int RPC = 1024 / TB, XR = 1024 / XTB;  // rows per copy
    constexpr int BM = 16 * MB, BN = 16 * NB;
    constexpr int WC = BN / RPC;                 // weight copies per tile
    constexpr int SC = WK == kW4A16 ? TB / 64 : 0;  // group scale copies (one scale per lane)
    constexpr int C = WC + XC + SC;
    constexpr int XROWS = XC * XR;               // activation rows held
    static_assert(XROWS == BM || (MB == 1 && !MT && XROWS < 16 && (XROWS & (XROWS - 1)) == 0), "activation rows");
    static_assert(WK != kW4A16 || BN <= 64, "a lane per column in a scale copy");
    constexpr int kStage = (WC + XC) * 1024 + SC * 256;
    constexpr int kSteps = TB / 64;
    constexpr int kH = WK == kW8A8 ? 1 : x_bytes(WK);  // 16-byte activation pieces per lane and step
    constexpr int T = 64 * KW;
    constexpr int NU = stream_units(NB, MT);
    // Column blocks whose partial sums are added at a time.
    constexpr int PJ = KW * MB * NB <= 32 ? NB : 1;
    constexpr int PN = 16 * PJ, kPart = BM * PN;  // partial sums per wave
    __shared__ __attribute__((aligned(1024))) uint8_t stages[KW * S * kStage];
    __shared__ Sum part[KW * kPart];
    __shared__ float s_scale[WK == kW8A8 ? (MT ? NU : 1) * BM : 1];
    __shared__ int s_sum[WK == kW8A8 ? (MT ? NU : 1) * BM : 1];
    __shared__ float s_ws[NU * BN];
    __shared__ int s_zero[WK == kW8A8 ? NU * BN : 1];
    __shared__ float s_bias[NU * BN];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int tiles_m = MT ? (int)((a.rows + BM - 1) / BM) : 1;
    const int units = (int)((a.columns + BN - 1) / BN) * tiles_m;
    // Units of one column block are neighbours, and neighbours share an XCD,
    // whose L2 then serves all but the first read of the weights.
    const int first = MT ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x, stride = gridDim.x;
    const int nu = (units - first + stride - 1) / stride;  // units of this workgroup (first < units)
    const int wrow = a.row_bytes, xrow = wrow * x_bytes(WK);
    const int ktiles = (wrow + TB - 1) / TB;
    const int lo = wave * ktiles / KW, mine = (wave + 1) * ktiles / KW - lo;
    const bool tail = wrow % TB != 0;
    auto unit_m0 = [&](int u) -> int64_t { return MT ? (int64_t)((first + u * stride) % tiles_m) * BM : 0; };
    auto unit_n0 = [&](int u) -> int64_t { return (int64_t)(MT ? (first + u * stride) / tiles_m : first + u * stride) * BN; };

    // 16-byte chunk slots are XOR-swizzled by the row's 256-byte window, on
    // the global side of the copies.
    constexpr int kW = 256 / TB > 0 ? 256 / TB : 1;    // rows per 256-byte window
    constexpr int kXW = 256 / XTB > 0 ? 256 / XTB : 1;
    constexpr int kWMask = (TB / 16 - 1) & 15, kXMask = (XTB / 16 - 1) & 15;
    auto w_row = [&](int c) { return c * RPC + lane / (TB / 16); };
    auto w_byte = [&](int c) { return ((lane % (TB / 16)) ^ ((w_row(c) / kW) & kWMask)) * 16; };
    auto x_row = [&](int c) { return c * XR + lane / (XTB / 16); };
    auto x_byte = [&](int c) { return ((lane % (XTB / 16)) ^ ((x_row(c) / kXW) & kXMask)) * 16; };
    // int4: a column's group scales (one group of 128 codes per 64 weight bytes).
    const int groups = wrow / 64;
    // The copies' sources in the unit being issued: wave-uniform bases and
    // per-lane offsets (rows past the matrix repeat the last one).
    const uint8_t *wbase = nullptr, *xbase = a.x;
    const uint16_t* sbase = nullptr;
    unsigned woff[WC], xoff[XC], soff = 0;
    auto set_unit = [&](int u) {
        const int64_t n0 = unit_n0(u), m0 = unit_m0(u);
        const int cols = (int)min((int64_t)BN, a.columns - n0) - 1;
        const int rows = (int)min((int64_t)BM, a.rows - m0) - 1;
        wbase = a.w + n0 * wrow;
        xbase = a.x + m0 * xrow;
#pragma unroll
        for (int c = 0; c < WC; ++c) woff[c] = (unsigned)(min(w_row(c), cols) * wrow + w_byte(c));
#pragma unroll
        for (int c = 0; c < XC; ++c) xoff[c] = (unsigned)(min(x_row(c), rows) * xrow + x_byte(c));
        if constexpr (SC != 0) {
            sbase = a.gscale + n0 * groups;
            soff = (unsigned)(min(lane, cols) * groups * 2);
        }
    };
    const unsigned st_lds = lds_addr(stages) + wave * (S * kStage);
    auto issue = [&](int tile, int slot) {
        const unsigned dst = st_lds + slot * kStage;
        const uint8_t* wb = wbase + tile * TB;
        const uint8_t* xb = xbase + tile * XTB;
        // A partial last tile: pieces past the row's end repeat its last one.
        const bool last = tail && tile == ktiles - 1;
        const int wend = wrow - 16 - tile * TB, xend = xrow - 16 - tile * XTB;
#pragma unroll
        for (int c = 0; c < WC; ++c) {
            unsigned off = woff[c];
            if (last) off -= max(w_byte(c) - wend, 0);
            if constexpr (MT)
                lds_copy16_saddr(off, wb, dst + c * 1024);
            else
                lds_copy16_nt(off, wb, dst + c * 1024);
        }
#pragma unroll
        for (int c = 0; c < SC; ++c)
            lds_copy2_saddr(soff, sbase + min(tile * SC + c, groups - 1), dst + (WC + XC) * 1024 + c * 256);
#pragma unroll
        for (int c = 0; c < XC; ++c) {
            unsigned off = xoff[c];
            if (last) off -= max(x_byte(c) - xend, 0);
            lds_copy16_saddr(off, xb, dst + (WC + c) * 1024);
        }
    };
    const int total = mine * nu;
    int iu = 0, it = 0, issued = 0;  // next tile to issue
    auto issue_next = [&](int slot) {
        issue(lo + it, slot);
        ++issued;
        if (++it == mine) {
            it = 0;
            if (++iu < nu) set_unit(iu);
        }
    };
    set_unit(0);
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < total) issue_next(s);

    const bool has_zero = a.w_zero != nullptr, has_bias = a.bias != nullptr;
    if constexpr (WK == kW8A8) {
        for (int i = tid; i < (MT ? nu : 1) * BM; i += T) {
            const int64_t row = min(unit_m0(i / BM) + i % BM, a.rows - 1);
            s_scale[i] = a.x_scale[row];
            s_sum[i] = has_zero ? a.x_sum[row] : 0;
        }
    }
    for (int i = tid; i < nu * BN; i += T) {
        const int64_t n = min(unit_n0(i / BN) + i % BN, a.columns - 1);
        if constexpr (WK == kW8A8) {
            s_ws[i] = a.w_scale[n];
            s_zero[i] = has_zero ? a.w_zero[n] : 0;
            s_bias[i] = has_bias ? a.bias[n] : -0.0f;  // x + -0.0 is x
        } else {
            s_ws[i] = a.scale16 ? (float)a.scale16[n] : 1.0f;
            s_bias[i] = a.bias16 ? (float)a.bias16[n] : 0.0f;
        }
    }

    const int wkey = (r16 / kW) & kWMask;
    const int xr = MB == 1 ? r16 & (XROWS - 1) : r16;
    const int xkey = (xr / kXW) & kXMask;
    int done = 0, slot = 0;
    for (int u = 0; u < nu; ++u) {
        Acc acc[NB][MB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[j][i] = Acc{};
        for (int t = 0; t < mine; ++t) {
            wait_tiles<C, S>(issued - done - 1);
            const uint8_t* st = stages + (wave * S + slot) * kStage;
            const uint8_t* ws = st + r16 * TB;
            const uint8_t* xs = st + WC * 1024 + xr * XTB;
            // Lane (r, g) holds weight bytes 64 s + 16 g .. +15 of column r's tile
            // (16 int8 codes, 32 int4 codes, 8 halves), and the activations of
            // row r at the same k.
            v4u w[kSteps][NB], x[kSteps][MB][kH];
            float sc[kSteps][NB];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    w[s][j] = *reinterpret_cast<const v4u*>(ws + j * 16 * TB + (((4 * s + g) ^ wkey) << 4));
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int q = 0; q < kH; ++q)
                        x[s][i][q] = *reinterpret_cast<const v4u*>(
                            xs + i * 16 * XTB + (((4 * kH * s + kH * g + q) ^ xkey) << 4));
            }
            if constexpr (SC != 0) {
#pragma unroll
                for (int s = 0; s < kSteps; ++s)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        sc[s][j] = bf16_to_f32(
                            *reinterpret_cast<const uint16_t*>(st + (WC + XC) * 1024 + s * 256 + (j * 16 + r16) * 4));
            }
            // Everything is read: the slot takes the next tile while this one
            // is multiplied.
            if (issued < total) {
                s_waitcnt_lgkm0();
                issue_next(slot);
            }
            if (tail && lo + t == ktiles - 1) {
                // Past the row's end both operands are zero (an infinity times
                // a zero weight would not be).
#pragma unroll
                for (int s = 0; s < kSteps; ++s)
                    if ((lo + t) * TB + s * 64 + g * 16 >= wrow) {
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            w[s][j] = v4u{0u, 0u, 0u, 0u};
                            if constexpr (SC != 0) sc[s][j] = 0.0f;
                        }
#pragma unroll
                        for (int i = 0; i < MB; ++i)
#pragma unroll
                            for (int q = 0; q < kH; ++q) x[s][i][q] = v4u{0u, 0u, 0u, 0u};
                    }
            }
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                if constexpr (WK == kW8A8) {
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, x[s][i][0]),
                                                                             __builtin_bit_cast(v4i, w[s][j]),
                                                                             acc[j][i], 0, 0, 0);
                } else {
                    v8h b[NB][kH];
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        const v4u wq = w[s][j];
                        v2h h[4 * kH];
                        if constexpr (WK == kF16) {
                            __builtin_memcpy(h, &wq, 16);
                        } else if constexpr (WK == kW8A16) {
                            i8x4_to_f16x4(wq.x, h[0], h[1]);
                            i8x4_to_f16x4(wq.y, h[2], h[3]);
                            i8x4_to_f16x4(wq.z, h[4], h[5]);
                            i8x4_to_f16x4(wq.w, h[6], h[7]);
                        } else {
                            const unsigned word[4] = {wq.x, wq.y, wq.z, wq.w};
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                v2h h4[4];
                                i4x8_to_f16x8(word[q], h4);
#pragma unroll
                                for (int e = 0; e < 4; ++e) h[4 * q + e] = h4[e];
                            }
                        }
#pragma unroll
                        for (int q = 0; q < kH; ++q)
                            b[j][q] = v8h{h[4 * q][0],     h[4 * q][1],     h[4 * q + 1][0], h[4 * q + 1][1],
                                          h[4 * q + 2][0], h[4 * q + 2][1], h[4 * q + 3][0], h[4 * q + 3][1]};
                    }
                    // int4: the step's 64 bytes are one group, whose sum takes its
                    // scale in f32, four FMAs per 16 x 16 block (a lane's sums are of
                    // one column). Scaling the codes in f16 first took 16 packed
                    // multiplies per column block and lost scales outside f16's
                    // normal range (3 rows of 4096 x 14336 10.6 against 11.4 us, 8 of
                    // 3584 x 18944 15.1 against 15.9, 16 17.5 against 18.2; 32 rows
                    // even).
                    Acc group[NB][MB];
#pragma unroll
                    for (int q = 0; q < kH; ++q)
#pragma unroll
                        for (int i = 0; i < MB; ++i)
#pragma unroll
                            for (int j = 0; j < NB; ++j) {
                                const bool first_of = WK == kW4A16 && q == 0;
                                Acc& to = WK == kW4A16 ? group[j][i] : acc[j][i];
                                to = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x[s][i][q]),
                                                                           b[j][q], first_of ? Acc{} : to, 0, 0, 0);
                            }
                    if constexpr (WK == kW4A16) {
#pragma unroll
                        for (int i = 0; i < MB; ++i)
#pragma unroll
                            for (int j = 0; j < NB; ++j)
#pragma unroll
                                for (int r = 0; r < 4; ++r)
                                    acc[j][i][r] = __builtin_fmaf(group[j][i][r], sc[s][j], acc[j][i][r]);
                    }
                }
            }
            ++done;
            if (++slot == S) slot = 0;
        }
        const int64_t m0 = unit_m0(u), n0 = unit_n0(u);
#pragma unroll
        for (int j0 = 0; j0 < NB; j0 += PJ) {
            if (u + j0 > 0) lds_barrier();  // the last partial sums are read
#pragma unroll
            for (int j = 0; j < PJ; ++j)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        part[wave * kPart + (i * 16 + 4 * g + r) * PN + j * 16 + r16] = acc[j0 + j][i][r];
            s_waitcnt_lgkm0();
            lds_barrier();
#pragma unroll
            for (int e0 = 0; e0 < kPart; e0 += T) {
                const int e = e0 + tid;
                const int row = e / PN, c = j0 * 16 + e % PN;
                const int64_t m = m0 + row, n = n0 + c;
                if (e < kPart && m < a.rows && n < a.columns) {
                    const int64_t idx = m * a.columns + n;
                    const int col = u * BN + c;
                    if constexpr (WK == kW8A8) {
                        unsigned sum = 0;
#pragma unroll
                        for (int k = 0; k < KW; ++k) sum += (unsigned)part[k * kPart + e];
                        if (a.acc_dump) a.acc_dump[idx] = (int)sum;
                        const int srow_i = (MT ? u * BM : 0) + row;
                        float o;
                        {
                            // crates/omni-kernel/src/int8_matmul.rs:156-158: wrapping
                            // int32, then two multiplies and the bias, each rounded.
#pragma clang fp contract(off)
                            const int centered = (int)(sum - (unsigned)s_sum[srow_i] * (unsigned)s_zero[col]);
                            const float t = (float)centered * s_scale[srow_i];
                            o = t * s_ws[col] + s_bias[col];
                        }
                        if (a.out_f16)
                            static_cast<_Float16*>(a.out)[idx] = (_Float16)o;
                        else
                            static_cast<float*>(a.out)[idx] = o;
                    } else {
                        float sum = 0.0f;
#pragma unroll
                        for (int k = 0; k < KW; ++k) sum += part[k * kPart + e];
                        static_cast<_Float16*>(a.out)[idx] = (_Float16)(sum * s_ws[col] + s_bias[col]);
                    }
                }
            }
            s_waitcnt_lgkm0();  // before the next barrier
        }
    }
}

template <int WK, int MB, int NB, int XC, int S, int KW, int TB, bool MT = false>
hipError_t launch_stream_cfg(const RowsArgs& a, int64_t cus, hipStream_t stream) {
    const int64_t tiles_m = MT ? (a.rows + 16 * MB - 1) / (16 * MB) : 1;
    const int64_t units = (a.columns + 16 * NB - 1) / (16 * NB) * tiles_m;
    constexpr int64_t kMost = stream_units(NB, MT);
    const int64_t least = (units + kMost - 1) / kMost;
    // As many workgroups as are resident at once: two per CU where LDS allows.
    constexpr int kLds = KW * (S * (16 * NB * TB / 1024 + XC) + MB * NB) * 1024 + 12 * 16 * NB * (int)kMost + 128 * MB;
    const int64_t cap = cus * (KW == 4 && kLds <= 80 * 1024 ? 2 : 1);
    const int64_t grid = units < cap ? units : (least > cap ? least : cap);
    if (grid > 0x7fffffff || units > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((rows_stream_kernel<WK, MB, NB, XC, S, KW, TB, MT>), dim3((unsigned)grid), dim3(64 * KW), 0,
                       stream, a);
    return hipGetLastError();
}

// Blocks of 16 columns outnumber the CUs.
bool is_wide(int64_t columns, int64_t cus) { return columns > 16 * cus; }

// One activation byte per weight byte (W8A8, f16 weights). Measured over K x
// N of 1152 ... 14336 x 1152 ... 28672 at 1 to 64 rows of W8A8. Where one block
// of 16 columns per CU covers the matrix, eight waves share it (from 17 rows
// on the rings leave LDS for four). On wider matrices up to 8 rows take two
// four-wave workgroups per CU (8 rows of 4096 x 6144 7.9 against 8.4 us, of
// 4096 x 28672 23.1 against 24.0), more rows blocks of 32 columns, which
// halve the activations' share of the copies (48 rows of 4096 x 6144 11.0
// against 13.9 us, of 4096 x 28672 36.0 against 43).
template <int WK>
hipError_t launch_even(const RowsArgs& a, hipStream_t st) {
    const int64_t cus = num_cus();
    const bool wide = is_wide(a.columns, cus);
    if constexpr (WK == kW8A8)  // (up to 4 rows of f16 weights take the GEMV)
        if (a.rows <= 4)
            return wide ? launch_stream_cfg<WK, 1, 1, 1, 2, 4, 256>(a, cus, st)
                        : launch_stream_cfg<WK, 1, 1, 1, 3, 8, 256>(a, cus, st);
    if (a.rows <= 8)
        return wide ? launch_stream_cfg<WK, 1, 1, 2, 2, 4, 256>(a, cus, st)
                    : launch_stream_cfg<WK, 1, 1, 2, 2, 8, 256>(a, cus, st);
    if (a.rows <= 16)
        return wide ? launch_stream_cfg<WK, 1, 2, 2, 2, 8, 128>(a, cus, st)
                    : launch_stream_cfg<WK, 1, 1, 4, 2, 8, 256>(a, cus, st);
    if (a.rows <= 32)
        return wide ? launch_stream_cfg<WK, 2, 2, 4, 3, 4, 128>(a, cus, st)
                    : launch_stream_cfg<WK, 2, 1, 8, 2, 4, 256>(a, cus, st);
    if (a.rows <= 48)
        return wide ? launch_stream_cfg<WK, 3, 2, 6, 3, 4, 128>(a, cus, st)
                    : launch_stream_cfg<WK, 3, 1, 6, 3, 4, 128>(a, cus, st);
    return wide ? launch_stream_cfg<WK, 4, 2, 8, 2, 4, 128>(a, cus, st)
                : launch_stream_cfg<WK, 4, 1, 8, 2, 4, 128>(a, cus, st);
}

// Row blocks per workgroup above 64 rows: the rows spread evenly over the
// fewest tiles of at most 64 (then 3 or 4 blocks of 16).
int row_blocks(int64_t rows) {
    const int64_t tiles = (rows + 63) / 64;
    return (int)(((rows + tiles - 1) / tiles + 15) / 16);
}
int64_t row_units(int64_t rows, int64_t columns, int nb) {
    const int64_t bm = 16 * row_blocks(rows);
    return (rows + bm - 1) / bm * ((columns + 16 * nb - 1) / (16 * nb));
}

// More than 64 rows: tiles of 48 or 64 rows by 16 NB columns, K split over
// four waves that each own a ring.
template <int NB>
hipError_t launch_tiles(const RowsArgs& a, hipStream_t st) {
    const int64_t cus = num_cus();
    return row_blocks(a.rows) == 3 ? launch_stream_cfg<kW8A8, 3, NB, 6, 2, 4, 128, true>(a, cus, st)
                                   : launch_stream_cfg<kW8A8, 4, NB, 8, 2, 4, 128, true>(a, cus, st);
}

RowsArgs f16_args(const W8A16Args& w, int64_t row_bytes) {
    RowsArgs a{};
    a.x = reinterpret_cast<const uint8_t*>(w.x);
    a.w = reinterpret_cast<const uint8_t*>(w.w);
    a.rows = w.rows;
    a.columns = w.columns;
    a.row_bytes = (int)row_bytes;
    a.out = w.out;
    a.scale16 = w.scale;
    a.bias16 = w.bias;
    a.gscale = w.gscale;
    return a;
}

// Byte offsets are 32-bit within 64 weight rows and within the activations.
constexpr int64_t kMaxRowBytes = 1 << 18;

}  // namespace

bool w8a8_rows_fits(const W8A8Args& a) {
    return a.rows <= 4096 && a.width % 16 == 0 && a.width >= 16 && a.width <= kMaxRowBytes;
}

hipError_t launch_w8a8_rows(const W8A8Args& w, int nb, hipStream_t st) {
    if (w.rows == 0 || w.columns == 0) return hipSuccess;
    RowsArgs a{};
    a.x = w.x;
    a.w = w.w;
    a.rows = w.rows;
    a.columns = w.columns;
    a.row_bytes = (int)w.width;
    a.out = w.out;
    a.x_scale = w.x_scale;
    a.x_sum = w.x_sum;
    a.w_scale = w.w_scale;
    a.w_zero = w.w_zero;
    a.bias = w.bias;
    a.acc_dump = w.acc_dump;
    a.out_f16 = w.out_f16;
    if (a.rows <= 64) return launch_even<kW8A8>(a, st);
    return nb == 2 ? launch_tiles<2>(a, st) : launch_tiles<4>(a, st);
}

// Time in us of 65 rows and more in blocks of 32 or 64 columns, fitted to 65
// to 1024 rows of thirteen K x N (1152 ... 14336 x 1152 ... 28672): each round
// of one tile per CU costs a fixed part and its K loop (within 10 % of 64 of
// the 78 timings, 20 % of the rest). Of 17 to 64 rows, for K from 6000 on: up
// to one block of 16 columns per CU the K loop of a block and its share of the
// weights' stream; wider, rounds of one block of 32 per CU, a partial last one
// from half a round up (1100 timings: within 4 % of half, 10 % of nine in
// ten). Rows of the weights that are not whole 128-byte lines take 1.3 times
// as long, above 64 rows 1.2 (1300 timings). Fewer rows are ahead of every other kernel (1).
double w8a8_rows_us(int64_t rows, int64_t columns, int64_t width, int* nb) {
    const int64_t cus = num_cus();
    *nb = 0;
    if (rows <= 16) return 1.0;
    const double K = 1e-3 * (double)width;
    const double line = width % 128 == 0 ? 1.0 : rows <= 64 ? 1.3 : 1.2;
    if (rows <= 64) {
        const int mb = (int)((rows + 15) / 16) - 2;
        if (!is_wide(columns, cus)) {
            constexpr double kLoop[3] = {0.58, 0.89, 1.06};
            return 3.8 + K * (kLoop[mb] * line + 1.05e-3 * (double)((columns + 15) / 16));
        }
        constexpr double kFull[3] = {1.55, 1.80, 2.16}, kPart[3] = {1.0, 1.12, 1.22};
        const int64_t units = (columns + 31) / 32, rem = units % cus;
        const double part = rem ? kPart[mb] + 0.65 * (double)rem / (double)cus : 0.0;
        return 3.3 + line * K * ((double)(units / cus) * kFull[mb] + part);
    }
    const int mb = row_blocks(rows);
    auto us = [&](int n, double fixed, double per_k) {
        const int64_t rounds = (row_units(rows, columns, n) + cus - 1) / cus;
        return 5.0 + (double)rounds * (fixed + per_k * line * K * (mb + n) / (4 + n));
    };
    const double t2 = us(2, 1.3, 1.5), t4 = us(4, 2.1, 2.06);
    *nb = t2 < t4 ? 2 : 4;
    return t2 < t4 ? t2 : t4;
}

// Five to 64 rows, against the skinny kernels and the GEMM (w8a16.hip):
// 8 rows of 14336 x 4096 14.0 against 19.9 us, 16 of 4096 x 14336 16.5
// against 21.3, 32 of 1536 x 17920 14.5 against 25.4, 48 of 8960 x 1536 18.7
// against 29.7; one and two rows of K > 16384 (the GEMV's limit) 15.4 against
// 21.4 (18944 x 3584). The others keep:
//  * up to 16 rows at K = 1024, 2048, 3072, 4096 in one round of workgroups,
//    the LDS skinny kernel built for that K (16 of 4096 x 4096 6.9 against
//    7.5 us, of 1024 x 4096 3.4 against 3.8), and past it while its second
//    round costs less than a few rows' wide blocks (5 of 1024 x 4112 3.2
//    against 3.6, of 1024 x 8192 4.0 against 4.3, 8 even; 12 of 1024 x 4112
//    3.5 against 3.9, from 4352 on even; 5 of 2048 x 4112 4.65 against 4.9,
//    of 2048 x 7168 5.45 against 5.55, 8 even; 5 of 3072 x 4112 7.3 against
//    5.9);
//  * three and four rows, the GEMV up to K = 4096 on up to 8192 columns (4 of
//    4096 x 4096 5.8 against 6.1, 3 of 5120 x 5120 9.0 against 9.4), up to K =
//    8192 on up to 2048 (3 of 7616 x 1344 5.4 against 6.8, 4 of 8192 x 2048 5.8
//    against 6.4) and at K = 4096 up to 64 M weights (4 of 4096 x 14336 13.9
//    against 14.5; beyond, 4 of 4096 x 28672 22.8 against 24.1, of 14336 x 4096
//    12.6 against 15.3); and where weight rows start within 64-byte pieces, which
//    the copies then straddle (4 of 4064 x 12736 13.4 against 15.5, of 5456 x
//    1928 5.5 against 6.6, of 11536 x 2176 10.4 against 11.4);
//  * 17 to 32 rows of long K, the GEMM where blocks of 32 columns leave a nearly
//    empty second round: 25 rows and more from K = 8300 on (32 of 12160 x 10048
//    44 against 48 us, 31 of 9856 x 9088 33 against 37), and where weight rows
//    are not whole 128-byte lines from K = 5300 (30 of 6080 x 8576 24 against
//    27, of 13760 x 9200 45 against 59), up to 24 from 8000 (20 of 10432 x 8832
//    35.5 against 39.5, 23 of 8128 x 8320 28 against 33);
//  * from 33 rows on, the GEMM where the matrix is large: each activation
//    copy is then read by too few columns (48 of 4096 x 14336 28.3 against
//    25.8 us, but of 4096 x 6144 15.1 against 29.2, of 14336 x 4096 29.9
//    against 32.8; 36 of 1984 x 16960 19.5 against 17.4; 64 of 2048 x 14336
//    18.6 against 17.4, of 4096 x 5120 15.7 against 17.5, of 8960 x 1536 24.4
//    against 37.1; 50 of 1088 x 18240 15.3 against 12.2).
bool w8a16_rows_take(const W8A16Args& a) {
    if (a.rows > 64 || a.width % 16 != 0 || a.width < 16 || a.width > kMaxRowBytes) return false;
    const int64_t cus = num_cus();
    const bool wide = is_wide(a.columns, cus);
    const double elems = (double)a.columns * (double)a.width;
    if (a.width > 16384 && a.rows <= 4) return true;
    if (a.rows <= 2) return false;
    if (a.rows <= 4) {
        if (a.width % 64 != 0 || (a.width == 4096 && elems <= (64 << 20))) return false;
        return wide ? a.columns >= 8192 : a.width > 8192 || (a.width > 4096 && a.columns > 8 * cus);
    }
    if (a.rows <= 16) {
        if (a.width > 4096 || a.width % 1024 != 0) return true;
        if (a.width == 1024) return a.columns > (a.rows <= 8 ? 32 : 17) * cus;
        return a.width == 2048 && a.rows < 8 ? a.columns >= 32 * cus : wide;
    }
    if (a.rows <= 32) {
        if (a.columns <= 32 * cus || a.columns > 42 * cus || a.width % 64 != 0) return true;  // (K % 64: no ring)
        if (a.width % 128 == 0) return a.rows <= 24 || a.width < 8300;
        return a.width < (a.rows <= 24 ? 8000 : 5300);
    }
    if (a.rows <= 48) return !wide || elems <= (a.columns > 64 * cus ? 32e6 : 36e6);
    return elems < 16e6 || (a.width <= 4096 && a.columns <= 64 * cus && elems <= 26e6);
}

hipError_t launch_w8a16_rows(const W8A16Args& w, hipStream_t st) {
    if (w.rows == 0 || w.columns == 0) return hipSuccess;
    const RowsArgs a = f16_args(w, w.width);
    const int64_t cus = num_cus();
    const bool wide = is_wide(a.columns, cus);
    // Wide: two four-wave workgroups per CU, or from K = 4096 and 9 rows on
    // blocks of 32 columns (8 rows of 4096 x 6144 7.7 against 8.8 us, of 1536
    // x 17920 9.7 against 8.7; 16 rows of 4096 x 14336 16.5 against 21.4).
    if (w.rows <= 4)
        return wide ? launch_stream_cfg<kW8A16, 1, 1, 2, 2, 4, 256>(a, cus, st)
                    : launch_stream_cfg<kW8A16, 1, 1, 1, 3, 8, 128>(a, cus, st);
    if (w.rows <= 8) {
        if (!wide) return launch_stream_cfg<kW8A16, 1, 1, 2, 3, 8, 128>(a, cus, st);
        return w.width >= 4096 ? launch_stream_cfg<kW8A16, 1, 2, 2, 2, 8, 128>(a, cus, st)
                               : launch_stream_cfg<kW8A16, 1, 1, 2, 3, 4, 128>(a, cus, st);
    }
    if (w.rows <= 16)
        return wide ? launch_stream_cfg<kW8A16, 1, 2, 4, 2, 8, 128>(a, cus, st)
                    : launch_stream_cfg<kW8A16, 1, 1, 4, 3, 8, 128>(a, cus, st);
    if (w.rows <= 32)
        return wide ? launch_stream_cfg<kW8A16, 2, 2, 8, 2, 4, 128>(a, cus, st)
                    : launch_stream_cfg<kW8A16, 2, 1, 8, 3, 4, 128>(a, cus, st);
    if (w.rows <= 48)
        return wide ? launch_stream_cfg<kW8A16, 3, 2, 6, 3, 4, 64>(a, cus, st)
                    : launch_stream_cfg<kW8A16, 3, 1, 12, 2, 4, 128>(a, cus, st);
    return wide ? launch_stream_cfg<kW8A16, 4, 2, 8, 2, 4, 64>(a, cus, st)
                : launch_stream_cfg<kW8A16, 4, 1, 8, 3, 4, 64>(a, cus, st);
}

// Groups of 128. Three to 64 rows, against the GEMV, the skinny kernels and the
// GEMM:
// 4 rows of 4096 x 6144 6.8 against 8.7 us, of 3584 x 18944 13.2 against
// 15.9, 8 of 4096 x 14336 12.2 against 21.6, 16 of 14336 x 4096 16.2 against
// 28.9, 32 of 3584 x 18944 29.8 against 40.3. The others keep:
//  * three and four rows, the GEMV on narrow matrices of long K (4 of 8960 x
//    1536 7.4 against 7.8; below 1408 columns 3 of 2432 x 1088 3.85 against
//    4.04); one and two rows of K > 32768 are past its limit;
//  * where weight rows are not whole 128-byte lines (K % 256 != 0), which the
//    copies then straddle: three and four rows in a nearly empty second round of
//    32-column blocks, the GEMV (4 of 7040 x 9216 15.3 against 17.8, 3 of 4480 x
//    10112 11.9 against 13.4); some rows of short K, the skinny kernel, whose
//    loads split K evenly over more waves (9 of 1152 x 8488 6.2 against 7.4, 17
//    of 1152 x 1792 4.13 against 4.50, 9 of 2176 x 2200 4.40 against 4.84);
//  * from 49 rows on (in blocks of 16 columns: 64 of 8960 x 1536 21.2 against
//    37.9, of 2048 x 8192 12.6 against 18.3, of 4096 x 6144 19.4 against 20.6),
//    the GEMM, what is wide and large (64 of 4096 x 14336 36.0 against 30.0; 61
//    of 5632 x 4416 25.8 against 23.3) or very wide (of 1024 x 18944 16.4
//    against 14.8). 48 rows of 4096 x 6144 12.5 against 32.2, of 8192 x 28672
//    80 against 93.
bool w4a16_rows_take(const W8A16Args& a) {
    if (a.rows > 64 || a.group != kInt4Group || a.width % kInt4Group != 0 || a.width <= 0 || a.width > kMaxRowBytes)
        return false;
    const int64_t cus = num_cus();
    const bool wide = is_wide(a.columns, cus), lines = a.width % 256 == 0;
    const bool second_round = a.columns > 32 * cus && a.columns <= 44 * cus;
    if (a.width > 32768 && a.rows <= 4) return true;
    if (a.rows <= 2) return false;
    if (a.rows <= 4) {
        if (!lines && second_round && a.width >= 4096) return false;
        return a.columns > 2048 || (a.width <= 4096 && a.columns >= 1408);
    }
    if (!lines && a.rows > 8 && a.rows <= 24 && a.width < 1280 && (!wide || second_round)) return false;
    if (!lines && a.rows > 8 && a.rows <= 12 && a.width > 2048 && a.width < 3584 && !wide) return false;
    return a.rows <= 48 || !wide ||
           (a.columns <= 40 * cus && (double)a.columns * (double)a.width <= (a.width <= 4096 ? 26e6 : 22e6));
}

hipError_t launch_w4a16_rows(const W8A16Args& w, hipStream_t st) {
    if (w.rows == 0 || w.columns == 0) return hipSuccess;
    const RowsArgs a = f16_args(w, w.width / 2);
    const int64_t cus = num_cus();
    const bool wide = is_wide(a.columns, cus);
    // Wide: blocks of 32 columns; up to 4 rows only where they still make a
    // few rounds of long K (4096 x 6144 6.8 against 7.5 us, of 1536 x 17920
    // 8.6 against 7.4).
    if (w.rows <= 4) {
        if (!wide) return launch_stream_cfg<kW4A16, 1, 1, 2, 3, 8, 128>(a, cus, st);
        return w.width >= 4096 && w.columns <= 16384 ? launch_stream_cfg<kW4A16, 1, 2, 2, 2, 8, 128>(a, cus, st)
                                                     : launch_stream_cfg<kW4A16, 1, 1, 2, 3, 4, 128>(a, cus, st);
    }
    if (w.rows <= 8)
        return wide ? launch_stream_cfg<kW4A16, 1, 2, 4, 2, 8, 128>(a, cus, st)
                    : launch_stream_cfg<kW4A16, 1, 1, 4, 2, 8, 128>(a, cus, st);
    if (w.rows <= 16)
        return wide ? launch_stream_cfg<kW4A16, 1, 2, 8, 2, 4, 128>(a, cus, st)
                    : launch_stream_cfg<kW4A16, 1, 1, 8, 3, 4, 128>(a, cus, st);
    // One 128-byte tile, not three of 64 (32 rows of 4096 x 14336 17.6 against
    // 18.7, of 8960 x 1536 13.0 against 13.6; 17 to 24 rows even).
    if (w.rows <= 32)
        return wide ? launch_stream_cfg<kW4A16, 2, 2, 16, 1, 4, 128>(a, cus, st)
                    : launch_stream_cfg<kW4A16, 2, 1, 16, 1, 4, 128>(a, cus, st);
    // (64 rows by 32 columns do not fit LDS.)
    if (w.rows <= 48)
        return wide ? launch_stream_cfg<kW4A16, 3, 2, 12, 2, 4, 64>(a, cus, st)
                    : launch_stream_cfg<kW4A16, 3, 1, 12, 2, 4, 64>(a, cus, st);
    return launch_stream_cfg<kW4A16, 4, 1, 16, 2, 4, 64>(a, cus, st);
}

// Five to 64 rows of f16 weights (up to 4 take the GEMV).
bool f16_rows_take(const W8A16Args& a) {
    return a.rows > 4 && a.rows <= 64 && a.width % 8 == 0 && a.width >= 8 && 2 * a.width <= kMaxRowBytes;
}

hipError_t launch_f16_rows(const W8A16Args& w, hipStream_t st) {
    if (w.rows == 0 || w.columns == 0) return hipSuccess;
    return launch_even<kF16>(f16_args(w, 2 * w.width), st);
}

}  // namespace omni
