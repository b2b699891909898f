// Linears of up to 64 rows on gfx950, bound by the stream of their weights
// (columns x width bytes; the matrix cores need a fraction of its time).
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
// 8 rows of 4304 x 1152 (K % 64 != 0) 5.6 against 48.
#include "common.hpp"
#include "kernels.hpp"

namespace omni {

namespace {

// The weights' kind. W8A8's activations are int8 codes.
enum : int { kW8A8 = 0 };

template <int WK>
struct Kind {
    static constexpr int kXBytes = 1;   // activation bytes per weight byte
    using Acc = v4i;
};

struct RowsArgs {
    const uint8_t* x;   // [rows][width] codes
    const uint8_t* w;   // [columns][width]
    int64_t rows, columns, width;
    // The epilogue, as in W8A8Args.
    const float* x_scale;
    const int32_t* x_sum;
    const float* w_scale;
    const int32_t* w_zero;
    const float* bias;
    void* out;
    int32_t* acc_dump;
    bool out_f16;
};

// lds_copy16_saddr as a nontemporal load: the weights are read once (4096 x
// 4096, the bare read: 4.05 against 4.45 us).
__device__ __forceinline__ void lds_copy16_nt(unsigned voff, const void* base, unsigned lds_byte) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(voff), "s"(base), "s"(lds_byte)
                 : "memory", "m0");
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

// Columns per workgroup, at most (their epilogue values are kept in LDS).
constexpr int kStreamColumns = 512;

// XC activation copies per tile hold XC * XR rows: 16 MB, or for MB = 1 a
// smaller power of two (the other rows of the block repeat them; they are
// never stored).
template <int WK, int MB, int NB, int XC, int S, int KW, int TB>
__global__ __launch_bounds__(64 * KW, KW / 4) void rows_stream_kernel(RowsArgs a) {
    using Kd = Kind<WK>;
    using Acc = typename Kd::Acc;
    constexpr int XTB = TB * Kd::kXBytes;        // activation bytes per row and tile
    constexpr int RPC = 1024 / TB, XR = 1024 / XTB;  // rows per copy
    constexpr int BN = 16 * NB;
    constexpr int WC = BN / RPC, C = WC + XC;    // copies per tile
    constexpr int XROWS = XC * XR;               // activation rows held
    static_assert(XROWS == 16 * MB || (MB == 1 && XROWS < 16 && (XROWS & (XROWS - 1)) == 0), "activation rows");
    constexpr int kStage = C * 1024;
    constexpr int kSteps = TB / 64;
    constexpr int T = 64 * KW;
    constexpr int kPart = MB * NB * 256;         // partial sums per wave
    __shared__ __attribute__((aligned(1024))) uint8_t stages[KW * S * kStage];
    __shared__ int part[KW * kPart];
    __shared__ float s_scale[16 * MB];
    __shared__ int s_sum[16 * MB];
    __shared__ float s_ws[kStreamColumns];
    __shared__ int s_zero[kStreamColumns];
    __shared__ float s_bias[kStreamColumns];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int units = (int)((a.columns + BN - 1) / BN);
    const int first = blockIdx.x, stride = gridDim.x;
    const int nu = (units - first + stride - 1) / stride;  // units of this workgroup (first < units)
    const int wrow = (int)a.width;
    const int ktiles = (wrow + TB - 1) / TB;
    const int lo = wave * ktiles / KW, mine = (wave + 1) * ktiles / KW - lo;
    const bool tail = wrow % TB != 0;

    // 16-byte chunk slots are XOR-swizzled by the row's 256-byte window, on
    // the global side of the copies.
    constexpr int kW = 256 / TB > 0 ? 256 / TB : 1;    // rows per 256-byte window
    constexpr int kXW = 256 / XTB > 0 ? 256 / XTB : 1;
    constexpr int kWMask = (TB / 16 - 1) & 15, kXMask = (XTB / 16 - 1) & 15;
    int wrow_l[WC], wch[WC];
    unsigned xoff[XC];
    int xch[XC];
#pragma unroll
    for (int c = 0; c < WC; ++c) {
        wrow_l[c] = c * RPC + lane / (TB / 16);
        wch[c] = ((lane % (TB / 16)) ^ ((wrow_l[c] / kW) & kWMask)) * 16;
    }
#pragma unroll
    for (int c = 0; c < XC; ++c) {
        const int r = c * XR + lane / (XTB / 16);
        xch[c] = ((lane % (XTB / 16)) ^ ((r / kXW) & kXMask)) * 16;
        xoff[c] = (unsigned)(min((int64_t)r, a.rows - 1) * wrow * Kd::kXBytes);
    }
    const unsigned st_lds = lds_addr(stages) + wave * (S * kStage);
    auto issue = [&](int unit, int tile, int slot) {
        const int64_t n0 = (int64_t)(first + unit * stride) * BN;
        const uint8_t* wb = a.w + n0 * wrow;
        const int cols = (int)min((int64_t)BN, a.columns - n0);
        const unsigned dst = st_lds + slot * kStage;
#pragma unroll
        for (int c = 0; c < WC; ++c) {
            const unsigned off = (unsigned)(min(wrow_l[c], cols - 1) * wrow + min(tile * TB + wch[c], wrow - 16));
            lds_copy16_nt(off, wb, dst + c * 1024);
        }
#pragma unroll
        for (int c = 0; c < XC; ++c) {
            const unsigned off = xoff[c] + (unsigned)min(tile * XTB + xch[c], wrow * Kd::kXBytes - 16);
            lds_copy16_saddr(off, a.x, dst + (WC + c) * 1024);
        }
    };
    const int total = mine * nu;
    int iu = 0, it = 0, issued = 0;  // next tile to issue
    auto issue_next = [&](int slot) {
        issue(iu, lo + it, slot);
        if (++it == mine) it = 0, ++iu;
        ++issued;
    };
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < total) issue_next(s);

    const bool has_zero = a.w_zero != nullptr, has_bias = a.bias != nullptr;
    for (int i = tid; i < 16 * MB; i += T) {
        const int64_t row = min((int64_t)i, a.rows - 1);
        s_scale[i] = a.x_scale[row];
        s_sum[i] = has_zero ? a.x_sum[row] : 0;
    }
    for (int i = tid; i < nu * BN; i += T) {
        const int64_t n = min((int64_t)(first + i / BN * stride) * BN + i % BN, a.columns - 1);
        s_ws[i] = a.w_scale[n];
        s_zero[i] = has_zero ? a.w_zero[n] : 0;
        s_bias[i] = has_bias ? a.bias[n] : -0.0f;  // x + -0.0 is x
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
            const uint8_t* ws = stages + (wave * S + slot) * kStage + r16 * TB;
            const uint8_t* xs = stages + (wave * S + slot) * kStage + WC * 1024 + xr * XTB;
            v4i b[kSteps][NB], x[kSteps][MB];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    b[s][j] = *reinterpret_cast<const v4i*>(ws + j * 16 * TB + (((4 * s + g) ^ wkey) << 4));
#pragma unroll
                for (int i = 0; i < MB; ++i)
                    x[s][i] = *reinterpret_cast<const v4i*>(xs + i * 16 * XTB + (((4 * s + g) ^ xkey) << 4));
            }
            if (tail && lo + t == ktiles - 1) {
#pragma unroll
                for (int s = 0; s < kSteps; ++s)
                    if ((lo + t) * TB + s * 64 + g * 16 >= wrow) {
#pragma unroll
                        for (int j = 0; j < NB; ++j) b[s][j] = v4i{0, 0, 0, 0};
                    }
            }
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i)
                        acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[s][i], b[s][j], acc[j][i], 0, 0, 0);
            if (issued < total) {
                s_waitcnt_lgkm0();  // the slot is read
                issue_next(slot);
            }
            ++done;
            if (++slot == S) slot = 0;
        }
        if (u > 0) lds_barrier();  // the last unit's sums are read
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    part[wave * kPart + (i * 16 + 4 * g + r) * BN + j * 16 + r16] = acc[j][i][r];
        s_waitcnt_lgkm0();
        lds_barrier();
#pragma unroll
        for (int e0 = 0; e0 < kPart; e0 += T) {
            const int e = e0 + tid;
            const int row = e / BN, col = u * BN + e % BN;
            const int64_t n = (int64_t)(first + u * stride) * BN + e % BN;
            if (e < kPart && row < a.rows && n < a.columns) {
                unsigned sum = 0;
#pragma unroll
                for (int k = 0; k < KW; ++k) sum += (unsigned)part[k * kPart + e];
                const int64_t idx = row * a.columns + n;
                if (a.acc_dump) a.acc_dump[idx] = (int)sum;
                float o;
                {
#pragma clang fp contract(off)
                    const int centered = (int)(sum - (unsigned)s_sum[row] * (unsigned)s_zero[col]);
                    const float t = (float)centered * s_scale[row];
                    o = t * s_ws[col] + s_bias[col];
                }
                if (a.out_f16)
                    static_cast<_Float16*>(a.out)[idx] = (_Float16)o;
                else
                    static_cast<float*>(a.out)[idx] = o;
            }
        }
        s_waitcnt_lgkm0();  // before the next unit's barrier
    }
}

template <int WK, int MB, int NB, int XC, int S, int KW, int TB>
hipError_t launch_stream_cfg(const RowsArgs& a, int64_t cus, hipStream_t stream) {
    const int64_t units = (a.columns + 16 * NB - 1) / (16 * NB);
    constexpr int64_t kMost = kStreamColumns / (16 * NB);
    const int64_t least = (units + kMost - 1) / kMost;
    // As many workgroups as are resident at once: two per CU where LDS allows.
    constexpr int kLds = KW * (S * (16 * NB * TB / 1024 + XC) + MB * NB) * 1024 + 12 * kStreamColumns + 128 * MB;
    const int64_t cap = cus * (KW == 4 && kLds <= 80 * 1024 ? 2 : 1);
    const int64_t grid = units < cap ? units : (least > cap ? least : cap);
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((rows_stream_kernel<WK, MB, NB, XC, S, KW, TB>), dim3((unsigned)grid), dim3(64 * KW), 0, stream, a);
    return hipGetLastError();
}

}  // namespace

// Byte offsets are 32-bit within 32 weight rows and within the activations.
bool w8a8_rows_fits(const W8A8Args& a) {
    return a.rows <= 64 && a.width % 16 == 0 && a.width >= 16 && a.width <= 131072;
}

// Measured over K x N of 1152 ... 14336 x 1152 ... 28672 at 1 to 64 rows. Where
// one block of 16 columns per CU covers the matrix, eight waves share it
// (16 rows and fewer; the rings of more rows leave LDS for four). On wider
// matrices up to 8 rows take two four-wave workgroups per CU (8 rows of 4096
// x 6144 7.9 against 8.4 us, of 4096 x 28672 23.1 against 24.0), more rows
// blocks of 32 columns, which halve the activations' share of the copies (48
// rows of 4096 x 6144 11.0 against 13.9 us, of 4096 x 28672 36.0 against 43).
hipError_t launch_w8a8_rows(const W8A8Args& w, hipStream_t st) {
    if (w.rows == 0 || w.columns == 0) return hipSuccess;
    RowsArgs a{w.x,       w.w,      w.rows, w.columns, w.width,    w.x_scale, w.x_sum,
               w.w_scale, w.w_zero, w.bias, w.out,     w.acc_dump, w.out_f16};
    const int64_t cus = num_cus();
    const bool wide = w.columns > 16 * cus;
    if (w.rows <= 4)
        return wide ? launch_stream_cfg<kW8A8, 1, 1, 1, 2, 4, 256>(a, cus, st)
                    : launch_stream_cfg<kW8A8, 1, 1, 1, 3, 8, 256>(a, cus, st);
    if (w.rows <= 8)
        return wide ? launch_stream_cfg<kW8A8, 1, 1, 2, 2, 4, 256>(a, cus, st)
                    : launch_stream_cfg<kW8A8, 1, 1, 2, 2, 8, 256>(a, cus, st);
    if (w.rows <= 16)
        return wide ? launch_stream_cfg<kW8A8, 1, 2, 2, 2, 8, 128>(a, cus, st)
                    : launch_stream_cfg<kW8A8, 1, 1, 4, 2, 8, 256>(a, cus, st);
    if (w.rows <= 32)
        return wide ? launch_stream_cfg<kW8A8, 2, 2, 4, 3, 4, 128>(a, cus, st)
                    : launch_stream_cfg<kW8A8, 2, 1, 8, 2, 4, 256>(a, cus, st);
    if (w.rows <= 48)
        return wide ? launch_stream_cfg<kW8A8, 3, 2, 6, 3, 4, 128>(a, cus, st)
                    : launch_stream_cfg<kW8A8, 3, 1, 6, 3, 4, 128>(a, cus, st);
    return wide ? launch_stream_cfg<kW8A8, 4, 2, 8, 2, 4, 128>(a, cus, st)
                : launch_stream_cfg<kW8A8, 4, 1, 8, 2, 4, 128>(a, cus, st);
}

}  // namespace omni
