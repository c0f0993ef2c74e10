// Index unpack and dequantized-tile kernels.
//
// unpack:  the flat nibble stream -> one uint8 per index
//          (epure/runtime.py:48-54 _unpack4; identity copy above 16 levels).
// dequant: W[n, k] = cb[idx] * scale[n, k / group] with the rounding of
//          epure/runtime.py:78-89 materialize(dtype):
//            f32:       f32(cb) * f32(scale)      (container.py:70-88)
//            f16/bf16:  dtype(dtype(cb) * dtype(scale))
//          The exact product of two fp16 (or two bf16) values fits in fp32,
//          so computing it in fp32 and rounding once is the torch result.
// embedding rows: the dequant of selected rows (PackedEmbedding).
// All read indices through the same flat-stream addressing as the GEMV
// fallback, so odd K with 4-bit packing is covered.
#include "ep_common.h"
#include "ep_internal.h"

namespace ep {
namespace {

__global__ void __launch_bounds__(256) unpack_kernel(const uint8_t *__restrict__ packed, int64_t n,
                                                     int four, uint8_t *__restrict__ idx)
{
    // Each thread expands 8 indices (4 packed bytes for 4-bit).
    const int64_t base = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
    if (base >= n)
        return;
    uint8_t out[8];
    if (four) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t p = base + 2 * i;
            const uint8_t b = p < n ? packed[p >> 1] : 0;
            out[2 * i] = b & 0x0f;
            out[2 * i + 1] = b >> 4;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            out[i] = base + i < n ? packed[base + i] : 0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (base + i < n)
            idx[base + i] = out[i];
}

__device__ __forceinline__ float round_to(int dt, float v)
{
    if (dt == EP_F16)
        return (float)(f16_t)v;
    if (dt == EP_BF16)
        return bf16_to_f32(f32_to_bf16(v));
    return v;
}

struct TileArgs {
    const uint8_t *packed;
    const void *scale;
    int scale_dtype;
    int64_t lds;
    const void *cb;
    int cb_dtype;
    int levels;
    int group;
    int64_t N, K;
    void *out;
    int out_dtype;
    int64_t ldo;
};

// Element (n, k) of the dequantized weight in out_dtype's rounding.
__device__ __forceinline__ float dequant_elem(const TileArgs &a, int64_t n, int64_t k)
{
    const bool four = a.levels <= 16;
    const int64_t p = n * a.K + k;
    const uint8_t byte = a.packed[four ? (p >> 1) : p];
    const int idx = four ? ((p & 1) ? (byte >> 4) : (byte & 15)) : byte;
    const float c = idx < a.levels ? load_as_f32(a.cb, a.cb_dtype, idx) : 0.0f;
    const float s = load_as_f32(a.scale, a.scale_dtype, n * a.lds + k / a.group);
    return round_to(a.out_dtype, c) * round_to(a.out_dtype, s);
}

__global__ void __launch_bounds__(256) dequant_tile_kernel(TileArgs a)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.K)
        return;
    for (int64_t n = blockIdx.y; n < a.N; n += gridDim.y)
        store_from_f32(a.out, a.out_dtype, n * a.ldo + k, dequant_elem(a, n, k));
}

// The same tile for 4-bit rows of whole 16-byte chunks (K % 32 == 0, groups
// of a multiple of 32), bound by its stores: a wave takes 4 x 64 consecutive
// dwords of the packed stream, a lane one dword (8 weights, one group scale)
// of each 64, four loads in flight, so a store instruction writes 1 KiB
// (2-byte types) in one piece wherever the rows are long enough.  With a
// thread per 32 weights its four stores lay 64 bytes from its neighbours':
// 6144 x 2048 to fp16 beside the backward's other product 23.8 us, 11 to 17
// now.  The waves go over the stream and not over the rows: with a wave per
// row a few long rows ran on a few waves (4 x 2^20 to bf16 1090 -> 6.7 us) and
// rows shorter than 512 weights left lanes idle (2^20 x 32 365 -> 19.8 us);
// between them 4096^2 13.8 -> 12.9, 14336 x 4096 29.6 -> 31.3.  The codebook is pre-rounded in LDS.  Same arithmetic as
// dequant_elem (round(c) * round(s) in fp32, rounded once).
// U: dwords per lane, all loaded before the first is expanded.
constexpr int kTile4 = 4;
template <int DT, int U>
__global__ void __launch_bounds__(256) dequant_tile4_kernel(TileArgs a, uint32_t dw, int64_t total)
{
    __shared__ float tab[16];
    const int lane = threadIdx.x & 63;
    const int64_t f0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * U) + lane;
    // row and dword of the row of the lane's first dword; 64 dwords on are
    // d64 rows and r64 dwords on
    uint32_t row, i;
    if (total <= 0xffffffff) {  // uniform
        row = (uint32_t)f0 / dw;
        i = (uint32_t)f0 - row * dw;
    } else {
        row = (uint32_t)(f0 / dw);
        i = (uint32_t)(f0 - (int64_t)row * dw);
    }
    const uint32_t d64 = 64 / dw, r64 = 64 % dw;
    uint32_t w[U], at[U], rows[U];
    float sc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const bool in = f0 + 64 * u < total;  // past the end: dword 0, not stored
        rows[u] = in ? row : 0;
        at[u] = in ? i : 0;
        w[u] = ((const uint32_t *)a.packed)[in ? f0 + 64 * u : 0];
        sc[u] = load_as_f32(a.scale, a.scale_dtype, (int64_t)rows[u] * a.lds + at[u] * 8u / (uint32_t)a.group);
        row += d64;
        i += r64;
        if (i >= dw) {
            i -= dw;
            ++row;
        }
    }
    if (threadIdx.x < 16)
        tab[threadIdx.x] = threadIdx.x < a.levels ? round_to(DT, load_as_f32(a.cb, a.cb_dtype, threadIdx.x)) : 0.0f;
    lds_barrier();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (f0 + 64 * u >= total)
            break;
        char *dst = (char *)a.out + ((int64_t)rows[u] * a.ldo + (int64_t)at[u] * 8) * (DT == EP_F32 ? 4 : 2);
        const float s = round_to(DT, sc[u]);
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            v[t] = tab[(w[u] >> (4 * t)) & 15] * s;
        if constexpr (DT == EP_F32) {
            ((f32x4_t *)dst)[0] = (f32x4_t){v[0], v[1], v[2], v[3]};
            ((f32x4_t *)dst)[1] = (f32x4_t){v[4], v[5], v[6], v[7]};
        } else {
            u32x4_t o;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float lo = v[2 * t], hi = v[2 * t + 1];
                if constexpr (DT == EP_F16)
                    o[t] = (uint32_t)f16_bits((f16_t)lo) | ((uint32_t)f16_bits((f16_t)hi) << 16);
                else
                    o[t] = (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16);
            }
            *(u32x4_t *)dst = o;
        }
    }
}

template <int DT>
void launch_tile4(const TileArgs &a, hipStream_t stream)
{
    const uint32_t dw = (uint32_t)(a.K / 8);  // dwords per row
    const int64_t total = a.N * dw;
    // one dword per lane while four would leave fewer than two workgroups per
    // CU: 256 x 256 to bf16 5.2 -> 4.3 us
    if (total < (int64_t)2 * 256 * kTile4 * device_cus())
        hipLaunchKernelGGL((dequant_tile4_kernel<DT, 1>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                           a, dw, total);
    else
        hipLaunchKernelGGL((dequant_tile4_kernel<DT, kTile4>),
                           dim3((unsigned)((total + 256 * kTile4 - 1) / (256 * kTile4))), dim3(256), 0, stream, a, dw,
                           total);
}

// out[i, :] = dequantized row ids[i] (epure/runtime.py:139-156
// PackedEmbedding.forward: only the rows a batch asks for are expanded);
// an id outside [0, N) gives a row of zeros.
__global__ void __launch_bounds__(256) embedding_rows_kernel(TileArgs a, const int64_t *ids, int64_t n_ids)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.K)
        return;
    for (int64_t i = blockIdx.y; i < n_ids; i += gridDim.y) {
        const int64_t n = ids[i];
        const float w = (n >= 0 && n < a.N) ? dequant_elem(a, n, k) : 0.0f;
        store_from_f32(a.out, a.out_dtype, i * a.ldo + k, w);
    }
}

}  // namespace

int launch_unpack(const uint8_t *packed, int64_t n, int levels, uint8_t *idx, hipStream_t stream)
{
    if (n <= 0)
        return EP_OK;
    const int64_t threads = (n + 7) / 8;
    const int64_t grid = (threads + 255) / 256;
    hipLaunchKernelGGL(unpack_kernel, dim3((unsigned)grid), dim3(256), 0, stream, packed, n,
                       levels <= 16 ? 1 : 0, idx);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

int launch_dequant_tile(const PackedDesc &w, void *out, int out_dtype, int64_t ldo,
                        hipStream_t stream)
{
    if (w.N <= 0 || w.K <= 0)
        return EP_OK;
    TileArgs a{w.packed, w.scale, w.scale_dtype, w.ld_scale, w.cb, w.cb_dtype, w.levels,
               w.group, w.N, w.K, out, out_dtype, ldo};
    const int esz = out_dtype == EP_F32 ? 4 : 2;
    const bool fast = w.levels <= 16 && w.K % 32 == 0 && w.group % 32 == 0 &&
                      ((uintptr_t)w.packed & 15) == 0 && ((uintptr_t)out & 15) == 0 &&
                      (ldo * esz) % 16 == 0 && w.K <= 0x7fffffff &&
                      w.N <= 0x7fffffff && w.N * (w.K / 8) <= (int64_t)256 * kTile4 * 0x7fffffff;
    if (fast) {
        if (out_dtype == EP_F16)
            launch_tile4<EP_F16>(a, stream);
        else if (out_dtype == EP_BF16)
            launch_tile4<EP_BF16>(a, stream);
        else
            launch_tile4<EP_F32>(a, stream);
        EP_HIP_CHECK(hipGetLastError());
        return EP_OK;
    }
    dim3 grid((unsigned)((w.K + 255) / 256), (unsigned)(w.N < 65535 ? w.N : 65535));
    hipLaunchKernelGGL(dequant_tile_kernel, grid, dim3(256), 0, stream, a);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

int launch_embedding_rows(const PackedDesc &w, const int64_t *ids, int64_t n_ids, void *out,
                          int out_dtype, int64_t ldo, hipStream_t stream)
{
    if (n_ids <= 0 || w.K <= 0)
        return EP_OK;
    TileArgs a{w.packed, w.scale, w.scale_dtype, w.ld_scale, w.cb, w.cb_dtype, w.levels,
               w.group, w.N, w.K, out, out_dtype, ldo};
    dim3 grid((unsigned)((w.K + 255) / 256), (unsigned)(n_ids < 65535 ? n_ids : 65535));
    hipLaunchKernelGGL(embedding_rows_kernel, grid, dim3(256), 0, stream, a, ids, n_ids);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

}  // namespace ep
