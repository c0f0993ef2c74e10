// Prefill (M > 64 rows; f32 group scales: M > 4) fused codebook dequant-matmul on gfx950 MFMA.
//
// y[M, N] = x[M, K] . W[N, K]^T, W[n, k] = cb[idx[n, k]] * scale[n, k / group],
// for row counts where the contraction is compute-bound (and, with f32 group
// scales, from a few rows up).  Reference
// behaviour: the table kernel epure/kernels/_triton.py:54-107 (fp16 operands,
// fp32 accumulation) and, for the dense tile, materialize(float16)
// (runtime.py:78-89): the weight enters the product as fp16(fp16(cb) * fp16(scale)).
//
// Layout of the work (v_mfma_f32_32x32x16_f16):
//  * a workgroup is WAVES waves and covers WAVES x 32 NT weight rows x BM
//    activation rows; each wave owns NT 32-row N tiles and all BM rows, so
//    every weight is dequantized exactly once per workgroup, in registers,
//    straight into the B operand -- the dense weight never reaches LDS or
//    global memory.  From M = 128 (8-bit) or 160 (4-bit): 8 waves x BM = 128
//    (8-bit: one N tile per wave, as two would not fit 256 VGPRs; 4-bit: one
//    tile at M < 1024 and on small grids, else two), one workgroup per CU.  What bounds these tilings is the
//    bytes a CU pulls from L2 per k step (weights + the activation tile: a
//    CU keeps ~32 KiB of loads in flight), so wider workgroups -- more weight
//    rows per staged activation tile -- measured faster than 4-wave ones
//    (8-bit 1.1-1.15x) and than two weight tiles at 64 activation rows
//    (8-bit 1.25x); smaller M runs 8 waves x BM = 64 x one tile, two
//    workgroups per CU (M <= 32: 4 waves x 32 rows x two tiles);
//  * lane (j = lane & 31, h = lane >> 5) of a wave holds, per 64-k step and
//    N tile, 32 consecutive weights of row j (k = 32 h .. 32 h + 31 of the
//    step: one 16-byte load at 4 bits, two at 8 bits); MFMA sub-step s takes
//    weights 8 s .. 8 s + 7 of them as its k slots 8 h .. 8 h + 7, and the
//    activation operand is read from LDS with the same k mapping;
//  * dequantization is one LDS lookup per packed byte in a 256-entry table
//    replicated 32 times (lane & 31 reads its own copy: no bank conflicts),
//    addressed by one v_perm of the packed word, then the group scale is
//    applied in fp16 (v_pk_mul_f16);
//  * group scales are read as stored, fp16 or f32 (SF32: a fine-tuned
//    store's, rounded to fp16 where they enter the product as the generic
//    tiles did): 4-bit 2048 x 6144 at M = 201 with f32 scales 139.7 -> 41.5
//    us against mm_kernel, 6144 x 2048 at M = 2048 131.8 -> 99.9 us (36.2 and
//    88.4 since);
//  * activations are converted once to fp16 after the exact per-row
//    power-of-two rescale by a pre-kernel (row_prep_kernel, into the
//    workspace) and staged in LDS as they are, double buffered: step k + 1
//    is stored while step k is multiplied;
//  * weight loads run PD steps ahead in registers (buffer loads: a row past
//    N or a step past K reads zeros without touching memory);
//  * the step is software pipelined and its LDS reads are spread between its
//    MFMAs (step, interleave): in one phase after another the matrix cores
//    and the LDS were each under half busy (28% / 48% at 8-bit 2048 x 14336
//    x 4096).  Next to bind were the L1's line accesses (65% busy): staging
//    loads of eight threads per row read whole lines, and with groups of a
//    multiple of 128 one scale load serves two steps (a load of 32 rows'
//    scales touches 32 lines).  Together 8-bit 2048 x 14336 x 4096: 390 ->
//    354 us, 2048 x 4096 x 14336: 366 -> 319, 512 x 14336 x 4096: 106 -> 97;
//    4-bit 2048 x 14336 x 4096: 309 -> 281, 333 x 6656 x 2560: 44.7 -> 40.7
//    (graph replays, all launches);
//  * when the grid of (N / (32 WAVES NT)) x (M / BM) workgroups cannot fill the device,
//    K is split and the f32 partials are summed in split order by the
//    reduction shared with the small-M path (deterministic).
#include "ep_common.h"
#include "ep_internal.h"
#include "gemv_core.h"

#include <type_traits>

namespace ep {
namespace {

// A workgroup is WAVES waves (4 or 8), 32 * NT weight rows each.
constexpr int kPfBK = 64;              // k per step
constexpr int kPfCopies = 32;          // LDS table replicas
// A buffer offset past every buffer's end (buffers are at most this long);
// sums of two such parts plus a piece offset stay below 2^32.
constexpr uint32_t kPfOut = 0x7fffff00u;

struct PfArgs {
    const void *x;
    int64_t ldx;
    int M;
    const uint8_t *packed;
    uint32_t row_bytes;
    const void *scale;
    int64_t lds;
    const void *cb;
    int cb_dtype;
    int levels;
    int N;
    int K;
    int group;
    int gk_mul, gk_shift;  // k step kt starts in group (kt * gk_mul) >> gk_shift
    int ksteps;   // k steps per split (even)
    const int *rexp;
    uint32_t xbytes, wbytes, sbytes, cbbytes;
    void *y;
    int y_dtype;
    int64_t ldy;
    int accumulate;  // with one split: y += result (read in the epilogue)
    float *part;     // [S][M][N] partials (null: results go straight to y)
    // grouped experts (pf_kernel<..., true>): row tile blockIdx.y is entry
    // tiles[4 y ..] = (expert, first sorted row, rows, 0) while y < *ntiles;
    // sorted row p is token perm[p]; expert e's weight rows start
    // e * estride_w bytes and its scales e * estride_s elements further
    const int *perm;
    const int *tiles;
    const int *ntiles;
    int64_t estride_w, estride_s;
};

// Pieces of 8 values of a row for row_prep_kernel.
template <int XDT>
EP_DEV void prep_load(const char *base, int q, u32x4_t (&v)[XDT == EP_F32 ? 2 : 1])
{
#pragma unroll
    for (int i = 0; i < (XDT == EP_F32 ? 2 : 1); ++i)
        v[i] = *(const __attribute__((address_space(1))) u32x4_t *)(base + (int64_t)q * (XDT == EP_F32 ? 32 : 16) +
                                                                   16 * i);
}

template <int XDT>
EP_DEV void prep_values(const u32x4_t (&r)[XDT == EP_F32 ? 2 : 1], float (&v)[8])
{
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if constexpr (XDT == EP_F32) {
            v[t] = __uint_as_float(r[0][t]);
            v[4 + t] = __uint_as_float(r[1][t]);
        } else {
            unpack_pair<XDT>(r[0][t], v[2 * t], v[2 * t + 1]);
        }
    }
}

template <int XDT>
EP_DEV float prep_max(const u32x4_t (&r)[XDT == EP_F32 ? 2 : 1], float amax)
{
    float v[8];
    prep_values<XDT>(r, v);
#pragma unroll
    for (int t = 0; t < 8; ++t)
        amax = fmaxf(amax, fabsf(v[t]));
    return amax;
}

template <int XDT>
EP_DEV f16x8_t prep_round(const u32x4_t (&r)[XDT == EP_F32 ? 2 : 1], float pw)
{
    float v[8];
    prep_values<XDT>(r, v);
    f16x8_t h;
#pragma unroll
    for (int t = 0; t < 8; ++t)
        h[t] = (f16_t)(v[t] * pw);
    return h;
}

// Per-row exponent of the largest |x| (row_exponent), then the row rescaled
// by 2^-e and rounded to fp16 into xh [M][K]: converting once here saves the
// main kernel a conversion per N tile.  Bound by the latency of a row's
// loads, not by their bytes: a workgroup takes one row and each thread holds
// its PP pieces of 8 values in registers from the maximum to the rescale (a
// wave per row read the row twice, in a chain of loads and waits).
// bf16 rows: 201 x 6144 8.9 -> 3.3 us, 4096 x 2048 9.3 -> 7.3, 2048 x 2048
// 6.4 -> 5.4.
// Pieces past the row's end are clamped to its last one; those of rows
// beyond 8 pieces per thread are read again for the rescale.
template <int XDT, int PP>
__global__ void __launch_bounds__(256) row_prep_kernel(const void *x, int64_t ldx, int K, int *rexp, f16_t *xh)
{
    __shared__ float s_max[4];
    const int tid = threadIdx.x, nt = blockDim.x, row = blockIdx.x;
    const int pieces = K / 8;
    const char *base = (const char *)x + (int64_t)row * ldx * (XDT == EP_F32 ? 4 : 2);
    u32x4_t v[PP][XDT == EP_F32 ? 2 : 1];
#pragma unroll
    for (int p = 0; p < PP; ++p)
        prep_load<XDT>(base, min(tid + p * nt, pieces - 1), v[p]);
    float amax = 0.0f;
#pragma unroll
    for (int p = 0; p < PP; ++p)
        amax = prep_max<XDT>(v[p], amax);
    for (int q = tid + PP * nt; q < pieces; q += nt) {
        u32x4_t r[XDT == EP_F32 ? 2 : 1];
        prep_load<XDT>(base, q, r);
        amax = prep_max<XDT>(r, amax);
    }
    amax = wave_max(amax);
    if (nt > 64) {  // uniform
        if ((tid & 63) == 0)
            s_max[tid >> 6] = amax;
        __syncthreads();
        for (int w = 0; w < nt / 64; ++w)
            amax = fmaxf(amax, s_max[w]);
    }
    const int e = row_exponent(amax);
    if (tid == 0)
        rexp[row] = e;
    const float pw = ldexpf(1.0f, -e);
    f16x8_t *dst = (f16x8_t *)(xh + (int64_t)row * K);
#pragma unroll
    for (int p = 0; p < PP; ++p)
        if (tid + p * nt < pieces)
            dst[tid + p * nt] = prep_round<XDT>(v[p], pw);
    for (int q = tid + PP * nt; q < pieces; q += nt) {
        u32x4_t r[XDT == EP_F32 ? 2 : 1];
        prep_load<XDT>(base, q, r);
        dst[q] = prep_round<XDT>(r, pw);
    }
}

template <int XDT>
void row_prep_x(const void *x, int64_t ldx, int64_t M, int64_t K, int *rexp, f16_t *xh, hipStream_t stream)
{
    // as many waves (up to four) as the row has 64 pieces, then as few
    // pieces per thread as cover it
    const int64_t pieces = K / 8;
    const int nt = pieces <= 64 ? 64 : (pieces <= 128 ? 128 : 256);
    const int64_t pp = (pieces + nt - 1) / nt;
    const dim3 grid((unsigned)M), block((unsigned)nt);
    if (pp <= 1)
        hipLaunchKernelGGL((row_prep_kernel<XDT, 1>), grid, block, 0, stream, x, ldx, (int)K, rexp, xh);
    else if (pp <= 2)
        hipLaunchKernelGGL((row_prep_kernel<XDT, 2>), grid, block, 0, stream, x, ldx, (int)K, rexp, xh);
    else if (pp <= 4)
        hipLaunchKernelGGL((row_prep_kernel<XDT, 4>), grid, block, 0, stream, x, ldx, (int)K, rexp, xh);
    else
        hipLaunchKernelGGL((row_prep_kernel<XDT, 8>), grid, block, 0, stream, x, ldx, (int)K, rexp, xh);
}

// Waves per SIMD that the registers have to leave room for: two workgroups
// per CU (what the table's LDS allows) at 64 rows of eight waves and at four
// waves, one at 128 rows.
constexpr int pf_min_waves(int BM, int WAVES) { return BM == 64 && WAVES == 8 ? 4 : 8 / WAVES; }

template <int BITS, int BM, int PF, int NT, int WAVES, bool GR, bool SF32, bool G128>
__global__ void __launch_bounds__(WAVES * 64, pf_min_waves(BM, WAVES)) pf_kernel(PfArgs a)
{
    // steps of weights in flight: PF, but two where a scale load per piece
    // and step would not leave room for the second workgroup (8-bit 64-row
    // tiles of eight waves, groups below 128: 130 to 136 registers, one
    // workgroup per CU).  8-bit group 64, four steps and one workgroup / two
    // and two: 14336 x 4096 at M = 100 63.4 -> 57.4 us, 8192^2 at 127 69.8 ->
    // 62.4, 64 x 2048 x 1024 grouped, 4096 rows 97.5 -> 79.7; four steps at
    // two workgroups spill and took 58.5, 64.5 and 109
    constexpr int PD = BITS == 8 && BM == 64 && WAVES == 8 && !G128 ? 2 : PF;
    constexpr int SB = SF32 ? 4 : 2;             // bytes of a group scale
    constexpr int MT = BM / 32;                  // 32-row M tiles per wave
    constexpr int THREADS = WAVES * 64;
    constexpr int XE = 2;  // activations: fp16, pre-scaled per row (row_prep_kernel)
    constexpr int XROWS = THREADS / 8;           // activation rows per staging load (8 threads a row)
    constexpr int XP = BM / XROWS;               // 16-byte pieces per staging thread and step
    constexpr int WL = BITS == 4 ? 1 : 2;        // 16-byte weight loads per lane, N tile and step
    constexpr int NB = PD;                       // register sets of weights
    constexpr int UN = 4;  // unrolled steps (a multiple of PD; two register sets of activations and of scale pairs)
    static_assert(UN % PD == 0 && BM % XROWS == 0, "register sets rotate with the unroll");
    static_assert(THREADS >= 256, "one table entry per thread");
    static_assert(BM <= 128, "two activation buffers in the table's gaps");

    // 256-byte table entries: the lower 128 bytes hold entry b's 32 copies
    // (copy c at byte (b << 8) | (c << 2), the address one v_perm builds from
    // the packed byte); the upper 128 bytes of entry q * 128 + r hold row r
    // of activation buffer q (64 fp16 values), 16-byte piece p at position
    // p ^ (r & 7) so a 32-row operand read and the staging stores are free
    // of bank conflicts.
    __shared__ __align__(16) uint32_t tab[256 * 64];
    __shared__ uint32_t s_cbraw[256];
    __shared__ uint16_t s_cb16[256];
    __shared__ int s_e[BM];
    __shared__ int s_row[GR ? BM : 1];  // grouped: token of each tile row (-1: none)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, h = lane >> 5;
    const int nw = blockIdx.x * (WAVES * 32 * NT) + wave * (32 * NT);  // the wave's first weight row
    const int m0 = blockIdx.y * BM;
    const int kt0 = blockIdx.z * a.ksteps;
    const int nk = a.K / kPfBK;
    int gstart = 0, gcount = 0;
    if constexpr (GR) {
        // tiles past the sorted expert runs do nothing (uniform exit)
        if ((int)blockIdx.y >= *a.ntiles)
            return;
        const int *tl = a.tiles + 4 * blockIdx.y;
        const int e = tl[0];
        gstart = tl[1];
        gcount = tl[2];
        a.packed += (int64_t)e * a.estride_w;
        a.scale = (const char *)a.scale + e * a.estride_s * SB;
    }
    const auto rx = buffer_rsrc(a.x, a.xbytes), rw = buffer_rsrc(a.packed, a.wbytes);
    const auto rs = buffer_rsrc(a.scale, a.sbytes), rcb = buffer_rsrc(a.cb, a.cbbytes);

    // ---- first loads: codebook, row exponents, step 0's activations
    const uint32_t cbraw = __builtin_amdgcn_raw_buffer_load_b32(rcb, tid * 4, 0, 0);
    // row r of the tile: its token (row of x), -1 past M or the expert's run
    auto row_token = [&](int r) -> int {
        if constexpr (GR)
            return r < gcount ? a.perm[gstart + r] : -1;
        else
            return m0 + r < a.M ? m0 + r : -1;
    };
    const int xr = tid / 8, xq = tid % 8;  // staging: piece xq of rows xr, xr + XROWS, ..
    const int em = tid < BM ? row_token(tid) : -1;
    const int ex = *(const __attribute__((address_space(1))) int *)(a.rexp + (em >= 0 ? em : 0));

    // Load offsets = a per-lane part fixed for the whole loop (kPfOut for a
    // row past M or N) + a per-step part that is uniform (kPfOut for a step
    // past K or the split): one add per load.  Both parts stay below 2^31,
    // so a sum with either at kPfOut is past the buffer and reads zeros
    // (the bounds check covers the per-lane offset, which holds the sum).
    uint32_t xlo[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) {
        const int xm = row_token(xr + p * XROWS);
        xlo[p] = xm >= 0 ? (uint32_t)(((int64_t)xm * a.ldx + xq * 8) * XE) : kPfOut;
    }
    uint32_t wlo[NT][WL], slo[NT][WL];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = nw + nt * 32 + j;
#pragma unroll
        for (int l = 0; l < WL; ++l) {
            const int kl = 32 * h + 16 * l;  // first k of the piece within the step
            wlo[nt][l] = n < a.N ? (uint32_t)n * a.row_bytes + (uint32_t)(BITS == 4 ? kl / 2 : kl) : kPfOut;
            // the group divides 64 or is 64 * 2^i: the piece's group is the
            // step's (kt * gk_mul) >> gk_shift plus kl / group
            slo[nt][l] = n < a.N ? (uint32_t)(((int64_t)n * a.lds + kl / a.group) * SB) : kPfOut;
        }
    }
    const int kend = kt0 + a.ksteps < nk ? kt0 + a.ksteps : nk;
    auto issue_x = [&](int kt, u32x4_t (&xv)[XP]) {
        const uint32_t ks = kt < kend ? (uint32_t)(kt * kPfBK * XE) : kPfOut;
#pragma unroll
        for (int p = 0; p < XP; ++p)
            xv[p] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(xlo[p] + ks), 0, 0);
    };
    auto load_scale = [&](uint32_t off) -> uint32_t {
        if constexpr (SF32)
            return __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0);
        else
            return __builtin_amdgcn_raw_buffer_load_b16(rs, (int)off, 0, 0);
    };
    auto group_off = [&](int kt) -> uint32_t {
        return kt < kend ? (uint32_t)(((kt * a.gk_mul) >> a.gk_shift) * SB) : kPfOut;
    };
    auto issue_w = [&](int kt, u32x4_t (&w)[NT][WL], uint32_t (&sr)[NT][WL]) {
        const uint32_t kw = kt < kend ? (uint32_t)(kt * (BITS == 4 ? kPfBK / 2 : kPfBK)) : kPfOut;
        const uint32_t kg = group_off(kt);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int l = 0; l < WL; ++l) {
                w[nt][l] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(wlo[nt][l] + kw), 0, 0);
                if constexpr (!G128)
                    sr[nt][l] = load_scale(slo[nt][l] + kg);
            }
    };
    // G128 (groups of a multiple of 128): one scale serves the two steps
    // kt, kt + 1 (kt - kt0 even) and both pieces of each
    auto issue_s = [&](int kt, uint32_t (&sr)[NT]) {
        const uint32_t kg = group_off(kt);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            sr[nt] = load_scale(slo[nt][0] + kg);
    };

    // register sets, rotated with static indices: weights up to PD steps
    // ahead, activations two steps ahead (stored to LDS one step ahead)
    u32x4_t xv[2][XP];
    u32x4_t wb[NB][NT][WL];
    uint32_t sb[NB][NT][WL];
    uint32_t sp[2][NT];  // G128: the scales of two pairs of steps
    issue_x(kt0, xv[0]);
    issue_x(kt0 + 1, xv[1]);
    if constexpr (G128) {
        issue_s(kt0, sp[0]);
        issue_s(kt0 + 2, sp[1]);
    }
#pragma unroll
    for (int d = 0; d < PD; ++d)
        issue_w(kt0 + d, wb[d], sb[d]);
    __builtin_amdgcn_sched_barrier(0);

    // staged activation row r, buffer q, 16-byte piece p (see the layout above)
    auto xs_off = [](int q, int r, int p) -> uint32_t {
        return ((uint32_t)(q * 128 + r) << 8) + 128u + ((uint32_t)(p ^ (r & 7)) << 4);
    };
    auto store_x = [&](const u32x4_t (&v4)[XP], int q) {
#pragma unroll
        for (int p = 0; p < XP; ++p)
            *(u32x4_t *)((char *)tab + xs_off(q, xr + p * XROWS, xq)) = v4[p];
    };

    // codebook -> fp16 -> the replicated table; step 0's activations -> LDS
    if (tid < 256)
        s_cbraw[tid] = cbraw;
    if (tid < BM) {
        s_e[tid] = em >= 0 ? ex : 0;
        if constexpr (GR)
            s_row[tid] = em;
    }
    lds_barrier();
    {
        float c = 0.0f;
        if (tid < a.levels) {
            if (a.cb_dtype == EP_F32) {
                c = __uint_as_float(s_cbraw[tid]);
            } else {
                const uint16_t hb = (uint16_t)(s_cbraw[tid >> 1] >> (16 * (tid & 1)));
                c = a.cb_dtype == EP_F16 ? (float)f16_from_bits(hb) : bf16_to_f32(hb);
            }
        }
        // fp16 bits of the entries (past levels: 0, the Rust LUT's zeros)
        if (tid < 256)
            s_cb16[tid] = tid < a.levels ? f16_bits((f16_t)c) : (uint16_t)0;
        lds_barrier();
        // entry t: (cb[t & 15], cb[t >> 4]) at 4 bits, cb[t] twice at 8 bits
        if (tid < 256) {
            const uint32_t v = BITS == 4 ? ((uint32_t)s_cb16[tid & 15] | ((uint32_t)s_cb16[tid >> 4] << 16))
                                         : ((uint32_t)s_cb16[tid] | ((uint32_t)s_cb16[tid] << 16));
            u32x4_t *row = (u32x4_t *)(tab + tid * 64);
#pragma unroll
            for (int i = 0; i < kPfCopies / 4; ++i)
                row[i] = (u32x4_t){v, v, v, v};
        }
    }
    store_x(xv[0], 0);
    lds_barrier();

    f32x16_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[mt][nt][r] = 0.0f;

    const uint32_t c4 = (uint32_t)(lane & 31) << 2;  // the lane's table copy
    // Operand s of step register set r: the 8 weights of each lane for MFMA
    // sub-step s, in two parts with the MFMAs of another sub-step between
    // them: the table lookups, and their pairs times the group scale.
    constexpr int LQ = BITS == 4 ? 4 : 8;  // lookups per sub-step and N tile
    f16x2_t pr[NT][16];
    uint32_t tq[NT][LQ];
    auto lookup = [&](const u32x4_t (&w)[NT][WL], int s) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int b = 0; b < LQ; ++b) {
                const uint32_t word = BITS == 4 ? w[nt][0][s] : w[nt][WL == 2 ? s / 2 : 0][2 * (s % 2) + b / 4];
                tq[nt][b] = lds_read_u32(tab, __builtin_amdgcn_perm(word, c4, kSelByte[b % 4]));
            }
    };
    auto scaled = [&](int r, int s) {  // operand s of unrolled step r
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const uint32_t raw = G128 ? sp[(r / 2) % 2][nt] : sb[r % NB][nt][WL == 2 ? s / 2 : 0];
            const f16_t s16 = SF32 ? (f16_t)__uint_as_float(raw) : f16_from_bits((uint16_t)raw);
            const f16x2_t s2 = (f16x2_t){s16, s16};
#pragma unroll
            for (int p = 0; p < 4; ++p)
                pr[nt][4 * s + p] = as_f16x2(BITS == 4 ? tq[nt][p]
                                                       : __builtin_amdgcn_perm(tq[nt][(2 * p + 1) % LQ], tq[nt][(2 * p) % LQ],
                                                                               0x05040100u)) * s2;
        }
    };
    f16x8_t av[2][MT];
    auto read_a = [&](int q, int s, f16x8_t (&v)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            v[mt] = *(const f16x8_t *)((const char *)tab + xs_off(q, mt * 32 + j, 4 * h + s));
    };
    auto mfmas = [&](int s, const f16x8_t (&v)[MT]) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f16x8_t bv = {pr[nt][4 * s][0],     pr[nt][4 * s][1],     pr[nt][4 * s + 1][0],
                                pr[nt][4 * s + 1][1], pr[nt][4 * s + 2][0], pr[nt][4 * s + 2][1],
                                pr[nt][4 * s + 3][0], pr[nt][4 * s + 3][1]};
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[mt], bv, acc[mt][nt], 0, 0, 0);
        }
    };
    // One step (r = (kt - kt0) % UN), software pipelined.  Beside the MFMAs
    // of sub-step s run the activation reads of sub-step s + 1, the lookups
    // of operand s - 1 of step kt + 1 (s = 0: operand 3 of step kt) and the
    // scaling of the operand looked up a sub-step before; the step's one
    // barrier sits before its last MFMAs.  The LDS reads are spread between
    // the MFMAs (interleave): issued ahead of them, the eight waves' reads
    // filled the LDS queue while the matrix cores waited, then the other way
    // round (both under half busy).
    auto interleave = [&]() {
        constexpr int NM = MT * NT, ND = (MT + NT * LQ + NM - 1) / NM;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                              // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, ND, 0);  // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);                              // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](int kt, auto rc) {
        constexpr int r = decltype(rc)::value;
        constexpr int wc = r % NB, wn = (r + 1) % NB, q = r & 1;
        issue_x(kt + 2, xv[q]);
        __builtin_amdgcn_sched_barrier(0);
        scaled(r, 2);
        mfmas(0, av[0]);
        read_a(q, 1, av[1]);
        lookup(wb[wc], 3);
        interleave();
        scaled(r, 3);
        mfmas(1, av[1]);
        read_a(q, 2, av[0]);
        lookup(wb[wn], 0);
        interleave();
        issue_w(kt + PD, wb[wc], sb[wc]);  // the set that operand 3 was the last of
        if constexpr (G128 && r % 2 == 1)
            issue_s(kt + 3, sp[r / 2]);  // two pairs on, into the pair this step ends
        store_x(xv[q ^ 1], q ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        scaled(r + 1, 0);
        mfmas(2, av[0]);
        read_a(q, 3, av[1]);
        lookup(wb[wn], 1);
        interleave();
        // LDS-only barrier: __syncthreads() would also wait for the loads in
        // flight.  Every wave has read its operands of buffer q and stored
        // its part of buffer q ^ 1.
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        scaled(r + 1, 1);
        mfmas(3, av[1]);
        read_a(q ^ 1, 0, av[0]);
        lookup(wb[wn], 2);
        interleave();
    };

    // operands 0 and 1 of the first step, the lookups of operand 2
    lookup(wb[0], 0);
    scaled(0, 0);
    lookup(wb[0], 1);
    scaled(0, 1);
    lookup(wb[0], 2);
    read_a(0, 0, av[0]);
    // steps past the split's end load zeros and are not run
    for (int kt = kt0;; kt += UN) {
        step(kt, std::integral_constant<int, 0>{});
        if (kt + 1 >= kend)
            break;
        step(kt + 1, std::integral_constant<int, 1>{});
        if (kt + 2 >= kend)
            break;
        step(kt + 2, std::integral_constant<int, 2>{});
        if (kt + 3 >= kend)
            break;
        step(kt + 3, std::integral_constant<int, 3>{});
        if (kt + 4 >= kend)
            break;
    }

    // D[row][col] of a 32x32 tile: lane col + 32 * ((row / 4) % 2), register
    // (row % 4) + 4 * (row / 8)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int n = nw + nt * 32 + j;
            if (n >= a.N)
                continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = mt * 32 + (r % 4) + 4 * h + 8 * (r / 4);
                const int m = GR ? s_row[row] : m0 + row;
                if (GR ? m < 0 : m >= a.M)
                    continue;
                const float v = ldexpf(acc[mt][nt][r], s_e[row]);
                if (a.part) {
                    *(__attribute__((address_space(1))) float *)(a.part + ((int64_t)blockIdx.z * a.M + m) * a.N + n) = v;
                } else {
                    const int64_t off = (int64_t)m * a.ldy + n;
                    store_from_f32(a.y, a.y_dtype, off, a.accumulate ? v + load_as_f32(a.y, a.y_dtype, off) : v);
                }
            }
        }
}

// Tile rows, weight prefetch depth and K split for a shape.
// M from which the 8-wave 128-row tilings run (measured: 8-bit gains from
// M = 128, 4-bit only above it)
#ifndef EP_PF_BIG4_M
#define EP_PF_BIG4_M 160
#endif
#ifndef EP_PF_BIG8_M
#define EP_PF_BIG8_M 128
#endif
#ifndef EP_PF_PD8
#define EP_PF_PD8 4
#endif
struct PfPlan {
    int bm, nt, waves, S, ksteps;
};

// Activation rows of a tile.
int pf_rows(int bits, int64_t M)
{
    return M >= (bits == 4 ? EP_PF_BIG4_M : EP_PF_BIG8_M) ? 128 : M > 32 ? 64 : 32;
}

PfPlan pf_plan(int bits, int64_t M, int64_t N, int64_t K)
{
    PfPlan p;
    // measured: 128 x 2 tiles lead from M = 1024 (4-bit), 128 x 1 below, and
    // above while its grid is at most one round of workgroups on rows of up
    // to 96 steps: two tiles leave CUs idle there (f32 scales, 8192 x 1024
    // at M = 1024 63.7 -> 40.4 us, 50.6 on the generic tiles; 2048 x 1024 at
    // 2048 49.4 -> 34.6, 39.5; fp16 scales, 4096^2 at 1024 75.3 -> 60.9,
    // 6144^2 115.7 -> 107.0; longer rows gain more from the wider tile:
    // 5120 x 14336 at 1024 194 against 208).  The
    // 64-row tile on eight waves of one weight tile, two workgroups per CU
    // (four waves of two left a SIMD two waves to hide a step's lookups and
    // loads behind): 4-bit 4096^2 at M = 100 28.2 -> 24.3 us a call, 8192 x
    // 4096 at 65 31.6 -> 28.9, 8-bit 4096 x 14336 at 100 46.0 -> 40.3, 14336 x
    // 4096 at 127 48.1 -> 44.6.
    p.bm = pf_rows(bits, M);
    const bool one_round = ((N + 255) / 256) * ((M + 127) / 128) <= device_cus() && K <= 96 * kPfBK;
    p.nt = p.bm == 32 || (p.bm == 128 && bits == 4 && M >= 1024 && !one_round) ? 2 : 1;
    p.waves = p.bm == 32 ? 4 : 8;
    const int bn = p.waves * 32 * p.nt;
    const int64_t tiles = ((N + bn - 1) / bn) * ((M + p.bm - 1) / p.bm);
    const int nk = (int)(K / kPfBK);
    // K split in two while the grid stays within one round of resident
    // workgroups (one per CU at 128 rows, else two): a split past that only
    // adds partials (14336 x 4096 at M = 512, 224 tiles: 132.7 us with 2 splits, 110.5
    // with none; M = 256, 112 tiles: 93.6 us with 4, 80.9 with 2)
    const int target = (p.bm == 128 ? 1 : 2) * device_cus();
    int S = 1;
    while (tiles * S * 2 <= target && S < 8 && nk / (S * 2) >= 8)
        S *= 2;
    const int ks = ((nk + S - 1) / S + 1) / 2 * 2;
    p.S = (nk + ks - 1) / ks;
    p.ksteps = ks;
    return p;
}

template <int BITS, int BM, int PD, int NT, int WAVES>
int pf_launch(const PfArgs &a, const PfPlan &p, bool sf32, hipStream_t s)
{
    constexpr int BN = WAVES * 32 * NT;
    const dim3 grid((unsigned)((a.N + BN - 1) / BN), (unsigned)((a.M + BM - 1) / BM), (unsigned)p.S);
    const bool g128 = a.group % 128 == 0;
    const auto kern = sf32 ? (g128 ? pf_kernel<BITS, BM, PD, NT, WAVES, false, true, true>
                                   : pf_kernel<BITS, BM, PD, NT, WAVES, false, true, false>)
                           : (g128 ? pf_kernel<BITS, BM, PD, NT, WAVES, false, false, true>
                                   : pf_kernel<BITS, BM, PD, NT, WAVES, false, false, false>);
    hipLaunchKernelGGL(kern, grid, dim3(WAVES * 64), 0, s, a);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

template <int BITS, int BM, int PD, int NT, int WAVES>
int pf_launch_grouped(const PfArgs &a, unsigned tiles_y, bool sf32, hipStream_t s)
{
    constexpr int BN = WAVES * 32 * NT;
    const dim3 grid((unsigned)((a.N + BN - 1) / BN), tiles_y, 1u);
    const bool g128 = a.group % 128 == 0;
    const auto kern = sf32 ? (g128 ? pf_kernel<BITS, BM, PD, NT, WAVES, true, true, true>
                                   : pf_kernel<BITS, BM, PD, NT, WAVES, true, true, false>)
                           : (g128 ? pf_kernel<BITS, BM, PD, NT, WAVES, true, false, true>
                                   : pf_kernel<BITS, BM, PD, NT, WAVES, true, false, false>);
    hipLaunchKernelGGL(kern, grid, dim3(WAVES * 64), 0, s, a);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

}  // namespace

bool prefill_grouped_serves(const PackedDesc &w, const ActDesc &x, int64_t T)
{
    // one expert's rows and scales, and the T token rows of x, in buffer range
    return prefill_serves(w, x, T);
}

size_t prefill_grouped_workspace(int64_t T, int64_t K)
{
    return (size_t)((T * 4 + 255) / 256 * 256) + (size_t)((T * K * 2 + 255) / 256 * 256);
}

// Stacked experts grouped by expert (tiles from the device sort): the fp16
// copy of every token row, then pf_kernel over each expert's row tiles (bm
// 32, 64 or 128 rows, the whole K per workgroup), results at the tokens' rows.
int launch_prefill_grouped(const PackedDesc &w, const ActDesc &x, int64_t T, const int *perm,
                           const int *tiles, const int *ntiles, int64_t experts, int bm, unsigned tiles_y,
                           const OutDesc &y, void *ws, hipStream_t stream)
{
    const int bits = w.bits();
    const bool sf32 = w.scale_dtype == EP_F32;
    int *rexp = (int *)ws;
    f16_t *xh = (f16_t *)((char *)ws + (T * 4 + 255) / 256 * 256);
    if (const int rc = launch_row_prep(x, T, w.K, rexp, xh, stream); rc != EP_OK)
        return rc;
    PfArgs a{};
    a.xbytes = (uint32_t)(T * w.K * 2);
    a.wbytes = (uint32_t)(w.N * (bits == 4 ? w.K / 2 : w.K));
    a.sbytes = (uint32_t)(((w.N - 1) * w.ld_scale + (w.K + w.group - 1) / w.group) * (sf32 ? 4 : 2));
    a.cbbytes = (uint32_t)(w.levels * (w.cb_dtype == EP_F32 ? 4 : 2));
    a.x = xh;
    a.ldx = w.K;
    a.M = (int)T;
    a.packed = w.packed;
    a.row_bytes = (uint32_t)(bits == 4 ? w.K / 2 : w.K);
    a.scale = w.scale;
    a.lds = w.ld_scale;
    a.cb = w.cb;
    a.cb_dtype = w.cb_dtype;
    a.levels = w.levels;
    a.N = (int)w.N;
    a.K = (int)w.K;
    a.group = w.group;
    a.gk_mul = w.group <= kPfBK ? kPfBK / w.group : 1;
    a.gk_shift = 0;
    while (w.group > kPfBK && (kPfBK << a.gk_shift) < w.group)
        ++a.gk_shift;
    const int nk = (int)(w.K / kPfBK);
    a.rexp = rexp;
    a.y = y.ptr;
    a.y_dtype = y.dtype;
    a.ldy = y.ld;
    a.accumulate = 0;
    a.part = nullptr;
    a.perm = perm;
    a.tiles = tiles;
    a.ntiles = ntiles;
    a.estride_w = w.N * (int64_t)a.row_bytes;
    a.estride_s = w.N * w.ld_scale;
    a.ksteps = (nk + 1) / 2 * 2;  // the whole K per workgroup
    // 64-row tiles: one 32-row weight tile per wave, so that a SIMD has four
    // waves to hide a step's lookups and loads behind (four waves of two
    // tiles left it two); eight waves, or four (128 weight rows) where those
    // workgroups, two per CU, are all resident at the experts' mean rows.
    // Whole calls, 4-bit: 128 x 768 x 2048, 4096 rows, four waves of two
    // tiles / eight / four of one: 73.8 / 67.9 / 72.8 us; 64 x 2048 x 1024
    // 85.4 / 71.0 / 78.2; 8 x 2048 x 3072, 300 rows 52.2 / 44.1 / 38.5; 8-bit
    // 128 x 768 x 2048 92.3 / 83.7 / 81.7; 32 x 1024 x 2048, 1200 rows 60.7 /
    // 49.6 / 43.1.  32-row tiles take four waves: of one weight tile by the
    // same rule (4-bit 8 x 2048 x 3072, 120 rows 43.8 -> 33.7 us; past it two
    // stay ahead: 128 x 1536 x 2048, 3200 rows 99.3 against 102.0), and with
    // 8-bit indices, a lookup per weight, always (32 x 1024 x 2048, 400 rows
    // 50.8 -> 36.8; 128 x 768 x 2048, 1024 rows 69.2 -> 64.6).
    const int64_t mean = (T + experts - 1) / experts;
    const bool narrow = experts * ((mean + bm - 1) / bm) * ((w.N + 127) / 128) <= 2 * (int64_t)device_cus();
    if (bits == 4) {
        if (bm == 128) {
            return pf_launch_grouped<4, 128, 4, 1, 8>(a, tiles_y, sf32, stream);
        }
        if (bm == 32)
            return narrow ? pf_launch_grouped<4, 32, 4, 1, 4>(a, tiles_y, sf32, stream)
                          : pf_launch_grouped<4, 32, 4, 2, 4>(a, tiles_y, sf32, stream);
        return narrow ? pf_launch_grouped<4, 64, 4, 1, 4>(a, tiles_y, sf32, stream)
                      : pf_launch_grouped<4, 64, 4, 1, 8>(a, tiles_y, sf32, stream);
    }
    if (bm == 128) {
        return pf_launch_grouped<8, 128, EP_PF_PD8, 1, 8>(a, tiles_y, sf32, stream);
    }
    if (bm == 32)
        return pf_launch_grouped<8, 32, 4, 1, 4>(a, tiles_y, sf32, stream);
    return narrow ? pf_launch_grouped<8, 64, 4, 1, 4>(a, tiles_y, sf32, stream)
                  : pf_launch_grouped<8, 64, 4, 1, 8>(a, tiles_y, sf32, stream);
}

int launch_row_prep(const ActDesc &x, int64_t M, int64_t K, int *rexp, void *xh, hipStream_t stream)
{
    if (x.dtype == EP_F32)
        row_prep_x<EP_F32>(x.ptr, x.ld, M, K, rexp, (f16_t *)xh, stream);
    else if (x.dtype == EP_F16)
        row_prep_x<EP_F16>(x.ptr, x.ld, M, K, rexp, (f16_t *)xh, stream);
    else
        row_prep_x<EP_BF16>(x.ptr, x.ld, M, K, rexp, (f16_t *)xh, stream);
    EP_HIP_CHECK(hipGetLastError());
    return EP_OK;
}

bool prefill_serves(const PackedDesc &w, const ActDesc &x, int64_t M)
{
    const int bits = w.bits();
    if (M < 1 || M > ((int64_t)1 << 24) || w.N < 1 || w.K < kPfBK || w.K % kPfBK != 0)
        return false;
    if ((w.scale_dtype != EP_F16 && w.scale_dtype != EP_F32) || w.group % (bits == 4 ? 32 : 16) != 0)
        return false;
    // groups that divide the 64-wide k step or are 64 * 2^i (others: the
    // generic MFMA path)
    if (64 % w.group != 0 && (w.group % 64 != 0 || ((w.group / 64) & (w.group / 64 - 1)) != 0))
        return false;
    const int esz = x.dtype == EP_F32 ? 4 : 2;
    const int64_t rb = bits == 4 ? w.K / 2 : w.K;
    const int64_t G = (w.K + w.group - 1) / w.group;
    if (w.N * rb > kPfOut || ((M - 1) * x.ld + w.K) * esz > kPfOut || ((w.N - 1) * w.ld_scale + G) * (w.scale_dtype == EP_F32 ? 4 : 2) > kPfOut)
        return false;
    if (((uintptr_t)w.packed & 15) != 0 || ((uintptr_t)x.ptr & 15) != 0)
        return false;
    return (x.ld * esz) % 16 == 0;
}

// f32 group scales: whether the tiles lead the generic ones, which have no
// rescaled copy of x and no 64 KiB table to write before the first step and
// so win short rows, less so where the weight rows alone give every CU a
// workgroup.  Tiles / generic at N of 64 to 16384 (65536): 32-row tiles
// 4-bit M = 32 K = 384 1.16-1.21 (0.97), 512 1.1-1.15 (0.92), 768 1.0-1.06,
// 832 0.97-1.0; 8-bit K = 640 (1.01), 768 (0.98), 960 0.98-1.06, 1024
// 0.66-0.78; 64-row tiles at M = 48 K = 128 0.9-1.07, 256 0.81-0.97, from M =
// 65 0.7-0.85 at every K (there the generic kernel takes 128-row tiles);
// 128-row tiles K = 256 (0.87-1.09), 384 0.9-1.09 (0.82-1.01), 512 4-bit
// 0.89-1.04, 8-bit 0.9-1.08, 640 8-bit 0.83-1.03.
bool prefill_leads_f32(int bits, int64_t M, int64_t N, int64_t K)
{
    const int bm = pf_rows(bits, M);
    const int64_t steps = K / kPfBK;
    const bool wide = (N + 255) / 256 >= device_cus();
    if (bm == 32)
        return steps >= (bits == 4 ? (wide ? 8 : 13) : (wide ? 12 : 16));
    if (bm == 64)
        return M > 64 || steps >= 4;
    return steps >= (wide ? 6 : bits == 4 ? 8 : 10);
}

// The same for grouped experts of bm rows per tile: 32 rows 4-bit K = 128
// 0.97-1.27, 256 0.9-1.05; 8-bit K = 256 0.9-1.14, 384 0.85-1.0; 64 rows K =
// 128 0.78-1.15, 256 0.74-1.12; 128 rows K = 256 1.01-1.08, 384 0.95-1.04.
bool prefill_grouped_leads_f32(int bits, int bm, int64_t K)
{
    return K / kPfBK >= (bm == 64 || (bm == 32 && bits == 4) ? 4 : 6);
}

// Workspace: row exponents, the fp16 activations, then the split partials;
// none for rows shorter than a k step, which the tiles do not serve.
size_t prefill_workspace(int64_t M, int64_t N, int64_t K, int levels)
{
    if (K < kPfBK)
        return 0;
    const PfPlan p = pf_plan(levels <= 16 ? 4 : 8, M, N, K);
    const size_t ex = (size_t)((M * 4 + 255) / 256 * 256);
    const size_t xh = (size_t)((M * K * 2 + 255) / 256 * 256);
    return ex + xh + (p.S > 1 ? (size_t)p.S * (size_t)M * (size_t)N * sizeof(float) : 0);
}

int launch_prefill(const PackedDesc &w, const ActDesc &x, int64_t M, const OutDesc &y, void *ws,
                   size_t ws_bytes, hipStream_t stream)
{
    if (!prefill_serves(w, x, M))
        return EP_DECLINE_SHAPE;
    const int bits = w.bits();
    const bool sf32 = w.scale_dtype == EP_F32;
    const PfPlan p = pf_plan(bits, M, w.N, w.K);
    const bool partials = p.S > 1;
    const size_t ex = (size_t)((M * 4 + 255) / 256 * 256);
    const size_t xhb = (size_t)((M * w.K * 2 + 255) / 256 * 256);
    const size_t need = ex + xhb + (partials ? (size_t)p.S * (size_t)M * (size_t)w.N * sizeof(float) : 0);
    if (!ws || ws_bytes < need)
        return set_error(EP_ERR_WORKSPACE, "workspace of %zu bytes needed, %zu given", need, ws_bytes);
    int *rexp = (int *)ws;
    f16_t *xh = (f16_t *)((char *)ws + ex);
    if (const int rc = launch_row_prep(x, M, w.K, rexp, xh, stream); rc != EP_OK)
        return rc;
    PfArgs a{};
    a.xbytes = (uint32_t)(M * w.K * 2);
    a.wbytes = (uint32_t)(w.N * (bits == 4 ? w.K / 2 : w.K));
    a.sbytes = (uint32_t)(((w.N - 1) * w.ld_scale + (w.K + w.group - 1) / w.group) * (sf32 ? 4 : 2));
    a.cbbytes = (uint32_t)(w.levels * (w.cb_dtype == EP_F32 ? 4 : 2));
    a.x = xh;
    a.ldx = w.K;
    a.M = (int)M;
    a.packed = w.packed;
    a.row_bytes = (uint32_t)(bits == 4 ? w.K / 2 : w.K);
    a.scale = w.scale;
    a.lds = w.ld_scale;
    a.cb = w.cb;
    a.cb_dtype = w.cb_dtype;
    a.levels = w.levels;
    a.N = (int)w.N;
    a.K = (int)w.K;
    a.group = w.group;
    a.gk_mul = w.group <= kPfBK ? kPfBK / w.group : 1;
    a.gk_shift = 0;
    while (w.group > kPfBK && (kPfBK << a.gk_shift) < w.group)
        ++a.gk_shift;
    a.ksteps = p.ksteps;
    a.rexp = rexp;
    a.y = y.ptr;
    a.y_dtype = y.dtype;
    a.ldy = y.ld;
    a.accumulate = y.accumulate;
    a.part = partials ? (float *)((char *)ws + ex + xhb) : nullptr;
    int rc;
    if (bits == 4)
        rc = p.bm == 128  ? (p.nt == 1 ? pf_launch<4, 128, 4, 1, 8>(a, p, sf32, stream)
                                       : pf_launch<4, 128, 2, 2, 8>(a, p, sf32, stream))
             : p.bm == 64 ? pf_launch<4, 64, 4, 1, 8>(a, p, sf32, stream)
                          : pf_launch<4, 32, 4, 2, 4>(a, p, sf32, stream);
    else
        rc = p.bm == 128  ? pf_launch<8, 128, EP_PF_PD8, 1, 8>(a, p, sf32, stream)
             : p.bm == 64 ? pf_launch<8, 64, 4, 1, 8>(a, p, sf32, stream)
                          : pf_launch<8, 32, 4, 2, 4>(a, p, sf32, stream);
    if (rc != EP_OK || !partials)
        return rc;
    return launch_split_reduce(a.part, p.S, M, w.N, y, stream);
}

}  // namespace ep
