// gemm_chunk.hip — the GEMM of a prompt chunk (more than 32 rows) over panel
// weights, for gfx950.
//
// y[b][r] = sum over blocks of scale(r, blk) * sum_i q(r, blk, i) * x[b][i],
// the reference's q8_gemv (crates/engine/src/q8_gemv.rs:234-242) for every row
// b of a chunk at once; the reference runs its prompt projections token by
// token on the ANE (crates/cli/src/main.rs:1168-1429).
#include "panel.h"


namespace anehip {

namespace {

// 8 signed bytes q (Q8_0) as fp16 q, exactly: q + 128 placed in the
// mantissa of 1024 (fp16 0x64xx is 1024 + xx), minus 1152
__device__ __forceinline__ h8v q8_fragment(uint32_t w0, uint32_t w1) {
    const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
    const u32x4 p = {__builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u),
                     __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u),
                     __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u),
                     __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)};
    const h8v k = {1152, 1152, 1152, 1152, 1152, 1152, 1152, 1152};
    return __builtin_bit_cast(h8v, p) - k;
}
// 8 nibbles (Q4_0: the low, shift 0, or high, shift 4, nibbles of 8 bytes)
// as fp16 nibble - 8, exactly (1024 + nibble, minus 1032)
__device__ __forceinline__ h8v q4_fragment(uint32_t w0, uint32_t w1, int shift) {
    const uint32_t n0 = (w0 >> shift) & 0x0f0f0f0fu, n1 = (w1 >> shift) & 0x0f0f0f0fu;
    const u32x4 p = {__builtin_amdgcn_perm(0x64646464u, n0, 0x04010400u),
                     __builtin_amdgcn_perm(0x64646464u, n0, 0x04030402u),
                     __builtin_amdgcn_perm(0x64646464u, n1, 0x04010400u),
                     __builtin_amdgcn_perm(0x64646464u, n1, 0x04030402u)};
    const h8v k = {1032, 1032, 1032, 1032, 1032, 1032, 1032, 1032};
    return __builtin_bit_cast(h8v, p) - k;
}

constexpr int kXcds = 8;
constexpr int kRowBlock = 64;   // x rows of a workgroup (two 32-row groups)
constexpr int kTileRows = 256;  // weight rows of a workgroup (one 64-row tile per wave)
constexpr int kStages = 3;      // LDS buffers of 64 columns (2 quant blocks) each
constexpr int kStageBytes = 2 * 4 * 4096;  // [K half][row group, plane][4 KiB: 4 column steps of 1 KiB]

// One wave's weight operands for one stage: its tile's quant bytes as stored
// (16-byte chunk c of row lane; Q8_0: column step c, Q4_0: block c) and the
// row's two block scales.
template <uint32_t T> struct StageW {
    static constexpr int kVecs = T == ANEHIP_GGML_Q8_0 ? 4 : 2;
    u32x4 q[kVecs];
    uint32_t d;
};

// Lane l of the MFMA's B operand holds 8 columns of one row: rows 0-31 of the
// tile in one fragment, 32-63 in the other, columns 0-7 of a 16-byte chunk in
// lanes 0-31 and 8-15 in lanes 32-63.  Swapping the upper lanes of a chunk's
// first 8 bytes with the lower lanes of its last 8 gives both:
// lo = rows 0-31, hi = rows 32-63.
__device__ __forceinline__ void chunk_halves(u32x4 q, u32x2 &lo, u32x2 &hi) {
    const auto s0 = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
    lo = u32x2{s0[0], s1[0]};
    hi = u32x2{s0[1], s1[1]};
}

// Workgroup: 64 rows of x (two 32-row plane groups) against 256 weight rows.
// Wave w: tile w % 4, and the first or second half of the workgroup's columns
// (w / 4), its 64 x 64 sums in registers; the halves are added through LDS at
// the end.  Per stage of 64 columns:
//  * x fragments (hi and lo of both groups, 16 KiB per half) go from global
//    memory straight to LDS two stages ahead (each wave 4 loads of 1 KiB), in
//    the order the MFMA's A operand is read;
//  * each wave loads its own tile's bytes three stages ahead and turns them into
//    B fragments of q as fp16 (exact) in registers: no two waves of the
//    workgroup need the same ones;
//  * c = x_hi q + x_lo q over a 32-column block's two column steps on
//    v_mfma_f32_32x32x16_f16, then sums += c d on the VALU: the block's
//    (sum q x) d of q8_gemv.rs:234-242.
// What bounds it: a block costs 8 MFMAs (256 cycles) and 32 scale FMAs + ~24
// conversion instructions (~230 cycles) per 32 x rows and wave, so the matrix
// cores and the VALU are both near full; a copy without the scale FMAs takes
// 85 us where the kernel takes 96 (12288 x 2048, 960 rows), without weight
// loads 88.  Hence the tile: a 64 x 64 wave tile converts each weight once per
// 64 rows, and reads 8 KiB of x from LDS per 16 MFMAs (a 128 x 32 tile reads
// twice that, past the LDS rate; two waves sharing converted weights through
// LDS likewise); K halves rather than smaller tiles give 2 waves per SIMD.
// 16-byte weight loads with a lane swap, three stages ahead, against 8-byte
// ones of the fragment two stages ahead: 96 against 103 us; scheduling the
// FMAs between the next tile's MFMAs: 95, raised wave priority over the
// MFMAs: 103.  Measured on MI355X (Q8_0): 12288 x 2048, 256 / 960 rows 31.4 /
// 96 us = 410 / 505 TFLOP/s (two passes: 1.0 PFLOP/s of fp16 MFMA, against
// 1.24 of a large library matrix product); the kernel before it (32-row waves
// reading x from L2, one loader wave converting for 8) 42 us at 256 rows.
// The planes' exponent has to be one per row (Planes::uniform); the sums go
// out times 2^E.  With SILU (interleaved [gate; up] panels, m = 2 F, one K
// split) lane l of a wave holds feature l % 32's gate sums in the first 32
// columns and its up sums in the other: h = SiLU(g) u to out[row][F].
template <uint32_t T, bool SILU>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_chunk(
    const uint8_t *__restrict__ Wp, Planes xp, float *__restrict__ out, int m, int n, int rows, int nblocks,
    int rblocks, int ksplit, size_t split_stride) {
    constexpr int CH = Panel<T>::kChunks, SUB = CH / 4 * 1024;  // a stage's quant bytes
    constexpr int V = StageW<T>::kVecs;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kStages * kStageBytes];
    __shared__ float esc[kRowBlock];
    // workgroups go to the XCDs in turn; each XCD takes one contiguous range
    // of (weight tile block, K split, row block) with the row blocks
    // innermost, so that a tile block's bytes are shared in one L2
    const int total = nblocks * ksplit * rblocks, per_xcd = (total + kXcds - 1) / kXcds;
    const int L = ((int)blockIdx.x % kXcds) * per_xcd + (int)blockIdx.x / kXcds;
    if (L >= total) return;
    const int rb = L % rblocks, pair = L / rblocks, ks = pair % ksplit, nb = pair / ksplit;
    const int nsb = n >> 8, ptiles = (m + kWave - 1) / kWave;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int kh = wave >> 2, w4 = wave & 3;
    const int hs = 2 * (nsb / ksplit);        // stages per half
    const int g0 = (2 * ks + kh) * hs;        // this half's first stage of the row
    if (threadIdx.x < kRowBlock) {
        const int row = min(kRowBlock * rb + (int)threadIdx.x, rows - 1);
        esc[threadIdx.x] = ldexpf(1.0f, (int)xp.xe[(size_t)row * xe_stride(n)]);
    }

    // x: wave w4 of a half copies one 4 KiB block (group w4 / 2, plane w4 % 2)
    // per stage; a stage's 4 column steps are consecutive in the planes
    const int groups = (rows + 31) >> 5;
    const uint8_t *xsrc = reinterpret_cast<const uint8_t *>((w4 & 1 ? xp.lo : xp.hi) +
                                                            (size_t)min(2 * rb + (w4 >> 1), groups - 1) * xf_plane_len(n));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t xdst = lds0 + (uint32_t)(kh * 16384 + w4 * 4096);
    const uint32_t xoff = 16u * (uint32_t)lane;
    auto load_x = [&](int s, int buf) {
        const uint8_t *src = xsrc + (size_t)(g0 + min(s, hs - 1)) * 4096;
        // the instruction offset moves both the source and the LDS address
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dwordx4 %1, %2\n\t"
            "global_load_lds_dwordx4 %1, %2 offset:1024\n\t"
            "global_load_lds_dwordx4 %1, %2 offset:2048\n\t"
            "global_load_lds_dwordx4 %1, %2 offset:3072"
            :
            : "s"(xdst + (uint32_t)(buf * kStageBytes)), "v"(xoff), "s"(src)
            : "memory");
    };
    // weights: buffer loads, the lane's offset in a chunk, the stage's wave-uniform
    const int tile = min(4 * nb + w4, ptiles - 1);
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(Wp), 0, (int)((size_t)ptiles * nsb * Panel<T>::kBytes), kBufferWord3);
    const int wbase = tile * nsb * Panel<T>::kBytes;
    StageW<T> ring[3];
    auto stage_off = [&](int s, int &qo, int &so) {
        const int g = g0 + min(s, hs - 1), p = wbase + (g >> 2) * Panel<T>::kBytes;
        qo = p + (g & 3) * SUB;
        so = p + CH * 1024 + (g & 3) * 4;
    };
    auto load_block = [&](StageW<T> &u, int qo, int b) {
#pragma unroll
        for (int v = V / 2 * b; v < V / 2 * (b + 1); v++)
            u.q[v] =
                __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, 16 * lane + v * 1024, qo, 0));
    };
    auto load_scales = [&](StageW<T> &u, int so) { u.d = __builtin_amdgcn_raw_buffer_load_b32(wrsrc, 16 * lane, so, 0); };

    f32x16 acc[2][2] = {{f32x16{}, f32x16{}}, {f32x16{}, f32x16{}}};  // [row group][32-row half of the tile]
    // x of the next stage has landed: its 4 loads (this wave's) are followed
    // by at least 4 + 2 (V + 1) younger ones
    auto x_landed = [&]() {
        if constexpr (V == 4) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    };
    const u32x4 *xl = reinterpret_cast<const u32x4 *>(lds + kh * 16384) + lane;
    // One stage: the products of stage s (x in buffer b0), while x of stage
    // s + 2 is on its way to buffer b2 and weights of s + 3 to the registers
    // that this stage's leave.
    auto stage = [&](StageW<T> &u, int s, int b0, int b2) {
        int qo, so;
        stage_off(s + 3, qo, so);
        load_x(s + 2, b2);
        const u32x4 *xs = xl + b0 * (kStageBytes / 16);
        const auto ds = __builtin_amdgcn_permlane32_swap(u.d, u.d, false, false);
#pragma unroll
        for (int b = 0; b < 2; b++) {
            h8v a[2][2][2];  // [group][plane][column step]
#pragma unroll
            for (int i = 0; i < 8; i++)
                a[i >> 2][(i >> 1) & 1][i & 1] =
                    __builtin_bit_cast(h8v, xs[((i >> 1) * 4096 + (2 * b + (i & 1)) * 1024) / 16]);
            u32x2 q0[2], q1[2];
            chunk_halves(u.q[V / 2 * b], q0[0], q0[1]);
            if constexpr (T == ANEHIP_GGML_Q8_0) chunk_halves(u.q[V / 2 * b + 1], q1[0], q1[1]);
#pragma unroll
            for (int cb = 0; cb < 2; cb++) {
                h8v w0, w1;
                if constexpr (T == ANEHIP_GGML_Q8_0) {
                    w0 = q8_fragment(q0[cb].x, q0[cb].y);
                    w1 = q8_fragment(q1[cb].x, q1[cb].y);
                } else {
                    w0 = q4_fragment(q0[cb].x, q0[cb].y, 0);
                    w1 = q4_fragment(q0[cb].x, q0[cb].y, 4);
                }
                const float d = __half2float(__ushort_as_half((unsigned short)(ds[cb] >> (16 * b))));
                f32x16 c[2];
#pragma unroll
                for (int g = 0; g < 2; g++) c[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[g][0][0], w0, f32x16{}, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 2; g++) c[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[g][1][0], w0, c[g], 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 2; g++) c[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[g][0][1], w1, c[g], 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 2; g++) c[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[g][1][1], w1, c[g], 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 2; g++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[g][cb][r] = fmaf(c[g][r], d, acc[g][cb][r]);
            }
            load_block(u, qo, b);
        }
        load_scales(u, so);
        x_landed();
        lds_barrier();
    };
#pragma unroll
    for (int s = 0; s < 3; s++) {
        int qo, so;
        if (s < 2) load_x(s, s);
        stage_off(s, qo, so);
        load_block(ring[s], qo, 0);
        load_block(ring[s], qo, 1);
        load_scales(ring[s], so);
    }
    x_landed();
    lds_barrier();
    for (int s = 0;;) {
        stage(ring[0], s, 0, 2);
        if (++s >= hs) break;
        stage(ring[1], s, 1, 0);
        if (++s >= hs) break;
        stage(ring[2], s, 2, 1);
        if (++s >= hs) break;
    }
    // the two halves' sums: half kh finishes row group kh, the other group's
    // sums cross through LDS once every copy into it has landed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    float *red = reinterpret_cast<float *>(lds);
    auto park = [&](const f32x16 (&v)[2]) {
#pragma unroll
        for (int i = 0; i < 32; i++) red[(wave * 32 + i) * kWave + lane] = v[i >> 4][i & 15];
    };
    if (kh == 0) park(acc[1]);
    else park(acc[0]);
    lds_barrier();
    auto finish = [&](f32x16 (&v)[2]) {
        const float *o = red + (size_t)((wave ^ 4) * 32) * kWave + lane;
#pragma unroll
        for (int i = 0; i < 32; i++) v[i >> 4][i & 15] += o[i * kWave];
        if (4 * nb + w4 >= ptiles) return;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int lr = 32 * kh + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), row = kRowBlock * rb + lr;
            if (row >= rows) continue;
            const float sc = esc[lr];
            if constexpr (SILU) {
                const float g = v[0][r] * sc, up = v[1][r] * sc;
                out[(size_t)row * (m >> 1) + 32 * (4 * nb + w4) + (lane & 31)] = (g / (1.0f + expf(-g))) * up;
            } else {
                float *o = out + (size_t)ks * split_stride + (size_t)row * m;
#pragma unroll
                for (int cb = 0; cb < 2; cb++) {
                    const int col = kWave * (4 * nb + w4) + 32 * cb + (lane & 31);
                    if (col < m) o[col] = v[cb][r] * sc;
                }
            }
        }
    };
    if (kh == 0) finish(acc[0]);
    else finish(acc[1]);
}

// fp32 x[rows][n] -> uniform fragment-order planes (Planes::uniform), one
// workgroup per row: the row's largest |x|, then hi + lo of x 2^-E, 8
// consecutive columns (one 16-byte fragment of each plane) per thread.  Rows
// of up to 256 x 8 x kHold columns are read once and held in registers.
// A row's fragments lie 512 bytes apart, 8 rows to a line: workgroups go to the
// XCDs in turn, so each XCD takes per_xcd consecutive rows (a multiple of 8) and a
// line is written in one L2.  2048 columns, 64 / 128 rows: 3.0 / 3.6 us, with the
// rows dealt out in turn 3.6 / 4.6 (a split without the row's maximum, coalesced
// over the rows, 2.8 / 3.1).
constexpr int kSplitThreads = 256;
constexpr int kHold = 4;
__global__ __launch_bounds__(kSplitThreads) void split_rows_kernel(const float *__restrict__ x, Planes xp, int n, int rows,
                                                                    int per_xcd) {
    __shared__ float red[kSplitThreads / kWave];
    const int b = ((int)blockIdx.x % kXcds) * per_xcd + (int)blockIdx.x / kXcds;
    if (b >= rows) return;
    const int t = threadIdx.x, vecs = n >> 3;
    const float4 *src = reinterpret_cast<const float4 *>(x + (size_t)b * n);
    float4 v[kHold][2];
    float amax = 0.0f;
    auto top = [](float4 a) { return fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))); };
    // (fmaxf drops a NaN: kept apart so that a row with one has no exponent)
    bool bad = false;
    auto see = [&](float4 a) {
        amax = fmaxf(amax, top(a));
        bad |= !(a.x == a.x && a.y == a.y && a.z == a.z && a.w == a.w);
    };
    // (past the row: zeros, without a memory access)
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(src), 0, 4 * n, kBufferWord3);
#pragma unroll
    for (int i = 0; i < kHold; i++)
#pragma unroll
        for (int k = 0; k < 2; k++)
            v[i][k] = __builtin_bit_cast(
                float4, __builtin_amdgcn_raw_buffer_load_b128(rs, 32 * (t + kSplitThreads * i) + 16 * k, 0, 0));
#pragma unroll
    for (int i = 0; i < kHold; i++) {
        see(v[i][0]);
        see(v[i][1]);
    }
    for (int c = t + kSplitThreads * kHold; c < vecs; c += kSplitThreads) {
        see(src[2 * c]);
        see(src[2 * c + 1]);
    }
    if (bad) amax = INFINITY;
    amax = wave_max64(amax);
    if ((t & (kWave - 1)) == 0) red[t / kWave] = amax;
    __syncthreads();
    const int E = group_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
    auto put = [&](int c, float4 a0, float4 a1) {
        const float f[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        h8v h, l;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            _Float16 hh, ll;
            split_scaled(f[e], E, hh, ll);
            h[e] = hh;
            l[e] = ll;
        }
        const size_t o = xf_index(b, 8 * c, n);
        *reinterpret_cast<h8v *>(xp.hi + o) = h;
        *reinterpret_cast<h8v *>(xp.lo + o) = l;
    };
#pragma unroll
    for (int i = 0; i < kHold; i++) {
        const int c = t + kSplitThreads * i;
        if (c < vecs) put(c, v[i][0], v[i][1]);
    }
    for (int c = t + kSplitThreads * kHold; c < vecs; c += kSplitThreads) put(c, src[2 * c], src[2 * c + 1]);
    for (int g = t; g < n / kXeGroup; g += kSplitThreads) xp.xe[xe_index(b, g * kXeGroup, n)] = (int8_t)E;
}

template <bool SILU>
int launch_chunk(anehip_ctx *ctx, hipStream_t stream, uint32_t ggml_type, const void *wp, uint32_t m, uint32_t n,
                 const Planes &xp, uint32_t rows, float *out, int ksplit) {
    const int nsb = (int)(n / 256), ptiles = (int)((m + kWave - 1) / kWave);
    if (rows <= 32 || ksplit < 1 || nsb % ksplit || m % 4 || !xp.hi || !xp.lo || !xp.xe || !xp.uniform)
        return set_error(ctx->err, ANEHIP_EINVAL, "gemm_rows: %u rows, K split %d of %d panels, m %u, %s planes", rows,
                         ksplit, nsb, m, xp.uniform ? "uniform" : "grouped");
    // (offsets are 64-bit; the FFN's rows, two sums to a value, may take twice
    // the 1 GiB of a plain product, so that a chunk of 960 rows takes any F that
    // one of 256 did)
    if ((SILU ? 1.0 : 4.0) * rows * m > 1073741824.0)
        return set_error(ctx->err, ANEHIP_ESHAPE, "gemm_rows: output of %u x %u floats too large", rows, m);
    // the weights are addressed with 32-bit buffer offsets
    if ((double)ptiles * nsb * Panel<ANEHIP_GGML_Q8_0>::kBytes > 2147483647.0)
        return set_error(ctx->err, ANEHIP_ESHAPE, "gemm_rows: %u x %u weights too large (2 GiB of panels at most)", m, n);
    const int nblocks = (ptiles + 3) / 4, rblocks = (int)((rows + kRowBlock - 1) / kRowBlock);
    const int total = nblocks * rblocks * ksplit;
    const dim3 grid((unsigned)((total + kXcds - 1) / kXcds * kXcds)), block(512);
    const uint8_t *w = static_cast<const uint8_t *>(wp);
    const size_t ss = (size_t)rows * m;
    if (ggml_type == ANEHIP_GGML_Q8_0)
        hipLaunchKernelGGL((gemm_chunk<ANEHIP_GGML_Q8_0, SILU>), grid, block, 0, stream, w, xp, out, (int)m, (int)n,
                           (int)rows, nblocks, rblocks, ksplit, ss);
    else
        hipLaunchKernelGGL((gemm_chunk<ANEHIP_GGML_Q4_0, SILU>), grid, block, 0, stream, w, xp, out, (int)m, (int)n,
                           (int)rows, nblocks, rblocks, ksplit, ss);
    ANEHIP_HIP_TRY(ctx->err, hipGetLastError());
    return ANEHIP_OK;
}

// K split of gemm_chunk: a divisor of the panel count (at most 16, the
// partial slices a consumer sums) minimising an estimate of the launch:
// rounds of workgroups (one per CU) at 3.5 us + 3.5 us per panel (measured:
// 31.4 us for 8 panels, 45-47 for 12), the traffic of the extra partial
// slices (written here, read by the consumer: 2 x 4 bytes per row and output
// at ~2 TB/s), and a launch that adds them.  Over 190 products of 1024..16384
// x 1024..8192 at 33-960 rows, every split timed, the one chosen costs 0.1 % more
// than the best on average and 5 % at most (5 TB/s and 3 us for the launch: 1.2 %
// and 16 %; 4096 x 2048 at 128 rows 8 splits 26.9 us, 4 24.2; 6144 x 1024 at 256
// 2 splits 26.9, 1 23.2).
int gemm_chunk_ksplit(const anehip_ctx *ctx, uint32_t m, uint32_t n, uint32_t rows) {
    const int nsb = (int)(n / 256), cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const int wgs = (int)((m + kTileRows - 1) / kTileRows) * (int)((rows + kRowBlock - 1) / kRowBlock);
    const double fixed_us = 3.5, panel_us = 3.5, sum_us = 4.0, part_us = 8.0 / 2.0e6 * (double)rows * m;
    int best = 1;
    double best_cost = -1.0;
    for (int k = 1; k <= nsb && k <= 16; k++) {
        if (nsb % k) continue;
        const double cost = (double)((wgs * k + cus - 1) / cus) * (fixed_us + (nsb / k) * panel_us) +
                            (k > 1 ? sum_us + (k - 1) * part_us : 0.0);
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best = k;
        }
    }
    return best;
}

}  // namespace

int launch_split_rows(anehip_ctx *ctx, hipStream_t stream, const float *x, uint32_t rows, uint32_t n, const Planes &xp) {
    if (n % kXeGroup || !xp.uniform)
        return set_error(ctx->err, ANEHIP_EINVAL, "split_rows: n=%u not a multiple of %d, or grouped planes", n, kXeGroup);
    const int per_xcd = (int)(rows + 8 * kXcds - 1) / (8 * kXcds) * 8;
    hipLaunchKernelGGL(split_rows_kernel, dim3(kXcds * per_xcd), dim3(kSplitThreads), 0, stream, x, xp, (int)n, (int)rows,
                       per_xcd);
    ANEHIP_HIP_TRY(ctx->err, hipGetLastError());
    return ANEHIP_OK;
}

int gemm_rows_ksplit(const anehip_ctx *ctx, uint32_t m, uint32_t n, uint32_t rows) {
    return rows <= 32 ? gemm_packed_ksplit(ctx, m, n, rows) : gemm_chunk_ksplit(ctx, m, n, rows);
}

int launch_gemm_rows(anehip_ctx *ctx, hipStream_t stream, uint32_t ggml_type, const void *wp, uint32_t m, uint32_t n,
                     const Planes &xp, uint32_t rows, float *out, int ksplit) {
    if (rows <= 32) return launch_gemm_packed(ctx, stream, ggml_type, wp, m, n, xp, rows, out, ksplit);
    return launch_chunk<false>(ctx, stream, ggml_type, wp, m, n, xp, rows, out, ksplit);
}

int launch_gemm_rows_silu(anehip_ctx *ctx, hipStream_t stream, uint32_t ggml_type, const void *wp, uint32_t m,
                          uint32_t n, const Planes &xp, uint32_t rows, float *h) {
    return launch_chunk<true>(ctx, stream, ggml_type, wp, m, n, xp, rows, h, 1);
}

}  // namespace anehip
