// attention.hip — GQA decode attention over an fp16 KV cache for gfx950.
//
// Replaces q_gate_split, rmsnorm_gated (q/k norm use), rope_apply, the KV
// append gpu_memcpys, sdpa_causal and sigmoid_gate (crates/engine/metal/
// attention.metal:9-121, deltanet.metal:184-220; dispatched at
// gpu_full_decode.rs:628-903) and the CPU core of full_attn_decode_step
// (crates/engine/src/deltanet.rs:565-669).
//
// Split-K ("flash-decoding"): the positions 0..pos of one sequence are cut
// into tiles of 64, and the live tiles are spread evenly over the launch's
// chunks (chunk_count(): at most 128 per sequence and kv head, about one
// workgroup per CU over the whole batch); one workgroup per (chunk, kv head,
// sequence) streams its tiles' K and V rows once for all G query heads that
// share the kv head (the next tile's loads in flight while the current one is
// used), with an online softmax, and writes an unnormalised partial output
// with its running max and sum.  attn_combine_kernel merges the chunks with a
// log-sum-exp rescale and applies sigmoid(gate).  Each workgroup derives its
// tile range from the device-resident position (chunk_tiles()), so the work
// follows the live length, not the cache's capacity, while one launch shape
// serves every position and can be captured in a graph; with fewer live
// tiles than chunks the chunks past the tile count exit at once.
//
// The KV cache keeps fp16 values (round-to-nearest-even) in the reference's
// per-sequence layout [kv_head][max_seq][head_dim] (kv_cache.rs:7-27).  The
// current position's k/v are rounded to fp16 before use, exactly as if they
// had been written to the cache and read back (the reference writes first,
// deltanet.rs:625, then reads every position).
#include "panel.h"

namespace anehip {

namespace {

constexpr int kHd = 256;       // head_dim
constexpr int kCh = 64;        // positions per workgroup
constexpr int kThreads = 256;

// RMSNorm (eps 1e-6, deltanet.rs:575-598) + RoPE (deltanet.rs:600-623) of one
// 256-dim head by one wave: lane l owns dims 4l..4l+3 = rotary pairs 2l, 2l+1.
// The same arithmetic as the decode kernel's preparation (rsqrt, one sincos
// per pair), so prefill and decode append identical k rows.
__device__ __forceinline__ void norm_rope_head(const MixIn &mix, int b, int base, const float *__restrict__ w,
                                               const float *__restrict__ inv_freq, uint32_t pos, int lane,
                                               float *dst) {
    float4 x = mix.at4(b, base + 4 * lane);
    float ss = wave_sum(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w);
    const float inv_rms = rsqrtf(ss / (float)kHd + 1e-6f);
    float4 wv = *reinterpret_cast<const float4 *>(w + 4 * lane);
    float a0 = (x.x * inv_rms) * wv.x, a1 = (x.y * inv_rms) * wv.y;
    float a2 = (x.z * inv_rms) * wv.z, a3 = (x.w * inv_rms) * wv.w;
    const float fpos = (float)pos;
    float s0, c0, s1, c1;
    sincosf(fpos * inv_freq[2 * lane], &s0, &c0);
    sincosf(fpos * inv_freq[2 * lane + 1], &s1, &c1);
    dst[0] = a0 * c0 - a1 * s0;
    dst[1] = a0 * s0 + a1 * c0;
    dst[2] = a2 * c1 - a3 * s1;
    dst[3] = a2 * s1 + a3 * c1;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kWord3 = 0x00020000;  // raw buffer resource word 3 (gfx9 family)
constexpr float kPScale = 16384.0f;  // 2^14: probabilities in the PV MFMA operands
// Cache-policy bit nt of the K / V cache loads, for launches whose caches
// (capacity) reach kNtKvBytes: each cached row is read once per step and the
// caches of a batch exceed the L2s and the MALL.  Measured on MI355X (caches
// rotated past the MALL): batch 32 ctx 1k / 8k / 32k 19.1 / 94-98 / 364-369
// -> 17.1 / 82.3 / 307.3 us, batch 1 ctx 32k 18.6 -> 17.4, batch 1 ctx 1k
// 6.8 -> 7.0; batch-1 decode ctx 1k / 8k / 32k with the bit on every launch
// 1248 / 1241 / 1166 tok/s against 1254 / 1245 / 1130 with it on none.
constexpr int kCpolNt = 2;
constexpr size_t kNtKvBytes = (size_t)32 << 20;

// Sharing of the launch's workgroups over sequences of different lengths (2
// to 64 of them): every chunk gets at most `s` tiles, s the smallest (to 3 %)
// for which the chunks of all sequences and kv heads fit the W workgroups, so
// that a long sequence gets more of them than a short one.  (Chunks per
// sequence fixed by the batch alone, the longest sequence's set the time:
// batch 32, 2 kv heads, lengths spread over 2k-8k: 77 us a step against 65.)
// Lane b of each wave holds sequence b's chunks per kv head (n) and its first
// workgroup (start): kv head k's chunk c is workgroup start + k n + c.  Where
// that takes no tile off the longest chunk the fixed split stands (even): two
// sequences of 24.5k and 24.2k positions, 4 kv heads, 41.1 us a step with the
// plan all the same, 39.7 without, 39.0 by kernels that have none.
struct AttnPlan {
    int pos, tiles, n, start;
    bool even;
};
constexpr int kMaxPlanBatch = 64;
constexpr int kPlanTiles = 8;
// inclusive sum over the lanes of the wave up to this one
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31 into rows 2, 3
    return v;
}
// pos: plan_pos(), loaded by the caller ahead of its other loads (vector loads
// complete in order: behind them, the plan would wait for all of them).
__device__ __forceinline__ uint32_t plan_pos(const uint32_t *__restrict__ pos_arr, int batch) {
    return pos_arr[min((int)threadIdx.x & 63, batch - 1)];
}
__device__ __forceinline__ AttnPlan attn_plan(uint32_t pos, int batch, int n_kv, int nch, int max_tiles) {
    const int lane = threadIdx.x & 63, W = batch * n_kv * nch;
    AttnPlan P;
    P.pos = (int)pos;
    P.tiles = min(P.pos / kCh + 1, max_tiles);
    P.even = __ballot(P.tiles != __builtin_amdgcn_readfirstlane(P.tiles)) == 0;
    P.n = P.start = 0;
    if (P.even) return P;
    if (lane >= batch) P.tiles = 0;
    const int total = __builtin_amdgcn_readlane(wave_scan(P.tiles), 63) * n_kv;
    int s = (total + W - 1) / W;
    P.even = __ballot(P.tiles > s * nch) == 0;
    if (P.even) return P;
    // ends at s = max_tiles at the latest: one chunk each, and batch x n_kv <= W
    for (;; s += 1 + s / 32) {
        P.n = (P.tiles + s - 1) / s;
        const int end = wave_scan(P.n * n_kv);
        P.start = end - P.n * n_kv;
        if (__builtin_amdgcn_readlane(end, 63) <= W || s >= max_tiles) return P;
    }
}

// grid = (chunks, n_kv_heads, batch); chunk c takes the live tiles
// [tb, te) of 64 positions that chunk_tiles() gives it.  mix: per
// sequence [q_full | k | v] rows (K-split partial slices); q_full is
// [n_heads][q(256) | gate(256)].
//
// Wave w takes positions 16 w .. 16 w + 15 of every tile and keeps its own
// online softmax and output for them; the 4 waves merge once, at the end.
// Per tile and wave, on MFMA (16 x 16 x K f16 forms: operands A[i][k] /
// B[k][j] in lane i (j) + 16 (k / (K / 4)), elements k % (K / 4); D[i][j]
// in lane j + 16 (i / 4), element i % 4):
//  * scores S[pos][head] = K q^T / 16 (K = 32): A = the wave's 16 K rows,
//    loaded straight from the cache (lane l: row l % 16, dims 32 s + 8 (l /
//    16) of k-step s), B = q as fp16 hi + lo fragments (columns = the G
//    query heads, others zero), so K is read once for all G heads;
//  * lane l then holds the scores of head l % 16 at positions 4 (l / 16) ..
//    + 3: the max and sum over the wave's 16 positions are two lane swaps
//    (v_permlane16_swap / v_permlane32_swap), no LDS and no barrier;
//  * O[head][dim] += P V (K = 16): those probabilities (x 2^14, fp16 hi +
//    lo) are already the A operand; B = V rows 4 (l / 16) .. + 3 of the
//    wave, loaded as 8-byte pieces (dims 64 q + 4 (l % 16) .. + 3), and MFMA
//    (q, c) takes element c of each piece, so its output column l % 16 is
//    dim 64 q + 4 (l % 16) + c: 16 MFMA column blocks cover the 256 dims
//    with no transpose of V.
// The next tile's K / V loads are in flight while a tile is processed; the
// buffer resources cover positions [0, pos) only, so rows >= pos read zeros
// without a memory access (row pos takes this step's k / v), which also makes
// the prefetch of a tile past the chunk free.  One unnormalised partial per
// (chunk, query head) with its running max and sum.
//
// With one or two tiles per workgroup (batch 1 at short contexts) the kernel
// is a chain of dependent steps on one wave per SIMD, so the q / k
// preparation issues every input load before the position is known, shares
// one sincos per rotary pair and writes the q fragments straight from the
// wave that normalised the head.
//
// PLAN: where the sequences' lengths differ, the launch's W workgroups (their
// linear index) are shared out by attn_plan(); partials in workgroup order.
//
// Cache addressing: row b's cache is at cache_off + b * row_stride halves
// (decode: every row its own sequence; prefill: row_stride 0, every row a
// token of one sequence whose K / V rows the prefill append kernel wrote
// before this launch -- then `append` is false and no row is written here).
template <int G, bool NT, bool PLAN>
__global__ __launch_bounds__(kThreads) void attn_partial_kernel(
    MixIn mix, const float *__restrict__ q_norm, const float *__restrict__ k_norm,
    const float *__restrict__ inv_freq, const uint32_t *__restrict__ pos_arr, __half *__restrict__ k_cache,
    __half *__restrict__ v_cache, int max_seq, int n_heads, int n_kv, float *__restrict__ part_o,
    float *__restrict__ part_ml, size_t cache_off, size_t row_stride, bool append, int batch) {
    __shared__ __align__(16) h8v qf[8][2][64];
    __shared__ __align__(16) __half knew[kHd], vnew[kHd];
    __shared__ int qexp[G];
    __shared__ __align__(16) float ob[4][G][kHd];
    __shared__ float wm[4][G], wl[4][G];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int li = lane & 15, lg = lane >> 4;
    int c = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const int nch = gridDim.x, slot0 = (b * n_kv + kvh) * nch + c;
    // inputs that do not depend on the position first: this wave's q head
    // (wave < G) or k / v rows (wave G % 4, used by the chunk holding pos),
    // the norm weights and the RoPE frequencies
    const bool is_q = wave < G, is_k = wave == G % 4;
    int hq, kin, vin;
    uint32_t lane_pos = 0;
    if constexpr (PLAN) lane_pos = plan_pos(pos_arr, batch);
    float4 aq[8], ak[8], av[8];
    auto load_inputs = [&]() {
        hq = kvh * G + (wave < G ? wave : 0);
        kin = n_heads * 2 * kHd + kvh * kHd;
        vin = n_heads * 2 * kHd + n_kv * kHd + kvh * kHd;
        const float *r0 = mix.p + (size_t)b * mix.stride + 4 * lane;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (q < mix.kp) {
                const float *rq = r0 + (size_t)q * mix.split;
                if (is_q) aq[q] = *reinterpret_cast<const float4 *>(rq + hq * 2 * kHd);
                if (is_k) {
                    ak[q] = *reinterpret_cast<const float4 *>(rq + kin);
                    av[q] = *reinterpret_cast<const float4 *>(rq + vin);
                }
            }
    };
    load_inputs();
    const float4 wq = *reinterpret_cast<const float4 *>(q_norm + 4 * lane);
    const float4 wk = *reinterpret_cast<const float4 *>(k_norm + 4 * lane);
    const float2 fr = *reinterpret_cast<const float2 *>(inv_freq + 2 * lane);
    uint32_t pos;
    int tb = 0, te = 0;  // tiles [tb, te)
    bool shared_out = false;
    if constexpr (PLAN) {
        const AttnPlan P = attn_plan(lane_pos, batch, n_kv, nch, (max_seq + kCh - 1) / kCh);
        if (!P.even) {
            shared_out = true;
            b = 63 - __builtin_clzll(__ballot(P.start <= slot0 && lane < batch));
            const int n = __builtin_amdgcn_readlane(P.n, b), r = slot0 - __builtin_amdgcn_readlane(P.start, b);
            const int tiles = __builtin_amdgcn_readlane(P.tiles, b);
            kvh = r / n;
            c = r % n;
            if (kvh >= n_kv) return;  // uniform exit: past the last chunk
            load_inputs();
            // 32-bit: c < 256 and tiles < 2^15 (a cache row is below 1 GiB)
            tb = (int)((uint32_t)(c * tiles) / (uint32_t)n);
            te = (int)((uint32_t)((c + 1) * tiles) / (uint32_t)n);
        }
        pos = (uint32_t)__builtin_amdgcn_readlane(P.pos, b);
    } else {
        pos = pos_arr[b];
    }
    const int len = (int)pos + 1;
    if (!shared_out && !chunk_tiles(len, nch, c, &tb, &te)) return;  // uniform exit: nothing of this sequence here
    const size_t cache_base = cache_off + (size_t)b * row_stride + (size_t)kvh * max_seq * kHd;
    const bool has_new = (int)pos < te * kCh;
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc(k_cache + cache_base, 0, (int)pos * kHd * 2, kWord3);
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc(v_cache + cache_base, 0, (int)pos * kHd * 2, kWord3);
    const int kFar = max_seq;
    auto load_k = [&](u32x4 *kr, int row0) {
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int off = ((row0 + 16 * wave + li) * kHd + 32 * s + 8 * lg) * 2;
            kr[s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, off, 0, NT ? kCpolNt : 0));
        }
    };
    // V rows row0 + 16 wave + 4 lg + r, dims 64 q + 4 li .. + 3 in vr[4 q + r]
    auto load_v = [&](u32x2 *vr, int row0) {
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int off = ((row0 + 16 * wave + 4 * lg + r) * kHd + 64 * q + 4 * li) * 2;
                vr[4 * q + r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vrs, off, 0, NT ? kCpolNt : 0));
            }
    };
    auto row_of = [&](int ti) { return ti < te ? ti * kCh : kFar; };
    u32x4 ka[8], kb[8];
    u32x2 va[16], vb[16];
    load_k(ka, tb * kCh);
    load_v(va, tb * kCh);
    load_k(kb, row_of(tb + 1));
    load_v(vb, row_of(tb + 1));

    // preparation, every input load issued first: wave w < G normalises and
    // rotates q head kvh G + w and writes its MFMA B fragments (scaled by
    // 1/16 and 2^-qe, fp16 hi + lo); in the chunk holding pos, wave G % 4
    // also prepares this step's k (RMSNorm + RoPE) and v, rounded to fp16.
    const bool do_q = is_q, do_k = has_new && is_k;
    // rows of the q fragments that belong to no head are zero
    for (int e = t; e < 8 * 64; e += kThreads) {
        const int fl = e & 63;
        if ((fl & 15) >= G) {
            qf[e >> 6][0][fl] = h8v{};
            qf[e >> 6][1][fl] = h8v{};
        }
    }
    float sn0, cs0, sn1, cs1;
    sincosf((float)pos * fr.x, &sn0, &cs0);
    sincosf((float)pos * fr.y, &sn1, &cs1);
    // slices in ascending order; the GEMMs at batch > 1 split K up to 16
    // ways, slices past the 8 held in registers are loaded here
    auto sum4 = [&](const float4 *a, int off) {
        float4 x = a[0];
#pragma unroll
        for (int q = 1; q < 8; q++)
            if (q < mix.kp) x = make_float4(x.x + a[q].x, x.y + a[q].y, x.z + a[q].z, x.w + a[q].w);
        for (int q = 8; q < mix.kp; q++) {
            const float4 v = *reinterpret_cast<const float4 *>(
                mix.p + (size_t)b * mix.stride + 4 * lane + (size_t)q * mix.split + off);
            x = make_float4(x.x + v.x, x.y + v.y, x.z + v.z, x.w + v.w);
        }
        return x;
    };
    auto norm_rope = [&](float4 x, float4 wv, float *dst) {
        const float ss = wave_sum(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w);
        const float inv_rms = rsqrtf(ss / (float)kHd + 1e-6f);
        const float a0 = (x.x * inv_rms) * wv.x, a1 = (x.y * inv_rms) * wv.y;
        const float a2 = (x.z * inv_rms) * wv.z, a3 = (x.w * inv_rms) * wv.w;
        dst[0] = a0 * cs0 - a1 * sn0;
        dst[1] = a0 * sn0 + a1 * cs0;
        dst[2] = a2 * cs1 - a3 * sn1;
        dst[3] = a2 * sn1 + a3 * cs1;
    };
    if (do_q) {
        float q4[4];
        norm_rope(sum4(aq, hq * 2 * kHd), wq, q4);
        const float qm = wave_max64(fmaxf(fmaxf(fabsf(q4[0]), fabsf(q4[1])), fmaxf(fabsf(q4[2]), fabsf(q4[3]))));
        const int qe = group_exp(qm * 0.0625f);
        if (lane == 0) qexp[wave] = qe;
        // dims 4 lane .. + 3 = k-step lane / 8, lane group (lane % 8) / 2, half lane % 2
        h4v hi, lo;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float x = ldexpf(q4[i] * 0.0625f, -qe);
            hi[i] = (_Float16)x;
            lo[i] = (_Float16)(x - (float)hi[i]);
        }
        const int fs = lane >> 3, fl = wave + 16 * ((lane & 7) >> 1), half = lane & 1;
        reinterpret_cast<h4v *>(&qf[fs][0][fl])[half] = hi;
        reinterpret_cast<h4v *>(&qf[fs][1][fl])[half] = lo;
    }
    if (do_k) {
        float k4[4];
        norm_rope(sum4(ak, kin), wk, k4);
        const float4 v4 = sum4(av, vin);
        const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            knew[4 * lane + i] = __float2half_rn(k4[i]);
            vnew[4 * lane + i] = __float2half_rn(vv[i]);
        }
        if (append) {
            __half *kd = k_cache + cache_base + (size_t)pos * kHd + 4 * lane;
            __half *vd = v_cache + cache_base + (size_t)pos * kHd + 4 * lane;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                kd[i] = knew[4 * lane + i];
                vd[i] = vnew[4 * lane + i];
            }
        }
    }
    lds_barrier();
    const int qe_li = li < G ? qexp[li] : 0;

    float m_run = -INFINITY, l_run = 0.f;
    f32x4 o[16] = {};
    auto process = [&](u32x4 *kr, u32x2 *vr, int ti, bool first) {
        const int row0 = ti * kCh;
        if (row0 + 16 * wave + li == (int)pos) {
#pragma unroll
            for (int s = 0; s < 8; s++) kr[s] = *reinterpret_cast<const u32x4 *>(&knew[32 * s + 8 * lg]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (row0 + 16 * wave + 4 * lg + r == (int)pos) {
#pragma unroll
                for (int q = 0; q < 4; q++) vr[4 * q + r] = *reinterpret_cast<const u32x2 *>(&vnew[64 * q + 4 * li]);
            }
        f32x4 s0 = {}, s1 = {};
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const h8v a = __builtin_bit_cast(h8v, kr[s]);
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[s][0][lane], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[s][1][lane], s1, 0, 0, 0);
        }
        load_k(kr, row_of(ti + 2));
        const int p0 = row0 + 16 * wave + 4 * lg;
        float sv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) sv[e] = p0 + e < len ? ldexpf(s0[e] + s1[e], qe_li) : -INFINITY;
        const float tm = lanes_max4(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));
        const float mn = fmaxf(m_run, tm);
        const float mref = mn == -INFINITY ? 0.0f : mn;
        const float scale = expf(m_run - mref);
        float pe[4], ps = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            pe[e] = (li < G && p0 + e < len) ? expf(sv[e] - mref) : 0.0f;
            ps += pe[e];
        }
        l_run = l_run * scale + lanes_sum4(ps);
        m_run = mn;
        float rs[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            rs[e] = e < G ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, scale), e)) : 0.0f;
        if (!first) {
#pragma unroll
            for (int k = 0; k < 16; k++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[k][e] *= rs[e];
        }
        h4v ph, pl;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float x = pe[e] * kPScale;
            ph[e] = (_Float16)x;
            pl[e] = (_Float16)(x - (float)ph[e]);
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int cc = 0; cc < 4; cc++) {
                const int w = cc >> 1;
                const uint32_t x0 = vr[4 * q][w], x1 = vr[4 * q + 1][w], x2 = vr[4 * q + 2][w], x3 = vr[4 * q + 3][w];
                u32x2 bw;
                if (cc & 1) {
                    bw[0] = (x0 >> 16) | (x1 & 0xffff0000u);
                    bw[1] = (x2 >> 16) | (x3 & 0xffff0000u);
                } else {
                    bw[0] = (x0 & 0xffffu) | (x1 << 16);
                    bw[1] = (x2 & 0xffffu) | (x3 << 16);
                }
                const h4v bv = __builtin_bit_cast(h4v, bw);
                o[4 * q + cc] = __builtin_amdgcn_mfma_f32_16x16x16f16(ph, bv, o[4 * q + cc], 0, 0, 0);
                o[4 * q + cc] = __builtin_amdgcn_mfma_f32_16x16x16f16(pl, bv, o[4 * q + cc], 0, 0, 0);
            }
        load_v(vr, row_of(ti + 2));
    };
    process(ka, va, tb, true);
    int ti = tb + 1;
    while (ti + 1 < te) {
        process(kb, vb, ti, false);
        process(ka, va, ti + 1, false);
        ti += 2;
    }
    if (ti < te) process(kb, vb, ti, false);
    // merge the 4 waves: lanes 0-15 hold heads e < G, dims 64 q + 4 li + cc
    if (lane < G) {
        wm[wave][lane] = m_run;
        wl[wave][lane] = l_run;
    }
    if (lg == 0) {
#pragma unroll
        for (int e = 0; e < G; e++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<float4 *>(&ob[wave][e][64 * q + 4 * li]) =
                    make_float4(o[4 * q][e], o[4 * q + 1][e], o[4 * q + 2][e], o[4 * q + 3][e]);
    }
    lds_barrier();
    for (int idx = t; idx < G * 64; idx += kThreads) {
        const int hh = idx >> 6, d4 = idx & 63;
        float M = wm[0][hh];
#pragma unroll
        for (int w = 1; w < 4; w++) M = fmaxf(M, wm[w][hh]);
        float L = 0.f;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float sw = expf(wm[w][hh] - M);
            const float4 v = *reinterpret_cast<const float4 *>(&ob[w][hh][4 * d4]);
            L += sw * wl[w][hh];
            acc = make_float4(acc.x + sw * v.x, acc.y + sw * v.y, acc.z + sw * v.z, acc.w + sw * v.w);
        }
        const size_t slot = (size_t)slot0 * G + hh;
        const float inv = 1.0f / kPScale;
        *reinterpret_cast<float4 *>(part_o + slot * kHd + 4 * d4) =
            make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
        if (d4 == 0) {
            part_ml[slot * 2] = M;
            part_ml[slot * 2 + 1] = L;
        }
    }
}

// Prefill: the k / v rows of T consecutive tokens of one sequence (row t at
// position pos_arr[t]) -- RMSNorm + RoPE of k, both rounded to fp16 -- written
// to the cache at cache_off, as the decode kernel appends one row.  odd (when
// not null): [n_kv][T], 1 where the row's v holds an infinity or NaN (fp16
// overflows from 65520), 0 else.  grid = (n_kv, T), one wave.
__global__ __launch_bounds__(64) void attn_append_kernel(MixIn mix, const float *__restrict__ k_norm,
                                                         const float *__restrict__ inv_freq,
                                                         const uint32_t *__restrict__ pos_arr,
                                                         __half *__restrict__ k_cache, __half *__restrict__ v_cache,
                                                         size_t cache_off, int max_seq, int n_heads, int n_kv,
                                                         uint32_t *__restrict__ odd) {
    const int lane = threadIdx.x, kvh = blockIdx.x, b = blockIdx.y;
    const uint32_t pos = pos_arr[b];
    const int kin = n_heads * 2 * kHd + kvh * kHd;
    const int vin = n_heads * 2 * kHd + n_kv * kHd + kvh * kHd;
    float k4[4];
    norm_rope_head(mix, b, kin, k_norm, inv_freq, pos, lane, k4);
    const float4 v4 = mix.at4(b, vin + 4 * lane);
    const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
    const size_t o = cache_off + ((size_t)kvh * max_seq + pos) * kHd + 4 * lane;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const __half v = __float2half_rn(vv[i]);
        k_cache[o + i] = __float2half_rn(k4[i]);
        v_cache[o + i] = v;
        bad |= (__half_as_ushort(v) & 0x7c00) == 0x7c00;
    }
    if (odd) {
        const bool any = __ballot(bad) != 0;
        if (lane == 0) odd[(size_t)kvh * gridDim.y + b] = any;
    }
}

// grid = (n_heads, batch), 64 GR threads: thread (g = t / 64, l = t % 64) takes
// dims 4l..4l+3 of chunks g, g + GR, g + 2 GR, ...; merges them with a
// log-sum-exp rescale against the maximum over all chunks, adds the GR groups
// through LDS, normalises and multiplies by sigmoid(gate) (deltanet.rs:667-669).
// GR = 16 where a head has more than kManyChunks chunks, 8 above kSomeChunks (up
// to 8 per group, all loaded at once; with 4 groups of 32 chunks one after the
// other batch 1 at 32k positions took 14.6 us; a step there 30.6 -> 22.5), 4
// else: every 16 chunks past the first 16 cost those ~1.5 us, a workgroup of 16
// groups ~3 (20 chunks of 2 sequences 6.8 us traced, against 4.0).  Steps of 2
// sequences, 4 heads on 2 kv heads, capacity 3300 (52 chunks), 4 / 8 / 16 groups:
// 1.2k and 2.3k positions 11.1 / 10.8 / 11.9 us, 1.8k and 3.0k 11.7 / 10.7 / 12.0.
constexpr int kSomeChunks = 32, kManyChunks = 64;
constexpr int kMaxChunks = 128;  // the most chunk_count() gives; a plan may give a head more
// out: [batch][n_heads * 256] fp32, or range-safe fragment-order planes xp
// (Planes) when xp.hi is not null.  PLAN: the partials of a launch whose
// workgroups attn_plan() may have shared out.
template <int G, int GR, bool PLAN>
__global__ __launch_bounds__(64 * GR) void attn_combine_kernel(MixIn mix, const uint32_t *__restrict__ pos_arr,
                                                               const float *__restrict__ part_o,
                                                               const float *__restrict__ part_ml, int nch,
                                                               int n_heads, int n_kv, float *__restrict__ out,
                                                               Planes xp, int max_seq) {
    constexpr int PRE = GR >= 8 ? 8 : 4;  // chunks of a group loaded before the maximum is known
    constexpr bool MORE = PLAN || GR * PRE < kMaxChunks;
    __shared__ float red[GR];
    __shared__ float4 accs[GR][64];
    __shared__ float dens[GR][64];
    const int t = threadIdx.x, g = t >> 6, l = t & 63, h = blockIdx.x, b = blockIdx.y;
    const int kvh = h / G, hh = h % G;
    // the gate's K-split slices (independent of the partials) and this
    // group's first PRE chunks are loaded together, before the maximum is known
    float4 gq[8];
    uint32_t lane_pos = 0;
    int nc;
    size_t base = ((size_t)b * n_kv + kvh) * nch;
    if constexpr (PLAN) lane_pos = plan_pos(pos_arr, (int)gridDim.y);
    else nc = active_chunks((int)pos_arr[b] + 1, nch);
    {
        const float *g0 = mix.p + (size_t)b * mix.stride + h * 2 * kHd + kHd + 4 * l;
#pragma unroll
        for (int q = 0; q < 8; q++) gq[q] = *reinterpret_cast<const float4 *>(g0 + (size_t)min(q, mix.kp - 1) * mix.split);
    }
    if constexpr (PLAN) {
        const AttnPlan P = attn_plan(lane_pos, (int)gridDim.y, n_kv, nch, (max_seq + kCh - 1) / kCh);
        if (P.even) {
            nc = active_chunks(__builtin_amdgcn_readlane(P.pos, b) + 1, nch);
        } else {
            nc = __builtin_amdgcn_readlane(P.n, b);
            base = (size_t)(__builtin_amdgcn_readlane(P.start, b) + kvh * nc);
        }
    }
    float4 p4[PRE];
    float pm[PRE], pl[PRE];
#pragma unroll
    for (int i = 0; i < PRE; i++) {
        const size_t slot = (base + min(g + GR * i, nc - 1)) * G + hh;
        p4[i] = *reinterpret_cast<const float4 *>(part_o + slot * kHd + 4 * l);
        pm[i] = part_ml[slot * 2];
        pl[i] = part_ml[slot * 2 + 1];
    }
    float4 gate = gq[0];
#pragma unroll
    for (int q = 1; q < 8; q++)
        if (q < mix.kp) gate = make_float4(gate.x + gq[q].x, gate.y + gq[q].y, gate.z + gq[q].z, gate.w + gq[q].w);
    for (int q = 8; q < mix.kp; q++) {
        const float4 v = *reinterpret_cast<const float4 *>(mix.p + (size_t)b * mix.stride + h * 2 * kHd + kHd + 4 * l +
                                                           (size_t)q * mix.split);
        gate = make_float4(gate.x + v.x, gate.y + v.y, gate.z + v.z, gate.w + v.w);
    }
    // maximum over the chunks: each group's (the same in all its lanes), then
    // over the groups
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PRE; i++) mx = g + GR * i < nc ? fmaxf(mx, pm[i]) : mx;
    for (int c2 = g + GR * PRE; MORE && c2 < nc; c2 += GR) mx = fmaxf(mx, part_ml[((base + c2) * G + hh) * 2]);
    if (l == 0) red[g] = mx;
    __syncthreads();
    float M = red[0];
#pragma unroll
    for (int k = 1; k < GR; k++) M = fmaxf(M, red[k]);
    // this group's chunks in order: those loaded above, then 4 per trip with
    // their loads issued together (selects, not branches, on what is past the
    // last chunk: the compiler moves a load into the branch that uses it)
    float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < PRE; i++) {
        if (g + GR * i < nc) {
            const float w = expf(pm[i] - M);
            num = make_float4(num.x + w * p4[i].x, num.y + w * p4[i].y, num.z + w * p4[i].z, num.w + w * p4[i].w);
            den += w * pl[i];
        }
    }
    for (int cc = g + GR * PRE; MORE && cc < nc; cc += 4 * GR) {
        float4 o4[4];
        float m4[4], l4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t slot = (base + min(cc + GR * i, nc - 1)) * G + hh;
            o4[i] = *reinterpret_cast<const float4 *>(part_o + slot * kHd + 4 * l);
            m4[i] = part_ml[slot * 2];
            l4[i] = part_ml[slot * 2 + 1];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool in = cc + GR * i < nc;
            const float w = expf(m4[i] - M);
            num = make_float4(num.x + (in ? w * o4[i].x : 0.0f), num.y + (in ? w * o4[i].y : 0.0f),
                              num.z + (in ? w * o4[i].z : 0.0f), num.w + (in ? w * o4[i].w : 0.0f));
            den += in ? w * l4[i] : 0.0f;
        }
    }
    accs[g][l] = num;
    dens[g][l] = den;
    __syncthreads();
    if (g != 0) return;
    float4 s = accs[0][l];
    float dsum = dens[0][l];
#pragma unroll
    for (int k = 1; k < GR; k++) {
        const float4 o = accs[k][l];
        s = make_float4(s.x + o.x, s.y + o.y, s.z + o.z, s.w + o.w);
        dsum += dens[k][l];
    }
    const float gv[4] = {gate.x, gate.y, gate.z, gate.w};
    const float sv[4] = {s.x, s.y, s.z, s.w};
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = (sv[i] / dsum) * (1.0f / (1.0f + expf(-gv[i])));
    if (xp.hi) {
        // the head is two 128-column groups: lanes 0-31 and 32-63
        const int e = group_exp(half_max32(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])))));
        h4v vh, vl;  // 4 consecutive columns of a fragment-order plane
        split4_scaled(v, e, vh, vl);
        const size_t o = xf_index(b, h * kHd + 4 * l, n_heads * kHd);
        *reinterpret_cast<h4v *>(xp.hi + o) = vh;
        *reinterpret_cast<h4v *>(xp.lo + o) = vl;
        if ((l & 31) == 0) xp.xe[xe_index(b, h * kHd + 4 * l, n_heads * kHd)] = (int8_t)e;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) out[(size_t)b * n_heads * kHd + (size_t)h * kHd + 4 * l + i] = v[i];
    }
}

// Prefill: T consecutive tokens of one sequence (row t at position pos_arr[t],
// its K / V row already appended) against the cache.  A workgroup takes 32
// query rows of one kv head -- 32 / G tokens x the G query heads -- so that the
// K / V rows they share are read once for all of them; its 4 waves take every
// fourth tile of 32 positions, each with an online softmax of its own, and
// merge at the end.  On v_mfma_f32_32x32x16_f16 (operands A[i][k] / B[k][j] in
// lane i (j) + 32 (k / 8), elements k % 8; D[i][j] in lane j + 32 (i / 4 % 2),
// element 4 (i / 8) + i % 4), the query row always the lane's column:
//  * scores S[pos][row] = K q^T / 16: A = 32 K rows straight from the cache, B =
//    q as range-scaled fp16 hi + lo from LDS;
//  * O[dim][row] += V^T P^T: the lane's 16 scores of a tile are two steps' B
//    operand as they are (x 2^14, fp16 hi + lo) if step u's k slot (h, j) means
//    position 16 u + 8 (j / 4) + 4 h + j % 4; A = V rows loaded as 8-byte pieces
//    (dims 128 q + 4 i .. + 3), MFMA (q, c) taking element c of the 8 rows' pieces,
//    so that its row i is dim 128 q + 4 i + c.
// K and V of the wave's next tile are in flight while a tile is processed
// (sums 128, K 64 and V 64 registers: one wave per SIMD; q beside them spilled).
//
// The decode kernel with one row per workgroup read every position's K / V
// once per row and ran 4 of 16 MFMA columns: 130 us at 960 rows of 8 heads from
// position 0 and 158 at 540 from 960 on, plus 17 for its merge; here 39 and 51,
// 64 MFMAs of 32 cycles per wave and tile, the rest the softmax between the two
// products, which one wave per SIMD doesn't hide.
// A row's masked scores weigh 0, and the V rows of later tokens of its group
// enter the product with that 0, so that an infinity or NaN among them would
// make this row NaN, and not only the rows from that token on (the earlier
// tokens' K / V rows in the layers after outlive it where the sequence is
// rewound).  A group with such a row (odd, of attn_append_kernel) goes token by
// token: no tile then holds a V row that its query rows don't see.
constexpr int kQRows = 32;    // query rows per workgroup
constexpr int kPTile = 32;    // positions per tile
constexpr int kMergeF = 66;   // LDS row of the merge: reads along the dims hit all banks

// Tokens t0 .. T - 1 (at most 32 / G) of kv head kvh; row t is at position p0 + t.
// False, with nothing written, where a lane's bad is not 0 (looked at once the
// first tiles' loads are on their way).
template <int G>
__device__ __forceinline__ bool prefill_tokens(MixIn mix, const float *__restrict__ q_norm,
                                               const float *__restrict__ inv_freq,
                                               int p0, const __half *__restrict__ k_cache,
                                               const __half *__restrict__ v_cache, size_t cache_off, int max_seq,
                                               int n_heads, int kvh, int t0, int T, uint32_t bad,
                                               float *__restrict__ out) {
    __shared__ __align__(16) h8v qs[16 * 2 * 64];             // q fragments [k-step][hi, lo][lane]
    __shared__ __align__(16) float lds[4 * 4 * 16 * kMergeF];  // the merge's [wave][c][element][lane]
    __shared__ int qexp[kQRows];
    __shared__ float wm[4][kQRows], wl[4][kQRows];
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));  // not invariant in the kernel's loop: what it gives would be held in registers and spill
    const int lane = t & 63, col = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t base = cache_off + (size_t)kvh * max_seq * kHd;
    const int last = p0 + T - 1, plim = p0 + min(t0 + col / G, T - 1);
    const int tiles = last / kPTile + 1;
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(k_cache) + base, 0, (last + 1) * kHd * 2, kWord3);
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(v_cache) + base, 0, (last + 1) * kHd * 2, kWord3);
    u32x4 kr[16];
    u32x2 vr[2][2][8];  // [step][q][slot]
    // positions past `last` read zeros without a memory access
    auto load_k = [&](int ti) {
#pragma unroll
        for (int s = 0; s < 16; s++)
            kr[s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  krs, ((ti * kPTile + col) * kHd + 16 * s + 8 * h) * 2, 0, 0));
    };
    auto load_v = [&](int ti) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int q = 0; q < 2; q++)
                    vr[u][q][j] = __builtin_bit_cast(
                        u32x2, __builtin_amdgcn_raw_buffer_load_b64(
                                   vrs, ((ti * kPTile + 16 * u + 8 * (j >> 2) + 4 * h + (j & 3)) * kHd + 128 * q + 4 * col) * 2,
                                   0, 0));
    };
    load_k(wave);
    load_v(wave);
    // wave w normalises and rotates query rows 8 w .. + 7 (every row's loads
    // first, one sincos per rotary pair and token) and writes their B
    // fragments (scaled by 1/16 and 2^-qe, fp16 hi + lo)
    constexpr int QR = kQRows / 4;
    float4 xq[QR];
    auto row_in = [&](int i) {
        const int r = QR * wave + i, tok = min(t0 + r / G, T - 1);
        return mix.p + (size_t)tok * mix.stride + (kvh * G + r % G) * 2 * kHd + 4 * lane;
    };
#pragma unroll
    for (int i = 0; i < QR; i++) xq[i] = *reinterpret_cast<const float4 *>(row_in(i));
    for (int q = 1; q < mix.kp; q++)
#pragma unroll
        for (int i = 0; i < QR; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(row_in(i) + (size_t)q * mix.split);
            xq[i] = make_float4(xq[i].x + v.x, xq[i].y + v.y, xq[i].z + v.z, xq[i].w + v.w);
        }
    const float4 wv = *reinterpret_cast<const float4 *>(q_norm + 4 * lane);
    const float2 fr = *reinterpret_cast<const float2 *>(inv_freq + 2 * lane);
    float sn0 = 0.0f, cs0 = 0.0f, sn1 = 0.0f, cs1 = 0.0f;
#pragma unroll
    for (int i = 0; i < QR; i++) {
        const int r = QR * wave + i;
        if (i % G == 0) {
            const float fpos = (float)(p0 + min(t0 + r / G, T - 1));
            sincosf(fpos * fr.x, &sn0, &cs0);
            sincosf(fpos * fr.y, &sn1, &cs1);
        }
        // norm_rope_head's arithmetic
        const float4 x4 = xq[i];
        const float inv_rms =
            rsqrtf(wave_sum(x4.x * x4.x + x4.y * x4.y + x4.z * x4.z + x4.w * x4.w) / (float)kHd + 1e-6f);
        const float a0 = (x4.x * inv_rms) * wv.x, a1 = (x4.y * inv_rms) * wv.y;
        const float a2 = (x4.z * inv_rms) * wv.z, a3 = (x4.w * inv_rms) * wv.w;
        const float q4[4] = {a0 * cs0 - a1 * sn0, a0 * sn0 + a1 * cs0, a2 * cs1 - a3 * sn1, a2 * sn1 + a3 * cs1};
        const float qm = wave_max64(fmaxf(fmaxf(fabsf(q4[0]), fabsf(q4[1])), fmaxf(fabsf(q4[2]), fabsf(q4[3]))));
        const int qe = group_exp(qm * 0.0625f);
        if (lane == 0) qexp[r] = qe;
        h4v hi, lo;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float x = ldexpf(q4[c] * 0.0625f, -qe);
            hi[c] = (_Float16)x;
            lo[c] = (_Float16)(x - (float)hi[c]);
        }
        // dims 4 lane .. + 3: k-step lane / 4, lane group (lane % 4) / 2, half lane % 2
        const int o = (lane >> 2) * 128 + r + 32 * ((lane & 3) >> 1);
        reinterpret_cast<h4v *>(&qs[o])[lane & 1] = hi;
        reinterpret_cast<h4v *>(&qs[o + 64])[lane & 1] = lo;
    }
    lds_barrier();
    if (__ballot(bad != 0)) return false;
    const int qe = qexp[col];
    float m_run = -INFINITY, l_run = 0.0f;
    f32x16 o[2][4] = {};  // [q][c]: dims 128 q + 4 i + c
    for (int ti = wave; ti < tiles; ti += 4) {
        asm volatile("" ::: "memory");  // q is read again for every tile, not kept in registers
        // two steps' q fragments are read while the two before are multiplied
        f32x16 sc = {}, sl = {};
        h8v qa[2][4];
#pragma unroll
        for (int i = 0; i < 4; i++) qa[0][i] = qs[i * 64 + lane];
#pragma unroll
        for (int s = 0; s < 16; s += 2) {
            const int k = (s >> 1) & 1;
            if (s < 14) {
#pragma unroll
                for (int i = 0; i < 4; i++) qa[k ^ 1][i] = qs[(2 * s + 4 + i) * 64 + lane];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const h8v a = __builtin_bit_cast(h8v, kr[s + i]);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qa[k][2 * i], sc, 0, 0, 0);
                sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qa[k][2 * i + 1], sl, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        load_k(ti + 4);
        float tm = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int pos = ti * kPTile + 8 * (e >> 2) + 4 * h + (e & 3);
            sc[e] = pos <= plim ? ldexpf(sc[e] + sl[e], qe) : -INFINITY;
            tm = fmaxf(tm, sc[e]);
        }
        const float mn = fmaxf(m_run, lanes_max2(tm));
        const float mref = mn == -INFINITY ? 0.0f : mn;
        const float scale = expf(m_run - mref);
        float ps = 0.0f;
        h8v ph[2], pl[2];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float pe = expf(sc[e] - mref);
            ps += pe;
            const float x = pe * kPScale;
            ph[e >> 3][e & 7] = (_Float16)x;
            pl[e >> 3][e & 7] = (_Float16)(x - (float)ph[e >> 3][e & 7]);
        }
        l_run = l_run * scale + lanes_sum2(ps);
        // the sums need scaling only where a row's maximum moved
        if (__ballot(mn != m_run)) {
#pragma unroll
            for (int k = 0; k < 8; k++) o[k >> 2][k & 3] *= scale;
        }
        m_run = mn;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    u32x4 w;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        w[k] = __builtin_amdgcn_perm(vr[u][q][2 * k + 1][c >> 1], vr[u][q][2 * k][c >> 1],
                                                     c & 1 ? 0x07060302u : 0x05040100u);
                    const h8v a = __builtin_bit_cast(h8v, w);
                    o[q][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph[u], o[q][c], 0, 0, 0);
                    o[q][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl[u], o[q][c], 0, 0, 0);
                }
        load_v(ti + 4);
    }
    // merge: every wave's sums times exp(m - M) / L of the row, added over the
    // waves 128 dims at a time, times sigmoid(gate) (deltanet.rs:667-669).
    // Thread (i = t % 32) finishes dims 128 q + 4 i .. + 3 of rows t / 32 + 8 k;
    // its gates are loaded ahead of the exchange.
    const int mi = t & 31;
    float4 gate[2][kQRows / 8];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int k = 0; k < kQRows / 8; k++) {
            const int r = (t >> 5) + 8 * k;
            gate[q][k] = mix.at4(min(t0 + r / G, T - 1), (kvh * G + r % G) * 2 * kHd + kHd + 128 * q + 4 * mi);
        }
    if (h == 0) {
        wm[wave][col] = m_run;
        wl[wave][col] = l_run;
    }
    lds_barrier();
    float M = wm[0][col];
#pragma unroll
    for (int w = 1; w < 4; w++) M = fmaxf(M, wm[w][col]);
    float L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) L += expf(wm[w][col] - M) * wl[w][col];
    const float f = expf(m_run - M) / (L * kPScale);
#pragma unroll
    for (int q = 0; q < 2; q++) {
        if (q) lds_barrier();  // the first half's sums were read
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int e = 0; e < 16; e++) lds[((wave * 4 + c) * 16 + e) * kMergeF + lane] = o[q][c][e] * f;
        lds_barrier();
#pragma unroll
        for (int k = 0; k < kQRows / 8; k++) {
            const int r = (t >> 5) + 8 * k, tok = t0 + r / G, head = kvh * G + r % G;
            const int at = ((mi >> 3) * 4 + (mi & 3)) * kMergeF + r + 32 * ((mi >> 2) & 1);
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                v[c] = 0.0f;
#pragma unroll
                for (int w = 0; w < 4; w++) v[c] += lds[(w * 4 + c) * 16 * kMergeF + at];
            }
            const float4 g = gate[q][k];
            if (tok < T)
                *reinterpret_cast<float4 *>(out + ((size_t)tok * n_heads + head) * kHd + 128 * q + 4 * mi) =
                    make_float4(v[0] * (1.0f / (1.0f + expf(-g.x))), v[1] * (1.0f / (1.0f + expf(-g.y))),
                                v[2] * (1.0f / (1.0f + expf(-g.z))), v[3] * (1.0f / (1.0f + expf(-g.w))));
        }
    }
    return true;
}

template <int G>
__global__ __launch_bounds__(kThreads, 1) void attn_prefill_kernel(
    MixIn mix, const float *__restrict__ q_norm, const float *__restrict__ inv_freq,
    const uint32_t *__restrict__ pos_arr, const __half *__restrict__ k_cache, const __half *__restrict__ v_cache,
    size_t cache_off, int max_seq, int n_heads, int T, const uint32_t *__restrict__ odd, float *__restrict__ out) {
    constexpr int QT = kQRows / G;  // tokens per workgroup
    // the last tokens see the most positions: they go first
    const int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * QT, kvh = blockIdx.y, end = min(t0 + QT, T);
    const int p0 = (int)pos_arr[0];
    uint32_t bad = odd[(size_t)kvh * T + min(t0 + ((int)threadIdx.x & (QT - 1)), end - 1)];
#pragma unroll 1
    for (int a = t0, step = QT; a < end;) {
        if (prefill_tokens<G>(mix, q_norm, inv_freq, p0, k_cache, v_cache, cache_off, max_seq, n_heads, kvh, a,
                              min(a + step, end), bad, out)) {
            a += step;
            if (a < end) lds_barrier();  // the tokens before are done with the LDS
        } else {
            step = 1;
            bad = 0;
        }
    }
}

// Chunks per (sequence, kv head): at most 128, at most one per 64-position
// tile of the cache, and about one workgroup per CU over the launch
// (kAttnWorkgroups / (batch x kv heads): batch 32 with 2 kv heads 4 chunks,
// batch 1 with 2 kv heads 128, with 4 kv heads 64).  256 chunks at batch 1
// were slower at 32k (the o_proj prologue merges twice the partials:
// 1049 against 1064 tok/s).  Longer chunks at batch > 1 amortise each
// workgroup's q / k preparation and partial write (batch 32, capacity =
// context 1k / 8k / 32k: 20.6k / 15.4k / 8.4k tok/s at ~256 workgroups
// against 20.1–20.3k / 14.7–14.9k / 8.4k at ~2048).
int chunk_count(int max_seq, int batch, int n_kv) {
    const int tiles = (max_seq + kCh - 1) / kCh;
    const int fill = std::max(1, kAttnWorkgroups / std::max(1, batch * n_kv));
    return std::max(1, std::min(std::min(tiles, kMaxChunks), fill));
}

}  // namespace

int attn_chunks(int max_seq, int batch, int n_kv) { return chunk_count(max_seq, batch, n_kv); }

size_t attn_partial_floats(int batch, int n_kv, int max_seq, int G) {
    return (size_t)batch * n_kv * chunk_count(max_seq, batch, n_kv) * G * (kHd + 2);
}

namespace {

int attention_impl(anehip_ctx *ctx, hipStream_t stream, int batch, int n_heads, int n_kv, int max_seq,
                   const MixIn &mix, const float *q_norm, const float *k_norm, const float *inv_freq,
                   const uint32_t *pos, __half *k_cache, __half *v_cache, float *part, float *out, const Planes &xp,
                   size_t cache_off, size_t row_stride, bool append) {
    const int G = n_heads / n_kv;
    const int nch = chunk_count(max_seq, batch, n_kv);
    if ((size_t)max_seq * kHd * 2 >= (size_t)1 << 30)
        return set_error(ctx->err, ANEHIP_EUNSUPPORTED, "attention: max_seq %d too large", max_seq);
    float *part_o = part;
    float *part_ml = part + (size_t)batch * n_kv * nch * G * kHd;
    dim3 g1(nch, n_kv, batch), g2(n_heads, batch);
    // the caches this launch can read (prefill rows share one sequence's)
    const bool nt = (size_t)(row_stride ? batch : 1) * n_kv * max_seq * 2 * kHd * sizeof(__half) >= kNtKvBytes;
    // sequences of their own, at least two workgroups each to share out, and
    // chunks that can grow to kPlanTiles tiles: equal lengths pay the plan
    // without a use for it (20.0 against 19.4 us at batch 32, 5 tiles a chunk).
    // Their caches hold 80 MiB and more, so that plans come with nt.
    const bool plan = row_stride && batch >= 2 && batch <= kMaxPlanBatch && nch >= 2 &&
                      (max_seq + kCh - 1) / kCh >= kPlanTiles * nch;
#define ANEHIP_ATTN_PART(GG, NT, PLAN)                                                                          \
    hipLaunchKernelGGL((attn_partial_kernel<GG, NT, PLAN>), g1, dim3(kThreads), 0, stream, mix, q_norm, k_norm, \
                       inv_freq, pos, k_cache, v_cache, max_seq, n_heads, n_kv, part_o, part_ml, cache_off,     \
                       row_stride, append, batch)
#define ANEHIP_ATTN_COMBINE(GG, GR, PLAN)                                                                       \
    hipLaunchKernelGGL((attn_combine_kernel<GG, GR, PLAN>), g2, dim3(64 * GR), 0, stream, mix, pos, part_o,     \
                       part_ml, nch, n_heads, n_kv, out, xp, max_seq)
#define ANEHIP_ATTN_CASE(GG)                                                                                    \
    case GG:                                                                                                    \
        if (plan) ANEHIP_ATTN_PART(GG, true, true);                                                             \
        else if (nt) ANEHIP_ATTN_PART(GG, true, false);                                                         \
        else ANEHIP_ATTN_PART(GG, false, false);                                                                \
        ANEHIP_HIP_TRY(ctx->err, hipGetLastError());                                                            \
        if (!out && !xp.hi) return ANEHIP_OK; /* partials only */                                               \
        if (nch > kManyChunks && plan) ANEHIP_ATTN_COMBINE(GG, 16, true);                                       \
        else if (nch > kManyChunks) ANEHIP_ATTN_COMBINE(GG, 16, false);                                         \
        else if (nch > kSomeChunks && plan) ANEHIP_ATTN_COMBINE(GG, 8, true);                                   \
        else if (nch > kSomeChunks) ANEHIP_ATTN_COMBINE(GG, 8, false);                                          \
        else if (plan) ANEHIP_ATTN_COMBINE(GG, 4, true);                                                        \
        else ANEHIP_ATTN_COMBINE(GG, 4, false);                                                                 \
        ANEHIP_HIP_TRY(ctx->err, hipGetLastError());                                                            \
        return ANEHIP_OK;
    switch (G) {
        ANEHIP_ATTN_CASE(1)
        ANEHIP_ATTN_CASE(2)
        ANEHIP_ATTN_CASE(4)
        default:
            return set_error(ctx->err, ANEHIP_EUNSUPPORTED, "attention: %d query heads per kv head (1, 2 or 4)", G);
    }
#undef ANEHIP_ATTN_CASE
#undef ANEHIP_ATTN_COMBINE
#undef ANEHIP_ATTN_PART
}

}  // namespace

// part: workspace of attn_partial_floats() floats.
int launch_attention(anehip_ctx *ctx, hipStream_t stream, int batch, int n_heads, int n_kv, int max_seq,
                     const MixIn &mix, const float *q_norm, const float *k_norm, const float *inv_freq,
                     const uint32_t *pos, __half *k_cache, __half *v_cache, float *part, float *out,
                     const Planes &xp) {
    return attention_impl(ctx, stream, batch, n_heads, n_kv, max_seq, mix, q_norm, k_norm, inv_freq, pos, k_cache,
                          v_cache, part, out, xp, 0, (size_t)n_kv * max_seq * kHd, true);
}

int launch_attention_prefill(anehip_ctx *ctx, hipStream_t stream, int rows, int n_heads, int n_kv, int max_seq,
                             const MixIn &mix, const float *q_norm, const float *k_norm, const float *inv_freq,
                             const uint32_t *pos, __half *k_cache, __half *v_cache, size_t cache_off, float *part,
                             float *out, const Planes &xp) {
    if ((size_t)max_seq * kHd * 2 >= (size_t)1 << 30)
        return set_error(ctx->err, ANEHIP_EUNSUPPORTED, "attention: max_seq %d too large", max_seq);
    // few rows: one workgroup of the decode kernel per row and kv head has less
    // to set up (16 rows from position 0: 8.8 + 4.1 us with its merge, against
    // 23.8 + 4.6 with the planes' launch); above, both sides' launches are those
    // of the uniform planes, and 33 rows of a 4-layer model take 535 us against 659
    const bool few = !xp.uniform;
    uint32_t *odd = reinterpret_cast<uint32_t *>(part);  // [n_kv][rows]
    if (rows > (few ? kPrefillFewRows : kPrefillFewRows * (kHd + 2)))
        return set_error(ctx->err, ANEHIP_EINVAL, "attention: %d rows into %s planes", rows, few ? "grouped" : "uniform");
    hipLaunchKernelGGL(attn_append_kernel, dim3(n_kv, rows), dim3(64), 0, stream, mix, k_norm, inv_freq, pos, k_cache,
                       v_cache, cache_off, max_seq, n_heads, n_kv, few ? nullptr : odd);
    ANEHIP_HIP_TRY(ctx->err, hipGetLastError());
    if (few)
        return attention_impl(ctx, stream, rows, n_heads, n_kv, max_seq, mix, q_norm, k_norm, inv_freq, pos, k_cache,
                              v_cache, part, nullptr, xp, cache_off, 0, false);
    const int G = n_heads / n_kv;
#define ANEHIP_ATTN_PREFILL(GG)                                                                                      \
    hipLaunchKernelGGL(attn_prefill_kernel<GG>, dim3((rows * GG + kQRows - 1) / kQRows, n_kv), dim3(kThreads), 0,     \
                       stream, mix, q_norm, inv_freq, pos, k_cache, v_cache, cache_off, max_seq, n_heads, rows, odd, \
                       out)
    if (G == 4) ANEHIP_ATTN_PREFILL(4);
    else if (G == 2) ANEHIP_ATTN_PREFILL(2);
    else if (G == 1) ANEHIP_ATTN_PREFILL(1);
    else return set_error(ctx->err, ANEHIP_EUNSUPPORTED, "attention: %d query heads per kv head (1, 2 or 4)", G);
#undef ANEHIP_ATTN_PREFILL
    ANEHIP_HIP_TRY(ctx->err, hipGetLastError());
    return launch_split_rows(ctx, stream, out, (uint32_t)rows, (uint32_t)(n_heads * kHd), xp);
}

}  // namespace anehip
