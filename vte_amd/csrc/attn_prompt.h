// Attention of many query columns over one cache (prompt chunks), gfx950.
//
// Algorithm: online softmax per chunk as in
// vte/compiler/templates/rdna/flash_attention_split_kv_partial.hip.template:31-120
// (which runs once per query head and token; here a block serves 64 rows).
//
// A row is one (column, query head of the KV head); rows are numbered column
// by column, so a GQA group of any size packs 16-row MFMA tiles without
// padding.  A block's four waves own 16 rows each and walk the same tokens,
// 64 at a time: K and V rows are copied to LDS once per block (LDS-direct
// loads, the next 64 tokens' under this step's products), scores are K.Q^T
// (lane = row, so the softmax state is per lane), the probabilities are the
// A operand of P.V as they stand, and V's operand comes from the transposing
// LDS read.  A wave stops at its own longest row.  In the steps where rows of
// the block end, tokens past a row have probability 0, and 0 * Inf and 0 * NaN
// are NaN: when such a step leaves a non-finite sum, its products are formed
// again by ap_pv_masked, which multiplies a row only with the tokens it sees
// (the check is 32 fmas; reading the V tile for it took 1 us).  The tokens up to
// the block's longest column are cut into nsp equal shares, one per grid.z, so
// every block of a launch does about the same work wherever the chunk lies in
// the prompt; the shares' partial results meet in attn_prompt_combine.
//
// Bound by instruction issue: per 16 rows and 64 tokens 48 MFMAs (768 matrix
// cycles) stand beside about 300 other instructions.  32 rows per wave halve
// the LDS reads but leave one wave per SIMD: 24.5 against 23.0 us (512 columns
// of 12 heads after 1536 rows, probabilities in one part), 15.8 against 13.3
// (128 columns).
#pragma once
#include <type_traits>

#include "attn_tile.h"

#define AP_ROWS 64  // rows of a block
#define AP_TOK 64   // tokens of a step
#define AP_MAX_SPLITS 8

// Probabilities are held as 2^14 exp(score - running maximum) and enter P.V as
// two fp16 parts, hi (rounded down) and lo (the rest): about 21 bits down to
// 2^-38 of the maximum.  One fp16 part relative to a whole share's maximum was
// up to twice as far from the 64-bit result as the other forms, whose reference
// is a 32-token tile's (fp32 results, 1500 rows, scores of standard deviation
// 0.5 / 8: 2.0e-4 / 1.8e-5 against 1.8e-4 / 0.9e-5; two parts 3.4e-7 / 7.0e-7).
// The second part costs 16 MFMAs a step (512 columns after 1536 rows: 21.5 ->
// 23.0 us).  lo's last bit is set, so both parts of a seen token are positive and
// Inf in V stays Inf (0 * Inf is NaN).
#define AP_P_LOG2 14.0f
typedef __fp16 ap_h2 __attribute__((ext_vector_type(2)));
union ApP {
    half8_t v;
    ap_h2 h[4];
    uint32_t u[4];
};

typedef short ap_s4 __attribute__((ext_vector_type(4)));
typedef unsigned ap_u2 __attribute__((ext_vector_type(2)));

// Over the four lanes of a row (lane groups of 16): every lane gets the result.
__device__ __forceinline__ float ap_max4(float v) {
    ap_u2 a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float ap_sum4(float v) {
    ap_u2 a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// 64 tokens' K and V rows, 16-byte chunks permuted inside a row so that the
// rows an operand read touches lie in distinct banks: K chunk ^ (row & 15)
// (16 rows per read), V chunk ^ 2 (row & 7) (pairs of chunks of 16 rows).
struct alignas(16) ApTile {
    _Float16 k[AP_TOK * ATT_D], v[AP_TOK * ATT_D];
};
__device__ __forceinline__ void ap_stage(ApTile& T, const __half* kb, const __half* vb, size_t row_stride, int t0,
                                         int t_last, int wv, int lane) {
    const int r4 = lane >> 4, slot = lane & 15;
#pragma unroll
    for (int j = 0; j < AP_TOK / (4 * ATT_WAVES); ++j) {
        const int r0 = (j * ATT_WAVES + wv) * 4, row = r0 + r4;  // a wave's load fills four rows
        const size_t src = (size_t)min(t0 + row, t_last) * row_stride;
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(kb + src + 8 * (slot ^ (row & 15))),
            (__attribute__((address_space(3))) void*)(T.k + r0 * ATT_D), 16, 0, 0);
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(vb + src + 8 * (slot ^ (2 * (row & 7)))),
            (__attribute__((address_space(3))) void*)(T.v + r0 * ATT_D), 16, 0, 0);
    }
}

// Whether any lane's sums hold an Inf or a NaN (the same answer in every lane).
__device__ __forceinline__ bool ap_nonfinite(const floatx4_t (&o)[ATT_D / 16]) {
    float z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < ATT_D / 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] = fmaf(o[dt][i], 0.f, z[i]);
    return __any(!((z[0] + z[1]) + (z[2] + z[3]) == 0.f));
}

// o += P.V on the vector units, row 4 grp + i over its first cnt[i] tokens only
// (rare: see above).  e[tt][i]: probability of row col, token 16 tt + 4 grp + i.
__device__ __forceinline__ void ap_pv_masked(const ApTile& T, const floatx4_t (&e)[4], const int (&cnt)[4],
                                             floatx4_t (&o)[ATT_D / 16], int lane) {
    const int col = lane & 15, grp = lane >> 4;
#pragma unroll 1
    for (int t = 0; t < AP_TOK; ++t) {
        float ev = e[0][0];
#pragma unroll
        for (int j = 1; j < 16; ++j) ev = (4 * (t >> 4) + (t & 3)) == j ? e[j >> 2][j & 3] : ev;
        float pr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) pr[i] = __shfl(ev, 4 * grp + i + 16 * ((t >> 2) & 3), 64);
#pragma unroll
        for (int dt = 0; dt < ATT_D / 16; ++dt) {
            const float v = (float)T.v[t * ATT_D + 8 * ((2 * dt + (col >> 3)) ^ (2 * (t & 7))) + (col & 7)];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[dt][i] = t < cnt[i] ? fmaf(pr[i], v, o[dt][i]) : o[dt][i];
        }
    }
}

// grid (row blocks, n_kv, nsp), block 256.  max_ctx: rows of the cache that
// may be read.  nsp == 1: out holds the results; else part_m / part_l / part_o
// [n_cols][n_q][max_splits] (x 128) hold share z's at index z < nsp.
template <typename TQ, typename TO>
__global__ __launch_bounds__(256, 2) void attn_prompt_kernel(
    const TQ* __restrict__ q, const __half* __restrict__ k_cache, const __half* __restrict__ v_cache,
    float* __restrict__ part_m, float* __restrict__ part_l, float* __restrict__ part_o, TO* __restrict__ out, int n_q,
    int n_kv, float scale, const int* __restrict__ kv_offset, int n_cols, int max_ctx, int max_splits) {
    __shared__ ApTile tile[2];
    __shared__ int red[2][ATT_WAVES];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int G = n_q / n_kv, kvh = blockIdx.y, sp = blockIdx.z, nsp = gridDim.z;
    const int rows = n_cols * G, r0 = blockIdx.x * AP_ROWS;
    const size_t row_stride = (size_t)n_kv * ATT_D;
    const __half* kb = k_cache + (size_t)kvh * ATT_D;
    const __half* vb = v_cache + (size_t)kvh * ATT_D;

    // this lane's row: query operands and length; the wave's longest length, the block's shortest and longest
    half8_t qb[ATT_D / 32];
    int len;
    {
        const int row = min(r0 + wv * 16 + col, rows - 1), c = row / G, h = row - c * G;
        const TQ* qp = q + ((size_t)c * n_q + kvh * G + h) * ATT_D + 8 * grp;
        len = min(kv_offset[c] + 1, max_ctx);
#pragma unroll
        for (int s = 0; s < ATT_D / 32; ++s) qb[s] = att_load_q8(qp + 32 * s);
    }
    int longest = len, shortest = len;
    for (int i = 1; i < 16; i *= 2) {
        longest = max(longest, __shfl_xor(longest, i, 64));
        shortest = min(shortest, __shfl_xor(shortest, i, 64));
    }
    longest = __builtin_amdgcn_readfirstlane(longest);
    if (lane == 0) {
        red[0][wv] = longest;
        red[1][wv] = shortest;
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(max(max(red[0][0], red[0][1]), max(red[0][2], red[0][3])));
    const int share = ((total + nsp - 1) / nsp + AP_TOK - 1) / AP_TOK * AP_TOK;
    const int t_begin = sp * share, t_end = min(total, t_begin + share);
    const int all_end = __builtin_amdgcn_readfirstlane(
        min(min(min(red[1][0], red[1][1]), min(red[1][2], red[1][3])), t_end));  // every row reaches this far

    float neg1 = -1.f;
    asm volatile("" : "+v"(neg1));  // keeps a - hi one mixed-precision fma (a conversion and a subtraction else)
    const float c2 = scale * 1.44269504088896340736f;  // exp(scale s) = 2^(c2 s)
    float m_run = -1e30f, l_run = 0.f;  // raw score maximum of the row; this lane's share of its sum
    floatx4_t o[ATT_D / 16];            // rows 4 grp + i, dim 16 dt + col
#pragma unroll
    for (int dt = 0; dt < ATT_D / 16; ++dt) o[dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // operand addresses: K row 16 tt + col, chunk 4 s + grp; V token 16 tt + 4 grp + col / 4, dims 16 dt + 4 (col % 4) ..
    int ko[ATT_D / 32], vo[ATT_D / 16];
#pragma unroll
    for (int s = 0; s < ATT_D / 32; ++s) ko[s] = col * ATT_D + 8 * ((4 * s + grp) ^ col);
    const int vtok = 4 * grp + (col >> 2), vx = 2 * (vtok & 7);
#pragma unroll
    for (int dt = 0; dt < ATT_D / 16; ++dt)
        vo[dt] = vtok * ATT_D + 8 * ((2 * dt + ((col & 3) >> 1)) ^ vx) + 4 * (col & 1);

    if (t_begin < t_end) {
        ap_stage(tile[0], kb, vb, row_stride, t_begin, t_end - 1, wv, lane);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    // One step over tile T.  ENDS: some row of the block ends in it (or the share does).
    auto step = [&](const ApTile& T, int t0, auto ends) {
        constexpr bool ENDS = decltype(ends)::value;
        // ---- scores: lane holds S[row col][token 16 tt + 4 grp + i] ----
        floatx4_t s[4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
            s[tt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < ATT_D / 32; ++d)
                s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    *reinterpret_cast<const half8_t*>(T.k + 16 * tt * ATT_D + ko[d]), qb[d], s[tt], 0, 0, 0);
        }
        // ---- online softmax ----
        if constexpr (ENDS) {
            const int end = min(len, t_end) - t0 - 4 * grp;
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[tt][i] = 16 * tt + i < end ? s[tt][i] : -INFINITY;
        }
        float mx = m_run;
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[tt][i]);
        mx = ap_max4(mx);
        if (__any(mx > m_run)) {  // else every factor is 1
            const float corr = __builtin_amdgcn_exp2f((m_run - mx) * c2);
            l_run *= corr;
            m_run = mx;
            float cr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) cr[i] = __shfl(corr, 4 * grp + i, 64);
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[dt][i] *= cr[i];
        }
        const float mc = fmaf(-mx, c2, AP_P_LOG2);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[tt][i] = __builtin_amdgcn_exp2f(fmaf(s[tt][i], c2, mc));
                l_run += s[tt][i];
            }
        ApP hi[2], lo[2];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float a = s[j >> 1][2 * (j & 1)], b = s[j >> 1][2 * (j & 1) + 1];
            const ap_h2 h = __builtin_amdgcn_cvt_pkrtz(a, b);
            hi[j >> 2].h[j & 3] = h;
            lo[j >> 2].h[j & 3] = __builtin_amdgcn_cvt_pkrtz(fmaf((float)h[0], neg1, a), fmaf((float)h[1], neg1, b));
            if constexpr (!ENDS) lo[j >> 2].u[j & 3] |= 0x00010001u;
        }
        floatx4_t before[ATT_D / 16];
        if constexpr (ENDS) {
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt) before[dt] = o[dt];
        }
        // ---- P.V: V[token slots][dim 16 dt + col] by transposing reads of 4 tokens x 16 dims ----
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            union {
                ap_s4 h[2];
                half8_t v;
            } vf[ATT_D / 16];
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt) {
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    vf[dt].h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) ap_s4*)(T.v + (2 * u + e) * 16 * ATT_D + vo[dt]));
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[u].v, vf[dt].v, o[dt], 0, 0, 0);
            }
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt)
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[u].v, vf[dt].v, o[dt], 0, 0, 0);
        }
        if constexpr (ENDS) {
            if (ap_nonfinite(o)) {
                int cnt[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) cnt[i] = min(__shfl(len, 4 * grp + i, 64), t_end) - t0;
#pragma unroll
                for (int dt = 0; dt < ATT_D / 16; ++dt) o[dt] = before[dt];
                ap_pv_masked(T, s, cnt, o, lane);
            }
        }
    };
    int t0 = t_begin, cur = 0;
    auto stage_next = [&] {
        if (t0 + AP_TOK < t_end) ap_stage(tile[cur ^ 1], kb, vb, row_stride, t0 + AP_TOK, t_end - 1, wv, lane);
    };
    auto next = [&] {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tokens' copies
        __syncthreads();
        t0 += AP_TOK;
        cur ^= 1;
    };
    while (t0 + AP_TOK <= all_end) {
        stage_next();
        step(tile[cur], t0, std::false_type{});
        next();
    }
    while (t0 < t_end) {
        stage_next();
        if (t0 < longest) step(tile[cur], t0, std::true_type{});  // past its rows a wave only takes part in the copies
        next();
    }

    // ---- results: rows 4 grp + i of the wave's tile ----
    const float l = ap_sum4(l_run);
    const int row0 = r0 + wv * 16;
    if (nsp > 1 && grp == 0 && row0 + col < rows) {
        const int c = (row0 + col) / G, h = (row0 + col) - c * G;
        const size_t st = ((size_t)c * n_q + kvh * G + h) * max_splits + sp;
        part_m[st] = m_run * scale;
        part_l[st] = l;
    }
    const float inv = 1.0f / fmaxf(l, 1e-20f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + 4 * grp + i;
        const float f = __shfl(inv, 4 * grp + i, 64);
        if (row >= rows) continue;
        const int c = row / G, h = row - c * G;
        const size_t hd = (size_t)c * n_q + kvh * G + h;
        if (nsp == 1) {
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt) st_act<TO>(out + hd * ATT_D + 16 * dt + col, o[dt][i] * f);
        } else if (t_begin < t_end) {  // an empty share's sums are not read
#pragma unroll
            for (int dt = 0; dt < ATT_D / 16; ++dt) part_o[(hd * max_splits + sp) * ATT_D + 16 * dt + col] = o[dt][i];
        }
    }
}

// Log-sum-exp combine of the nsp <= AP_MAX_SPLITS shares: 32 threads per
// (column, head), four dims each, every load requested at once.  Shares with
// nothing in them (l = 0) are left out.
template <typename TO>
__global__ __launch_bounds__(256) void attn_prompt_combine(const float* __restrict__ part_m,
                                                           const float* __restrict__ part_l,
                                                           const float* __restrict__ part_o, TO* __restrict__ out,
                                                           int heads, int nsp, int max_splits) {
    const int hd = blockIdx.x * 8 + (threadIdx.x >> 5), d = 4 * (threadIdx.x & 31);
    if (hd >= heads) return;
    const size_t st = (size_t)hd * max_splits;
    float m[AP_MAX_SPLITS], l[AP_MAX_SPLITS];
    float4 o[AP_MAX_SPLITS];
#pragma unroll
    for (int j = 0; j < AP_MAX_SPLITS; ++j) {
        const int s = min(j, nsp - 1);
        m[j] = part_m[st + s];
        l[j] = part_l[st + s];
        __builtin_memcpy(&o[j], part_o + (st + s) * ATT_D + d, sizeof(float4));  // part_o: any float's alignment
    }
    float M = -1e30f;
#pragma unroll
    for (int j = 0; j < AP_MAX_SPLITS; ++j) M = j < nsp ? fmaxf(M, m[j]) : M;
    float L = 0.f, r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < AP_MAX_SPLITS; ++j) {
        const bool has = j < nsp && l[j] != 0.f;
        const float w = has ? __expf(m[j] - M) : 0.f;
        L = has ? fmaf(l[j], w, L) : L;
        const float v[4] = {o[j].x, o[j].y, o[j].z, o[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = has ? fmaf(v[e], w, r[e]) : r[e];
    }
    L = fmaxf(L, 1e-20f);
#pragma unroll
    for (int e = 0; e < 4; ++e) st_act<TO>(out + (size_t)hd * ATT_D + d + e, r[e] / L);
}
