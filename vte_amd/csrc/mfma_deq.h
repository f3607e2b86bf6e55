// Quantised weights as exact MFMA operands (Q4_K / Q6_K super-blocks) and the
// k-slot map shared by the batched MFMA kernels, gfx950.
//
//  * v_mfma_f32_16x16x32_f16 with the activations as the A operand (M = 16
//    batch columns) and the weights as the B operand (N = 16 weight rows),
//    K = 32: C[m][n] lands in lane (n, g) as batch columns 4g .. 4g+3 of
//    weight row n, the lane that loaded row n's super-block, so the
//    super-block scales apply lane-locally.
//  * Exact weight operands: a super-block's weights are d * (sc_j * q) -
//    dmin * m_j (Q4_K) or d * (sc_j * (q - 32)) (Q6_K), with 4/6-bit codes
//    q and 6/8-bit sub-block scales sc_j, m_j.  The operands are the integer
//    products sc_j * q (<= 945) and sc_j * (q - 32) (exact in fp16 while
//    |sc_j| <= 64, one rounding of an integer product beyond), made with
//    packed fp16 math from the code bytes (nibble -> 0x64xx magic = 1024 + q);
//    the Q4_K minimum term is either one MFMA per k-step of the activations
//    against the splat 6-bit minimum (launches of at most 16 columns) or one
//    MFMA of the activations' sub-block sums (formed once per super-block and
//    wave, q4_xmin) against the row's eight minima (longer batches).  The MFMA sums a super-block in fp32 and the fp32
//    scales d, dmin are applied once per super-block (sb_mfma).  The weights
//    therefore enter the sums exactly as the reference's fp32 dequantisation
//    defines them (vte/compiler/dequantizer.py:26-70, 129-169); only the fp16
//    activations and the fp32 sums round.
//  * K-slot permutation: MFMA pairs A and B by (lane group, slot), so any
//    bijection of super-block elements to (k-step, group, slot) is valid as
//    long as A and B use the same one.  The map is chosen so each lane's 8
//    slots are 8 contiguous elements sharing one sub-block scale:
//      Q4_K step t, group g: qs chunk c = g + 4*(t>>2), nibble (t>>1)&1, half t&1
//           (sub-block 2 * ((g>>1) + 2*(t>>2)) + ((t>>1)&1); steps 2s, 2s+1 share one)
//      Q6_K step t, group g: half h = g>>1, quarter q = t>>1, l = 16 (g&1) + 8 (t&1) .. +7
//           (16-element sub-block 8h + 2q + (g&1)); a lane's codes for all 8
//           steps come from three 16-byte runs of its row's block (ql, ql + 32, qh)
#pragma once
#include <cstdlib>
#include "quant.h"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

union H8 {
    half8_t v;
    uint32_t u[4];
    half2_t h2[4];
};

#define MF_WAVES 8

// bytes b0..b3 of `u` (each < 256) -> two fp16 pairs 1024+b.
__device__ __forceinline__ void bytes_to_f16magic(uint32_t u, uint32_t& lo, uint32_t& hi) {
    lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
}

// 8 codes in the bytes of (u0, u1) -> 8 fp16 values (1024 + q) * s + c: with
// c = -1024 s the exact integer q * s, with c = -1056 s the integer (q - 32) * s.
__device__ __forceinline__ half8_t codes8(uint32_t u0, uint32_t u1, half2_t s2, half2_t c2) {
    H8 r;
    bytes_to_f16magic(u0, r.u[0], r.u[1]);
    bytes_to_f16magic(u1, r.u[2], r.u[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.h2[i] = __builtin_elementwise_fma(r.h2[i], s2, c2);  // one rounding: exact
    return r.v;
}

__device__ __forceinline__ half2_t splat2(float v) { return half2_t{(_Float16)v, (_Float16)v}; }

template <typename TI>
__device__ __forceinline__ half8_t load_x8(const TI* p, bool valid);
template <>
__device__ __forceinline__ half8_t load_x8<__half>(const __half* p, bool valid) {
    if (!valid) return half8_t{0, 0, 0, 0, 0, 0, 0, 0};
    return *reinterpret_cast<const half8_t*>(p);
}
template <>
__device__ __forceinline__ half8_t load_x8<float>(const float* p, bool valid) {
    half8_t r = {0, 0, 0, 0, 0, 0, 0, 0};
    if (!valid) return r;
    const float4 a = reinterpret_cast<const float4*>(p)[0];
    const float4 b = reinterpret_cast<const float4*>(p)[1];
    r[0] = (_Float16)a.x; r[1] = (_Float16)a.y; r[2] = (_Float16)a.z; r[3] = (_Float16)a.w;
    r[4] = (_Float16)b.x; r[5] = (_Float16)b.y; r[6] = (_Float16)b.z; r[7] = (_Float16)b.w;
    return r;
}

// Element offset (within a super-block) of step t, group g.
template <int FMT>
__device__ __forceinline__ int kslot_base(int t, int g) {
    if (FMT == 4) {
        const int c = g + 4 * (t >> 2);
        return 64 * (c >> 1) + 16 * (c & 1) + 32 * ((t >> 1) & 1) + 8 * (t & 1);
    } else {
        return 128 * (g >> 1) + 32 * (t >> 1) + 16 * (g & 1) + 8 * (t & 1);
    }
}


// The eight MFMA A operands (k-steps t = 4*hh + q) of one lane for a Q6_K
// super-block read straight from global memory: the lane's 8-byte slices of
// ql, qh and the scales of each half.  Q6_K blocks are only 2-byte aligned;
// the unaligned 8-byte loads stream as fast as aligned ones on gfx950.
__device__ __forceinline__ uint2 q6_ld8(const uint8_t* p) {
    uint2 v;
    __builtin_memcpy(&v, p, 8);
    return v;
}
// A lane's raw bytes of one Q6_K super-block (both halves), loaded ahead of
// the dequantisation so several super-blocks can be in flight.
struct Q6Raw {
    uint4 la, lb, hq;  // ql[64h + 16j ..], ql[64h + 32 + 16j ..], qh[32h + 16j ..] (h = g>>1, j = g&1)
    uint2 sc;          // scales 8h .. 8h+7
    uint32_t d;
};
__device__ __forceinline__ uint4 q6_ld16(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
__device__ __forceinline__ void q6_raw_load(const uint8_t* blk, int grp, Q6Raw& r) {
    const int h = grp >> 1, j = grp & 1;
    r.la = q6_ld16(blk + 64 * h + 16 * j);
    r.lb = q6_ld16(blk + 64 * h + 32 + 16 * j);
    r.hq = q6_ld16(blk + 128 + 32 * h + 16 * j);
    r.sc = q6_ld8(blk + 192 + 8 * h);
    r.d = ((const __attribute__((address_space(1))) uint16_t*)(blk + 208))[0];
}
// Exact operands of one super-block for one lane: the 8 k-steps' weight
// operands and the fp32 scales (Q4_K: also the 4 sub-block minima, splat).
struct Q6Ops {
    half8_t w[8];
    float d;
};
struct Q4Ops {
    half8_t w[8];
    half8_t mins;   // XM: lane groups 0-1 the row's eight sub-block minima m_0..m_7, groups 2-3 zero
    uint32_t mnb;   // !XM: byte s = m_j of the lane's sub-block of steps 2s, 2s+1
    float d, dmin;
};

// Operand of k-step t.
__device__ __forceinline__ half8_t q6_step_operand(const Q6Raw& r, int t, int grp) {
    const uint32_t la[4] = {r.la.x, r.la.y, r.la.z, r.la.w};
    const uint32_t lb[4] = {r.lb.x, r.lb.y, r.lb.z, r.lb.w};
    const uint32_t hq[4] = {r.hq.x, r.hq.y, r.hq.z, r.hq.w};
    const uint64_t sc = ((uint64_t)r.sc.y << 32) | r.sc.x;
    const int q = t >> 1, w0 = 2 * (t & 1);  // quarter; first code word of the step's 8 codes
    uint32_t u[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const uint32_t l = (q & 1) ? lb[w0 + e] : la[w0 + e];
        const uint32_t nib = (q < 2) ? (l & 0x0F0F0F0Fu) : ((l >> 4) & 0x0F0F0F0Fu);
        u[e] = nib | (((hq[w0 + e] >> (2 * q)) & 0x03030303u) << 4);
    }
    const float scq = (float)(int8_t)((sc >> (8 * (2 * q + (grp & 1)))) & 0xFF);
    // (1024 + u) - 1056 = u - 32 exactly, then one multiply by the integer scale
    H8 v;
    bytes_to_f16magic(u[0], v.u[0], v.u[1]);
    bytes_to_f16magic(u[1], v.u[2], v.u[3]);
    const half2_t off = splat2(-1056.0f), s2 = splat2(scq);
#pragma unroll
    for (int i = 0; i < 4; ++i) v.h2[i] = (v.h2[i] + off) * s2;
    return v.v;
}
__device__ __forceinline__ void q6_exact_operands(const Q6Raw& r, int grp, Q6Ops& o) {
    o.d = h2f_bits(r.d);
#pragma unroll
    for (int t = 0; t < 8; ++t) o.w[t] = q6_step_operand(r, t, grp);
}

// Q4_K: the header and the lane's two 16-byte code chunks; operands for the
// k-slot map of kslot_base<4>.
struct Q4Raw {
    uint4 h, q0, q1;
};
__device__ __forceinline__ void q4_raw_load(const uint8_t* blk, int grp, Q4Raw& r) {
    r.h = *reinterpret_cast<const uint4*>(blk);
    r.q0 = *reinterpret_cast<const uint4*>(blk + 16 + 16 * grp);
    r.q1 = *reinterpret_cast<const uint4*>(blk + 16 + 16 * (grp + 4));
}
// Byte b of u (< 256) as a splat fp16 pair, exactly.
__device__ __forceinline__ half2_t byte_splat(uint32_t u, int b) {
    const uint32_t v = __builtin_amdgcn_perm(0x64646464u, u, 0x04000400u + 0x00010001u * (uint32_t)b);
    return __builtin_bit_cast(half2_t, v) + splat2(-1024.0f);
}
// The eight 6-bit scales of a Q4_K header, four to a word (get_scale_min_k4 on
// all bytes at once), and its eight minima.
__device__ __forceinline__ void q4_scale_words(const uint4& h, uint32_t (&sc)[2]) {
    sc[0] = h.y & 0x3F3F3F3Fu;
    sc[1] = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
}
__device__ __forceinline__ void q4_min_words(const uint4& h, uint32_t (&mn)[2]) {
    mn[0] = h.z & 0x3F3F3F3Fu;
    mn[1] = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
}
// Q4Ops::mins of a lane.
__device__ __forceinline__ half8_t q4_mins(const uint4& h, int grp) {
    uint32_t mn[2];
    q4_min_words(h, mn);
    H8 v;
    bytes_to_f16magic(grp < 2 ? mn[0] : 0u, v.u[0], v.u[1]);
    bytes_to_f16magic(grp < 2 ? mn[1] : 0u, v.u[2], v.u[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) v.h2[i] = v.h2[i] + splat2(-1024.0f);
    return v.v;
}
// Operand of the k-step that takes nibble `part`, half `e` of code chunk qc.
__device__ __forceinline__ half8_t q4_step_operand(const uint4& qc, int part, int e, half2_t s2, half2_t c2) {
    const uint32_t wa = e == 0 ? qc.x : qc.z, wb = e == 0 ? qc.y : qc.w;
    const uint32_t u0 = part ? ((wa >> 4) & 0x0F0F0F0Fu) : (wa & 0x0F0F0F0Fu);
    const uint32_t u1 = part ? ((wb >> 4) & 0x0F0F0F0Fu) : (wb & 0x0F0F0F0Fu);
    return codes8(u0, u1, s2, c2);
}
template <bool XM>
__device__ __forceinline__ void q4_exact_operands(const Q4Raw& r, int grp, Q4Ops& o) {
    o.d = h2f_bits(r.h.x);
    o.dmin = h2f_bits(r.h.x >> 16);
    uint32_t sc[2];
    q4_scale_words(r.h, sc);
    const int b0 = 2 * (grp >> 1);  // byte of the lane's first sub-block in either word
    if constexpr (!XM) {
        uint32_t mn[2];
        q4_min_words(r.h, mn);
        o.mnb = __builtin_amdgcn_perm(mn[1], mn[0], 0x05040100u + 0x02020202u * (uint32_t)(grp >> 1));
    } else {
        o.mins = q4_mins(r.h, grp);
    }
#pragma unroll
    for (int ci = 0; ci < 2; ++ci)
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            const half2_t s2 = byte_splat(sc[ci], b0 + part), c2 = s2 * splat2(-1024.0f);  // exact: sc <= 63
#pragma unroll
            for (int e = 0; e < 2; ++e)
                o.w[4 * ci + 2 * part + e] = q4_step_operand(ci == 0 ? r.q0 : r.q1, part, e, s2, c2);
        }
}

// Sub-block sums of the activations of one super-block, X[m][j] = sum of
// x[m][k] over sub-block j (Q4_K: 8 sub-blocks of 32), for the minimum term
// dmin * sum_j m_j X[m][j], which is the same for every weight row of the
// tile and so is formed once per super-block and wave: eight MFMAs of the
// activation operands against 0/1 sub-block indicators (exact fp32 sums),
// then, through the wave's LDS scratch `xl` [NT][16][8], the A-operand layout
// with X split into fp16 hi (lane group 0) and lo (group 1) parts, so the
// single MFMA against the row minima (Q4Ops::mins) sums hi + lo to ~2^-22.
// This form (XM) pays off where several row tiles or column tiles share the
// sums (weight-stationary and multi-tile launches).  With one row tile and
// one column tile per super-block and wave (the batched decode launches) its
// serial chain (indicator MFMAs, LDS round trip) lies on the critical path,
// and the !XM form instead adds one MFMA per k-step of the activations
// against the splat minimum of the step's sub-block, independent of the
// weight MFMAs.  The two forms round the minimum term differently (both sum
// in fp32; results agree to fp32 rounding, not bit for bit).
template <int NT, bool XM>
struct XMin {
    half8_t xa[NT];
};
template <int NT>
struct XMin<NT, false> {};
template <int NT>
__device__ __forceinline__ void q4_xmin(const half8_t (&bx)[8][NT], float* xl, XMin<NT, true>& xm) {
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    floatx4_t cx[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) cx[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int sub = 2 * ((grp >> 1) + 2 * (t >> 2)) + ((t >> 1) & 1);  // sub-block of step t, group grp
        const _Float16 one = col == sub ? (_Float16)1.0f : (_Float16)0.0f;
        const half8_t ind = {one, one, one, one, one, one, one, one};
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) cx[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bx[t][nt], ind, cx[nt], 0, 0, 0);
    }
    // C layout: lane (j, grp) holds X[4 grp + i][j]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (col < 8) xl[(nt * 16 + 4 * grp + i) * 8 + col] = cx[nt][i];
    // a wave's LDS operations complete in order: wait for the stores (LDS
    // counter only, the weight prefetches stay in flight) before the reads
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float4 a = *reinterpret_cast<const float4*>(xl + (nt * 16 + col) * 8);
        const float4 b = *reinterpret_cast<const float4*>(xl + (nt * 16 + col) * 8 + 4);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        half8_t h;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const _Float16 hi = (_Float16)v[j];
            const _Float16 lo = (_Float16)(v[j] - (float)hi);
            h[j] = grp == 0 ? hi : (grp == 1 ? lo : (_Float16)0.0f);
        }
        xm.xa[nt] = h;
    }
    asm volatile("" ::: "memory");  // xl is rewritten by the next call
}

// One super-block of MFMA work for NT 16-column activation tiles bx[t][nt]
// (A operands, k-slot map of the format) against one lane's exact weight
// operands: acc[nt] += d * sum(w x) [- dmin * sum_j m_j X_j], the sums in fp32
// over the super-block's 8 k-steps in order.  The launches of 17 to 32 columns,
// the weight-stationary and the streaming kernels go through these functions
// (one-tile launches through sb_staged, with the same sums; the tiled kernels
// through mt_loop, which rounds a scaled super-block before it adds it).  So for
// a given minimum-term form (XM) a weight row's result depends only on which
// super-blocks a wave sums and the order the waves' partials are added, and the
// tiled kernels agree bit for bit where each of those waves has at most one
// super-block (K of at most 2048, or that share of K), not beyond.
template <int NT, bool XM>
__device__ __forceinline__ void sb_mfma(const Q6Ops& o, const half8_t (&bx)[8][NT], const XMin<NT, XM>&,
                                        floatx4_t (&acc)[NT]) {
    floatx4_t aw[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) aw[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) aw[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bx[t][nt], o.w[t], aw[nt], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[nt][i] = fmaf(o.d, aw[nt][i], acc[nt][i]);
}
template <int NT>
__device__ __forceinline__ void sb_mfma(const Q4Ops& o, const half8_t (&bx)[8][NT], const XMin<NT, true>& xm,
                                        floatx4_t (&acc)[NT]) {
    floatx4_t aw[NT], am[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        aw[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        am[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xm.xa[nt], o.mins, floatx4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) aw[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bx[t][nt], o.w[t], aw[nt], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[nt][i] = fmaf(-o.dmin, am[nt][i], fmaf(o.d, aw[nt][i], acc[nt][i]));
}

template <int NT>
__device__ __forceinline__ void sb_mfma(const Q4Ops& o, const half8_t (&bx)[8][NT], const XMin<NT, false>&,
                                        floatx4_t (&acc)[NT]) {
    floatx4_t aw[NT], am[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) aw[nt] = am[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const half2_t m = byte_splat(o.mnb, t >> 1);
        const half8_t mv = {m[0], m[1], m[0], m[1], m[0], m[1], m[0], m[1]};
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            aw[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bx[t][nt], o.w[t], aw[nt], 0, 0, 0);
            am[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bx[t][nt], mv, am[nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[nt][i] = fmaf(-o.dmin, am[nt][i], fmaf(o.d, aw[nt][i], acc[nt][i]));
}

// The minimum-term sums where the format has one (Q4_K), else nothing.
template <int FMT, int NT, bool XM>
__device__ __forceinline__ void sb_xmin(const half8_t (&bx)[8][NT], float* xl, XMin<NT, XM>& xm) {
    if constexpr (FMT == 4 && XM) q4_xmin<NT>(bx, xl, xm);
}

// Raw bytes -> operands for either format.
template <int FMT> struct SbRaw;
template <> struct SbRaw<4> { using Raw = Q4Raw; using Ops = Q4Ops; };
template <> struct SbRaw<6> { using Raw = Q6Raw; using Ops = Q6Ops; };
__device__ __forceinline__ void sb_load(const uint8_t* blk, int grp, Q4Raw& r) { q4_raw_load(blk, grp, r); }
__device__ __forceinline__ void sb_load(const uint8_t* blk, int grp, Q6Raw& r) { q6_raw_load(blk, grp, r); }
template <bool XM>
__device__ __forceinline__ void sb_ops(const Q4Raw& r, int grp, Q4Ops& o) { q4_exact_operands<XM>(r, grp, o); }
template <bool XM>
__device__ __forceinline__ void sb_ops(const Q6Raw& r, int grp, Q6Ops& o) { q6_exact_operands(r, grp, o); }

// LDS of one wave of a batched kernel: its partial C tiles, summed over the
// waves by the epilogue, over its staged activations (ST, 16 columns), and the
// minimum-term scratch (q4_xmin).
template <int RT, int NT, bool ST>
struct alignas(16) MfWave {
    union {
        _Float16 x[ST ? 16 * QK_K : 8];
        float red[RT][NT][4][64];
    };
    float xl[ST ? 4 : NT * 128];
};

#define MT_GLOBAL(p) ((const __attribute__((address_space(1))) void*)(p))
#define MT_SHARED(p) ((__attribute__((address_space(3))) void*)(p))

// 16 (or 8) bytes at a 2-byte aligned LDS address.
template <int N>
__device__ __forceinline__ void lds_words(const uint8_t* p, uint32_t (&v)[N]) {
    const uint32_t a = (uint32_t)(uintptr_t)MT_SHARED(p);
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p - (a & 2));
    uint32_t w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; ++i) w[i] = q[i];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], a & 2);
}
// A lane's raw bytes of its row's super-block from the staged copy.
__device__ __forceinline__ void mt_raw(const uint8_t* blk, int grp, Q4Raw& r) { q4_raw_load(blk, grp, r); }
__device__ __forceinline__ void mt_raw(const uint8_t* blk, int grp, Q6Raw& r) {
    const int h = grp >> 1, j = grp & 1;
    uint32_t a[4], b[4], c[4], s[2], d[1];
    lds_words<4>(blk + 64 * h + 16 * j, a);
    lds_words<4>(blk + 64 * h + 32 + 16 * j, b);
    lds_words<4>(blk + 128 + 32 * h + 16 * j, c);
    lds_words<2>(blk + 192 + 8 * h, s);
    d[0] = *reinterpret_cast<const uint16_t*>(blk + 208);
    r.la = make_uint4(a[0], a[1], a[2], a[3]);
    r.lb = make_uint4(b[0], b[1], b[2], b[3]);
    r.hq = make_uint4(c[0], c[1], c[2], c[3]);
    r.sc = make_uint2(s[0], s[1]);
    r.d = d[0];
}


// RT row tiles' raw Q6_K bytes of super-block sb (row r at w + r * row_bytes,
// rows from n_rows on: the last) into a wave's LDS, 14 16-byte chunks a row from
// the aligned-down start (a super-block's 210 bytes start 0..14 past it; every
// chunk holds a byte of it), then each lane's share.  LDS-direct loads write a
// lane's chunk at 16 * lane, so the copy is wlds[row * 224 + chunk * 16].
#define Q6_STAGE_ROW 224
template <int RT>
__device__ __forceinline__ void q6_stage_w(const uint8_t* w, size_t row_bytes, int sb, int row0, int n_rows,
                                           uint8_t* wlds, int lane) {
    constexpr int CH = Q6_STAGE_ROW / 16, TOTAL = RT * 16 * CH;
#pragma unroll
    for (int j = 0; j < (TOTAL + 63) / 64; ++j) {
        const int idx = j * 64 + lane, r = idx / CH, c = idx % CH;
        const uintptr_t p = reinterpret_cast<uintptr_t>(w + (size_t)min(row0 + r, n_rows - 1) * row_bytes +
                                                        (size_t)sb * Q6K_BYTES);
        if (idx < TOTAL)
            __builtin_amdgcn_global_load_lds(MT_GLOBAL((p & ~(uintptr_t)15) + 16 * c), MT_SHARED(wlds + j * 1024), 16,
                                             0, 0);
    }
}

// 16 columns' activations of super-block sb into a wave's LDS as fp16 rows of
// 256, 16-byte chunks permuted by chunk ^ column so an operand read's 16
// columns lie in distinct banks; columns past M stay as they are (results
// unused).  Consecutive lanes take consecutive bytes, and fp16 goes straight
// to LDS, holding no registers (wait for vmcnt before reading it).  The copy
// waits for the wave's reads of what it overwrites (their products have been
// issued by then, so the wait is free).
__device__ __forceinline__ void sb_stage_x(const __half* x, int K, int sb, int M, _Float16* lds, int lane) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(lane)::"memory");  // (and addresses made here, not kept across the loop)
    const int hi = lane >> 5, slot = lane & 31;
    const char* base = reinterpret_cast<const char*>(x + sb * QK_K);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (2 * j >= M) break;
        const uint32_t off = 2u * (uint32_t)(min(2 * j + hi, M - 1) * K) + 16u * (uint32_t)(slot ^ (2 * j + hi));
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off),
                                         (__attribute__((address_space(3))) void*)(lds + 2 * j * QK_K), 16, 0, 0);
    }
}
// The same through registers, for rows of any alignment (the reference-ABI
// symbols take any pointer; an LDS-direct load wants an aligned one).
__device__ __forceinline__ void sb_stage_x_any(const __half* x, int K, int sb, int M, _Float16* lds, int lane) {
    const int hi = lane >> 5, slot = lane & 31;
    uint4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
        v[j] = q6_ld16(reinterpret_cast<const uint8_t*>(x + (size_t)min(2 * j + hi, M - 1) * K + sb * QK_K +
                                                        8 * (slot ^ (2 * j + hi))));
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<uint4*>(lds + 2 * j * QK_K + 8 * lane) = v[j];
}
__device__ __forceinline__ void sb_stage_x(const float* x, int K, int sb, int M, _Float16* lds, int lane) {
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    float4 v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j)  // (a repeated row costs less than the branches that would skip it)
        v[j] = reinterpret_cast<const float4*>(x + (size_t)min(j, M - 1) * K + sb * QK_K)[lane];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int slot = (lane >> 1) ^ j;
        *reinterpret_cast<half4_t*>(lds + j * QK_K + 8 * slot + 4 * (lane & 1)) =
            half4_t{(_Float16)v[j].x, (_Float16)v[j].y, (_Float16)v[j].z, (_Float16)v[j].w};
    }
}

// The eight operands of a staged column tile.
template <int FMT, int NT>
__device__ __forceinline__ void sb_read_x(const _Float16* x, int col, int grp, half8_t (&bx)[8][NT]) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
        bx[t][0] = *reinterpret_cast<const half8_t*>(x + col * QK_K + 8 * ((kslot_base<FMT>(t, grp) >> 3) ^ col));
}

// One super-block of sb_mfma's work (minimum term per k-step) for RT row tiles
// and 16 staged columns, each k-step's operands made as they are needed.
template <int RT>
__device__ __forceinline__ void sb_staged(const Q4Raw (&r)[RT], const _Float16* x, int col, int grp,
                                          floatx4_t (&acc)[RT][1]) {
    floatx4_t aw[RT], am[RT];
    uint32_t sc[RT][2], mn[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        aw[rt] = am[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        q4_scale_words(r[rt].h, sc[rt]);
        q4_min_words(r[rt].h, mn[rt]);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int ci = t >> 2, part = (t >> 1) & 1, b = 2 * (grp >> 1) + part;
        const half8_t xv = *reinterpret_cast<const half8_t*>(x + col * QK_K + 8 * ((kslot_base<4>(t, grp) >> 3) ^ col));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const half2_t s2 = byte_splat(sc[rt][ci], b), m = byte_splat(mn[rt][ci], b);
            const half8_t wv = q4_step_operand(ci == 0 ? r[rt].q0 : r[rt].q1, part, t & 1, s2, s2 * splat2(-1024.0f));
            const half8_t mv = {m[0], m[1], m[0], m[1], m[0], m[1], m[0], m[1]};
            aw[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, wv, aw[rt], 0, 0, 0);
            am[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, mv, am[rt], 0, 0, 0);
        }
        if (t & 1) __builtin_amdgcn_sched_barrier(0);  // two steps' operands at a time, not all eight
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float d = h2f_bits(r[rt].h.x), dmin = h2f_bits(r[rt].h.x >> 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][0][i] = fmaf(-dmin, am[rt][i], fmaf(d, aw[rt][i], acc[rt][0][i]));
    }
}
template <int RT>
__device__ __forceinline__ void sb_staged(const Q6Raw (&r)[RT], const _Float16* x, int col, int grp,
                                          floatx4_t (&acc)[RT][1]) {
    floatx4_t aw[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) aw[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const half8_t xv = *reinterpret_cast<const half8_t*>(x + col * QK_K + 8 * ((kslot_base<6>(t, grp) >> 3) ^ col));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            aw[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, q6_step_operand(r[rt], t, grp), aw[rt], 0, 0, 0);
        if (t & 1) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][0][i] = fmaf(h2f_bits(r[rt].d), aw[rt][i], acc[rt][0][i]);
}

// C tile element of weight row rw (0..15) and batch column cc (0..15): lane
// rw + 16 * (cc / 4), register cc % 4.
__device__ __forceinline__ int c_lane(int rw, int cc) { return rw + 16 * (cc >> 2); }
__device__ __forceinline__ int c_reg(int cc) { return cc & 3; }

// Column groups for a weight-stationary launch of `tiles` row tiles over M
// batch columns, 32 at a time: each group re-reads and re-dequantises the
// weights, each block walks its group's 32-column chunks one after another,
// and `slots` blocks run at once.  Picks the group count with the least
// (rounds of blocks) x (chunks per block), weighted by 1 + groups / 16 for
// the repeated weight reads.
static inline int ws_column_groups(int tiles, int M, int slots) {
    const int chunks = (M + 31) / 32;
    if (const char* v = getenv("VTE_WS_GROUPS")) {  // tuning: pin the group count
        const int g = atoi(v);
        if (g >= 1) return g < chunks ? g : chunks;
    }
    int best = 1;
    double best_cost = 1e30;
    for (int g = 1; g <= chunks; ++g) {
        const int per = (chunks + g - 1) / g;
        const int used = (chunks + per - 1) / per;  // groups that hold columns
        const int rounds = (tiles * used + slots - 1) / slots;
        const double cost = (double)rounds * per * (1.0 + used / 16.0);
        if (cost < best_cost - 1e-9) {
            best_cost = cost;
            best = used;
        }
    }
    return best;
}
