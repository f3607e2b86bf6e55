// Batched (3 or more columns) projections with the decode-step glue fused in, on MFMA
// (gfx950).  One launch per group of projections that read the same
// (already RMSNorm-ed, fp16) activations:
//
//   q/k/v (+bias) -> RoPE(q, k) -> K/V cache append       => one launch
//   gate/up -> SwiGLU                                       => one launch
//
// (reference nodes: vte/compiler/qwen_compute.py:100-282, captured by
// vte/core/hip_graph_executor.py:504-738), with the rounding points of those
// nodes: projections (+bias) and rotated q/k are fp16 values computed in fp32,
// SwiGLU is fp16(g / (1 + exp(-g)) * u) on fp16 g and u
// (rope.hip.template:82-97, swiglu.hip.template:11-25).
//
// Tiles are 16 * RT weight rows; paired tiles hold 8 * RT rows and their
// partners (RoPE: d and d + 64 of one head; SwiGLU: gate row j and up row j),
// so a pair's two sums finish in the same block.  The weight operand of each
// lane comes from its tile row's weight row; everything else is the batched
// MFMA GEMM (waves split K, partial C tiles summed through LDS), whose k-slot
// map, exact operands and per-super-block scaling it shares (mfma_deq.h).
#include <cstdlib>
#include <cstring>

#include "mm_tile.h"

#define MM_MAX_SEG 3


enum MmMode : int {
    MM_STORE = 0,        // out[m][row] = fp16(acc + bias)
    MM_ROPE_Q = 2,       // fp16(acc + bias), rotated -> out (q [m][rows])
    MM_ROPE_KCACHE = 3,  // fp16(acc + bias), rotated -> k_cache at kv_offset[m]
    MM_VCACHE = 4,       // fp16(acc + bias) -> v_cache at kv_offset[m]
    MM_SWIGLU = 5,       // gate rows of w, up rows of w2: out[m][j] = fp16(silu(g) * u)
};

struct MmSeg {
    const uint8_t* w;
    const uint8_t* w2;   // up rows (SwiGLU)
    __half* out;
    const __half* bias;  // nullable
    int fmt;             // 4 = Q4_K, 6 = Q6_K
    int n_rows;          // output rows (SwiGLU: outputs, i.e. gate rows)
    int mode;
    int tiles;
    int row_bytes;
};

struct MmPlan {
    MmSeg seg[MM_MAX_SEG];
    int nseg;
    int K, M;            // activations [M][K] fp16, M <= 16 * NT in one launch
    const __half* x;
    const __half* rope_cos;
    const __half* rope_sin;
    const int* kv_offset;  // [M] positions of this launch's columns
    __half* k_cache;       // sequence m at k_cache + m * kv_batch_stride
    __half* v_cache;
    int kv_batch_stride;
    int n_kv;
};

__host__ __device__ __forceinline__ bool mm_paired(int mode) {
    return mode == MM_ROPE_Q || mode == MM_ROPE_KCACHE || mode == MM_SWIGLU;
}

// Tile of a block: `pr` pairs (paired) or 16*RT rows starting at j0.
struct MmTile {
    const MmSeg* S;
    int j0;      // first row (paired: first A row)
    int nvalid;  // valid rows (not paired) or pairs (paired)
};

template <int RT>
__device__ __forceinline__ MmTile mm_tile(const MmPlan& P, int g) {
    MmTile T;
    const int t0 = P.seg[0].tiles, t1 = P.seg[1].tiles;
    int s = 0;
    if (P.nseg > 1 && g >= t0) {
        g -= t0;
        s = 1;
        if (P.nseg > 2 && g >= t1) {
            g -= t1;
            s = 2;
        }
    }
    const MmSeg& S = P.seg[s];
    T.S = &P.seg[s];
    if (!mm_paired(S.mode)) {
        T.j0 = g * 16 * RT;
        T.nvalid = min(16 * RT, S.n_rows - T.j0);
    } else if (S.mode == MM_SWIGLU) {
        T.j0 = g * 8 * RT;
        T.nvalid = min(8 * RT, S.n_rows - T.j0);
    } else {  // RoPE: 8 * RT pairs (d, d + 64) of one 128-row head
        const int tph = 64 / (8 * RT);  // tiles per head
        T.j0 = (g / tph) * 128 + (g % tph) * 8 * RT;
        T.nvalid = 8 * RT;
    }
    return T;
}

// Weight row of tile row rr (past the valid rows: a valid row, results unused).
template <int RT>
__device__ __forceinline__ const uint8_t* mm_row(const MmTile& T, int rr) {
    const MmSeg& S = *T.S;
    if (!mm_paired(S.mode)) return S.w + (size_t)(T.j0 + min(rr, T.nvalid - 1)) * S.row_bytes;
    const int p = rr % (8 * RT), pc = min(p, T.nvalid - 1);
    if (rr < 8 * RT) return S.w + (size_t)(T.j0 + pc) * S.row_bytes;
    if (S.mode == MM_SWIGLU) return S.w2 + (size_t)(T.j0 + pc) * S.row_bytes;
    return S.w + (size_t)(T.j0 + 64 + pc) * S.row_bytes;
}

template <int FMT, int RT, int NT, int NW>
__device__ __forceinline__ void mm_body(const MmPlan& P, const MmTile& T, MfWave<RT, NT, NT == 1>* L) {
    constexpr bool XM = NT > 1;  // minimum-term form (q4_xmin)
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int K = P.K, M = P.M, n_sb = K / QK_K;
    const int sb0 = (n_sb * wv) / NW, sb1 = (n_sb * (wv + 1)) / NW;
    const __half* x = P.x;

    floatx4_t acc[RT][NT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    const uint8_t* rowp[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) rowp[rt] = mm_row<RT>(T, rt * 16 + col);

    for (int sb = sb0; sb < sb1; ++sb) {
        if constexpr (NT == 1) {  // staged activations: no registers in flight, so more blocks per CU
            sb_stage_x(x, K, sb, M, L[wv].x, lane);
            typename SbRaw<FMT>::Raw raw[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                sb_load(rowp[rt] + (size_t)sb * (FMT == 4 ? Q4K_BYTES : Q6K_BYTES), grp, raw[rt]);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            sb_staged<RT>(raw, L[wv].x, col, grp, acc);
            continue;
        } else {
        half8_t bx[8][NT];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int kb = sb * QK_K + kslot_base<FMT>(t, grp);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int m = nt * 16 + col;
                bx[t][nt] = load_x8<__half>(x + (size_t)(m < M ? m : 0) * K + kb, m < M);
            }
        }
        // weights requested before the minimum-term LDS round trip, whose
        // memory clobber would otherwise hold them back
        typename SbRaw<FMT>::Raw raw[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            sb_load(rowp[rt] + (size_t)sb * (FMT == 4 ? Q4K_BYTES : Q6K_BYTES), grp, raw[rt]);
        XMin<NT, XM> xm;
        sb_xmin<FMT, NT, XM>(bx, L[wv].xl, xm);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            typename SbRaw<FMT>::Ops ops;
            sb_ops<XM>(raw[rt], grp, ops);
            sb_mfma<NT>(ops, bx, xm, acc[rt]);
        }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) L[wv].red[rt][nt][i][lane] = acc[rt][nt][i];
}

// Sum over the NW waves of tile row rr, batch column mc (C layout: lane
// (row rw, grp) holds batch columns 4*grp+i of a 16-column tile).
template <int RT, int NT, int NW, bool ST>
__device__ __forceinline__ float mm_sum(const MfWave<RT, NT, ST>* L, int rr, int mc) {
    const int rt = rr >> 4, rw = rr & 15, nt = mc >> 4, cc = mc & 15;
    const int ln = c_lane(rw, cc), i = c_reg(cc);
    float s = 0.f;
#pragma unroll
    for (int wq = 0; wq < NW; ++wq) s += L[wq].red[rt][nt][i][ln];
    return s;
}

__device__ __forceinline__ float mm_bias(const __half* b, int row) { return b ? __half2float(b[row]) : 0.f; }

// g / (1 + e^-g) with the library's exponential and a division, as every other
// SwiGLU of the decode path.  The hardware's exponential and reciprocal are
// faster (gate/up of 512 columns of 8960: 53.1 against 54.9 us), but several
// fp32 units off for gates of -8 and below, which flips fp16 results.
__device__ __forceinline__ float mm_silu(float g) { return g / (1.0f + expf(-g)); }

// Epilogue of one output (row, batch column m of the launch: position
// kv_offset[m], row m of the outputs) from its sum.
__device__ __forceinline__ void mm_put(const MmPlan& P, const MmSeg& S, int row, int m, float sum) {
    const __half v = __float2half(sum + mm_bias(S.bias, row));
    if (S.mode == MM_VCACHE) {
        const int pos = P.kv_offset[m];
        P.v_cache[(size_t)m * P.kv_batch_stride + ((size_t)pos * P.n_kv + row / 128) * 128 + (row % 128)] = v;
    } else {
        S.out[(size_t)m * S.n_rows + row] = v;
    }
}
// The same for a pair: gate row and up row `row`, or rows `row`, `row` + 64 of one head.
__device__ __forceinline__ void mm_put_pair(const MmPlan& P, const MmSeg& S, int row, int m, float a, float b) {
    if (S.mode == MM_SWIGLU) {
        const float g = __half2float(__float2half(a)), u = __half2float(__float2half(b));
        S.out[(size_t)m * S.n_rows + row] = __float2half(mm_silu(g) * u);
        return;
    }
    const float x1 = __half2float(__float2half(a + mm_bias(S.bias, row)));
    const float x2 = __half2float(__float2half(b + mm_bias(S.bias, row + 64)));
    const int pos = P.kv_offset[m], d = row & 127;
    const float c = __half2float(P.rope_cos[(size_t)pos * 128 + d]);
    const float sn = __half2float(P.rope_sin[(size_t)pos * 128 + d]);
    const __half o1 = __float2half(x1 * c - x2 * sn), o2 = __float2half(x1 * sn + x2 * c);
    if (S.mode == MM_ROPE_Q) {
        S.out[(size_t)m * S.n_rows + row] = o1;
        S.out[(size_t)m * S.n_rows + row + 64] = o2;
    } else {
        __half* kc = P.k_cache + (size_t)m * P.kv_batch_stride + ((size_t)pos * P.n_kv + row / 128) * 128;
        kc[d] = o1;
        kc[d + 64] = o2;
    }
}

// Epilogue of a block's C tiles: batch columns cb .. cb + mcount - 1.
// Neighbouring lanes take neighbouring rows: contiguous stores, and LDS reads
// of distinct banks.
template <int RT, int NT, int NW, bool ST>
__device__ __forceinline__ void mm_epilogue(const MmPlan& P, const MmTile& T, const MfWave<RT, NT, ST>* L, int cb,
                                            int mcount) {
    const MmSeg& S = *T.S;
    if (!mm_paired(S.mode)) {
        for (int o = threadIdx.x; o < 16 * RT * 16 * NT; o += blockDim.x) {
            const int rr = o % (16 * RT), mc = o / (16 * RT);
            if (rr < T.nvalid && mc < mcount) mm_put(P, S, T.j0 + rr, cb + mc, mm_sum<RT, NT, NW>(L, rr, mc));
        }
        return;
    }
    for (int o = threadIdx.x; o < 8 * RT * 16 * NT; o += blockDim.x) {
        const int p = o % (8 * RT), mc = o / (8 * RT);
        if (p < T.nvalid && mc < mcount)
            mm_put_pair(P, S, T.j0 + p, cb + mc, mm_sum<RT, NT, NW>(L, p, mc),
                        mm_sum<RT, NT, NW>(L, p + 8 * RT, mc));
    }
}

// NW waves per block split K (6 for K = 1536: one super-block each).
template <int RT, int NT, int NW, bool Q6>
__global__ __launch_bounds__(64 * NW, RT == 2 && NT == 1 && NW == 6 ? 5 : 1) void fused_mm_kernel(MmPlan P) {
    __shared__ MfWave<RT, NT, NT == 1> L[NW];
    const MmTile T = mm_tile<RT>(P, blockIdx.x);
    const MmSeg& S = *T.S;
    if (!Q6 || S.fmt == 4) mm_body<4, RT, NT, NW>(P, T, L);
    else mm_body<6, RT, NT, NW>(P, T, L);
    __syncthreads();

    mm_epilogue<RT, NT, NW>(P, T, L, 0, P.M);
}


// Weight-stationary form for batches above 32 columns with few row tiles, K = 6
// super-blocks:
// wave w decodes super-block w of its tile rows once, keeps the weight
// operands in registers and runs them against the block's columns
// [blockIdx.y * cols, ...) 16 at a time, the next columns' activations
// requested ahead.  Each C tile sums
// its eight k-steps in the same order as fused_mm_kernel, so both forms give
// the same bits.
template <int FMT, int RT>
__device__ __forceinline__ void mm_ws_body(const MmPlan& P, const MmTile& T, MfWave<RT, 1, false>* L,
                                           _Float16 (*xb)[16 * QK_K], int c0, int c1) {
    constexpr bool XM = true;  // minimum-term form (q4_xmin)
    constexpr int NW = 6, NT = 1;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int K = P.K;
    typename SbRaw<FMT>::Ops ops[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint8_t* rowp = mm_row<RT>(T, rt * 16 + col);
        typename SbRaw<FMT>::Raw raw;
        sb_load(rowp + (size_t)wv * (FMT == 4 ? Q4K_BYTES : Q6K_BYTES), grp, raw);
        sb_ops<XM>(raw, grp, ops[rt]);
    }
    auto load_b = [&](int m0) { sb_stage_x(P.x + (size_t)m0 * K, K, wv, c1 - m0, xb[wv], lane); };
    load_b(c0);
    for (int m0 = c0; m0 < c1; m0 += 16 * NT) {
        floatx4_t acc[RT][NT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        half8_t bx[8][NT];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies; no other wave reads them
        sb_read_x<FMT>(xb[wv], col, grp, bx);
        if (m0 + 16 < c1) load_b(m0 + 16);
        XMin<NT, XM> xm;
        sb_xmin<FMT, NT, XM>(bx, L[wv].xl, xm);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) sb_mfma<NT>(ops[rt], bx, xm, acc[rt]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) L[wv].red[rt][nt][i][lane] = acc[rt][nt][i];
        __syncthreads();
        mm_epilogue<RT, NT, NW>(P, T, L, m0, min(16 * NT, c1 - m0));
        __syncthreads();
    }
}

template <int RT>
__global__ __launch_bounds__(64 * 6) void fused_mm_ws_kernel(MmPlan P, int cols) {
    __shared__ MfWave<RT, 1, false> L[6];
    __shared__ alignas(16) _Float16 xb[6][16 * QK_K];
    const MmTile T = mm_tile<RT>(P, blockIdx.x);
    const int c0 = blockIdx.y * cols, c1 = min(P.M, c0 + cols);
    if (c0 >= c1) return;
    if (T.S->fmt == 4) mm_ws_body<4, RT>(P, T, L, xb, c0, c1);
    else mm_ws_body<6, RT>(P, T, L, xb, c0, c1);
}

// Eight SwiGLU outputs of column m from the sums of eight gate and up rows.
__device__ __forceinline__ half8_t mm_swiglu8(const float* g, const float* u) {
    half8_t v;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float a = __half2float(__float2half(g[e])), b = __half2float(__float2half(u[e]));
        v[e] = (_Float16)(mm_silu(a) * b);
    }
    return v;
}

// Long batches (prompt chunks): the tiled main loop of mm_tile.h, each wave on
// one 32-row tile (16 pairs, or 32 rows) of the plan.  SwiGLU launches store
// through LDS in 16-byte pieces (2-byte stores of 16 neighbouring rows took
// 13 of 78 us at 512 columns of 8960); the other modes store from the
// accumulators, where a pair's two sums are in one lane.
// WCH: chunks per staged weight row (9: Q4_K only, 14: some segment is Q6_K);
// SW: the SwiGLU plan.
template <int NT, int WCH, bool SW>
__global__ __launch_bounds__(64 * MT_WAVES, 2) void fused_mm_tile_kernel(
    MmPlan P, int row_blocks, int groups, int total) {
    __shared__ MtLds<NT, WCH> L;
    const MtTile bt = mt_tile(blockIdx.x, row_blocks, groups);
    if (bt.rb >= row_blocks) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int g = bt.rb * MT_WAVES + wv, c0 = bt.cg * 16 * NT;
    const MmTile T = mm_tile<2>(P, min(g, total - 1));  // waves past the last tile repeat it and store nothing
    const MmSeg& S = *T.S;
    const auto row = [&](int r) { return mm_row<2>(T, r); };
    floatx4_t acc[2][NT];
    if (WCH == 9 || __builtin_amdgcn_readfirstlane(S.fmt) == 4)
        mt_loop<4, NT, WCH>(P.x, P.K, c0, P.M, row, 0, P.K / QK_K, true, L, acc);
    else
        mt_loop<6, NT, WCH>(P.x, P.K, c0, P.M, row, 0, P.K / QK_K, true, L, acc);
    if constexpr (SW) {
        const MmSeg& S0 = P.seg[0];
        const bool vec = S0.n_rows % 8 == 0 && (reinterpret_cast<uintptr_t>(S0.out) & 15) == 0;
        mt_epilogue<NT, WCH>(L, acc, [&](int p0, int pc) {
            for (int o = threadIdx.x; o < pc * 2 * MT_WAVES; o += 64 * MT_WAVES) {
                const int mc = o / (2 * MT_WAVES), ch = o % (2 * MT_WAVES), m = c0 + p0 + mc;
                const int j = bt.rb * 16 * MT_WAVES + 8 * ch;
                if (m >= P.M || j >= S0.n_rows) continue;
                const float* c = L.c + mc * MT_LDC + 32 * (ch >> 1) + 8 * (ch & 1);
                const half8_t v = mm_swiglu8(c, c + 16);
                _Float16* dst = reinterpret_cast<_Float16*>(S0.out) + (size_t)m * S0.n_rows + j;
                if (vec) {
                    *reinterpret_cast<half8_t*>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (j + e < S0.n_rows) dst[e] = v[e];
                }
            }
        });
        return;
    }
    if (g >= total) return;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = c0 + nt * 16 + 4 * grp + i;
            if (m >= P.M) continue;
            if (!mm_paired(S.mode)) {
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    if (16 * rt + col < T.nvalid) mm_put(P, S, T.j0 + 16 * rt + col, m, acc[rt][nt][i]);
            } else if (col < T.nvalid) {
                mm_put_pair(P, S, T.j0 + col, m, acc[0][nt][i], acc[1][nt][i]);
            }
        }
}

namespace vte {

static MmSeg mm_seg(const void* w, const void* w2, void* out, const void* bias, int fmt, int n_rows, int mode, int K,
                    int RT) {
    MmSeg S;
    memset(&S, 0, sizeof(S));
    S.w = (const uint8_t*)w;
    S.w2 = (const uint8_t*)w2;
    S.out = (__half*)out;
    S.bias = (const __half*)bias;
    S.fmt = fmt;
    S.n_rows = n_rows;
    S.mode = mode;
    S.row_bytes = (K / QK_K) * (fmt == 4 ? Q4K_BYTES : Q6K_BYTES);
    if (mode == MM_SWIGLU) S.tiles = (n_rows + 8 * RT - 1) / (8 * RT);
    else if (mode == MM_ROPE_Q || mode == MM_ROPE_KCACHE) S.tiles = n_rows / (8 * RT) / 2;
    else S.tiles = (n_rows + 16 * RT - 1) / (16 * RT);
    return S;
}

static int mm_env(const char* name, int dflt) {
    const char* v = getenv(name);
    return v ? atoi(v) : dflt;
}

// Launch form of a batch of B columns, `tiles` 32-row tiles in all.  Above 32
// columns at K = 6 super-blocks the weight-stationary form, whose six waves each
// take a super-block, against the tiled one (the same bits there).  Its time goes
// with the 16-column steps that a CU takes one after another in blocks of 64 rows
// (a further round of blocks, which decodes its weights again, costs one more):
// gate/up 9.5 / 11.1 / 13.8 / 16.3 / 18.2 us for 2 / 3 / 4 / 5 / 6 steps, where the
// tiled form takes 12.8-14.2 with up to a block (of 128 rows x 32 columns) per CU and
// 17.7-18.9 with up to two; q/k/v 12.4 / 17.1 / 21.8 / 26.8 for 2 / 4 / 6 / 8 against
// 20-21, 24-25 and 28.5 beyond with Q6_K rows, 16.5 and 21.5 without.  Up to 128
// columns q/k/v takes smaller blocks (8.5 us at 2048 rows, where the tiled form
// takes 19), while the tiled form would not fill the chip.  Other K as in
// mt_beats_launches.
// VTE_MM_WS=0 selects the 32-column launches for every batch.
enum MmForm { MM_COLS32, MM_WS, MM_TILED };
static MmForm mm_form(int B, int tiles, int K, bool swiglu, bool q6) {
    if (B <= 32 || mm_env("VTE_MM_WS", 1) == 0) return MM_COLS32;
    const int row_blocks = (tiles + MT_WAVES - 1) / MT_WAVES, chunks = (B + 31) / 32, cus = device_cus();
    if (K == 6 * QK_K) {
        const int ws_tiles = (tiles + 1) / 2, g = ws_column_groups(ws_tiles, B, cus);
        const int cols = (chunks + g - 1) / g * 32, gy = (B + cols - 1) / cols, rounds = (ws_tiles * gy + cus - 1) / cus;
        const int full = ((B < cols ? B : cols) + 15) / 16, last = (B - (gy - 1) * cols + 15) / 16;
        const int steps = (rounds - 1) * (full + 1) + (ws_tiles * (gy - 1) <= cus * (rounds - 1) ? last : full);
        const bool fills = (long long)row_blocks * chunks > cus;
        if (!swiglu && B <= 128) return fills ? MM_TILED : MM_WS;
        return steps <= (q6 ? 5 : 3) + (fills ? 2 : 0) ? MM_WS : MM_TILED;
    }
    // (the launches' blocks: 24 pairs of gate/up rows, 16 rows of q/k/v; RoPE and
    // the cache writes cost the tiled form more than the small blocks)
    const MtCost cost = swiglu ? MtCost{3.9f, 1.55f, 5.1f, 0.3f, 0.008f} : MtCost{7.1f, 1.98f, 4.0f, 0.2f, 0.0105f};
    return mt_beats_launches(row_blocks, swiglu ? (tiles * 2 + 2) / 3 : 2 * tiles, B, K / QK_K, cus, cost) ? MM_TILED
                                                                                                          : MM_COLS32;
}
static hipError_t mm_run_tiled(MmPlan P, int B, hipStream_t st) {
    int total = 0;
    for (int s = 0; s < P.nseg; ++s) total += P.seg[s].tiles;
    P.M = B;
    const int rbs = (total + MT_WAVES - 1) / MT_WAVES, nt = mt_pick_nt(rbs, 1, B, device_cus());
    const int groups = (B + 16 * nt - 1) / (16 * nt);
    bool q6 = false;
    for (int s = 0; s < P.nseg; ++s) q6 = q6 || P.seg[s].fmt != 4;
#define MM_LAUNCH(NT_, W_, SW_) \
    hipLaunchKernelGGL((fused_mm_tile_kernel<NT_, W_, SW_>), dim3(mt_grid(rbs, groups)), dim3(64 * MT_WAVES), 0, st, P, \
                       rbs, groups, total)
#define MM_LAUNCH_NT(W_, SW_)            \
    do {                                 \
        if (nt == 6) MM_LAUNCH(6, W_, SW_); \
        else if (nt == 4) MM_LAUNCH(4, W_, SW_); \
        else MM_LAUNCH(2, W_, SW_);      \
    } while (0)
    if (P.seg[0].mode == MM_SWIGLU) MM_LAUNCH_NT(9, true);  // gate/up: Q4_K
    else if (q6) MM_LAUNCH_NT(14, false);
    else MM_LAUNCH_NT(9, false);
#undef MM_LAUNCH_NT
#undef MM_LAUNCH
    return hipGetLastError();
}

// Runs the plan over the batch: in chunks of 32 columns (one launch each), or
// in one weight-stationary launch.
template <int RT>
static hipError_t mm_run(MmPlan P, int B, MmForm form, size_t out_ld_elems[MM_MAX_SEG], hipStream_t st) {
    int total = 0;
    for (int s = 0; s < P.nseg; ++s) total += P.seg[s].tiles;
    const __half* x0 = P.x;
    const int* ko0 = P.kv_offset;
    __half* out0[MM_MAX_SEG];
    for (int s = 0; s < P.nseg; ++s) out0[s] = P.seg[s].out;
    __half* kc0 = P.k_cache;
    __half* vc0 = P.v_cache;
    bool q6 = false;
    for (int s = 0; s < P.nseg; ++s) q6 = q6 || P.seg[s].fmt != 4;
    if constexpr (RT != 3) if (form == MM_WS) {
        // 64 rows per block: one block per CU; fewer: two
        const int g = ws_column_groups(total, B, (RT == 4 ? 1 : 2) * device_cus());
        const int cols = ((B + 31) / 32 + g - 1) / g * 32, gy = (B + cols - 1) / cols;
        P.M = B;
        hipLaunchKernelGGL((fused_mm_ws_kernel<RT>), dim3(total, gy), dim3(64 * 6), 0, st, P, cols);
        return hipGetLastError();
    }
    for (int m0 = 0; m0 < B; m0 += 32) {
        const int mc = B - m0 < 32 ? B - m0 : 32;
        P.M = mc;
        P.x = x0 + (size_t)m0 * P.K;
        P.kv_offset = ko0 ? ko0 + m0 : nullptr;
        for (int s = 0; s < P.nseg; ++s) P.seg[s].out = out0[s] ? out0[s] + (size_t)m0 * out_ld_elems[s] : nullptr;
        P.k_cache = kc0 ? kc0 + (size_t)m0 * P.kv_batch_stride : nullptr;
        P.v_cache = vc0 ? vc0 + (size_t)m0 * P.kv_batch_stride : nullptr;
        // batches above 16 columns take the two-tile form for every chunk, a
        // short tail included, so all their columns share the minimum-term
        // form (and the bits) of the weight-stationary launch
#define MM_LAUNCH(NT_, NW_, Q6_) \
    hipLaunchKernelGGL((fused_mm_kernel<RT, NT_, NW_, Q6_>), dim3(total), dim3(64 * NW_), 0, st, P)
#define MM_LAUNCH_Q(NT_, NW_)                    \
    do {                                         \
        if (q6) MM_LAUNCH(NT_, NW_, true);       \
        else MM_LAUNCH(NT_, NW_, false);         \
    } while (0)
        if (P.K == 6 * QK_K) {
            if (B > 16) MM_LAUNCH_Q(2, 6);
            else MM_LAUNCH_Q(1, 6);
        } else {
            if (B > 16) MM_LAUNCH_Q(2, MF_WAVES);
            else MM_LAUNCH_Q(1, MF_WAVES);
        }
#undef MM_LAUNCH_Q
#undef MM_LAUNCH
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// q/k/v projections of RMSNorm-ed fp16 activations xn [B][K] with bias, RoPE
// on q and k, and the K/V rows written at kv_offset[b]; q_out [B][n_q*128].
hipError_t qkv_mm(const void* xn, const void* wq, const void* q_bias, int fmt_q, const void* wk, const void* k_bias,
                  int fmt_k, const void* wv, const void* v_bias, int fmt_v, void* q_out, void* k_cache, void* v_cache,
                  const int* kv_offset, int kv_batch_stride, const void* rope_cos, const void* rope_sin, int B, int K,
                  int n_q, int n_kv, hipStream_t st) {
    const MmForm form = mm_form(B, (n_q + 2 * n_kv) * 4, K, false, fmt_v != 4);
    // weight-stationary: 16, 32 or 64 rows per block up to 64, 128 and more
    // columns (2048 rows; 64 / 128 / 256 columns: 6.7 / 11.6 / 19.7 us with 16 rows,
    // 8.1 / 8.3 / 14.6 with 32, 11.5 / 11.6 / 11.7 with 64)
    const int ws_rt = B > 128 ? 4 : B > 64 ? 2 : 1;
    const int RT = form == MM_TILED ? 2 : mm_env("VTE_MM_RT_QKV", form == MM_WS ? ws_rt : 1);
    MmPlan P;
    memset(&P, 0, sizeof(P));
    P.K = K;
    P.x = (const __half*)xn;
    P.seg[0] = mm_seg(wq, nullptr, q_out, q_bias, fmt_q, n_q * 128, MM_ROPE_Q, K, RT);
    P.seg[1] = mm_seg(wk, nullptr, nullptr, k_bias, fmt_k, n_kv * 128, MM_ROPE_KCACHE, K, RT);
    P.seg[2] = mm_seg(wv, nullptr, nullptr, v_bias, fmt_v, n_kv * 128, MM_VCACHE, K, RT);
    P.nseg = 3;
    P.rope_cos = (const __half*)rope_cos;
    P.rope_sin = (const __half*)rope_sin;
    P.kv_offset = kv_offset;
    P.k_cache = (__half*)k_cache;
    P.v_cache = (__half*)v_cache;
    P.kv_batch_stride = kv_batch_stride;
    P.n_kv = n_kv;
    if (form == MM_TILED) return mm_run_tiled(P, B, st);
    size_t ld[MM_MAX_SEG] = {(size_t)n_q * 128, 0, 0};
    return RT == 4   ? mm_run<4>(P, B, form, ld, st)
           : RT == 2 ? mm_run<2>(P, B, form, ld, st)
                     : mm_run<1>(P, B, form, ld, st);
}

// out [B][ffn] = fp16(silu(W_gate xn) * (W_up xn)) for RMSNorm-ed fp16 xn [B][K].
hipError_t gate_up_mm(const void* xn, const void* w_gate, const void* w_up, int fmt, void* out, int B, int K, int ffn,
                      hipStream_t st) {
    // 16 gate/up pairs per block (half the blocks of 8, activations read half
    // as often); 24 for 17-32 columns (measured: batch 32 2.26 -> 2.18 ms per
    // step, batch 8-16 slightly slower); 32 in the weight-stationary form
    const MmForm form = mm_form(B, (ffn + 15) / 16, K, true, false);
    const int RT = form == MM_TILED ? 2 : mm_env("VTE_MM_RT_FFN", form == MM_WS ? 4 : B > 16 ? 3 : 2);
    MmPlan P;
    memset(&P, 0, sizeof(P));
    P.K = K;
    P.x = (const __half*)xn;
    P.seg[0] = mm_seg(w_gate, w_up, out, nullptr, fmt, ffn, MM_SWIGLU, K, RT);
    P.nseg = 1;
    if (form == MM_TILED) return mm_run_tiled(P, B, st);
    size_t ld[MM_MAX_SEG] = {(size_t)ffn, 0, 0};
    return RT == 4   ? mm_run<4>(P, B, form, ld, st)
           : RT == 3 ? mm_run<3>(P, B, form, ld, st)
           : RT == 2 ? mm_run<2>(P, B, form, ld, st)
                     : mm_run<1>(P, B, form, ld, st);
}

}  // namespace vte
