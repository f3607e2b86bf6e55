// Tiled quantised GEMM for batches above 32 columns (prompt chunks), gfx950.
//
// A block of MT_WAVES waves owns MT_WAVES x 32 weight rows and 16 * NT batch
// columns.  Per super-block (256 of K) the columns' activations and each
// wave's raw weight blocks are copied to LDS with 16-byte LDS-direct loads of
// consecutive addresses (an MFMA operand's own lane order, 16 rows apart in
// neighbouring lanes, costs one address cycle per lane: reading Q6_K weights
// that way took half of the kernel), every wave turns its two 16-row tiles
// into exact MFMA operands once and runs them against all NT column tiles, so
// a super-block is decoded once per 16 * NT columns and an activation operand
// read from LDS serves two row tiles.  The next super-block's raw weights are
// requested as soon as this one's are decoded; the blocks of a CU overlap one
// block's copies with another's products.
//
// Q4_K's minimum term needs the activations' sub-block sums (XMin): the waves
// share the column tiles, each tile's sums are formed once per block and
// super-block and read by every wave.
//
// Sums: one C tile per super-block (its eight k-steps in order, then the fp32
// scales), added to the running sum in super-block order.  That is the order
// of the kernels that give every super-block of a split its own wave and add
// the waves in order, so the results have the same bits as theirs; where a wave
// of theirs sums several super-blocks (a share of K above 2048) it folds them
// into one fma chain, and the results agree to fp32 rounding.
#pragma once
#include "mfma_deq.h"

#define MT_WAVES 4
#define MT_ROWS (32 * MT_WAVES)

// Raw bytes of one row's super-block in LDS: Q4_K 9 chunks of 16 bytes; Q6_K
// the 14 aligned chunks that hold its 210 bytes (blocks are 2-byte aligned).
template <int FMT>
struct MtRaw {
    static constexpr int BPB = FMT == 4 ? Q4K_BYTES : Q6K_BYTES;
    static constexpr int CHUNKS = FMT == 4 ? 9 : 14;
    static constexpr int ROUNDS = (32 * CHUNKS + 63) / 64;  // loads of a wave for its 32 rows
};

// LDS of one block: activations [16 NT][256] fp16, 16-byte chunks of a row
// permuted by chunk ^ (row & 15) so the 16 rows an operand read touches lie in
// distinct banks; sub-block sums [16 NT] x fp16 hi[8], lo[8]; each wave's raw
// weights.  The C tile of the epilogue overlays them, columns of MT_LDC floats.
#define MT_LDC (MT_ROWS + 4)
#define MT_CT 4  // column tiles of an epilogue pass
template <int NT, int WCH>
struct alignas(16) MtLds {
    union {
        struct {
            _Float16 x[16 * NT * 256];
            _Float16 xs[16 * NT * 16];
            uint8_t w[MT_WAVES][32 * WCH * 16];
        };
        float c[16 * (NT < MT_CT ? NT : MT_CT) * MT_LDC];
    };
};

// Activations of super-block sb, columns c0 .. c0 + 16 NT - 1 (past M: column
// M - 1, results unused), into LDS.  A wave's load fills two rows.  Where all
// columns exist the row advance is scalar and a lane keeps two offsets.
template <int NT>
__device__ __forceinline__ void mt_stage(const __half* x, int K, int sb, int c0, int M, _Float16* lds, int wv,
                                         int lane) {
    constexpr int STEP = 2 * MT_WAVES;  // rows per round of the block's waves
    static_assert(STEP == 8, "rows of a lane alternate between two values of row & 15");
    const int r = 2 * wv + (lane >> 5), slot = lane & 31;
    if (c0 + 16 * NT <= M) {
        const char* base = reinterpret_cast<const char*>(x + (size_t)c0 * K + sb * QK_K);
        const uint32_t off[2] = {2u * (uint32_t)(r * K + 8 * (slot ^ r)), 2u * (uint32_t)(r * K + 8 * (slot ^ (r + 8)))};
#pragma unroll
        for (int j = 0; j < 16 * NT / STEP; ++j)
            __builtin_amdgcn_global_load_lds(MT_GLOBAL(base + (size_t)j * STEP * 2 * K + off[j & 1]),
                                             MT_SHARED(lds + (j * STEP + 2 * wv) * 256), 16, 0, 0);
        return;
    }
#pragma unroll 1
    for (int j = 0; j < 16 * NT / STEP; ++j) {
        const int row = j * STEP + r;
        const __half* src = x + (size_t)min(c0 + row, M - 1) * K + sb * QK_K + 8 * (slot ^ (row & 15));
        __builtin_amdgcn_global_load_lds(MT_GLOBAL(src), MT_SHARED(lds + (j * STEP + 2 * wv) * 256), 16, 0, 0);
    }
}
template <int NT>
__device__ __forceinline__ void mt_stage(const float* x, int K, int sb, int c0, int M, _Float16* lds, int wv,
                                         int lane) {
#pragma unroll
    for (int j = 0; j < 16 * NT / (2 * MT_WAVES); ++j) {
        const int row = (j * MT_WAVES + wv) * 2 + (lane >> 5), slot = lane & 31;
        const int chunk = slot ^ (row & 15);
        const half8_t v = load_x8<float>(x + (size_t)min(c0 + row, M - 1) * K + sb * QK_K + 8 * chunk, true);
        *reinterpret_cast<half8_t*>(lds + row * 256 + 8 * slot) = v;
    }
}

// Sub-block sums of column tile nt (q4_xmin's sums), shared by the block: the
// indicators are the A operand, so a lane gets four sub-blocks of one column.
template <int NT, int WCH>
__device__ __forceinline__ void mt_xsum(MtLds<NT, WCH>& L, int nt, int col, int grp) {
    asm volatile("" : "+v"(col));  // the indicators are rebuilt here, not kept in registers across the products
    floatx4_t cx = {0.f, 0.f, 0.f, 0.f};
    half8_t b[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
        b[t] = *reinterpret_cast<const half8_t*>(L.x + (nt * 16 + col) * 256 + 8 * ((kslot_base<4>(t, grp) >> 3) ^ col));
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int sub = 2 * ((grp >> 1) + 2 * (t >> 2)) + ((t >> 1) & 1);
        const _Float16 one = col == sub ? (_Float16)1.0f : (_Float16)0.0f;
        const half8_t ind = {one, one, one, one, one, one, one, one};
        cx = __builtin_amdgcn_mfma_f32_16x16x32_f16(ind, b[t], cx, 0, 0, 0);
    }
    if (grp < 2) {  // lane (column col, grp): sub-blocks 4 grp .. 4 grp + 3
        typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
        half4_t hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            hi[i] = (_Float16)cx[i];
            lo[i] = (_Float16)(cx[i] - (float)hi[i]);
        }
        _Float16* p = L.xs + (nt * 16 + col) * 16 + 4 * grp;
        *reinterpret_cast<half4_t*>(p) = hi;
        *reinterpret_cast<half4_t*>(p + 8) = lo;
    }
}

// acc += this super-block's scaled C tile.  The product with d, the fma of
// the minimum and the add round one after another (no contraction), as in the
// kernels whose waves each hold one super-block's sum.
__device__ __forceinline__ void mt_add(const Q4Ops& o, const floatx4_t& aw, const floatx4_t& am, floatx4_t& acc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float t = fmaf(-o.dmin, am[i], o.d * aw[i]);
        acc[i] = acc[i] + t;
    }
}
__device__ __forceinline__ void mt_add(const Q6Ops& o, const floatx4_t& aw, const floatx4_t&, floatx4_t& acc) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float t = o.d * aw[i];
        acc[i] = acc[i] + t;
    }
}

// Sums of a wave's two row tiles over super-blocks sb0 .. sb1 - 1 for the
// block's columns; row(r): the weight row (raw bytes of super-block 0) of the
// wave's tile row r, 0 <= r < 32.  xsum: some wave of the launch holds Q4_K
// rows (uniform over the block; every wave takes the same barriers).
template <int FMT, int NT, int WCH, typename TI, typename Row>
__device__ __forceinline__ void mt_loop(const TI* __restrict__ x, int K, int c0, int M, Row row, int sb0, int sb1,
                                        bool xsum, MtLds<NT, WCH>& L, floatx4_t (&acc)[2][NT]) {
    using W = MtRaw<FMT>;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // lane's operand chunks: row col of a column tile, k-step t
    // (Q4_K: steps 4..7 read 128 elements past steps 0..3)
    constexpr int XO = FMT == 4 ? 4 : 8;
    int xoff[XO];
#pragma unroll
    for (int t = 0; t < XO; ++t) xoff[t] = col * 256 + 8 * ((kslot_base<FMT>(t, grp) >> 3) ^ col);

    // the wave's raw weights of super-block sb -> L.w[wv], chunk c of row r at (r * CHUNKS + c) * 16
    const uint8_t* wp[W::ROUNDS];
    int wsh[2];  // Q6_K: bytes before the super-block in its first chunk
#pragma unroll
    for (int j = 0; j < W::ROUNDS; ++j) {
        const int idx = min(j * 64 + lane, 32 * W::CHUNKS - 1), r = idx / W::CHUNKS, c = idx % W::CHUNKS;
        wp[j] = row(r) + 16 * c;
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) wsh[rt] = FMT == 4 ? 0 : (int)(reinterpret_cast<uintptr_t>(row(16 * rt + col)) & 15);
    auto stage_w = [&](int sb) {
#pragma unroll
        for (int j = 0; j < W::ROUNDS; ++j) {
            const uint8_t* p = wp[j] + (size_t)sb * W::BPB;
            // aligned down, row by row: a row's chunk c starts 16 c past its first aligned chunk
            if (FMT != 4) p = reinterpret_cast<const uint8_t*>(reinterpret_cast<uintptr_t>(p) & ~(uintptr_t)15);
            if ((j + 1) * 64 <= 32 * W::CHUNKS || lane < 32 * W::CHUNKS - j * 64)
                __builtin_amdgcn_global_load_lds(MT_GLOBAL(p), MT_SHARED(&L.w[wv][j * 1024]), 16, 0, 0);
        }
    };
    stage_w(sb0);
    for (int sb = sb0; sb < sb1; ++sb) {
        mt_stage<NT>(x, K, sb, c0, M, L.x, wv, lane);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the LDS-direct loads of this wave
        __syncthreads();
        if (xsum) {
#pragma unroll
            for (int nt = 0; nt < NT; nt += MT_WAVES)
                if (nt + wv < NT) mt_xsum<NT, WCH>(L, nt + wv, col, grp);
        }
        typename SbRaw<FMT>::Ops ops[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            typename SbRaw<FMT>::Raw raw;
            const int sh = FMT == 4 ? 0 : (wsh[rt] + sb * W::BPB) & 15;
            mt_raw(&L.w[wv][(16 * rt + col) * W::CHUNKS * 16 + sh], grp, raw);
            sb_ops<true>(raw, grp, ops[rt]);
            __builtin_amdgcn_sched_barrier(0);  // one tile's temporaries at a time
        }
        // the raw weights are in registers (the operands depend on them): their LDS is free
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        stage_w(min(sb + 1, sb1 - 1));
        if (xsum) {  // the sums are in LDS; not __syncthreads, which would wait for the weights just requested
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
        // Products, half a super-block (four k-steps) at a time: under this half's
        // MFMAs the next half's operands are requested from LDS and a row tile of
        // the column tile before is scaled (an MFMA leaves two issue slots free
        // while it runs; the group barriers put the other instructions there).
        half8_t b0[4], b1[4], xa = {0, 0, 0, 0, 0, 0, 0, 0};
        auto fetch = [&](half8_t (&b)[4], int nt, int h) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                b[t] = *reinterpret_cast<const half8_t*>(L.x + nt * 16 * 256 + (FMT == 4 ? xoff[t] + 128 * h : xoff[4 * h + t]));
        };
        auto fetch_xs = [&](int nt) {  // groups 2, 3 read them too: their minima are zero
            if constexpr (FMT == 4) xa = *reinterpret_cast<const half8_t*>(L.xs + (nt * 16 + col) * 16 + 8 * (grp & 1));
        };
        auto interleave = [] {
#pragma unroll
            for (int i = 0; i < 10; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_s_setprio(1);
        floatx4_t aw[2], am[2], pw[2], pm[2];
        fetch_xs(0);
        fetch(b0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            fetch(b1, nt, 1);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                aw[rt] = am[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
                if constexpr (FMT == 4) am[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa, ops[rt].mins, am[rt], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    aw[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0[t], ops[rt].w[t], aw[rt], 0, 0, 0);
            if (nt > 0) mt_add(ops[0], pw[0], pm[0], acc[0][nt - 1]);
            interleave();
            if (nt + 1 < NT) {
                fetch_xs(nt + 1);
                fetch(b0, nt + 1, 0);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    aw[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b1[t], ops[rt].w[4 + t], aw[rt], 0, 0, 0);
            if (nt > 0) mt_add(ops[1], pw[1], pm[1], acc[1][nt - 1]);
            interleave();
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                pw[rt] = aw[rt];
                pm[rt] = am[rt];
            }
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) mt_add(ops[rt], pw[rt], pm[rt], acc[rt][NT - 1]);
        __builtin_amdgcn_s_setprio(0);
        // the products are done with this super-block's LDS
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last (repeated) weight copy, before the C tile reuses its LDS
}

// The block's C tile through LDS, MT_CT column tiles at a time: column m of a
// pass at L.c + m * MT_LDC, tile row r of wave w at element 32 w + r; then
// store(first column of the pass within the group, its columns).
template <int NT, int WCH, typename Store>
__device__ __forceinline__ void mt_epilogue(MtLds<NT, WCH>& L, const floatx4_t (&acc)[2][NT], Store store) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int p = 0; p < NT; p += MT_CT) {
        __syncthreads();  // the weight copies, or the pass before, are done with this LDS
#pragma unroll
        for (int nt = p; nt < NT && nt < p + MT_CT; ++nt)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    L.c[((nt - p) * 16 + 4 * grp + i) * MT_LDC + 32 * wv + 16 * rt + col] = acc[rt][nt][i];
        __syncthreads();
        store(16 * p, 16 * (NT - p < MT_CT ? NT - p : MT_CT));
    }
}

// Tile of a block: blocks go to the 8 XCDs round-robin, so XCD x takes the
// tiles x * per .. of the list (row block, column group), column groups
// innermost: equal shares, and a row block's weights come into one L2.
struct MtTile {
    int rb, cg;
};
__device__ __forceinline__ MtTile mt_tile(int idx, int row_blocks, int groups) {
    const int per = (row_blocks * groups + 7) / 8, i = (idx & 7) * per + (idx >> 3);
    return MtTile{i / groups, i % groups};
}
// Blocks of a launch (tiles rounded up to the XCD count; the surplus exits).
static inline int mt_grid(int row_blocks, int groups) { return (row_blocks * groups + 7) / 8 * 8; }

// Column tiles per block.  Four decode a super-block for the fewest
// instructions per column that still leave 8 waves per CU (gate/up of 17920
// rows, 512 columns: 67.5 / 57.0 / 58.3 us with 2 / 4 / 6); two where four give
// less than a block per CU (8960 -> 1536 in 5 splits, Q4_K, 256 columns: 21.3
// against 23.5 us); six where that saves a second round of two blocks per CU
// (gate/up, 256 columns: 30.8 against 36.6 us).
static inline int mt_pick_nt(int row_blocks, int splits, int M, int cus) {
    const auto blocks = [&](int nt) { return (long long)row_blocks * splits * ((M + 16 * nt - 1) / (16 * nt)); };
    if (blocks(4) < cus) return 2;
    return blocks(4) > 2 * cus && blocks(6) <= 2 * cus ? 6 : 4;
}

// Whether one tiled launch beats a launch per 32 columns whose waves split K.
// Always where its blocks (of 32 columns here) outnumber the CUs.  With fewer it
// still takes the super-blocks one after another, against launches that each
// cost a start and grow with the super-blocks and their columns (and with the
// rounds of their blocks): both linear, us, fitted to 3060 shapes of 33 to 200
// columns, where the form picked is at most 1.13 times the other (mean 1.001).
struct MtCost {
    float tile, tile_sb;                   // tiled: a + b n_sb
    float launch, launch_sb, launch_col;   // launches (c + d n_sb) + e n_sb M
};
// vte_gemm_mfma: Q6_K weights and fp32 activations take longer in either form;
// tall: 32-row blocks in the launches.
static inline MtCost mt_gemm_cost(bool q6, bool f32, bool tall) {
    return MtCost{3.5f, 1.5f + (q6 ? 0.25f : 0.f) + (f32 ? 0.25f : 0.f),
                  3.1f + (f32 ? 0.6f : 0.f) - (q6 ? 0.5f : 0.f) + (tall ? 0.55f : 0.f),
                  q6 ? (tall ? 0.47f : 0.29f) : (tall ? 0.25f : 0.19f), f32 ? 0.022f : 0.011f};
}
static inline bool mt_beats_launches(int row_blocks, int launch_blocks, int M, int n_sb, int cus, const MtCost& c) {
    const int launches = (M + 31) / 32;
    if ((long long)row_blocks * launches > cus) return true;
    const int rounds = (launch_blocks + cus - 1) / cus;
    return rounds * (launches * (c.launch + c.launch_sb * n_sb) + c.launch_col * n_sb * M) > c.tile + c.tile_sb * n_sb;
}
