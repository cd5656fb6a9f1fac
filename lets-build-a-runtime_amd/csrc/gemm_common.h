// gemm_common.h — what the GEMM kernels share: their arguments, the tile order and
// the epilogue of the LDS-tiled kernels (gemm.hip, gemm_split.hip).
#pragma once

#include "lbr_device.h"

#include <algorithm>

constexpr int N_XCD = 8;
constexpr int GROUP_M = 8;   // tile rows per L2 group

struct GemmArgs {
    const float* A;
    const float* B;
    float* C;
    const float* bias;
    int M, N, K;
    long long sA, sB, sC;     // batch strides (elements)
    float alpha;
    int tiles_m, tiles_n;
    float* W;                 // split-K partial sums [ksplit][batches][M][N] (ksplit > 1)
    int ksplit, kchunk;       // number of K ranges, K per range (multiple of BK)
    // Fused epilogues (set only by the plan's peephole fusion; all null/0 otherwise).
    const float* resid;       // C += resid (same layout as C): a following same-shape ADD
    int n_split;              // >0: C columns are scattered as attention heads, see epi_store
    int col_begin[5];         // split k owns columns [col_begin[k], col_begin[k+1])
    float* dst[4];            // split k's output, laid out [B, H, S, hd]
    const float* sbias[4];    // split k's bias row (indexed by column - col_begin[k]) or null
    int Hs[4], hd, S;         // heads of each split, head dim, rows per batch (M = B·S)
    int frag;                 // bit k: split k is stored fragment-major (lbr_frag_offset)
    // Head prologue in the epilogue (lbr_merge_gemm_head_prologue; 64×128 DMA tile, hd =
    // 128 = TN): C columns [hp_col[p], hp_col[p] + hp_H[p]·128) of part p hold heads of
    // 128; each tile's C values (+ bias) go round through LDS, get the part's bias,
    // per-head RMSNorm (weight hp_w[p], eps hp_eps[p]) and rotate-half RoPE (cos/sin row
    // of token (b, s) at b·hp_tst[0] + s·hp_tst[1]) and are stored as [B, H, S, 128] at
    // hp_out[p] (C's columns of the parts are not written); hp_flags: 1 norm, 2 RoPE
    int hp_parts, hp_flags, hp_S;
    int hp_col[2], hp_H[2];
    float* hp_out[2];
    const float* hp_w[2];
    const float* hp_b[2];
    float hp_eps[2];
    const float* hp_cos;
    const float* hp_sin;
    long long hp_tst[2];
    int act;                  // LBR_ACT_*: a following RELU / GELU / SILU applied to C (DMA kernel)
    // Gated pair (DMA kernel): the GEMM's columns hold a gate half and an up half
    // of gF columns each; the kernel writes out[m][j] = act(gate[m][j] (+ gbias[j]))·up[m][j]
    // to C as [M, gF]
    int gF;                   // 0: off
    int gbase;                // first column of the gate half (0 or gF; up is the other half)
    int gact;                 // 0: SiLU, 1: GELU (GATED_ACT extras[1])
    const float* gbias;       // GATED_ACT bias (applied to gate) or null
    // A in head layout (DMA kernel): A is stored [B, aH, aS, ahd] and read as the
    // [B·aS, aH·ahd] matrix its TRANSPOSE(1, 2) would give (aH = 0: A is row-major)
    int aH, aS, ahd;
    // Norm prologue (DMA kernel, NORM template argument): A is the input of a
    // RMSNORM / LAYERNORM over its K columns whose output was this GEMM's A;
    // nw = weight (γ), nb = LayerNorm bias (β), neps = eps
    const float* nw;
    const float* nb;
    float neps;
    // Norm after the split-K reduce (lbr_merge_reduce_norm): the reduce, one row
    // at a time, also normalises C's row into nt_out (RMSNORM / LAYERNORM over
    // the N columns, weight nt_w, LayerNorm bias nt_b)
    float* nt_out;
    const float* nt_w;
    const float* nt_b;
    float nt_eps;
    int group;                // split-bf16 kernel: K steps between changes of the sum's sign
};

// Final store of one C element (row m, column n of batch bz) with the fused
// epilogues applied in the order the unfused nodes would: v (already
// alpha-scaled or bias-added) + resid, then the scattered split's bias.
__device__ __forceinline__ void epi_store(const GemmArgs& g, long long bz, int m, int n, float v) {
    if (g.resid) v = v + g.resid[bz * g.sC + (long long)m * g.N + n];
    if (g.n_split == 0) {
        g.C[bz * g.sC + (long long)m * g.N + n] = v;
        return;
    }
    if (n < g.col_begin[0] || n >= g.col_begin[g.n_split]) return;   // columns no split reads
    int k = 0;
    while (k + 1 < g.n_split && n >= g.col_begin[k + 1]) ++k;
    const int c = n - g.col_begin[k];
    if (g.sbias[k]) v = v + g.sbias[k][c];
    const int h = c / g.hd, d = c - h * g.hd;
    const int b = m / g.S, s = m - b * g.S;
    const long long head = ((long long)b * g.Hs[k] + h) * g.S * g.hd;
    g.dst[k][head + (((g.frag >> k) & 1) ? lbr_frag_offset(s, d, g.hd) : (long long)s * g.hd + d)] = v;
}

__device__ __forceinline__ void tile_coords(const GemmArgs& g, int& tm, int& tn) {
    // XCD-aware remap: hardware places workgroup id w on XCD w % 8.
    const int tiles = g.tiles_m * g.tiles_n;
    int w = blockIdx.x;
    if (tiles % N_XCD == 0) {
        const int per = tiles / N_XCD;
        w = (w % N_XCD) * per + (w / N_XCD);
    }
    // grouped ordering: GROUP_M tile-rows advance together along N
    const int group_size = GROUP_M * g.tiles_n;
    const int gid = w / group_size;
    const int first_m = gid * GROUP_M;
    const int gm = min(g.tiles_m - first_m, GROUP_M);
    const int in_group = w % group_size;
    tm = first_m + in_group % gm;
    tn = in_group / gm;
}

// Accumulator element (row group i of 4 rows, column block j, row r of the group) of
// the 16×16 and the 32×32 MFMA blocks; their row and column of a lane follow in
// gemm_epilogue.
template <int FM, int FN>
__device__ __forceinline__ float acc_at(const floatx4 (&a)[FM][FN], int i, int j, int r) {
    return a[i][j][r];
}
template <int FM, int FN>
__device__ __forceinline__ float acc_at(const floatx16 (&a)[FM][FN], int i, int j, int r) {
    return a[i >> 2][j][(i & 3) * 4 + r];
}

// Stores the C tile at (m0, n0) with the fused epilogues.  CB: edge of the MFMA blocks
// (16: register r of lane l holds row 4·(l/16) + r, column l%16; 32: register q holds row
// 8·(q/4) + 4·(l/32) + q%4, column l%32).  HEADP: the 64×128 tile has the head-prologue
// form; `lds` holds LDSF floats, free once every wavefront has passed its last fragment read.
template <int TM, int TN, int WGM, int WGN, int CB, bool HAS_BIAS, bool HEADP, int LDSF, typename ACC>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, float* lds, const ACC& acc, int m0, int n0, int tn,
                                              int wave, int lane, long long bz, int ks) {
    constexpr int NW = WGM * WGN;
    constexpr int RG = TM / WGM / (CB == 16 ? 16 : 8), CG = TN / WGN / CB;
    // the fields the loops use, read once (the stores below may alias what g refers to, so the
    // compiler would read them again after each)
    const int M = g.M, N = g.N, act = g.act, seq = g.S, hdim = g.hd, gact = g.gact;
    const float alpha = g.alpha;
    const float* __restrict__ bias = g.bias;
    const float* __restrict__ gbias = g.gbias;
    const int wm = wave / WGN, wn = wave % WGN;
    const int cl = lane & (CB - 1);
    // a lane's row group i starts at row mw + i·RS
    constexpr int RS = CB == 16 ? 16 : 8;
    const int lr = CB == 16 ? (lane >> 4) * 4 : (lane >> 5) * 4;
    const int mw = m0 + wm * (TM / WGM) + lr, nw = n0 + wn * (TN / WGN);
    if constexpr (HEADP && TM == 64 && TN == 128 && WGM == 2 && WGN == 2) {
        int p = -1;
        for (int q = 0; q < g.hp_parts; ++q)
            if (n0 >= g.hp_col[q] && n0 < g.hp_col[q] + g.hp_H[q] * TN) p = q;
        if (p >= 0) {
            // one head per tile: C (+ bias) through LDS, then each wavefront takes 16 rows,
            // two a pass, a row over 32 lanes of 4 columns each — the lanes, sums and
            // partner swaps of head_rows4 at HD = 128, so the values are the same bits
            constexpr int TS = TN + 4;
            static_assert(TM * TS <= LDSF, "the tile fits in the stages");
            __syncthreads();   // every wavefront's last fragment reads are done
#pragma unroll
            for (int j = 0; j < CG; ++j) {
                const int c = wn * (TN / WGN) + j * CB + cl;
                const float bv = HAS_BIAS ? bias[n0 + c] : 0.f;
#pragma unroll
                for (int i = 0; i < RG; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        lds[(wm * (TM / WGM) + i * RS + lr + r) * TS + c] =
                            HAS_BIAS ? (acc_at(acc, i, j, r) + bv) : alpha * acc_at(acc, i, j, r);
            }
            __syncthreads();
            const int H = g.hp_H[p], h = (n0 - g.hp_col[p]) / TN, S = g.hp_S;
            const int l = lane & 31, d = 4 * l;
            const bool norm = g.hp_flags & 1, rope = g.hp_flags & 2;
            const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 wv = norm ? *reinterpret_cast<const float4*>(g.hp_w[p] + d) : zero;
            const float* __restrict__ pbias = g.hp_b[p];
            const float4 pb = pbias ? *reinterpret_cast<const float4*>(pbias + h * TN + d) : zero;
            const float eps = g.hp_eps[p];
#pragma unroll 2
            for (int pass = 0; pass < TM / NW / 2; ++pass) {
                const int row = wave * (TM / NW) + 2 * pass + (lane >> 5);
                const int m = m0 + row, mc = min(m, M - 1);
                const int b = mc / S, s = mc - b * S;
                const float4 x = *reinterpret_cast<const float4*>(&lds[row * TS + d]);
                float4 v = x;
                if (pbias) {
                    v.x = v.x + pb.x;
                    v.y = v.y + pb.y;
                    v.z = v.z + pb.z;
                    v.w = v.w + pb.w;
                }
                float4 c4 = zero, s4 = zero;
                if (rope) {
                    const long long t = b * g.hp_tst[0] + s * g.hp_tst[1] + d;
                    c4 = *reinterpret_cast<const float4*>(g.hp_cos + t);
                    s4 = *reinterpret_cast<const float4*>(g.hp_sin + t);
                }
                const float4 y = lbr_head_row<32, TN>(v, norm, wv, eps, rope, c4, s4, lane);
                if (m < M)
                    *reinterpret_cast<float4*>(g.hp_out[p] + (((long long)b * H + h) * S + s) * TN + d) = y;
            }
            return;
        }
    }
    if (g.ksplit > 1) {
        float* __restrict__ Wp = g.W + ((long long)ks * gridDim.z + bz) * (long long)M * N;
#pragma unroll
        for (int j = 0; j < CG; ++j) {
            const int n = nw + j * CB + cl;
            if (n >= N) continue;
#pragma unroll
            for (int i = 0; i < RG; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mw + i * RS + r;
                    if (m < M) Wp[(long long)m * N + n] = acc_at(acc, i, j, r);
                }
        }
        return;
    }
    if (g.n_split) {
        // head scatter: the column fixes split, head, d and split bias; the
        // row fixes (b, s) = divmod(m, S), stepped from each 4-row group's first row; a group's
        // values before its stores (512×2304×768 in its layer: 0.6 µs less than row by row)
#pragma unroll
        for (int j = 0; j < CG; ++j) {
            const int n = nw + j * CB + cl;
            if (n >= N || n < g.col_begin[0] || n >= g.col_begin[g.n_split]) continue;
            int k = 0;
            while (k + 1 < g.n_split && n >= g.col_begin[k + 1]) ++k;
            const int c = n - g.col_begin[k];
            const int h = c / hdim, d = c - h * hdim;
            const float bv = HAS_BIAS ? bias[n] : 0.f;
            const bool has_sb = g.sbias[k] != nullptr;
            const float sb = has_sb ? g.sbias[k][c] : 0.f;
            const bool fr = (g.frag >> k) & 1;
            float* __restrict__ col = g.dst[k] + ((long long)h * seq) * hdim + (fr ? lbr_frag_offset(0, d, hdim) : d);
            const long long bstride = (long long)g.Hs[k] * seq * hdim;
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const int mb = mw + i * RS;
                int b = mb / seq, s = mb - b * seq;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = HAS_BIAS ? (acc_at(acc, i, j, r) + bv) : alpha * acc_at(acc, i, j, r);
                    if (has_sb) v[r] = v[r] + sb;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (mb + r < M) col[b * bstride + (fr ? lbr_frag_offset(s, 0, hdim) : (long long)s * hdim)] = v[r];
                    if (++s == seq) {
                        s = 0;
                        ++b;
                    }
                }
            }
        }
        return;
    }
    if (CG % 2 == 0 && g.gF) {   // tiles with an odd block count never take a gated pair
        // gated pair: blocks j (gate) and j+1 (up) of this wave hold the same 16
        // output columns; out = act(gate (+ gated bias))·up, rounded like the
        // unfused GEMM → SLICE → GATED_ACT chain
        const int F = g.gF;
        float* __restrict__ C = g.C + bz * (long long)M * F;
#pragma unroll
        for (int j = 0; j + 1 < CG; j += 2) {
            const int o = tn * (TN / 2) + ((wn * CG + j) >> 1) * CB + cl;
            if (o >= F) continue;
            const float bg = HAS_BIAS ? bias[g.gbase + o] : 0.f;
            const float bu = HAS_BIAS ? bias[(g.gbase ? 0 : F) + o] : 0.f;
            const float gb = gbias ? gbias[o] : 0.f;
#pragma unroll
            for (int i = 0; i < RG; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mw + i * RS + r;
                    if (m >= M) continue;
                    float x = HAS_BIAS ? (acc_at(acc, i, j, r) + bg) : alpha * acc_at(acc, i, j, r);
                    const float u = HAS_BIAS ? (acc_at(acc, i, j + 1, r) + bu) : alpha * acc_at(acc, i, j + 1, r);
                    if (gbias) x = x + gb;
                    const float a = gact == 0 ? lbr_silu(x) : lbr_gelu_tanh(x);
                    C[(long long)m * F + o] = a * u;
                }
        }
        return;
    }
    float* __restrict__ C = g.C + bz * g.sC;
    if (g.resid) {   // never with a fused activation
        // As many residual loads as 16 registers (or one block column) hold go out before the
        // first store, rows and columns clamped, not skipped: a load that follows a store waits
        // for it.  Two 333-token sequences of width 768, masked attention layer (64×64 fp32
        // tiles): 77.1 µs, against 77.8 with four loads at a time, 78.9 with loads skipped.
#pragma clang fp contract(off)   // as the unfused nodes round
        const float* __restrict__ R = g.resid + bz * g.sC;
        constexpr int JC = std::clamp(4 / RG, 1, CG);   // block columns at a time
#pragma unroll
        for (int j0 = 0; j0 < CG; j0 += JC) {
            float rv[JC][RG][4];
#pragma unroll
            for (int j = 0; j < JC && j0 + j < CG; ++j) {
                const int n = min(nw + (j0 + j) * CB + cl, N - 1);
#pragma unroll
                for (int i = 0; i < RG; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) rv[j][i][r] = R[(long long)min(mw + i * RS + r, M - 1) * N + n];
            }
#pragma unroll
            for (int j = 0; j < JC && j0 + j < CG; ++j) {
                const int n = nw + (j0 + j) * CB + cl;
                if (n >= N) continue;
                const float bv = HAS_BIAS ? bias[n] : 0.f;
#pragma unroll
                for (int i = 0; i < RG; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int m = mw + i * RS + r;
                        if (m >= M) continue;
                        const float v = HAS_BIAS ? (acc_at(acc, i, j0 + j, r) + bv) : alpha * acc_at(acc, i, j0 + j, r);
                        C[(long long)m * N + n] = v + rv[j][i][r];
                    }
            }
        }
        return;
    }
    // One loop for GELU, so that its elements' chains overlap, and one for the rest (GELU MLP layer
    // of 512 tokens and width 768: 59.85 µs, against 60.3 with the choice made element by element).
    auto store = [&](auto f) {
#pragma unroll
        for (int j = 0; j < CG; ++j) {
            const int n = nw + j * CB + cl;
            if (n >= N) continue;
            const float bv = HAS_BIAS ? bias[n] : 0.f;
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    v[r] = f(HAS_BIAS ? (acc_at(acc, i, j, r) + bv) : alpha * acc_at(acc, i, j, r));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = mw + i * RS + r;
                    if (m < M) C[(long long)m * N + n] = v[r];
                }
            }
        }
    };
    if (act == LBR_ACT_GELU) store([](float v) { return lbr_gelu_tanh(v); });
    else store([act](float v) { return lbr_act(act, v); });
}

// Kernel arguments of a decoded or fused GEMM step, and its split-K reduction (gemm.hip).
GemmArgs gemm_make_args(const Step& s);
void gemm_reduce_ksplit(const Step& s, const GemmArgs& g, hipStream_t st);

// Launcher of the split-bf16 GEMM (gemm_split.hip) with its tile number `shape`; `heads`: A
// in head layout.
step_fn gemm_split_launcher(int shape, bool has_bias, bool heads);
