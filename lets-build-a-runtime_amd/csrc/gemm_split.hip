// gemm_split.hip — the fp32 GEMM C = A · Bᵀ on the bf16 matrix cores.
//
// An fp32 value is the exact sum of three bf16 values (8 + 8 + 8 significand bits):
// h = bf16(x), m = bf16(x − h), l = x − h − m (the splitting of a float into an unevaluated
// sum of shorter ones, Dekker 1971).  A product a·b is then the sum of nine bf16 products,
// each exact in the MFMA's fp32 accumulator input; the six largest are taken and m·l, l·m and
// l·l left out, together at most 2⁻²⁴ of the product (0.09·2⁻²⁴ rms over 2·10⁶ pairs).  Six
// v_mfma_f32_32x32x16_bf16 replace sixteen v_mfma_f32_16x16x4_f32 in 6/16 of their time: 2.67×
// the fp32 matrix peak.  The sum rounds six times per 16 terms, smallest products first, the
// fp32 kernel's four times.  Measured, root mean square error against 64 bits in the results'
// rms, N(0,1) rows of K = 4 / 20 / 64 / 256 / 768 / 4096 / 16384: 3.2e-8 / 6.3e-8 / 1.1e-7 / 2.4e-7 /
// 2.4e-7 / 2.7e-7 / 5.3e-7 against the fp32 kernels' 4.1e-8 / 8.2e-8 / 1.4e-7 / 2.9e-7 / 2.9e-7 /
// 4.4e-7 / 6.2e-7, each on its own tile and K ranges; lower at all 16 values of K tried, and
// with GELU outputs for A too.
//
// Range: both operands are taken times 2²⁴ and the sum times 2⁻⁴⁸, all exact, so that the
// planes of every finite value below 2¹⁰⁴, subnormals included, are zero or normal bf16
// values (the smallest fp32 bit, 2⁻¹⁴⁹, becomes 2⁻¹²⁵) and no bit is lost.  Operands from
// 2¹⁰⁴ up, infinities and NaN, and sums from 2⁸⁰ up give an accumulator that is not finite,
// and the fp32 matrix cores recompute the 32×32 blocks that hold one.  Unscaled planes lost
// bits below 2⁻¹¹⁰ and all of them below 2⁻¹³⁴.  The scaling takes the place of the sign's
// XOR on A and costs B a multiplication an element: 1% of 4096×12288×4096 on 256×256 tiles
// (1776 → 1783 µs) and 3% of 1024×6144×2560 on 64×128, which steps in pairs (below) win back
// (1762, and 201 against 202).  A block that is recomputed reads its rows of A and B from
// memory for itself: a product with such values everywhere runs at a fraction of the rate.
//
// Structure: a WGM×WGN grid of wavefronts, each (TM/WGM)×(TN/WGN) of C in 32×32 blocks.  A
// step is 16 columns of K.  Each thread loads its float4s of the A and B tiles two steps
// ahead, splits them once for the whole workgroup (22 VALU instructions a float4, which
// issue beside the MFMAs: bf16 MFMAs leave the VALU free, the fp32 ones do not) and writes
// the three planes into the LDS stage the step before last has left; the next loads go out
// as soon as a float4 has been split.  One barrier a step.  A fragment (32 rows × 16
// columns of a plane) is 1 KiB of LDS in the order the lanes read it: half h (columns 8h ..
// 8h+7) of row r at 512·h + 16·(r ^ 12h), so that the 16-byte reads and the 8-byte writes
// of a wavefront hit every bank once (SQ_LDS_BANK_CONFLICT 0; row-major planes of 32 bytes
// a row had two conflict cycles a read and cost 2%).
//
// What bounds it: 4096×12288×4096 takes 1731 µs, 238 TFLOP/s (1.43 PFLOP/s of bf16
// products), against 2765 µs and 149 for the fp32 kernel; MFMAs alone, on such data, run at
// 295, the power limit (a library's bf16 product of 8192³: 1.28-1.37 PFLOP/s over cards, which
// differ by up to 8%).  Splitting costs 10% of that and the loads the rest.
#include "gemm_common.h"

#include <type_traits>

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

namespace {

__device__ __forceinline__ unsigned cvt_bf16x2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2{a, b}), bf16x2));
}

// The planes of two neighbours, packed: x = h + m + l exactly (l fits: after two
// round-to-nearest steps at most 8 significant bits are left).
__device__ __forceinline__ void split3(float x0, float x1, unsigned& h, unsigned& m, unsigned& l) {
#pragma clang fp contract(off)   // a subtraction is the shorter instruction
    h = cvt_bf16x2(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = cvt_bf16x2(r0, r1);
    l = cvt_bf16x2(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
}

// Powers of two that keep the planes of subnormal operands normal (see the top).
constexpr float UP = 0x1p24f, DOWN = 0x1p-48f;

__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7fffffffu) >= 0x7f800000u; }

// The bf16 MFMAs round their fp32 sum down, not to nearest: 4096 terms of N(0,1) rows came
// out 2.1e-7 of their rms too low on average, which an average over many of them (attention
// over its keys) would keep.  So the sum changes sign, accumulators and A alike, between
// groups of at most GROUP steps, an even number of about equal size (even themselves: the
// steps go in pairs), and the half of it that is negated rounds up.  Mean error of 512×512
// results in their rms, N(0,1) rows: -5e-10 / -3e-9 / 2e-9 / 1e-8 at K = 128 / 200 / 256 / 4096,
// against -9e-9 / -1.3e-8 / -1.5e-8 / -2.1e-7 where it does not change.  Two steps or less stay
// one group (-8e-9 at K = 16, of an error of 3.4e-8; the fp32 kernels' is 7.4e-8).
constexpr int GROUP = 16;
int sign_group(int nk) {   // steps a group, of nk
    const int n = (nk + 2 * GROUP - 1) / (2 * GROUP) * 2;   // groups
    return ((nk + n - 1) / n + 1) & ~1;
}

// K: any multiple of 4 with RAGGED (the last step's columns past K read as zero through
// the buffer views' range check), else a multiple of 16.
template <int TM, int TN, int WGM, int WGN, int OCC, bool HAS_BIAS, bool AHEADS, bool RAGGED>
__global__ __launch_bounds__(64 * WGM * WGN, OCC) void gemm_split_f32(GemmArgs g) {
    constexpr int NT = 64 * WGM * WGN;
    constexpr int WM = TM / WGM, WN = TN / WGN, FM = WM / 32, FN = WN / 32;
    // One MFMA block a wavefront: a step is a chain of latencies, which wants fewer VALU
    // instructions between the MFMAs and, with the ragged tail's selects, no steps in pairs
    // (231×200×712: 21.7 µs against 23.0 with both as on the other tiles).
    constexpr bool ONE = FM * FN == 1;
    constexpr int KB = 16, QR = KB / 4;                       // float4s ("quads") per tile row and step
    constexpr int NA = TM * QR / NT, NB = TN * QR / NT, NQ = NA + NB;   // quads per thread
    static_assert(NA * NT == TM * QR && NB * NT == TN * QR, "tile rows must split evenly over the threads");
    static_assert(FM * 32 * WGM == TM && FN * 32 * WGN == TN, "tile shape");
    constexpr int PA = TM * KB * 2, PB = TN * KB * 2, STAGE = 3 * (PA + PB);   // bytes of a plane, of a stage
    __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];

    int tm, tn;
    tile_coords(g, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    const long long bz = blockIdx.z;
    const int M = g.M, N = g.N, K = g.K;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(g.A + bz * g.sA), (short)0, M * K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(g.B + bz * g.sB), (short)0, N * K * 4, 0x00020000);

    // first float of row m of A (clamped to the matrix: rows past the edge are never stored)
    auto a_row = [&](int m) {
        m = min(m, M - 1);
        if (!AHEADS) return m * K;
        const int b = m / g.aS, s = m - b * g.aS;   // head layout [B, aH, aS, ahd]
        return ((b * g.aH) * g.aS + s) * g.ahd;
    };
    // first float of the row of B behind tile column c
    auto b_row = [&](int c) {
        if (g.gF) {
            // gated pair: tile column blocks of 32 alternate gate, up for the same TN/2
            // output columns starting at tn·TN/2 (clamped to the last one)
            const int jb = c >> 5;
            const int o = min(tn * (TN / 2) + (jb >> 1) * 32 + (c & 31), g.gF - 1);
            return ((jb & 1) ? (g.gbase ? 0 : g.gF) + o : g.gbase + o) * K;
        }
        return min(n0 + c, N - 1) * K;
    };
    // float offset of column k of A within its row
    auto a_col = [&](int k) { return AHEADS ? (k / g.ahd) * g.aS * g.ahd + k % g.ahd : k; };

    unsigned off[NQ];   // byte offset of the thread's quad t at K step 0
    int dst[NQ], kq[NQ];
#pragma unroll
    for (int t = 0; t < NQ; ++t) {
        const int o = tid + (t < NA ? t : t - NA) * NT, row = o / QR, q = o % QR, half = q >> 1;
        kq[t] = q * 4;
        off[t] = (unsigned)(t < NA ? a_row(m0 + row) + a_col(q * 4) : b_row(row) + q * 4) * 4u;
        dst[t] = (t < NA ? 0 : 3 * PA) + (row >> 5) * 1024 + half * 512 + (((row & 31) ^ (half * 12)) * 16) + (q & 1) * 8;
    }
    floatx4 raw[NQ];
    const int kbeg = blockIdx.y * g.kchunk, kend = min(K, kbeg + g.kchunk);
    const int nk = (kend - kbeg + KB - 1) / KB;
    auto load = [&](int t, int k) {   // quad t of the K step at column k
        unsigned o = off[t];
        if (RAGGED && k + kq[t] >= kend) o = 0x80000000u;   // past every view
        const unsigned so = (unsigned)(t < NA && AHEADS ? a_col(k) : k) * 4u;
        raw[t] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(t < NA ? ra : rb, o, so, 0));
    };
    unsigned ph[2], pm[2], pl[2];
    auto split = [&](int p, float up) {   // pair p: components 2·(p&1), 2·(p&1)+1 of quad p/2
#pragma clang fp contract(off)
        const float f = (p >> 1) < NA ? up : UP;   // A's sign is the group's (see GROUP)
        split3(raw[p >> 1][2 * (p & 1)] * f, raw[p >> 1][2 * (p & 1) + 1] * f, ph[p & 1], pm[p & 1], pl[p & 1]);
    };
    auto negate = [&](auto& a) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) a[i][j] = -a[i][j];
    };
    auto put = [&](char* st, int t) {
        char* d = st + dst[t];
        const int plane = t < NA ? PA : PB;
        *reinterpret_cast<uintx2*>(d) = uintx2{ph[0], ph[1]};
        *reinterpret_cast<uintx2*>(d + plane) = uintx2{pm[0], pm[1]};
        *reinterpret_cast<uintx2*>(d + 2 * plane) = uintx2{pl[0], pl[1]};
    };

    floatx16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int fr = lane & 31, fh = lane >> 5;
    const int fo = fh * 512 + ((fr ^ (fh * 12)) * 16);
    const int rdA = wm * WM * 32 + fo, rdB = 3 * PA + wn * WN * 32 + fo;
    bf16x8 fa[FM][3], fb[2][3];
    auto get_a = [&](const char* st) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int p = 0; p < 3; ++p) fa[i][p] = *reinterpret_cast<const bf16x8*>(st + rdA + p * PA + i * 1024);
    };
    auto get_b = [&](const char* st, int j, bf16x8* f) {
#pragma unroll
        for (int p = 0; p < 3; ++p) f[p] = *reinterpret_cast<const bf16x8*>(st + rdB + p * PB + j * 1024);
    };
    auto mma = [&](int j, const bf16x8* f) {
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};   // smallest products first
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int i = 0; i < FM; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][pa[q]], f[pb[q]], acc[i][j], 0, 0, 0);
    };

    if (nk > 0) {
#pragma unroll
        for (int t = 0; t < NQ; ++t) load(t, kbeg);
#pragma unroll
        for (int t = 0; t < NQ; ++t) {
            split(2 * t, UP);
            split(2 * t + 1, UP);
            put(lds, t);
            load(t, kbeg + min(1, nk - 1) * KB);
        }
        __syncthreads();
        // one step; CUR (0 or STAGE): where its planes are, the other stage takes the next step's
        auto step = [&](int kt, int kl, bool pos, auto CUR) {
            // steps past the last are re-fetches of the last one, into a stage nothing reads
            const char* st = lds + CUR;
            char* wr = lds + (STAGE - CUR);
            const int k2 = kbeg + min(kt + 2, nk - 1) * KB;
            // of the step being split: UP, negative in every other group
            const float up = (kt + 1 < kl) == pos ? UP : -UP;
            get_a(st);
            get_b(st, 0, fb[0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                constexpr int NP = 2 * NQ, VPM = ((NP + FN - 1) / FN * (ONE ? 9 : 13) + 6 * FM - 1) / (6 * FM);
                if (j + 1 < FN) get_b(st, j + 1, fb[(j + 1) & 1]);
                mma(j, fb[j & 1]);
#pragma unroll
                for (int p = 0; p < NP; ++p)   // this block's share of the next step's pairs
                    if (p * FN / NP == j) {
                        split(p, up);
                        if (p & 1) {
                            put(wr, p >> 1);
                            load(p >> 1, k2);
                        }
                    }
                if (j + 1 < FN) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // the fragment reads first
#pragma unroll
                for (int q = 0; q < 6 * FM; ++q) {   // then each MFMA with its share of the splitting
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
                }
                if (j + 1 < FN) __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        };
        bool pos = true;
        for (int kt = 0; kt < nk;) {
            const int kl = min(nk, kt + g.group);
            if constexpr (!(ONE && RAGGED))
                for (; kt + 1 < kl; kt += 2) {   // in pairs: the stages' addresses are constants
                    step(kt, kl, pos, std::integral_constant<int, 0>());
                    step(kt + 1, kl, pos, std::integral_constant<int, STAGE>());
                }
            for (; kt < kl; ++kt) step(kt, kl, pos, (kt & 1) * STAGE);
            if (kt < nk) {
                negate(acc);
                pos = !pos;
            }
        }
        const float down = pos ? DOWN : -DOWN;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = acc[i][j] * down;
    }

    // Blocks with a sum that is not finite: the whole block again on the fp32
    // matrix cores, fragments straight from memory (lane (fh, fr) reads 4 consecutive k of
    // its row, MFMA q takes k = 4·fh + q of an 8-wide chunk), and those results replaced.
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            bool bad = false;
#pragma unroll
            for (int r = 0; r < 16; ++r) bad = bad || not_finite(acc[i][j][r]);
            if (!__any(bad)) continue;
            const unsigned oa = (unsigned)a_row(m0 + wm * WM + i * 32 + fr) * 4u;
            const unsigned ob = (unsigned)b_row(wn * WN + j * 32 + fr) * 4u;
            floatx16 f;
#pragma unroll
            for (int r = 0; r < 16; ++r) f[r] = 0.f;
            for (int k = kbeg; k < kend; k += 8) {
                const int kl = k + 4 * fh;
                const bool in = kl < kend;   // kend is a multiple of 4
                const floatx4 x = __builtin_bit_cast(
                    floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra, in ? oa + (unsigned)a_col(kl) * 4u : 0x80000000u, 0, 0));
                const floatx4 y = __builtin_bit_cast(
                    floatx4, __builtin_amdgcn_raw_buffer_load_b128(rb, in ? ob + (unsigned)kl * 4u : 0x80000000u, 0, 0));
#pragma unroll
                for (int q = 0; q < 4; ++q) f = __builtin_amdgcn_mfma_f32_32x32x2f32(x[q], y[q], f, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (not_finite(acc[i][j][r])) acc[i][j][r] = f[r];
        }

    gemm_epilogue<TM, TN, WGM, WGN, 32, HAS_BIAS, !AHEADS, 2 * STAGE / 4>(g, reinterpret_cast<float*>(lds), acc, m0, n0,
                                                                          tn, wave, lane, bz, (int)blockIdx.y);
}

template <int TM, int TN, int WGM, int WGN, int OCC, bool HAS_BIAS, bool AHEADS>
void launch(const Step& s, hipStream_t st) {
    GemmArgs g = gemm_make_args(s);
    if (g.M <= 0 || g.N <= 0) return;
    g.tiles_m = (g.M + TM - 1) / TM;
    g.tiles_n = g.gF ? (g.gF + TN / 2 - 1) / (TN / 2) : (g.N + TN - 1) / TN;
    g.group = sign_group((g.kchunk + 15) / 16);
    const dim3 grid(g.tiles_m * g.tiles_n, g.ksplit, (unsigned)s.i[3]);
    if (g.K % 16 == 0)
        hipLaunchKernelGGL((gemm_split_f32<TM, TN, WGM, WGN, OCC, HAS_BIAS, AHEADS, false>), grid,
                           dim3(64 * WGM * WGN), 0, st, g);
    else if constexpr (!AHEADS)   // A in head layout: K is a multiple of 32
        hipLaunchKernelGGL((gemm_split_f32<TM, TN, WGM, WGN, OCC, HAS_BIAS, false, true>), grid,
                           dim3(64 * WGM * WGN), 0, st, g);
    if (g.ksplit > 1) gemm_reduce_ksplit(s, g, st);
}

template <bool HAS_BIAS, bool AHEADS>
step_fn pick(int shape) {
    switch (shape) {
        case 0: return launch<256, 256, 4, 2, 2, HAS_BIAS, AHEADS>;
        case 1: return launch<256, 128, 4, 2, 2, HAS_BIAS, AHEADS>;
        case 2: return launch<128, 256, 2, 4, 2, HAS_BIAS, AHEADS>;
        case 3: return launch<128, 128, 2, 2, 2, HAS_BIAS, AHEADS>;
        case 4: return launch<128, 64, 2, 2, 3, HAS_BIAS, AHEADS>;
        case 5: return launch<64, 128, 2, 2, 3, HAS_BIAS, AHEADS>;
        case 6: return launch<64, 64, 2, 2, 4, HAS_BIAS, AHEADS>;
        default: return nullptr;
    }
}

}  // namespace

step_fn gemm_split_launcher(int shape, bool has_bias, bool heads) {
    if (heads) return has_bias ? pick<true, true>(shape) : pick<false, true>(shape);
    return has_bias ? pick<true, false>(shape) : pick<false, false>(shape);
}
