// Weight-only bf16 x MXFP4 GEMM and its dual-batch form, for gfx950.
//
//   single:  C[m, n]  = sum_k A[m, k]  * deq(W)[n, k]
//   dual:    C0[m, n] = sum_k A0[m, k] * deq(W)[n, k],  C1 likewise with A1
//
// Semantics: the fake-quant forward of fp4_linear.py:40 with an unquantized
// activation (deq(W) = E2M1 value * 2^e, fp4.py:75-78), and dual_gemm.py:78-110
// _dual_separate_kernel used with one shared weight (train_step.py:52-53):
// two accumulators, one launch.  deq(W) is exact in bf16 (at most two
// significant bits times a power of two inside bf16's exponent range), so
// the products are exact and only fp32 accumulation rounds.
//
// Dequantization happens in registers: each lane pulls the 16 packed bytes
// (32 codes, one MX block) of its weight column for the stage from LDS and
// turns them into 32 bf16 values with v_cvt_scalef32_pk_bf16_fp4, which
// multiplies by the block scale on the way.  The MFMA is
// v_mfma_f32_32x32x16_bf16.  Its K positions are assigned so that, across
// the four K=16 steps of a 64-wide stage, lane half h covers block h of the
// stage: the A operand for step s reads A[row][32h + 8s .. +8].  A and W use
// the same assignment, so the sum is unchanged.
//
// Kernels, by the rules at launch_gemm_bf16f4: GEMV (1 row), decode and skinny
// (up to 32), tile and ring (E8M0 scales), gemm_bf16f4_kernel (what is left),
// gemm_xf4_kernel (fp32 / fp16 activations).  In the dual form of the ring
// kernel and gemm_bf16f4_kernel half of a tile's A rows are rows of A0 and half
// the same rows of A1: one weight tile in LDS feeds both batches and is read
// from memory once per stage.
#include <mutex>

#include "lsmx_dma.h"
#include "lsmx_store.h"
#include "lsmx_internal.h"
#include "lsmx_sched.h"

namespace lsmx {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace w4 {
constexpr int BK = 64;         // K per stage
constexpr int A_ROW_B = BK * 2;    // 128 bytes of bf16 per A row per stage
constexpr int W_ROW_B = BK / 2;    // 32 bytes of codes per W row per stage
constexpr int NT = 256;
constexpr int GROUP_M = 4;
}  // namespace w4

LSMX_DEV int a_swz(int row) { return (row ^ (row >> 3)) & 7; }

LSMX_DEV uint32_t bf16_rne_w(float f) {
    uint32_t u = f2u(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

template <int CT>
LSMX_DEV void store_cw(void *c, int64_t idx, float v) {
    if constexpr (CT == LSMX_F32) reinterpret_cast<float *>(c)[idx] = v;
    else if constexpr (CT == LSMX_BF16) reinterpret_cast<uint16_t *>(c)[idx] = (uint16_t)bf16_rne_w(v);
    else reinterpret_cast<_Float16 *>(c)[idx] = (_Float16)v;
}

LSMX_DEV void tile_coords_w(int pid, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int total = tiles_m * tiles_n;
    if ((total & 7) == 0) pid = (pid & 7) * (total >> 3) + (pid >> 3);
    const int per_group = w4::GROUP_M * tiles_n;
    const int group = pid / per_group;
    const int first_m = group * w4::GROUP_M;
    const int gsz = min(tiles_m - first_m, w4::GROUP_M);
    const int in_group = pid - group * per_group;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

template <bool SF32>
LSMX_DEV uint32_t load_scale2(const void *s, int64_t off) {
    // 2 consecutive block scales as E8M0 bytes in the low 16 bits
    if constexpr (SF32) {
        const u32x2 v = *reinterpret_cast<const u32x2 *>(reinterpret_cast<const float *>(s) + off);
        return f32_scale_e8m0(v[0]) | (f32_scale_e8m0(v[1]) << 8);
    } else {
        return *reinterpret_cast<const uint16_t *>(reinterpret_cast<const uint8_t *>(s) + off);
    }
}

// E8M0 byte -> fp32 scale: 2^(e - 127), with byte 0 -> 2^-127 (0x00400000)
// and byte 255 -> NaN (0x7FC00000), both of which are (e << 23) | 2^22.
// Written without selects: the compiler turned a select per special byte into
// branches on the exec mask in front of every conversion (against a 14336 x
// 4096 weight M = 1: 7.9 us with them, 7.3 without; M = 4096: 412 and 377).
LSMX_DEV float e8m0_scale_f32(uint32_t e) {
    const uint32_t special = ((((e + 1u) & 0xFEu) - 1u) >> 9) & 0x00400000u;
    return u2f((e << 23) | special);
}

// BR A rows (all batches) x BN weight columns per workgroup of 4 waves in a
// 2 x 2 grid: 256 x 256 for large M; 128 x 128 or 128 x 64 (several
// workgroups per CU) when larger tiles would leave CUs idle.
template <int NB, bool SF32, int CT, int BR, int BN>
__global__ __launch_bounds__(w4::NT, BR == 256 ? 1 : 2) void gemm_bf16f4_kernel(GemmArgs g) {
    using namespace w4;
    constexpr int RPB = BR / NB;           // A rows per batch per workgroup
    constexpr int RT = BR / 64 / NB;       // row tiles per batch per wave
    constexpr int WT = BN / 2;             // weight columns per wave
    constexpr int CTW = WT / 32;           // column tiles per wave
    constexpr int XA = BR * A_ROW_B / 16 / NT;   // A chunks per thread per stage
    constexpr int XW = BN * W_ROW_B / 16 / NT;   // W chunks per thread per stage (0 for BN = 64: threads
                                                 // t and t + 128 load the same chunk)
    static_assert(RT >= 1 && CTW >= 1, "tile too small");
    __shared__ __attribute__((aligned(16))) uint8_t sA[2][BR * A_ROW_B];   // 2 x 32 KiB
    __shared__ __attribute__((aligned(16))) uint8_t sW[2][BN * W_ROW_B];   // 2 x 8 KiB, [half][col][16B]
    __shared__ uint32_t sS[2][BN];

    const int tiles_m = (int)((g.M + RPB - 1) / RPB), tiles_n = (int)((g.N + BN - 1) / BN);
    int tm, tn;
    tile_coords_w(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * RPB, n0 = (int64_t)tn * BN;

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int nk = (int)(g.K / BK);

    // A staging: XA chunks of 16 B per thread; row = q >> 3, chunk = q & 7
    const uint8_t *ga[XA];
    int a_off[XA];
#pragma unroll
    for (int i = 0; i < XA; ++i) {
        const int q = i * NT + t;
        const int row = q >> 3, c = q & 7;
        const int b = row / RPB, r = row % RPB;
        const int64_t am = min(m0 + r, g.M - 1);
        const uint8_t *base = (NB == 2 && b == 1) ? g.a1 : g.a;
        ga[i] = base + am * g.lda * 2 + c * 16;
        a_off[i] = row * A_ROW_B + ((c ^ a_swz(row)) << 4);
    }
    // W staging: 2 chunks (one per block half) per weight row; with BN = 128
    // the 256 threads cover the 256 chunks once, with BN = 64 twice
    constexpr int XW1 = XW > 0 ? XW : 1;
    const uint8_t *gw[XW1];
    int w_off[XW1];
#pragma unroll
    for (int i = 0; i < XW1; ++i) {
        const int q = (i * NT + t) % (2 * BN);
        const int row = q >> 1, h = q & 1;
        const int64_t wn_ = min(n0 + row, g.N - 1);
        gw[i] = g.b + wn_ * g.ldb + h * 16;
        w_off[i] = h * (BN * 16) + row * 16;
    }
    // thread t < BN stages the scales of weight column t (threads past BN
    // load a clamped column and store nothing)
    const int64_t s_row = min(n0 + (t % BN), g.N - 1) * g.ld_sb;

    u32x4 ra[XA], rw[XW1];
    uint32_t rs;
    auto gload = [&](int kt) {
#pragma unroll
        for (int i = 0; i < XA; ++i) ra[i] = *reinterpret_cast<const u32x4 *>(ga[i] + (int64_t)kt * A_ROW_B);
#pragma unroll
        for (int i = 0; i < XW1; ++i) rw[i] = *reinterpret_cast<const u32x4 *>(gw[i] + (int64_t)kt * W_ROW_B);
        rs = load_scale2<SF32>(g.sb, s_row + (int64_t)kt * 2);
    };
    auto swrite = [&](int buf) {
#pragma unroll
        for (int i = 0; i < XA; ++i) *reinterpret_cast<u32x4 *>(&sA[buf][a_off[i]]) = ra[i];
#pragma unroll
        for (int i = 0; i < XW1; ++i) *reinterpret_cast<u32x4 *>(&sW[buf][w_off[i]]) = rw[i];
        if (BN == NT || t < BN) sS[buf][t % BN] = rs;
    };

    v16f acc[NB][RT][CTW];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CTW; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[b][i][j][e] = 0.0f;

    const int frow = lane & 31, half = lane >> 5;

    gload(0);
    swrite(0);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) gload(kt + 1);

        // dequantize this wave's CTW weight column tiles for the stage:
        // 32 codes of block `half` -> 32 bf16, 8 per K=16 step.
        v8bf fw[CTW][4];  // [col tile][step]
#pragma unroll
        for (int j = 0; j < CTW; ++j) {
            const int col = wn * WT + j * 32 + frow;
            const u32x4 pw = *reinterpret_cast<const u32x4 *>(&sW[buf][half * (BN * 16) + col * 16]);
            const float sc = e8m0_scale_f32((sS[buf][col] >> (8 * half)) & 0xFF);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pw[s], sc, 0);
                const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pw[s], sc, 1);
                const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pw[s], sc, 2);
                const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(pw[s], sc, 3);
                fw[j][s] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = half * 4 + s;  // 16-byte chunk: A[row][32h + 8s .. +8]
            v8bf fa[NB][RT];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const int row = b * RPB + wm * (RT * 32) + i * 32 + frow;
                    fa[b][i] = *reinterpret_cast<const v8bf *>(&sA[buf][row * A_ROW_B + ((c ^ a_swz(row)) << 4)]);
                }
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < CTW; ++j)
                        acc[b][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[b][i], fw[j][s], acc[b][i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) swrite(buf ^ 1);
        __syncthreads();
    }

#pragma unroll
    for (int b = 0; b < NB; ++b) {
        void *cb = (NB == 2 && b == 1) ? g.c1 : g.c;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CTW; ++j) {
                const int64_t col = n0 + wn * WT + j * 32 + frow;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int64_t row = m0 + wm * (RT * 32) + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
                    if (row < g.M && col < g.N) store_cw<CT>(cb, row * g.ldc + col, acc[b][i][j][e]);
                }
            }
    }
}

// ------------------------------------------------------------------ fp32 / fp16 activations
// Weight-only GEMM with wider activations: Y = X . deq(W)^T for X in fp32
// (the fake-quant forward of fp4_linear.py:40 with an unquantized fp32
// X, deq(W) of fp4.py:75-78) or fp16.  Each activation is
// split exactly into NTERM bf16 terms, each the bf16 truncation of what the
// terms before it leave,
//     hi = tr(x),  mid = tr(x - hi),  lo = x - hi - mid     (fp32: NTERM = 3)
// (x has 24 significant bits and each term holds 8; every subtraction and
// the last term are exact; fp16's 11 bits need hi and mid only), and each
// term runs through v_mfma_f32_32x32x16_bf16 against the exact bf16 weight.
// The products are exact in fp32, so only the fp32 accumulation rounds, as
// in an fp32 matmul.  Per K-step the terms are added hi, mid, lo.
// Tile: BR rows x BN weight columns per workgroup of 4 waves, 64-deep K
// stages, the widest tile whose grid still fills the CUs: 64 x 128 or
// 64 x 64 (2 x 2 waves of 32 x BN/2), or for small outputs 32 x 32 with the
// 4 waves splitting each stage's four 16-deep K-steps (cfg1's 256 x 1024
// output is 256 such workgroups); their partial tiles are added in wave
// order through LDS at the end.  The split happens once per element, as
// the activations are staged: each thread loads its 16-byte chunks two
// stages ahead into VGPRs and, after a stage's MFMAs, writes their terms to
// a double-buffered LDS tile of NTERM bf16 planes (128 bytes per row and
// plane per stage).  The K positions are those of the bf16 kernel above: at
// K-step s lane half h supplies X[row][32h + 8s .. +8] and codes 8s .. 8s+7
// of the weight's block h of the stage.
static int num_cus_w();

namespace xf {
constexpr int BK = 64, NT = 256;
constexpr int ROW_B = BK * 2;     // bytes per row of one bf16 term plane per stage
}  // namespace xf

// The bf16 terms of x (fp32 bits xb): hi = tr(x), mid = tr(x - hi),
// lo = tr(x - hi - mid), exact for |x| >= 2^-110 (there lo is at least a
// bf16 subnormal's ulp); Inf and NaN pass through hi alone (a NaN whose
// payload lies in the low 16 bits keeps a quiet bit).
LSMX_DEV void split_bf16_terms(uint32_t xb, uint32_t &hb, uint32_t &mb, uint32_t &lb) {
    const bool special = (xb & 0x7F800000u) == 0x7F800000u;
    hb = (xb >> 16) | (special && (xb & 0xFFFFu) ? 0x40u : 0u);
    const float r1 = special ? 0.0f : u2f(xb) - u2f(hb << 16);
    mb = f2u(r1) >> 16;
    lb = f2u(r1 - u2f(mb << 16)) >> 16;
}

template <int AT, bool SF32, int CT, int BR, int BN, int KS, int KG = 1>
__global__ __launch_bounds__(xf::NT * KG, KG == 1 ? 2 : 4) void gemm_xf4_kernel(GemmArgs g) {
    using namespace xf;
    static_assert(KG == 1 || KS == 4, "K groups split the 32 x 32 tile form");
    constexpr int ES = AT == LSMX_F32 ? 4 : 2;        // activation bytes
    constexpr int NTERM = AT == LSMX_F32 ? 3 : 2;     // bf16 terms per activation
    constexpr int WM = KS == 1 ? 2 : 1, WN = KS == 1 ? 2 : 1;  // wave grid over the tile
    static_assert(WM * WN * KS == 4 && BR == 32 * WM, "4 waves: 2 x 2 tiles, or one tile split 4 ways along K");
    constexpr int CTW = BN / 32 / WN;                 // 32-column MFMA tiles per wave
    constexpr int EPC = 16 / ES;                      // activations per 16-byte source chunk (4 or 8)
    constexpr int CPR = BK / EPC;                     // source chunks per row per stage (16 or 8)
    constexpr int XA = BR * CPR / NT;                 // source chunks per thread per stage (4 or 2)
    constexpr int WCH = BN * 2;                       // 16-byte W chunks per stage
    // K group kg's activation rows are rows kg * BR .. of each term plane,
    // its W chunks and scales the kg-th part of each buffer, so that every
    // LDS address is a per-lane offset (which includes kg) plus an immediate
    __shared__ __attribute__((aligned(16))) uint8_t sX[2][NTERM][KG * BR * ROW_B];  // 2 x 3 x 8 KiB per group (fp32)
    __shared__ __attribute__((aligned(16))) uint8_t sW[2][KG * BN * 32];            // [group][half][col][16 B]
    __shared__ uint32_t sS[2][KG * BN];

    const int tiles_m = (int)((g.M + BR - 1) / BR), tiles_n = (int)((g.N + BN - 1) / BN);
    int tm, tn;
    tile_coords_w(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t m0 = (int64_t)tm * BR, n0 = (int64_t)tn * BN;
    // K group kg (4 waves) runs stages kg * nkg .. + nkg - 1 on its own LDS
    // buffers; the groups meet only at the workgroup barriers, which they
    // reach in step
    const int kg = __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    const int t = (int)threadIdx.x % NT, lane = t & 63, wave = t >> 6;
    const int wm = KS == 1 ? wave >> 1 : 0, wn = KS == 1 ? wave & 1 : 0;
    const int wk = KS == 1 ? 0 : wave;                // this wave's K-steps: wk, wk + KS, ... of each stage
    const int frow = lane & 31, half = lane >> 5;
    const int nk = (int)(g.K / BK) / KG;              // stages of this K group (the launcher keeps KG | K / BK)
    const int64_t kg0 = (int64_t)kg * nk;             // its first stage

    // source chunk q = i * NT + t: row q / CPR, activations EPC * (q % CPR)
    // .. +EPC, i.e. 2 * EPC bytes of each term plane at byte 2 * EPC * (q %
    // CPR) of the row, whose 16-byte chunk sits at chunk ^ a_swz(row)
    const uint8_t *ga[XA];
    int x_off[XA];
#pragma unroll
    for (int i = 0; i < XA; ++i) {
        const int q = i * NT + t;
        const int row = q / CPR, c = q % CPR, lrow = kg * BR + row;
        ga[i] = g.a + min(m0 + row, g.M - 1) * g.lda * ES + c * 16;
        const int pb = 2 * EPC * c;  // byte in the plane row
        x_off[i] = lrow * ROW_B + (((pb >> 4) ^ a_swz(lrow)) << 4) + (pb & 15);
    }
    const int wq = t < WCH ? t : 0;  // W chunk of this thread (threads >= WCH load none)
    const uint8_t *gw = g.b + min(n0 + (wq >> 1), g.N - 1) * g.ldb + (wq & 1) * 16;
    const int w_off = (2 * kg + (wq & 1)) * (BN * 16) + (wq >> 1) * 16;
    const int64_t s_row = min(n0 + (t % BN), g.N - 1) * g.ld_sb;

    // two register slots of staged loads: stage k lives in slot k % 2 from
    // its load (issued two stages ahead) until its terms go to LDS
    u32x4 ra[2][XA], rw[2];
    uint32_t rs[2];
    auto gload = [&](int kt, auto slot) {
        constexpr int q = decltype(slot)::value;
#pragma unroll
        for (int i = 0; i < XA; ++i) ra[q][i] = *reinterpret_cast<const u32x4 *>(ga[i] + (kg0 + kt) * BK * ES);
        if (t < WCH) rw[q] = *reinterpret_cast<const u32x4 *>(gw + (kg0 + kt) * 32);
        rs[q] = load_scale2<SF32>(g.sb, s_row + (kg0 + kt) * 2);
    };
    auto swrite = [&](int buf, auto slot) {
        constexpr int q = decltype(slot)::value;
#pragma unroll
        for (int i = 0; i < XA; ++i) {
            if constexpr (ES == 4) {
                uint32_t tb[3][4];
#pragma unroll
                for (int e = 0; e < 4; ++e) split_bf16_terms(ra[q][i][e], tb[0][e], tb[1][e], tb[2][e]);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    *reinterpret_cast<u32x2 *>(&sX[buf][p][x_off[i]]) =
                        u32x2{tb[p][0] | (tb[p][1] << 16), tb[p][2] | (tb[p][3] << 16)};
            } else {
                uint32_t hw[4], mw[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t h0, m0_, l0, h1, m1, l1;
                    split_bf16_terms(f2u((float)__builtin_bit_cast(_Float16, (uint16_t)(ra[q][i][e] & 0xFFFFu))), h0, m0_, l0);
                    split_bf16_terms(f2u((float)__builtin_bit_cast(_Float16, (uint16_t)(ra[q][i][e] >> 16))), h1, m1, l1);
                    hw[e] = h0 | (h1 << 16);
                    mw[e] = m0_ | (m1 << 16);
                }
                *reinterpret_cast<u32x4 *>(&sX[buf][0][x_off[i]]) = u32x4{hw[0], hw[1], hw[2], hw[3]};
                *reinterpret_cast<u32x4 *>(&sX[buf][1][x_off[i]]) = u32x4{mw[0], mw[1], mw[2], mw[3]};
            }
        }
        if (t < WCH) *reinterpret_cast<u32x4 *>(&sW[buf][w_off]) = rw[q];
        if (t < BN) sS[buf][kg * BN + t] = rs[q];
    };

    v16f acc[CTW];
#pragma unroll
    for (int j = 0; j < CTW; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;

    // stage kt from LDS buffer kt % 2; stage kt + 1 (in slot `slot`) goes
    // to the other buffer and stage kt + 3 is loaded into the freed slot
    auto step = [&](int kt, auto slot) {
        const int buf = kt & 1;
        constexpr int NS = 4 / KS;                    // K-steps of 16 per wave per stage
        v8bf fw[CTW][NS];
#pragma unroll
        for (int j = 0; j < CTW; ++j) {
            const int col = wn * (BN / WN) + j * 32 + frow;
            const u32x4 pw = *reinterpret_cast<const u32x4 *>(&sW[buf][(2 * kg + half) * (BN * 16) + col * 16]);
            const float sc = e8m0_scale_f32((sS[buf][kg * BN + col] >> (8 * half)) & 0xFF);
#pragma unroll
            for (int ss = 0; ss < NS; ++ss) {
                const uint32_t cw = KS == 1 ? pw[ss] : pw[wk];
                const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(cw, sc, 0);
                const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(cw, sc, 1);
                const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(cw, sc, 2);
                const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(cw, sc, 3);
                fw[j][ss] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
            }
        }
        const int row = kg * BR + wm * 32 + frow;
#pragma unroll
        for (int ss = 0; ss < NS; ++ss) {
            const int s = wk + KS * ss;
            v8bf fa[NTERM];
#pragma unroll
            for (int p = 0; p < NTERM; ++p)
                fa[p] = *reinterpret_cast<const v8bf *>(&sX[buf][p][row * ROW_B + (((4 * half + s) ^ a_swz(row)) << 4)]);
#pragma unroll
            for (int j = 0; j < CTW; ++j)
#pragma unroll
                for (int p = 0; p < NTERM; ++p)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[p], fw[j][ss], acc[j], 0, 0, 0);
        }
        if (kt + 1 < nk) swrite(buf ^ 1, slot);
        if (kt + 3 < nk) gload(kt + 3, slot);
        __syncthreads();
    };
    constexpr SlotC<0> S0{};
    constexpr SlotC<1> S1{};
    gload(0, S0);
    swrite(0, S0);
    if (1 < nk) gload(1, S1);
    if (2 < nk) gload(2, S0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt += 2) {
        step(kt, S1);                   // stage kt + 1 sits in slot 1
        if (kt + 1 < nk) step(kt + 1, S0);
    }

    if constexpr (KS > 1) {
        // waves 1 .. KG * KS - 1 (wave wk of K group kg is kg * KS + wk)
        // hand their partial tiles to wave 0 through LDS (the staging planes
        // are free after the last barrier), which adds them in that order
        constexpr int NW = KG * KS;
        const int gwv = kg * KS + wk;
        float *red = reinterpret_cast<float *>(&sX[0][0][0]);
        static_assert(CTW == 1 && (NW - 1) * 16 * 64 * 4 <= (int)sizeof(sX), "reduction buffer");
        if (gwv > 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) red[((gwv - 1) * 16 + e) * 64 + lane] = acc[0][e];
        }
        __syncthreads();
        if (gwv > 0) return;
        // one partial tile at a time (unrolled over 15 tiles, the compiler
        // would issue all 240 reads at once and spill)
#pragma nounroll
        for (int w2 = 0; w2 < NW - 1; ++w2)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[0][e] += red[(w2 * 16 + e) * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < CTW; ++j) {
        const int64_t col = n0 + wn * (BN / WN) + j * 32 + frow;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int64_t row = m0 + wm * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
            if (row < g.M && col < g.N) store_cw<CT>(g.c, row * g.ldc + col, acc[j][e]);
        }
    }
}

hipError_t launch_gemm_xf4(const GemmArgs &g, int a_dtype, hipStream_t s) {
    // the widest tile whose grid still fills the CUs: 64 x 128, 64 x 64, or
    // 32 x 32 tiles split four ways along K
    auto tiles = [&](int br, int bn) { return ((g.M + br - 1) / br) * ((g.N + bn - 1) / bn); };
    const int cus = num_cus_w();
    // the 32 x 32 form: 4 K groups of 4 waves when the stage count allows
    // (each group runs a quarter of the stages; cfg1's 16 dependent stages
    // become 4)
    const int shape = tiles(64, 128) >= cus ? 0 : (tiles(64, 64) >= cus ? 1 : ((g.K / xf::BK) % 4 == 0 ? 3 : 2));
    const dim3 grid((unsigned)(shape == 0 ? tiles(64, 128) : shape == 1 ? tiles(64, 64) : tiles(32, 32))),
        blk(xf::NT), blk4(4 * xf::NT);
    const bool f = g.scale_fmt == LSMX_SCALE_F32;
#define LSMX_X(AT, F, CT)                                                                           \
    do {                                                                                            \
        if (shape == 0) hipLaunchKernelGGL((gemm_xf4_kernel<AT, F, CT, 64, 128, 1>), grid, blk, 0, s, g); \
        else if (shape == 1) hipLaunchKernelGGL((gemm_xf4_kernel<AT, F, CT, 64, 64, 1>), grid, blk, 0, s, g); \
        else if (shape == 3) hipLaunchKernelGGL((gemm_xf4_kernel<AT, F, CT, 32, 32, 4, 4>), grid, blk4, 0, s, g); \
        else hipLaunchKernelGGL((gemm_xf4_kernel<AT, F, CT, 32, 32, 4>), grid, blk, 0, s, g);       \
    } while (0)
#define LSMX_XC(AT, F)                                           \
    do {                                                         \
        if (g.c_dtype == LSMX_F32) LSMX_X(AT, F, LSMX_F32);      \
        else if (g.c_dtype == LSMX_BF16) LSMX_X(AT, F, LSMX_BF16); \
        else LSMX_X(AT, F, LSMX_F16);                            \
    } while (0)
    if (a_dtype == LSMX_F32) { if (f) LSMX_XC(LSMX_F32, true); else LSMX_XC(LSMX_F32, false); }
    else { if (f) LSMX_XC(LSMX_F16, true); else LSMX_XC(LSMX_F16, false); }
#undef LSMX_XC
#undef LSMX_X
    return hipGetLastError();
}

// ------------------------------------------------------------------ ring
// The large-M form: 256 "A rows" x 256 weight columns per workgroup of 8 waves
// (2 x 4, 128 x 64 per wave: two waves per SIMD, so one wave's MFMAs run
// while the other waits), a 3-slot LDS ring filled by direct-to-LDS loads
// (no VGPR staging), one barrier per 64-deep K stage.
//   - A stage is 128 bytes of every A row (64 bf16; 8 rows per load
//     instruction, chunk-swizzled) and 32 bytes of every W row (64 codes, two
//     MX blocks; 32 rows per load instruction).  Rows past the operand read
//     zeros through the buffer descriptor.
//   - At the barrier of stage u every wave has its own loads of stage u in
//     LDS and has finished stage u - 1, so the slot of stage u - 1 is free
//     and the loads of stage u + 2 go there, spread over the K-steps.
//     Stages past the end re-load the last stage (same slot pattern, no
//     branch), and the kernel waits for them before it exits.
//   - K positions: at K-step s lane half h supplies A[row][32h + 8s .. +8]
//     and the codes 8s .. 8s+7 of W's block h, so a lane dequantizes one
//     16-byte block per column tile per stage with one scale.
//   - A W load instruction covers 32 weight rows; its 1 KiB of LDS holds the
//     first 16-byte halves of those rows, then the second halves, so the 16
//     lanes a ds_read_b128 serves per cycle read 256 contiguous bytes.
//   - E8M0 block scales (row-major [N, K/32]) come 16 bytes per weight row =
//     8 stages at a time, into a 2-deep LDS buffer; the load for stages
//     8g .. 8g+7 is issued first in stage 8g - 2 (scale rows must be 16-byte
//     multiples: K % 512 == 0; fp32 scales use the VGPR-staged kernel).
namespace wr {
constexpr int BK = 64;
constexpr int NW = 8, NT = 64 * NW;
constexpr int WGM = 2, WGN = NW / WGM;      // 2 x 4 waves, 128 x 64 each
constexpr int NLW = 4;                      // loader waves
constexpr int BR = 256, BN = 256;           // A rows (all batches) x weight columns
constexpr int S = 3;                        // ring slots
constexpr int A_ROW_B = BK * 2, W_ROW_B = BK / 2;
constexpr int GROUP_M = 4;
LSMX_DEV int swz(int row) { return (row >> 1) & 7; }
}  // namespace wr

// Only waves 0-3 issue the stage loads: the two waves of a SIMD share its
// matrix core, the older one (0-3) wins issue arbitration and reaches the
// barrier first, so the younger one's instruction stream sets the stage's
// pace and is kept to LDS reads, dequantization and MFMAs.
template <bool V>
struct LoaderC {
    static constexpr bool value = V;
};
template <int NB, int CT>
__global__ __launch_bounds__(wr::NT, 1) void gemm_bf16f4_ring_kernel(GemmArgs g) {
    using namespace wr;
    constexpr int RPB = BR / NB;        // A rows per batch per workgroup
    constexpr int TM = BR / 32 / WGM, TN = BN / 32 / WGN;   // 32 x 32 tiles per wave
    static_assert(NB == 1 || TM * 32 <= RPB, "a wave's rows lie in one batch");
    constexpr int A_SLOT = BR * A_ROW_B, W_SLOT = BN * W_ROW_B;
    constexpr int XA = A_SLOT / 1024 / NLW;      // A load instructions per loader wave per stage
    constexpr int XW = BN / 32 / NLW;            // W load instructions (32 rows each)
    constexpr int L = XA + XW;                   // (scales: one more every 8 stages)
    static_assert(NLW * 64 == BN, "one scale load per loader wave");
    // The scales of stages 8g+8 .. 8g+15 are issued first among stage 8g+6's
    // loads and first read right after the barrier of stage 8g+8; the wait at
    // that barrier leaves (S - 2) L loads outstanding, which covers the scale
    // load only for this depth.
    static_assert(S == 3, "the scale prefetch distance assumes a 3-slot ring");
    __shared__ __attribute__((aligned(16))) uint8_t sA[S][A_SLOT];
    __shared__ __attribute__((aligned(16))) uint8_t sW[S][W_SLOT];
    __shared__ __attribute__((aligned(16))) uint8_t sS[2][BN * 16];   // [group & 1][row][16 scale bytes]

    const int tiles_m = (int)((g.M + RPB - 1) / RPB), tiles_n = (int)((g.N + BN - 1) / BN);
    const int tile = (int)blockIdx.x;
    int tm, tn;
    tile_coords(tile, tiles_m, tiles_n, GROUP_M, tm, tn);
    const int64_t m0 = (int64_t)tm * RPB, n0 = (int64_t)tn * BN;
    const int nk = (int)(g.K / BK);

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int frow = lane & 31, half = lane >> 5;

    // ---- DMA addressing (loader waves).  A load i of loader w covers slot
    // rows (i*NLW + w)*8 .. +7: lane -> row + lane/8, LDS chunk lane%8 holding
    // source chunk (lane%8) ^ swz(row).  All 8 rows of one instruction lie in
    // one batch.
    const int64_t lda_b = g.lda * 2;
    const int arow_l = lane >> 3;
    // Per load: the first byte and byte count of its rows at K offset 0,
    // loop-invariant, so that a stage's descriptors cost a 64-bit add and
    // subtract each (the scalar unit is shared by the CU's 8 waves).
    uint32_t a_off[XA];
    const uint8_t *a_base[XA];
    uint64_t a_bytes[XA];
#pragma unroll
    for (int i = 0; i < XA; ++i) {
        const int r0 = (i * NLW + wave) * 8;           // first slot row, wave-uniform
        const int b = NB == 2 ? r0 / RPB : 0;
        const int rb = r0 - b * RPB;                    // row inside the batch tile
        const int row = r0 + arow_l;
        a_off[i] = (uint32_t)(arow_l * lda_b + (((lane & 7) ^ swz(row)) << 4));
        a_base[i] = (b ? g.a1 : g.a) + (m0 + rb) * lda_b;
        // rows left in the operand from this instruction's first row, at most 8
        const int64_t left = g.M - (m0 + rb), rows = left < 8 ? (left > 0 ? left : 0) : 8;
        a_bytes[i] = rows > 0 ? (uint64_t)((rows - 1) * lda_b + g.K * 2) : 0;
    }
    // W: load j of loader w covers slot rows (j*NLW + w)*32 .. +31, lane -> row
    // lane%32, 16-byte half lane/32
    const uint32_t w_off = (uint32_t)((lane & 31) * g.ldb + (lane >> 5) * 16);
    const uint8_t *w_base[XW];
    uint64_t w_bytes[XW];
#pragma unroll
    for (int j = 0; j < XW; ++j) {
        const int wi = j * NLW + wave;
        w_base[j] = g.b + (n0 + wi * 32) * g.ldb;
        const int64_t left = g.N - (n0 + wi * 32), rows = left < 32 ? (left > 0 ? left : 0) : 32;
        w_bytes[j] = rows > 0 ? (uint64_t)((rows - 1) * g.ldb + g.K / 2) : 0;
    }
    // scales: loader w loads 16 bytes of weight rows 64 w + lane
    const int s_w = wave % NLW;
    const int64_t s_rows = g.N - n0;
    const uint8_t *s_base = reinterpret_cast<const uint8_t *>(g.sb) + n0 * g.ld_sb;
    const uint32_t s_off = (uint32_t)(((s_w * 64) + lane) * g.ld_sb);
    auto issue_scales = [&](int grp) __attribute__((always_inline)) {
        const int64_t ks = (int64_t)grp * 16;
        const int64_t rows = s_rows < BN ? s_rows : BN;
        const uint64_t bytes = (uint64_t)((rows - 1) * g.ld_sb + g.K / 32 - ks);
        dma_x4(s_off, buf_rsrc(s_base + ks, bytes), lds_u32(&sS[grp & 1][0]) + s_w * 1024);
    };

    auto issue = [&](int kt, int slot, int q) __attribute__((always_inline)) {
        const int64_t ko = (int64_t)kt * A_ROW_B;
        if (q < XA) {
            const uint64_t bytes = a_bytes[q] > 0 ? a_bytes[q] - (uint64_t)ko : 0;
            dma_x4(a_off[q], buf_rsrc(a_base[q] + ko, bytes),
                   lds_u32(&sA[0][0]) + slot * A_SLOT + (q * NLW + wave) * 1024);
        } else {
            const int j = q - XA;
            const int64_t kw = (int64_t)kt * W_ROW_B;
            const uint64_t bytes = w_bytes[j] > 0 ? w_bytes[j] - (uint64_t)kw : 0;
            dma_x4(w_off, buf_rsrc(w_base[j] + kw, bytes),
                   lds_u32(&sW[0][0]) + slot * W_SLOT + (j * NLW + wave) * 1024);
        }
    };


    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    int rowA[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) rowA[i] = wm * (TM * 32) + i * 32 + frow;
    auto body = [&](auto loader_c) __attribute__((always_inline)) {
    constexpr bool LOADER = decltype(loader_c)::value;
    // prologue: scales of stages 0..7, stages 0 .. S-2 in flight
    if constexpr (LOADER) {
        issue_scales(0);
#pragma unroll
        for (int p = 0; p < S - 1; ++p)
#pragma unroll
            for (int q = 0; q < L; ++q) issue(p < nk ? p : nk - 1, p, q);
    }
    // A stage's head: the W blocks and scales of this lane's columns and the
    // A fragments of its first K-step, read after its barrier; the rest of its
    // A fragments are read one K-step ahead.  (Reading the head during the
    // stage before needs that stage's loads one barrier earlier: the wait costs
    // more than the head read saves.)
    u32x4 wblk[TN];
    uint32_t sraw[TN];
    v8bf fa0[TM];
    auto read_head = [&](int uu) __attribute__((always_inline)) {
        const int sl = uu % S;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = wn * (TN * 32) + j * 32 + frow;
            wblk[j] = *reinterpret_cast<const u32x4 *>(&sW[sl][(wn * TN + j) * 1024 + half * 512 + frow * 16]);
            sraw[j] = sS[(uu >> 3) & 1][col * 16 + 2 * (uu & 7) + half];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int r = rowA[i];
            fa0[i] = *reinterpret_cast<const v8bf *>(&sA[sl][r * A_ROW_B + (((4 * half) ^ swz(r)) << 4)]);
        }
    };
    for (int u = 0; u < nk; ++u) {
        const int slot = u % S;
        // this thread's loads of stage u have landed (only the later stages up
        // to u + S - 2 may be outstanding, and a scale load issued before the
        // newest of them is waited for too); after the barrier everyone's
        // have, and slot (u + S - 1) % S = (u - 1) % S is no longer read (a
        // wave that issues no loads only meets the barrier)
        if constexpr (LOADER) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 2) * L) : "memory");
        else asm volatile("s_barrier" ::: "memory");
        read_head(u);
        const int kn = u + S - 1 < nk ? u + S - 1 : nk - 1;
        const int sn = (u + S - 1) % S;
        // scales of the next group of 8 stages, first of this stage's loads
        // (the next stage's vmcnt wait then also covers it)
        if constexpr (LOADER)
            if ((u & 7) == 6 && u + 2 < nk) issue_scales((u + 2) >> 3);
        u32x4 wcur[TN];
        float sc[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            wcur[j] = wblk[j];
            sc[j] = e8m0_scale_f32(sraw[j]);
        }
        v8bf fa[2][TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[0][i] = fa0[i];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            v8bf fw[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const uint32_t p = wcur[j][st];
                const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 0);
                const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 1);
                const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 2);
                const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 3);
                fw[j] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
            }
            // the next K-step's A fragments
            if (st < 3) {
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const int r = rowA[i];
                    fa[(st + 1) & 1][i] = *reinterpret_cast<const v8bf *>(
                        &sA[slot][r * A_ROW_B + (((4 * half + st + 1) ^ swz(r)) << 4)]);
                }
            }
            // loads of stage u + S - 1, spread over the K-steps
            if constexpr (LOADER)
#pragma unroll
                for (int q = 0; q < L; ++q)
                    if ((q * 4) / L == st) issue(kn, sn, q);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[st & 1][i], fw[j], acc[i][j], 0, 0, 0);
        }
    }
    };
    if (wave < NLW) body(LoaderC<true>{});
    else body(LoaderC<false>{});
    // no load may still be writing this workgroup's LDS when it exits
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // epilogue: acc element e of tile (i, j) is row i*32 + 8*(e/4) + 4*half + e%4, column j*32 + frow
    const int b = NB == 2 ? (wm * TM * 32) / RPB : 0;
    void *cb = b ? g.c1 : g.c;
    const int64_t rbase = m0 + wm * (TM * 32) - b * RPB;
    const int64_t cbase = n0 + wn * (TN * 32);
    if (((reinterpret_cast<uintptr_t>(cb) & 15) == 0) && g.ldc % 4 == 0 && g.ldc < ((int64_t)1 << 26) &&
        rbase + TM * 32 <= g.M && cbase + TN * 32 <= g.N) {
        // this wave's block lies inside C: a 4x4 transpose inside each quad
        // of lanes gives every lane 4 consecutive columns of one row (fp32
        // C: one 16-byte store each); for 16-bit C lanes 4 apart then trade
        // halves so each lane stores 8 columns (pack16_rows8).  Every store
        // is a wave-uniform row pointer plus a fixed lane offset.
        constexpr int EB = CT == LSMX_F32 ? 4 : 2;
        const int q = frow & 3;
        const uint8_t *cw = reinterpret_cast<const uint8_t *>(cb) + (rbase * g.ldc + cbase) * EB;
        if constexpr (CT == LSMX_F32) {
            const uint32_t loff = (uint32_t)(((4 * half + q) * g.ldc + (frow & ~3)) * EB);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    uint8_t *crow = const_cast<uint8_t *>(cw) + (i * 32 + 8 * gq) * g.ldc * EB;
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        float x[4] = {acc[i][j][4 * gq], acc[i][j][4 * gq + 1], acc[i][j][4 * gq + 2],
                                      acc[i][j][4 * gq + 3]};
                        quad_transpose(x, q);
                        *reinterpret_cast<u32x4 *>(crow + loff + j * 32 * EB) =
                            u32x4{f2u(x[0]), f2u(x[1]), f2u(x[2]), f2u(x[3])};
                    }
                }
        } else {
            const bool odd = (frow & 4) != 0;
            const uint32_t loff = (uint32_t)(((4 * half + q + (odd ? 8 : 0)) * g.ldc + (frow & ~7)) * EB);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    uint8_t *crow = const_cast<uint8_t *>(cw) + (i * 32 + 16 * p) * g.ldc * EB;
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const float x0[4] = {acc[i][j][8 * p], acc[i][j][8 * p + 1], acc[i][j][8 * p + 2],
                                             acc[i][j][8 * p + 3]};
                        const float x1[4] = {acc[i][j][8 * p + 4], acc[i][j][8 * p + 5], acc[i][j][8 * p + 6],
                                             acc[i][j][8 * p + 7]};
                        *reinterpret_cast<u32x4 *>(crow + loff + j * 32 * EB) = pack16_rows8<CT>(x0, x1, q, odd);
                    }
                }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t col = cbase + j * 32 + frow;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t row = rbase + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
                if (row < g.M && col < g.N) store_cw<CT>(cb, row * g.ldc + col, acc[i][j][e]);
            }
        }
}

template <int NB>
static hipError_t launch_ring(const GemmArgs &g, hipStream_t s) {
    constexpr int RPB = wr::BR / NB;
    const int tiles = (int)(((g.M + RPB - 1) / RPB) * ((g.N + wr::BN - 1) / wr::BN));
    const dim3 grid(tiles), blk(wr::NT);
#define LSMX_R(CT) hipLaunchKernelGGL((gemm_bf16f4_ring_kernel<NB, CT>), grid, blk, 0, s, g)
    if (g.c_dtype == LSMX_F32) LSMX_R(LSMX_F32);
    else if (g.c_dtype == LSMX_BF16) LSMX_R(LSMX_BF16);
    else LSMX_R(LSMX_F16);
#undef LSMX_R
    return hipGetLastError();
}

// the ring kernel reads E8M0 scales 16 bytes (8 stages) at a time
static bool ring_ok(const GemmArgs &g) {
    return g.scale_fmt == LSMX_SCALE_E8M0 && g.ld_sb % 16 == 0 && (reinterpret_cast<uintptr_t>(g.sb) & 15) == 0 &&
           g.K % 512 == 0;
}

// ------------------------------------------------------------------ skinny M
// For few activation rows (decode, M <= 32 per batch) the weight stream is the
// whole cost: N*K/2 bytes of codes against 2*M*K bytes of activations.  The
// 256-row tile above would leave most CUs idle, so this kernel spreads the
// weight over the chip instead:
//   - a workgroup owns 16*CT weight rows, its 8 waves split K: wave w takes
//     the 128-wide K chunks w, w + 8, w + 16, ...
//   - each lane loads one 16-byte MX block (32 codes) of one weight row per
//     chunk straight into registers, dequantizes it with
//     v_cvt_scalef32_pk_bf16_fp4, and feeds v_mfma_f32_16x16x32_bf16;
//   - the activation rows (MT tiles of 16, rows past M clamped) come straight
//     from global memory/L2, where they stay resident: they are tiny;
//   - the 8 partial sums are added in LDS in wave order and stored.
// K positions inside a chunk are assigned so that lane group q (lanes
// 16q..16q+15) of MFMA step s covers K = 128c + 32q + 8s .. +8 for both
// operands: one lane's 16 weight bytes are one block with one scale.
// Dual mode: virtual rows [0, M) are A0's and [M, 2M) are A1's, so the
// weight is streamed once for both batches.  The summation order of an
// output element depends on K only, so single and dual launches of the same
// M and K give identical bits.
namespace sk {
constexpr int WK = 8;  // waves per workgroup (K split)
constexpr int CHUNK = 128;
}  // namespace sk

typedef float v4f __attribute__((ext_vector_type(4)));

// MT <= 2: at most 128 VGPRs, so two workgroups (16 waves) share a CU.
template <int MT, int CT>
__global__ __launch_bounds__(64 * sk::WK, MT <= 2 ? 4 : 2) void gemm_bf16f4_skinny_kernel(GemmArgs g) {
    constexpr int U = MT == 1 ? 2 : 1;  // chunks in flight per wave
    __shared__ float red[sk::WK][MT * CT * 256];

    const int lane = threadIdx.x & 63, wk = threadIdx.x >> 6;
    const int j = lane & 15, grp = lane >> 4;
    const bool dual = g.a1 != nullptr;
    const int64_t VM = dual ? 2 * g.M : g.M;
    const int64_t nbase = (int64_t)blockIdx.x * (16 * CT);
    const bool sf32 = g.scale_fmt == LSMX_SCALE_F32;

    const uint8_t *arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int64_t v = min((int64_t)(16 * mt + j), VM - 1);
        const bool second = dual && v >= g.M;
        arow[mt] = (second ? g.a1 : g.a) + (second ? v - g.M : v) * g.lda * 2 + grp * 64;
    }
    const uint8_t *wrow[CT];
    int64_t srow[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int64_t n = min(nbase + 16 * ct + j, g.N - 1);
        wrow[ct] = g.b + n * g.ldb + grp * 16;
        srow[ct] = n * g.ld_sb + grp;
    }

    v4f acc[MT][CT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[mt][ct] = v4f{0.f, 0.f, 0.f, 0.f};

    const int nchunks = (int)(g.K / sk::CHUNK);
    for (int c0 = wk; c0 < nchunks; c0 += sk::WK * U) {
        u32x4 wv[U][CT], av[U][MT][4];
        uint32_t sv[U][CT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * sk::WK;
            if (c < nchunks) {
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    wv[u][ct] = *reinterpret_cast<const u32x4 *>(wrow[ct] + (int64_t)c * 64);
                    const int64_t so = srow[ct] + (int64_t)c * 4;
                    sv[u][ct] = sf32 ? f32_scale_e8m0(f2u(reinterpret_cast<const float *>(g.sb)[so]))
                                     : reinterpret_cast<const uint8_t *>(g.sb)[so];
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        av[u][mt][s] = *reinterpret_cast<const u32x4 *>(arow[mt] + (int64_t)c * 256 + s * 16);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u * sk::WK < nchunks) {
                float sc[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) sc[ct] = e8m0_scale_f32(sv[u][ct]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // dequantize step s of every column tile: codes 8s..8s+7 of the block
                    v8bf wf[CT];
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        const uint32_t p = wv[u][ct][s];
                        const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[ct], 0);
                        const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[ct], 1);
                        const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[ct], 2);
                        const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[ct], 3);
                        wf[ct] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        const v8bf fa = __builtin_bit_cast(v8bf, av[u][mt][s]);
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct)
                            acc[mt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa, wf[ct], acc[mt][ct], 0, 0, 0);
                    }
                }
            }
        }
    }

    // acc[mt][ct][r] = D[4*grp + r][j] of the 16 x 16 tile (rows: activation
    // rows of m-tile mt, columns: weight rows of col tile ct)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wk][(mt * CT + ct) * 256 + r * 64 + lane] = acc[mt][ct][r];
    __syncthreads();
    for (int p = wk; p < MT * CT; p += sk::WK) {
        const int mt = p / CT, ct = p % CT;
        const int64_t n = nbase + 16 * ct + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < sk::WK; ++w) v += red[w][p * 256 + r * 64 + lane];
            const int64_t vr = 16 * mt + 4 * grp + r;
            if (vr < VM && n < g.N) {
                const bool second = dual && vr >= g.M;
                void *cb = second ? g.c1 : g.c;
                const int64_t idx = (second ? vr - g.M : vr) * g.ldc + n;
                if (g.c_dtype == LSMX_F32) store_cw<LSMX_F32>(cb, idx, v);
                else if (g.c_dtype == LSMX_BF16) store_cw<LSMX_BF16>(cb, idx, v);
                else store_cw<LSMX_F16>(cb, idx, v);
            }
        }
    }
}

// ------------------------------------------------------------------ decode M
static int num_cus_w();
// Up to 16 activation rows per batch (dual: 32 virtual rows): the weight is
// read once, in whole 256-byte row pieces, with all of a workgroup's bytes in
// flight at once.
//   - a workgroup owns up to R weight rows (as many as spread the weight
//     evenly over the CUs, one workgroup each); its 8 waves split each
//     4096-deep K pass
//     into 512-deep slices (wave w: K = 512w .. 512w + 511, 256 bytes of
//     every row);
//   - at the start of a pass every wave issues its whole share: R/4 direct-
//     to-LDS loads of 4 rows x 256 contiguous bytes, the pass's E8M0 scales
//     (R rows x 128 E8M0 bytes, or 128 fp32 powers of two), and its
//     activation fragments into registers;
//     nothing is computed before they land, so a workgroup's latency is paid
//     once per pass while the other workgroups' loads keep HBM busy;
//   - lane (n, q) of MFMA step s (v_mfma_f32_16x16x32_bf16) reads 4 bytes
//     (8 codes) of weight row n: LDS chunk s of a row sits at 16 * (s ^ n),
//     which puts the 64 lanes of a ds_read_b32 on 64 distinct banks (the DMA
//     writes lanes in order, so the swizzle is applied by choosing each
//     lane's source chunk);
//   - v_cvt_scalef32_pk_bf16_fp4 expands the codes to bf16 with the block
//     scale (exact); the activation fragment of step s holds the same 8 K
//     positions (K = 32s + 8q .. +8 of the slice);
//   - the 8 waves' partial sums meet in LDS and are added in wave order.
// The summation order of an output element depends on K only, so single and
// dual launches of the same M give identical bits.
namespace dk {
constexpr int NW = 8, NT = 64 * NW;
constexpr int SLICE_K = 512;          // K per wave per pass
constexpr int PASS_K = NW * SLICE_K;  // 4096
constexpr int ROW_B = SLICE_K / 2;    // code bytes of one row per slice
}  // namespace dk

// 16-byte global load from inline asm: its completion is waited for with an
// explicit s_waitcnt, which counts it together with the direct-to-LDS loads.
LSMX_DEV u32x4 gload_x4(const void *p) {
    u32x4 v;
    asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(v) : "v"(p));
    return v;
}

// fp32 scale -> itself when it has an E8M0 form (a power of two in
// [2^-127, 2^127]), else NaN, without branches.
LSMX_DEV float f32_scale_nb(uint32_t b) {
    const bool ok = ((b & 0x807FFFFFu) == 0u && b - 0x00800000u <= 0x7E800000u) || b == 0x00400000u;
    return u2f(ok ? b : 0x7FC00000u);
}

// One workgroup per CU (the launcher gives each CU one share of the weight
// rows): 8 waves, two per SIMD, so up to 256 VGPRs per wave.
template <int MT, int R, int CT, bool SF32>
__global__ __launch_bounds__(dk::NT, 2) void gemm_bf16f4_decode_kernel(GemmArgs g) {
    using namespace dk;
    constexpr int TN = R / 16;                   // 16-column MFMA tiles
    constexpr int XW = R / 4;                    // weight loads per wave per pass
    constexpr int SV = SF32 ? 4 : 1;             // 16-byte scale vectors per row per slice
    static_assert(R % 16 == 0, "tile");
    __shared__ __attribute__((aligned(16))) uint8_t sW[NW][R * ROW_B];
    static_assert(sizeof(sW) >= (size_t)NW * MT * TN * 256 * 4, "reduction buffer");

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15, q = lane >> 4;
    const bool dual = g.a1 != nullptr;
    const int64_t VM = dual ? 2 * g.M : g.M;
    const int64_t n0 = (int64_t)blockIdx.x * g.rows_wg;
    const int64_t nend = min(n0 + g.rows_wg, g.N);   // rows past nend read zeros

    // activation rows of this lane (rows past VM repeat the last one; their
    // outputs are not stored)
    const uint8_t *arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int64_t v = min((int64_t)(16 * mt + n16), VM - 1);
        const bool second = dual && v >= g.M;
        arow[mt] = (second ? g.a1 : g.a) + (second ? v - g.M : v) * g.lda * 2 + q * 16;
    }
    // scale rows of this lane's weight rows (rows past nend repeat the last one)
    const uint8_t *srow[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t)
        srow[t] = reinterpret_cast<const uint8_t *>(g.sb) + min(n0 + 16 * t + n16, nend - 1) * g.ld_sb * (SF32 ? 4 : 1);
    // weight load j covers rows 4j .. 4j + 3: lane l -> row 4j + l/16, LDS
    // chunk l%16 holding source chunk (l%16) ^ (row & 15)
    uint32_t w_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 4 * j + (lane >> 4);
        w_off[j] = (uint32_t)((lane >> 4) * g.ldb + 16 * ((lane & 15) ^ (r & 15)));
    }

    // two accumulators per tile (even and odd K-steps), so that consecutive
    // MFMAs do not wait for each other's results; added at the end
    v4f acc[MT][TN][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[mt][t][0] = acc[mt][t][1] = v4f{0.f, 0.f, 0.f, 0.f};

#pragma nounroll
    for (int64_t kp = 0; kp < g.K; kp += PASS_K) {
        const int64_t k0 = kp + (int64_t)wave * SLICE_K;   // this wave's slice
        const bool live = k0 < g.K;                         // K % 512 == 0: whole slices
        if (kp > 0) __syncthreads();   // every wave is done with the previous pass's LDS
        if (live) {
            // The slice's 16 scales of each of this lane's weight rows and
            // its activation fragments, then its weight rows.  All are asm
            // loads counted by the explicit waits below: a compiler-visible
            // load would get a compiler wait that counts only its own loads
            // and so also waits for the weight loads issued after it.
            u32x4 sv[TN][SV];
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int v = 0; v < SV; ++v) sv[t][v] = gload_x4(srow[t] + (k0 / 32) * (SF32 ? 4 : 1) + 16 * v);
            u32x4 af[MT][16];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int s = 0; s < 16; ++s) af[mt][s] = gload_x4(arow[mt] + (k0 + 32 * s) * 2);
#pragma unroll
            for (int j = 0; j < XW; ++j) {
                const int64_t r0 = n0 + 4 * j, left = nend - r0;
                const uint64_t bytes = left > 0 ? (uint64_t)((left - 1) * g.ldb + (g.K - k0) / 2) : 0;
                dma_x4(w_off[j & 3], buf_rsrc(g.b + r0 * g.ldb + k0 / 2, bytes),
                       lds_u32(&sW[wave][0]) + j * 1024);
            }
            // The wave reads only the LDS its own loads wrote: no barrier.
            // Column tile t's rows are loads 4t .. 4t + 3, so its MFMAs start
            // once they (and everything issued before them) have landed,
            // while the later tiles' loads are still in flight.
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (TN - 1)) : "memory");
#pragma unroll
            for (int t = 0; t < TN; ++t)
#pragma unroll
                for (int v = 0; v < SV; ++v) asm volatile("" : "+v"(sv[t][v]));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int s = 0; s < 16; ++s) asm volatile("" : "+v"(af[mt][s]));
            // E8M0 bytes 0 and 255 need the exact conversion; any other byte
            // is 2^(e - 127) = e << 23.  Lane (n, q) tests dword q of its
            // row's 16 bytes, so the wave covers every byte once.
            bool exact = SF32;
            if constexpr (!SF32) {
                uint32_t hit = 0;
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    const uint32_t x = q == 0 ? sv[t][0].x : q == 1 ? sv[t][0].y : q == 2 ? sv[t][0].z : sv[t][0].w;
                    hit |= ((x - 0x01010101u) & ~x) | ((0xFEFEFEFEu - x) & x);   // a 00 or an FF byte
                }
                exact = __builtin_amdgcn_ballot_w64((hit & 0x80808080u) != 0u) != 0;
            }
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if (t > 0) {
                    // nothing moves across the wait: the tile before it
                    // computes while this tile's rows land
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (TN - 1 - t)) : "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                float sc[16];
                if (exact) {
#pragma unroll
                    for (int s = 0; s < 16; ++s)
                        sc[s] = SF32 ? f32_scale_nb(sv[t][s >> 2][s & 3])
                                     : e8m0_scale_f32((sv[t][0][s >> 2] >> (8 * (s & 3))) & 0xFFu);
                } else {
#pragma unroll
                    for (int s = 0; s < 16; ++s) sc[s] = u2f(((sv[t][0][s >> 2] >> (8 * (s & 3))) & 0xFFu) << 23);
                }
                // the tile's 16 code words in one batch of LDS reads (one
                // latency per tile instead of one per K-step)
                uint32_t pc[16];
#pragma unroll
                for (int s = 0; s < 16; ++s)
                    pc[s] = *reinterpret_cast<const uint32_t *>(&sW[wave][(16 * t + n16) * ROW_B + 16 * (s ^ n16) + 4 * q]);
                // dequantize four K-steps ahead of their MFMAs, into two
                // alternating register sets: an MFMA never waits for the
                // conversion just before it, and a conversion never
                // overwrites the operand of an MFMA still in flight
                v8bf wf[2][4];
                auto dequant = [&](int g4) __attribute__((always_inline)) {
#pragma unroll
                    for (int s1 = 0; s1 < 4; ++s1) {
                        const int s = 4 * g4 + s1;
                        const uint32_t p = pc[s];
                        const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[s], 0);
                        const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[s], 1);
                        const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[s], 2);
                        const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[s], 3);
                        wf[g4 & 1][s1] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
                    }
                };
                dequant(0);
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    if (g4 < 3) dequant(g4 + 1);
#pragma unroll
                    for (int s1 = 0; s1 < 4; ++s1) {
                        const int s = 4 * g4 + s1;
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            acc[mt][t][s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(v8bf, af[mt][s]), wf[g4 & 1][s1], acc[mt][t][s & 1], 0, 0, 0);
                    }
                }
            }
        }
    }

    // acc[mt][t][r] = D[4q + r][n16] of the 16 x 16 tile (rows: activation
    // rows of tile mt, columns: weight rows 16t ..); the 8 waves' partial
    // sums are added in wave order
    __syncthreads();
    float *red = reinterpret_cast<float *>(&sW[0][0]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[((wave * MT + mt) * TN + t) * 256 + r * 64 + lane] = acc[mt][t][0][r] + acc[mt][t][1][r];
    __syncthreads();
    for (int o = threadIdx.x; o < MT * TN * 256; o += NT) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += red[w * MT * TN * 256 + o];
        const int p = o >> 8, e = o & 255, r = e >> 6, l = e & 63;
        const int mt = p / TN, t = p % TN;
        const int64_t vr = 16 * mt + 4 * (l >> 4) + r, n = n0 + 16 * t + (l & 15);
        if (vr < VM && n < nend) {
            const bool second = dual && vr >= g.M;
            store_cw<CT>(second ? g.c1 : g.c, (second ? vr - g.M : vr) * g.ldc + n, v);
        }
    }
}

template <int R, int MT>
static hipError_t launch_decode_r(GemmArgs g, hipStream_t s) {
    // rows per workgroup: the weight spread evenly over the CUs, in whole
    // 4-row loads, at most R
    const int64_t cus = num_cus_w(), per = (g.N + cus - 1) / cus, rows = (per + 3) / 4 * 4;
    g.rows_wg = (int)(rows > R ? R : rows < 16 ? 16 : rows);
    const dim3 grid((unsigned)((g.N + g.rows_wg - 1) / g.rows_wg)), blk(dk::NT);
    const bool f = g.scale_fmt == LSMX_SCALE_F32;
#define LSMX_D(CT, F) hipLaunchKernelGGL((gemm_bf16f4_decode_kernel<MT, R, CT, F>), grid, blk, 0, s, g)
#define LSMX_DC(F)                                                    \
    do {                                                              \
        if (g.c_dtype == LSMX_F32) LSMX_D(LSMX_F32, F);               \
        else if (g.c_dtype == LSMX_BF16) LSMX_D(LSMX_BF16, F);        \
        else LSMX_D(LSMX_F16, F);                                     \
    } while (0)
    if (f) LSMX_DC(true);
    else LSMX_DC(false);
#undef LSMX_DC
#undef LSMX_D
    return hipGetLastError();
}

// up to 16 rows per batch (2 x 16 virtual rows for the dual form)
constexpr int64_t kDecodeMaxM = 16;
// up to 16 virtual rows: 64 weight rows per workgroup; 17 .. 32 (the dual
// form): 32, so that the second activation tile's registers fit
static hipError_t launch_decode(const GemmArgs &g, hipStream_t s) {
    const int64_t vm = g.a1 ? 2 * g.M : g.M;
    return vm <= 16 ? launch_decode_r<64, 1>(g, s) : launch_decode_r<32, 2>(g, s);
}

// The decode kernel's scale loads: 16-byte aligned rows of either format.  Up
// to one pass of K (PASS_K) E8M0 bytes and fp32 powers of two of the same
// scales run this kernel and give the same bits; past it, E8M0 calls with a
// workspace run K slices where gemm_bf16f4_slices says so.
static bool decode_ok(const GemmArgs &g) {
    return g.K % dk::SLICE_K == 0 && (reinterpret_cast<uintptr_t>(g.sb) & 15) == 0 && g.ld_sb % 16 == 0;
}

// ------------------------------------------------------------------ GEMV
// For one or two activation rows per batch (decode) the whole cost is reading
// W once, and the matrix cores have almost nothing to do.  This kernel reads
// W with fully contiguous loads and does the arithmetic on the VALU:
//   - the activation rows are staged once per workgroup in LDS;
//   - a wave owns RPW weight rows; lane l takes the MX blocks l, l + 64,
//     l + 128, ... of every row, so each load instruction reads 1 KiB of one
//     row in one piece, and all of a wave's weight loads are issued before
//     any arithmetic;
//   - v_cvt_scalef32_pk_bf16_fp4 expands a block to 32 bf16 (exact, block
//     scale applied) and v_dot2_f32_bf16 multiplies pairs with the
//     activations;
//   - the 64 lane partial sums of each (row, activation row) are added with a
//     fixed butterfly, so the order depends on K only.
// VM is the number of virtual activation rows (M, or 2M in dual mode).
namespace gv {
// 4 waves of 2 weight rows each (1792 workgroups at N = 14336): a 14336 x
// 4096 weight streams in 8.4 us against 8.9 us for 8-wave workgroups (896),
// 9.5 us for 2-wave ones and 9.5-9.8 us with 1 or 4 rows per wave.  Of the
// 8.4 us, the dequantize-and-dot arithmetic adds ~1.2 us and the activation
// staging ~0.5 us to the 6.8 us of the loads alone (a plain 31 MB read runs
// in 6.0 us); the lane sum on the vector ALU (wave_sum_fixed) took ~0.5 us
// off the arithmetic's share
constexpr int NT = 256;
constexpr int RPW = 2;
constexpr int UB = 2;     // groups of 64 blocks per lane in flight
}  // namespace gv

// Sum over the 64 lanes, the same in every lane, in a fixed tree on the
// vector ALU: pairs (l, l ^ 1), (l, l ^ 2) of each quad (DPP quad_perm), then
// the two quads of each 8 (row_half_mirror), the two halves of each row of
// 16 (row_mirror), then rows l, l ^ 16 and halves l, l ^ 32
// (v_permlane16_swap / v_permlane32_swap).  Each step adds a pair whose two
// lanes hold the same two values, and fp32 addition commutes, so all lanes
// end with the same bits.  Through __shfl_xor (LDS permutes) the six
// dependent steps cost ~0.5 us of the M = 1 GEMV.
LSMX_DEV float wave_sum_fixed(float v) {
    v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0xB1, 0xF, 0xF, false));
    v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0x4E, 0xF, 0xF, false));
    v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0x141, 0xF, 0xF, false));
    v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0x140, 0xF, 0xF, false));
    const auto s16 = __builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false);
    v = u2f(s16[0]) + u2f(s16[1]);
    const auto s32 = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false);
    return u2f(s32[0]) + u2f(s32[1]);
}

template <int VM, bool SF32, int CT>
__global__ __launch_bounds__(gv::NT) void gemv_bf16f4_kernel(GemmArgs g) {
    using namespace gv;
    extern __shared__ __attribute__((aligned(16))) uint8_t sact[];   // [VM][K] bf16
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t n0 = ((int64_t)blockIdx.x * (NT / 64) + wave) * RPW;
    const int nblk = (int)(g.K / 32);
    const bool dual = g.a1 != nullptr;

    // Stage the activation rows, 16 bytes per thread per step.  Lane l reads
    // the 64 bytes of block l (+ 64 k) as four 16-byte chunks, so 16 lanes
    // of one ds_read_b128 start 64 bytes apart; chunk q of block b is stored
    // at position (q + (b >> 2)) & 3 of the block, which puts those 16 lanes
    // on 16 distinct 16-byte bank groups (without it, 4-way conflicts).
    auto apos = [](int64_t b, int q) { return b * 64 + 16 * ((q + (int)(b >> 2)) & 3); };
    const int per_row = (int)(g.K / 8);   // 16-byte chunks per row
    // K % 512 == 0 (whole 64-chunk DMA instructions per row): the rows are
    // staged by direct-to-LDS loads issued before the weight loads.  A
    // staging load through registers would have to land before its LDS
    // store, and with vmcnt counting in issue order the weight stream could
    // only start after it; a DMA needs no register, so the weight loads go
    // out behind it at once and the wave waits for the DMA alone (all but
    // the newest 4 vector-memory operations: the first block group's weight
    // and scale loads, always issued) before the barrier.  Lane l of a DMA
    // writes chunk position p = its base + l; the swizzle is applied by
    // loading into position p the chunk that apos puts there.
    const bool dma_act = per_row % 64 == 0;
    if (dma_act) {
        for (int base = 64 * wave; base < VM * per_row; base += NT) {
            const int m = base / per_row;
            const bool second = dual && m >= (int)g.M;
            const uint8_t *row = (second ? g.a1 : g.a) + (int64_t)(second ? m - g.M : m) * g.lda * 2;
            const int p = base - m * per_row + lane, bk = p >> 2, slot = p & 3;
            const uint32_t voff = (uint32_t)((4 * bk + ((slot - (bk >> 2)) & 3)) * 16);
            dma_x4(voff, buf_rsrc(row, (uint64_t)g.K * 2),
                   lds_u32(sact) + (uint32_t)((int64_t)m * g.K * 2 + (int64_t)(base - m * per_row) * 16));
        }
    } else {
        for (int i = t; i < VM * per_row; i += NT) {
            const int m = i / per_row, c = i - m * per_row;
            const bool second = dual && m >= (int)g.M;
            const uint8_t *src = (second ? g.a1 : g.a) + (int64_t)(second ? m - g.M : m) * g.lda * 2 + c * 16;
            *reinterpret_cast<u32x4 *>(sact + ((int64_t)m * g.K * 2 + apos(c >> 2, c & 3))) =
                *reinterpret_cast<const u32x4 *>(src);
        }
    }

    const uint8_t *wrow[RPW];
    const uint8_t *srow[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int64_t n = min(n0 + r, g.N - 1);
        wrow[r] = g.b + n * g.ldb;
        srow[r] = reinterpret_cast<const uint8_t *>(g.sb) + n * g.ld_sb * (SF32 ? 4 : 1);
    }

    float acc[RPW][VM];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int m = 0; m < VM; ++m) acc[r][m] = 0.0f;

    u32x4 w[UB][RPW];
    uint32_t e[UB][RPW];
    // weight and scale loads of the UB block groups starting at b0 (blocks
    // past the row are skipped)
    auto wload = [&](int b0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const int b = b0 + 64 * u;
            if (b < nblk) {
#pragma unroll
                for (int r = 0; r < RPW; ++r) {
                    w[u][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wrow[r] + (int64_t)b * 16));
                    e[u][r] = SF32 ? f32_scale_e8m0(f2u(reinterpret_cast<const float *>(srow[r])[b])) : srow[r][b];
                }
            }
        }
    };
    wload(lane);       // the first weight loads are in flight across the barrier
    if (dma_act) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __syncthreads();
    for (int b0 = lane; b0 < nblk;) {
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const int b = b0 + 64 * u;
            if (b >= nblk) break;
            u32x4 av[VM][4];  // 32 bf16 of activation row m at K = 32b
#pragma unroll
            for (int m = 0; m < VM; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    av[m][q] = *reinterpret_cast<const u32x4 *>(sact + ((int64_t)m * g.K * 2 + apos(b, q)));
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const float sc = e8m0_scale_f32(e[u][r]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // dword q of the block: codes 8q .. 8q+7, low nibble first
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const v2bf d = p == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u][r][q], sc, 0)
                                     : p == 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u][r][q], sc, 1)
                                     : p == 2 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u][r][q], sc, 2)
                                              : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u][r][q], sc, 3);
#pragma unroll
                        for (int m = 0; m < VM; ++m) {  // activations 8q + 2p, 8q + 2p + 1 of the block
                            const u32x4 aq = av[m][q];
                            const uint32_t ap = p == 0 ? aq.x : p == 1 ? aq.y : p == 2 ? aq.z : aq.w;
                            acc[r][m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, ap), d, acc[r][m], false);
                        }
                    }
                }
            }
        }
        b0 += 64 * UB;
        if (b0 < nblk) wload(b0);
    }

#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int m = 0; m < VM; ++m) acc[r][m] = wave_sum_fixed(acc[r][m]);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int64_t n = n0 + r;
            if (n >= g.N) continue;
#pragma unroll
            for (int m = 0; m < VM; ++m) {
                if (m >= (dual ? 2 * g.M : g.M)) continue;
                const bool second = dual && m >= (int)g.M;
                const int64_t idx = (int64_t)(second ? m - g.M : m) * g.ldc + n;
                store_cw<CT>(second ? g.c1 : g.c, idx, acc[r][m]);
            }
        }
    }
}

// one activation row per batch (from two rows on the decode kernel is faster)
constexpr int64_t kGemvMaxM = 1;
constexpr int64_t kGemvMaxLds = 64 * 1024;   // activation bytes staged per workgroup

static hipError_t launch_gemv(const GemmArgs &g, hipStream_t s) {
    const int vm = (int)(g.a1 ? 2 * g.M : g.M);
    const int vmt = vm == 1 ? 1 : vm == 2 ? 2 : 4;
    const size_t lds = (size_t)vmt * g.K * 2;
    const int rows_per_wg = (gv::NT / 64) * gv::RPW;
    const dim3 grid((unsigned)((g.N + rows_per_wg - 1) / rows_per_wg)), blk(gv::NT);
    const bool f = g.scale_fmt == LSMX_SCALE_F32;
#define LSMX_V(VMT, F, CT) hipLaunchKernelGGL((gemv_bf16f4_kernel<VMT, F, CT>), grid, blk, lds, s, g)
#define LSMX_VC(VMT, F)                                               \
    do {                                                              \
        if (g.c_dtype == LSMX_F32) LSMX_V(VMT, F, LSMX_F32);          \
        else if (g.c_dtype == LSMX_BF16) LSMX_V(VMT, F, LSMX_BF16);   \
        else LSMX_V(VMT, F, LSMX_F16);                                \
    } while (0)
    if (vmt == 1) { if (f) LSMX_VC(1, true); else LSMX_VC(1, false); }
    else if (vmt == 2) { if (f) LSMX_VC(2, true); else LSMX_VC(2, false); }
    else { if (f) LSMX_VC(4, true); else LSMX_VC(4, false); }
#undef LSMX_VC
#undef LSMX_V
    return hipGetLastError();
}

// up to 32 rows per batch (M = 16 against a 14336 x 4096 weight: 20 us against 34 us for the 128-row
// ring tile, whose MFMAs would be 7/8 padding; from M = 64 the ring is faster)
constexpr int64_t kSkinnyMaxM = 32;

static int num_cus_w() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            cus = n;
        else
            cus = 256;
    }
    return cus;
}

// 16-row weight tiles per workgroup: two (the activation loads then serve
// twice the weight bytes) while that still gives every CU a workgroup and the
// activation tiles are at most 4; two workgroups are resident per CU either
// way with up to 2 of them
static int skinny_ct(int64_t vm, int64_t N) { return vm <= 64 && (N + 31) / 32 >= num_cus_w() ? 2 : 1; }
static hipError_t launch_skinny(const GemmArgs &g, hipStream_t s) {
    const int64_t vm = g.a1 ? 2 * g.M : g.M;
    const int mt = vm <= 16 ? 1 : vm <= 32 ? 2 : vm <= 64 ? 4 : 8;
    const int ct = skinny_ct(vm, g.N);
    const dim3 grid((unsigned)((g.N + 16 * ct - 1) / (16 * ct))), blk(64 * sk::WK);
#define LSMX_S(MT, CT) hipLaunchKernelGGL((gemm_bf16f4_skinny_kernel<MT, CT>), grid, blk, 0, s, g)
    switch (mt * 10 + ct) {
        case 11: LSMX_S(1, 1); break;
        case 12: LSMX_S(1, 2); break;
        case 21: LSMX_S(2, 1); break;
        case 22: LSMX_S(2, 2); break;
        case 41: LSMX_S(4, 1); break;
        case 42: LSMX_S(4, 2); break;
        default: LSMX_S(8, 1); break;
    }
#undef LSMX_S
    return hipGetLastError();
}

template <int NB, int BR, int BN>
static hipError_t launch_w4(const GemmArgs &g, hipStream_t s) {
    constexpr int RPB = BR / NB;
    const int tiles = (int)(((g.M + RPB - 1) / RPB) * ((g.N + BN - 1) / BN));
    const dim3 grid(tiles), blk(w4::NT);
    const bool f = g.scale_fmt == LSMX_SCALE_F32;
#define LSMX_W(F, CT) hipLaunchKernelGGL((gemm_bf16f4_kernel<NB, F, CT, BR, BN>), grid, blk, 0, s, g)
    if (f) {
        if (g.c_dtype == LSMX_F32) LSMX_W(true, LSMX_F32);
        else if (g.c_dtype == LSMX_BF16) LSMX_W(true, LSMX_BF16);
        else LSMX_W(true, LSMX_F16);
    } else {
        if (g.c_dtype == LSMX_F32) LSMX_W(false, LSMX_F32);
        else if (g.c_dtype == LSMX_BF16) LSMX_W(false, LSMX_BF16);
        else LSMX_W(false, LSMX_F16);
    }
#undef LSMX_W
    return hipGetLastError();
}

// What the tile kernel does not take (fp32 scales, rows that are not 4-byte
// aligned): the largest VGPR-staged tile that still gives every CU a
// workgroup: 256 x 256, then 128 x 128, then 128 x 64
template <int NB>
static hipError_t launch_w4_any(const GemmArgs &g, hipStream_t s) {
    auto tiles = [&](int br, int bn) { return ((g.M + br / NB - 1) / (br / NB)) * ((g.N + bn - 1) / bn); };
    const int64_t cus = num_cus_w();
    if (tiles(256, 256) >= cus) return launch_w4<NB, 256, 256>(g, s);
    if (tiles(128, 128) >= cus) return launch_w4<NB, 128, 128>(g, s);
    return launch_w4<NB, 128, 64>(g, s);
}

// ------------------------------------------------------------------ tiles
// 17 activation rows up to where the 256 x 256 ring fills the CUs: one tile of
// BM rows x BN weight columns of one batch per workgroup, WM x WN MFMA waves
// of TM x TN 32 x 32 tiles each, and 4 loader waves.
//
// What bounds it: at few rows the stream of weights and, per weight column
// tile, the re-reading of the activations from L2; at a few hundred rows the
// matrix cores, and before that tiles that do not divide the CUs evenly.  So
// the tile and the number of K slices are chosen by the shape (bf16f4_plan).
// A stage is 128 K: 256 bytes of every A row, 64 bytes (4 MX blocks) of every
// weight row.  The ring is as deep as the LDS allows and the loads come from
// waves of their own, since an MFMA behind a load that waits for a place in
// the memory pipeline would wait too.  E8M0 scales (row-major) come 16 bytes
// per weight row, 4 stages, at a time.
//
// K order: sub-stage g (64 K), K-step st: lane half h supplies A[row][64 g +
// 32 h + 8 st .. +8] and codes 8 st .. of W's block 2 g + h -- the ring
// kernel's order, so a whole-K output has the ring kernel's bits whatever
// the tile.  With g.splits > 1 workgroup (tile, slice) sums its run of
// stages and writes an fp32 partial tile; splitk_reduce_kernel adds the
// slices in slice order.
namespace wt {
constexpr int BK = 128, NLW = 4, GROUP_M = 4;
constexpr int A_ROW_B = BK * 2, W_ROW_B = BK / 2;
constexpr int lds(int bm, int bn, int s) { return s * (bm * A_ROW_B + bn * W_ROW_B) + ((s + 3) / 4 + 1) * bn * 16; }
// two workgroups per CU where the LDS holds both rings
constexpr int waves_per_simd(int bm, int bn, int s, int waves) { return waves / 4 * (2 * lds(bm, bn, s) <= 160 * 1024 ? 2 : 1); }
}  // namespace wt
// VEC: C starts at a multiple of 16 bytes, its rows at multiples of 4 elements
// (8 bytes of a 16-bit output, the width of its stores).
template <int CT, bool SPLITK, int WM, int WN, int TM, int TN, int S, int LA, bool VEC>
__global__ __launch_bounds__(64 * (WM * WN + wt::NLW), wt::waves_per_simd(32 * TM * WM, 32 * TN * WN, S, WM * WN + wt::NLW))
void gemm_bf16f4_tile_kernel(GemmArgs g) {
    using namespace wt;
    constexpr int NMW = WM * WN;
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
    constexpr int A_SLOT = BM * A_ROW_B, SLOT = A_SLOT + BN * W_ROW_B;
    constexpr int XA = BM / (4 * NLW), XW = BN / (16 * NLW), L = XA + XW;   // loads per loader lane per stage
    constexpr int NSB = (S + 3) / 4 + 1;            // scale buffers: groups of 4 stages in use or in flight
    constexpr int NSG = (BN + 63) / 64;             // 64-row scale loads per group
    static_assert(XA * 4 * NLW == BM && XW * 16 * NLW == BN, "whole DMA instructions");
    static_assert(lds(BM, BN, S) <= 160 * 1024 && (S - 1) * (L + 1) < 63, "LDS, vmcnt");
    constexpr int OFF_S = S * SLOT;
    __shared__ __attribute__((aligned(16))) uint8_t ring[lds(BM, BN, S)];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = g.a1 ? 2 : 1;
    const int tiles_m = (int)((g.M + BM - 1) / BM), tiles_n = (int)((g.N + BN - 1) / BN);
    // blockIdx -> (tile, batch, K slice): the batches of one (m, n) tile are
    // neighbours, which share its weights in L2
    int id = (int)blockIdx.x;
    if ((gridDim.x & 7) == 0) id = (id & 7) * ((int)gridDim.x >> 3) + (id >> 3);
    const int split = SPLITK ? id % g.splits : 0;
    if (SPLITK) id /= g.splits;
    const int batch = nb == 2 ? (id & 1) : 0;
    int tm, tn;
    group_coords(nb == 2 ? id >> 1 : id, make_tile_map(tiles_m, tiles_n, GROUP_M), tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    // this slice's stages
    const int nk_all = (int)(g.K / BK);
    const int k0 = SPLITK ? (int)((int64_t)nk_all * split / g.splits) : 0;
    const int nk = (SPLITK ? (int)((int64_t)nk_all * (split + 1) / g.splits) : nk_all) - k0;

    if (wave >= NMW) {
        // ---- loader waves
        __builtin_amdgcn_s_setprio(3);
        const int lw = wave - NMW;
        // A load i: rows (i * 4 + lw) * 4 + lane / 16, LDS chunk lane % 16
        // holding source chunk (lane % 16) ^ (row & 15)
        const int ar = lw * 4 + (lane >> 4);
        const uint32_t a_off = (uint32_t)(ar * g.lda * 2 + (((lane & 15) ^ (ar & 15)) << 4));
        const uint32_t a_step = (uint32_t)(4 * NLW * g.lda * 2);
        // W load i: rows (i * 4 + lw) * 16 + lane / 4, LDS chunk lane % 4
        // holding source chunk (lane % 4) ^ ((row >> 2) & 3)
        const int wrw = lw * 16 + (lane >> 2);
        const uint32_t w_off = (uint32_t)(wrw * g.ldb + (((lane & 3) ^ ((wrw >> 2) & 3)) << 4));
        const uint32_t w_step = (uint32_t)(16 * NLW * g.ldb);
        const int sg = lw < NSG ? lw : NSG - 1;     // this wave's 64 rows of scales (the last ones repeat)
        const uint32_t s_off = (uint32_t)((sg * 64 + lane) * g.ld_sb);
        const int64_t nrow = min(g.N - n0, (int64_t)BN);
        const uint8_t *pa = (batch ? g.a1 : g.a) + m0 * g.lda * 2 + (int64_t)k0 * A_ROW_B;
        const uint8_t *pw = g.b + n0 * g.ldb + (int64_t)k0 * W_ROW_B;
        const uint8_t *ps = reinterpret_cast<const uint8_t *>(g.sb) + n0 * g.ld_sb + (int64_t)k0 * (BK / 32);
        const int64_t kl = g.K - (int64_t)k0 * BK;  // K left from this slice's start
        const int64_t na = ((min(g.M - m0, (int64_t)BM) - 1) * g.lda + kl) * 2;
        const int64_t nw = (nrow - 1) * g.ldb + kl / 2;
        const int64_t ns = (nrow - 1) * g.ld_sb + kl / 32;
        const uint32_t ring0 = lds_u32(&ring[0]);
        auto load_stage = [&](int kt, uint32_t so) __attribute__((always_inline)) {
            const bool past = kt >= nk;   // refills past the end: empty descriptors, zeros
            // the scales of stages kt .. kt + 3, ahead of the first of them;
            // bytes past a row's end are other scales or zeros, never used
            if ((kt & 3) == 0) {
                const int64_t o = (int64_t)kt * (BK / 32);
                dma_x4(s_off, buf_rsrc(ps + (past ? 0 : o), past ? 0 : (uint64_t)(ns - o)),
                       ring0 + OFF_S + ((kt >> 2) % NSB) * (BN * 16) + sg * 1024);
            }
            const int64_t ao = (int64_t)kt * A_ROW_B, wo = (int64_t)kt * W_ROW_B;
            const v4i_rsrc ra = buf_rsrc(pa + (past ? 0 : ao), past ? 0 : (uint64_t)(na - ao));
            const v4i_rsrc rw = buf_rsrc(pw + (past ? 0 : wo), past ? 0 : (uint64_t)(nw - wo));
#pragma unroll
            for (int i = 0; i < XW; ++i) dma_x4(w_off + i * w_step, rw, ring0 + so + A_SLOT + (i * NLW + lw) * 1024);
#pragma unroll
            for (int i = 0; i < XA; ++i) dma_x4(a_off + i * a_step, ra, ring0 + so + (i * NLW + lw) * 1024);
        };
#pragma unroll
        for (int q = 0; q < S; ++q) load_stage(q, q * SLOT);
        // (the scale loads among the newest only make these waits stricter)
        wait_vm_barrier<(S - 1) * L>();
        uint32_t so = 0;
        for (int kt = 0; kt < nk; ++kt) {
            wait_vm_barrier<(S - 2) * L>();
            load_stage(kt + S, so);
            so = so + SLOT == S * SLOT ? 0 : so + SLOT;
        }
        // no load may still be writing this workgroup's LDS when it exits
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }

    // ---- MFMA waves
    const int wm = wave / WN, wn = wave % WN;
    const int frow = lane & 31, half = lane >> 5;
    uint32_t aoff[4];   // A chunk 4 half + st of row frow; sub-stage g flips bit 3 of the chunk
#pragma unroll
    for (int st = 0; st < 4; ++st)
        aoff[st] = (uint32_t)((wm * TM * 32 + frow) * A_ROW_B + (((4 * half + st) ^ (frow & 15)) << 4));
    uint32_t woff[2];   // W chunk 2 g + half of row frow
#pragma unroll
    for (int q = 0; q < 2; ++q)
        woff[q] = (uint32_t)(A_SLOT + (wn * TN * 32 + frow) * W_ROW_B + (((2 * q + half) ^ ((frow >> 2) & 3)) << 4));
    const uint32_t soff = (uint32_t)(OFF_S + (wn * TN * 32 + frow) * 16);
    v16f acc[TM][TN];
    v8bf fa[2][LA][TM];     // A fragments of LA K-steps, and of the next LA
    u32x4 wb[2][TN];        // weight blocks of the sub-stage in use and of the next one
    uint32_t sraw[TN], snext[TN];
    float sc[TN];
    auto read_a = [&](uint32_t so, int k, int i) __attribute__((always_inline)) {   // K-step k = 4 g + st
        fa[(k / LA) & 1][k % LA][i] = *reinterpret_cast<const v8bf *>(&ring[0] + so + i * 32 * A_ROW_B + (aoff[k & 3] ^ ((k >> 2) << 7)));
    };
    auto read_w = [&](uint32_t so, int gq, int j) __attribute__((always_inline)) {
        wb[gq][j] = *reinterpret_cast<const u32x4 *>(&ring[0] + so + j * 32 * W_ROW_B + woff[gq]);
    };
    auto read_s = [&](int kt, int j) __attribute__((always_inline)) {
        snext[j] = *reinterpret_cast<const uint32_t *>(&ring[0] + soff + ((kt >> 2) % NSB) * (BN * 16) + (kt & 3) * 4 +
                                                       j * 32 * 16);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int j = 0; j < TN; ++j) read_s(0, j);
#pragma unroll
    for (int j = 0; j < TN; ++j) read_w(0, 0, j);
#pragma unroll
    for (int k = 0; k < LA; ++k)
#pragma unroll
        for (int i = 0; i < TM; ++i) read_a(0, k, i);
    uint32_t so = 0;
    for (int kt = 0; kt < nk; ++kt) {
        const uint32_t sn = so + SLOT == S * SLOT ? 0 : so + SLOT;
#pragma unroll
        for (int j = 0; j < TN; ++j) sraw[j] = snext[j];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int gq = k >> 2, st = k & 3;
            if (k == 8 - LA) {
                // this wave's reads of the slot are complete; past the
                // barrier it may be refilled and stage kt + 1 has landed
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            v8bf fw[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if (st == 0) sc[j] = e8m0_scale_f32((sraw[j] >> (8 * (2 * gq + half))) & 0xFFu);
                const uint32_t p = wb[gq][j][st];
                const v2bf d0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 0);
                const v2bf d1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 1);
                const v2bf d2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 2);
                const v2bf d3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(p, sc[j], 3);
                fw[j] = v8bf{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
            }
            // every LA K-steps the A fragments of the next LA; the weight
            // blocks a sub-stage ahead; the next stage's scales with its first
            // fragments
            if (k % LA == 0) {
                if (k == 0)
#pragma unroll
                    for (int j = 0; j < TN; ++j) read_w(so, 1, j);
                if (k == 8 - LA)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        read_s(kt + 1, j);
                        read_w(sn, 0, j);
                    }
#pragma unroll
                for (int x = 0; x < LA; ++x)
#pragma unroll
                    for (int i = 0; i < TM; ++i) read_a(k < 8 - LA ? so : sn, (k + LA + x) & 7, i);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[(k / LA) & 1][k % LA][i], fw[j], acc[i][j], 0, 0, 0);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
        so = sn;
    }

    // ---- epilogue: acc element e of tile (i, j) sits at row i*32 + 8*(e/4) +
    //      4*half + e%4, column j*32 + frow; a 4x4 transpose inside each quad
    //      of lanes gives every lane 4 consecutive columns of one row
    const int q = frow & 3;
    if constexpr (SPLITK) {
        // partial tile of this slice: [splits][nb][Mp][Np], Mp and Np padded
        // to whole tiles, so every store is in bounds
        const int64_t Mp = (int64_t)tiles_m * BM, Np = (int64_t)tiles_n * BN;
        float *pt = g.ws + ((int64_t)split * nb + batch) * Mp * Np;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int gr = 0; gr < 4; ++gr) {
                const int64_t row = m0 + (wm * TM + i) * 32 + 8 * gr + 4 * half + q;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    float x[4] = {acc[i][j][4 * gr], acc[i][j][4 * gr + 1], acc[i][j][4 * gr + 2], acc[i][j][4 * gr + 3]};
                    quad_transpose(x, q);
                    const int64_t col = n0 + (wn * TN + j) * 32 + (frow & ~3);
                    // rows past M are never read by the reduction, which reads
                    // each other value once
                    if (row < g.M)
                        __builtin_nontemporal_store(u32x4{f2u(x[0]), f2u(x[1]), f2u(x[2]), f2u(x[3])},
                                                    reinterpret_cast<u32x4 *>(pt + row * Np + col));
                }
            }
    } else {
        void *c = batch ? g.c1 : g.c;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int gr = 0; gr < 4; ++gr) {
                const int64_t row = m0 + (wm * TM + i) * 32 + 8 * gr + 4 * half;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int64_t col = n0 + (wn * TN + j) * 32;
                    if constexpr (VEC) {
                        float x[4] = {acc[i][j][4 * gr], acc[i][j][4 * gr + 1], acc[i][j][4 * gr + 2], acc[i][j][4 * gr + 3]};
                        // all four lanes of a quad take part in the exchanges
                        quad_transpose(x, q);
                        const int64_t cq = col + (frow & ~3);
                        if (row + q < g.M && cq < g.N) {
                            if (cq + 4 <= g.N) store_c4<CT>(c, (row + q) * g.ldc + cq, x[0], x[1], x[2], x[3]);
                            else
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    if (cq + k < g.N) store_c<CT>(c, (row + q) * g.ldc + cq + k, x[k]);
                        }
                    } else {
                        // rows at any alignment: one element per lane, 32
                        // columns of 2 rows per store (as quads of 4
                        // columns each store touched 16 rows: 252 x 33771 x
                        // 384 21.7 us on this tile, 19.1 so)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (row + e < g.M && col + frow < g.N)
                                store_c<CT>(c, (row + e) * g.ldc + col + frow, acc[i][j][4 * gr + e]);
                    }
                }
            }
    }
}

// ------------------------------------------------------------------ plan
// Tile and K slices of a shape.  Output tiles (tile_time; us, stages of 128
// K): graph-replayed launches of every tile at 30 shapes, M 4 .. 4096, N 1000
// .. 16384, K 1024 .. 14336; kRingTile is the 256 x 256 ring.
//   M x N x K        32x128  64x128 128x128 128x256 192x256  ring (256 x 256)
//   20x4096x4096       13.2    16.4                                     us
//   128x14336x4096             19.9    26.5
//   200x14336x4096             34.5    28.5    44.1
//   600x4096x4096              33.1    25.7
//   300x14336x4096             50.1    50.6    44.4    60.5
//   600x14336x4096             85.5    83.3            68.7    85.0
//   1000x14336x4096                   113.3   103.4           104.1
//   4096x4096x4096                    121.3   111.9           107.4
// K slices: partials and their reduction add ~1.2 us and, per slice, 0.45 us +
// 0.6 us per MB, which pays where few tiles face a long K: 20x4096x14336 whole
// K 38 us, 7 or 8 slices 13.6 (8 is the plan's); 64x4096x14336 45 and 17;
// 200x1024x4096 16 and 12.3.
static const TileCost kTiles[] = {
    {32, 128, 2, 3.5f, 0.33f, 0.55f},  {64, 128, 2, 4.0f, 0.42f, 0.95f},  {128, 128, 1, 4.5f, 0.64f, 0.86f},
    {128, 256, 1, 4.5f, 1.20f, 1.66f}, {192, 256, 1, 5.5f, 1.80f, 2.05f}, {256, 256, 1, 8.0f, 2.20f, 3.05f},
};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]), kRingTile = kNumTiles - 1;
// The same tiles at K <= 512 (kShortStages), where ramp and stores of a round
// outweigh its stages and the fits above put the 256-column tiles 20 to 40% too
// low: fits of 590 shapes, M 33 .. 32768, N 64 .. 65536, that pick the fastest
// tile or one within 0.4% of it on average, 14% at worst.
//   M x N x K              64x128  192x256  ring (256 x 256)
//   30508x384x256            18.0     23.8             us
//   2309x48000x512 (dual)   332.5    320.9    247.6
//   12189x29056x512                    507      436
constexpr int kShortStages = 4;
static const TileCost kShortTiles[] = {
    {32, 128, 2, 4.10f, 0.13f, 0.634f, -0.41f}, {64, 128, 2, 4.41f, 0.27f, 0.94f, -1.18f},
    {128, 128, 1, 5.75f, 0.40f, 0.915f, -1.45f}, {128, 256, 1, 6.93f, 0.81f, 1.84f, -1.10f},
    {192, 256, 1, 8.27f, 1.14f, 2.72f, -0.62f},  {256, 256, 1, 9.67f, 2.35f, 3.21f, -3.00f},
};

// Bytes of fp32 partials a shape may use (one batch): what fills the CUs once
// with 128-row tiles of 256 or 128 columns in 2 or 4 slices.  0 where whole-K
// tiles do as well: half of the CUs filled already, one pass of the decode
// kernel (M <= 16, K <= 4096), or up to 64 rows against more than 16 weight
// rows per CU unless K is the long side.
static int64_t split_budget(int64_t M, int64_t N, int64_t K) {
    const int64_t mt = (M + 127) / 128, cus = num_cus_w();
    if (M <= 1 || (M <= kDecodeMaxM && K <= dk::PASS_K)) return 0;
    if (M <= 64 && N > 16 * cus && K <= 2 * N) return 0;
    if (2 * mt * ((N + 255) / 256) > cus) return 0;
    int64_t best_wg = 0, best_bytes = 0;
    for (int bn = 256; bn >= 128; bn /= 2)
        for (int sp = 2; sp <= 4; sp *= 2) {
            const int64_t nt = (N + bn - 1) / bn, wg = mt * nt * sp, bytes = sp * nt * bn;
            if (wg > cus || K < 512 * sp) continue;
            if (wg > best_wg || (wg == best_wg && bytes < best_bytes)) best_wg = wg, best_bytes = bytes;
        }
    return best_bytes * mt * 128 * 4;
}

struct Plan {
    int tile, splits;
    float us;
};
static int64_t partial_bytes(const TileCost &c, int64_t M, int64_t N, int splits) {
    return splits < 2 ? 0 : splits * ((M + c.bm - 1) / c.bm * c.bm) * ((N + c.bn - 1) / c.bn * c.bn) * 4;
}
// The fastest tile for `splits` slices (0: any number of slices) of nb batches
// within `budget` bytes of partials per batch.  The ring kernel counts its 256
// rows over both batches.
static Plan best_plan(int64_t M, int64_t N, int64_t K, int nb, int splits, int64_t budget, bool ring) {
    const int cus = num_cus_w();
    const int64_t nk = K / wt::BK;
    const int most = splits ? splits : imax(1, imin(16, (int)imin((int)nk, 1 << 20) / 2));
    Plan best{0, 1, 1e30f};
    for (int i = 0; i < kNumTiles; ++i) {
        if (i == kRingTile && (splits > 1 || !ring)) continue;
        const TileCost &c = nk <= kShortStages ? kShortTiles[i] : kTiles[i];
        const int64_t bm = i == kRingTile ? c.bm / nb : c.bm;
        const int64_t tiles = ((M + bm - 1) / bm) * ((N + c.bn - 1) / c.bn) * (i == kRingTile ? 1 : nb);
        const int64_t slice = partial_bytes(c, M, N, 2) / 2;
        for (int sp = splits ? splits : 1; sp <= (i == kRingTile ? 1 : most); ++sp) {
            if (sp > 1 && sp * slice > budget) break;
            float t = tile_time(c, tiles * sp, (nk + sp - 1) / sp, cus);
            if (sp > 1) t += 1.2f + (float)sp * (0.45f + 0.6e-6f * (float)(nb * M * N * 4));
            if (t < best.us) best = Plan{i, sp, t};
        }
    }
    return best;
}

// Time (us) of the skinny kernel at vm activation rows, a fit of 370 shapes,
// M 1 .. 32, N 64 .. 65536, K 128 .. 28672, within 10%: a launch, then per 1024 K
// one pass of 16 (32) weight rows per workgroup, and each further workgroup of
// a CU.
static float skinny_time(int64_t vm, int64_t N, int64_t K) {
    const int64_t cus = num_cus_w();
    const int ct = skinny_ct(vm, N);
    const float more = (float)((N + 16 * ct * cus - 1) / (16 * ct * cus) - 1), v = (float)vm;
    return 2.5f + 0.5f * more + (float)K / 1024.0f * (0.42f + 0.05f * v + more * (0.62f + 0.045f * v)) * (ct == 2 ? 1.32f : 1.0f);
}

// Route of a shape whose scales the tile kernel reads.
struct Route {
    bool skinny;
    int splits;   // K slices, given a workspace
};
static Route find_route(int64_t M, int64_t N, int64_t K) {
    // up to 32 rows against a small weight: the skinny kernel's 16-row tiles
    // spread it over more CUs (M = 32, 2048 x 2048: 7.3 us against 7.9)
    if (M <= kSkinnyMaxM && N <= 16 * (int64_t)num_cus_w() && K <= 2048) return Route{true, 1};
    const int64_t budget = split_budget(M, N, K);
    const bool few = M <= kDecodeMaxM && K % dk::SLICE_K != 0;
    const Plan one = budget > 0 || few ? best_plan(M, N, K, 1, 0, budget, K % 512 == 0) : Plan{0, 1, 0.0f};
    // up to 16 rows that the decode kernel does not take: the skinny kernel
    // where its time is less than the tiles', both forms weighed alike (M = 2,
    // 64 x 2944: 4.2 us against 9.7; M = 12, 2752 x 3328 6.9 and 12.0; M = 1,
    // 320 x 21888 12.8 and 56; M = 10, 59200 x 6784 61 and 40)
    if (few) {
        const Plan two = best_plan(M, N, K, 2, one.splits, budget, false);
        if (skinny_time(M, N, K) * skinny_time(2 * M, N, K) <= one.us * two.us) return Route{true, 1};
    }
    return Route{false, one.splits};
}
// A call asks twice, before it allocates a workspace and at its launch; the
// search (up to 1 us) runs once.
static Route route_of(int64_t M, int64_t N, int64_t K) {
    static thread_local int64_t last[3] = {0, 0, 0};
    static thread_local Route route;
    if (M != last[0] || N != last[1] || K != last[2]) {
        route = find_route(M, N, K);
        last[0] = M, last[1] = N, last[2] = K;
    }
    return route;
}

// The slices depend on M, N and K only, so the single and the dual launch of
// one M add the same partial sums and give identical bits; the tile of the
// dual form is chosen for its own number of tiles.
int gemm_bf16f4_slices(int64_t M, int64_t N, int64_t K) { return route_of(M, N, K).splits; }

// Workspace bytes to give: the budget, for each batch.
int64_t gemm_bf16f4_workspace(int64_t M, int64_t N, int64_t K, bool dual) {
    return split_budget(M, N, K) * (dual ? 2 : 1);
}

// C[b][m][n] = sum over slices s = 0, 1, ... of partial[s][b][m][n], in that
// order: 4 consecutive columns per thread, one 16-byte load per slice.  A
// workgroup covers 1024 columns of one output row: workgroup x is row
// x / cb (cb workgroups per row), so the row and batch come from scalar
// 32-bit divisions of uniform values and the loads issue at once (64-bit
// per-thread divisions put ~1 us of index arithmetic in front of them).
template <int CT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ ws, int splits, int nb,
                                                            int64_t Mp, int64_t Np, void *c0, void *c1, int64_t ldc,
                                                            int64_t M, int64_t N) {
    const uint32_t cb = (uint32_t)((Np / 4 + 255) / 256);   // workgroups per output row
    const uint32_t row = blockIdx.x / cb, b = row / (uint32_t)M;
    const int64_t m = row - b * (uint32_t)M;
    const int64_t n = ((int64_t)(blockIdx.x - row * cb) * 256 + threadIdx.x) * 4;
    if ((int)b >= nb || n >= N) return;
    const float *p = ws + (b * Mp + m) * Np + n;
    const int64_t slice = (int64_t)nb * Mp * Np;
    u32x4 v = *reinterpret_cast<const u32x4 *>(p);
    float x[4] = {u2f(v.x), u2f(v.y), u2f(v.z), u2f(v.w)};
    for (int s = 1; s < splits; ++s) {
        v = *reinterpret_cast<const u32x4 *>(p + s * slice);
        x[0] += u2f(v.x);
        x[1] += u2f(v.y);
        x[2] += u2f(v.z);
        x[3] += u2f(v.w);
    }
    void *c = b ? c1 : c0;
    const int64_t idx = m * ldc + n;
    if (n + 4 <= N && (((uintptr_t)c + idx * (CT == LSMX_F32 ? 4 : 2)) & (CT == LSMX_F32 ? 15 : 7)) == 0) {
        store_c4<CT>(c, idx, x[0], x[1], x[2], x[3]);
    } else {
        for (int k = 0; k < 4 && n + k < N; ++k) store_c<CT>(c, idx + k, x[k]);
    }
}

// The two launches of a sliced call, and no other thread's between them: all
// host threads on a stream share its workspace, and a call's partials must
// still be there when its reduction runs.
static std::mutex g_slices_mu;

// LA: 64 x 128 tiles have 128 registers per lane (two workgroups per CU), which
// LA = 4 overruns by two
template <int WM, int WN, int TM, int TN, int S, int LA>
static hipError_t launch_tile(GemmArgs g, int splits, hipStream_t s) {
    constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
    const int64_t tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
    const int nb = g.a1 ? 2 : 1;
    const dim3 grid((unsigned)(tm * tn * nb * splits)), blk(64 * (WM * WN + wt::NLW));
    g.splits = splits;
    const bool vec = ((reinterpret_cast<uintptr_t>(g.c) | reinterpret_cast<uintptr_t>(g.c1)) & 15) == 0 && g.ldc % 4 == 0;
    const int64_t Mp = tm * BM, Np = tn * BN;
    const dim3 rgrid((unsigned)(nb * g.M * ((Np / 4 + 255) / 256))), rblk(256);
#define LSMX_T(CT)                                                                                                 \
    do {                                                                                                           \
        if (splits > 1) {                                                                                          \
            std::lock_guard<std::mutex> lk(g_slices_mu);                                                           \
            hipLaunchKernelGGL((gemm_bf16f4_tile_kernel<LSMX_F32, true, WM, WN, TM, TN, S, LA, true>), grid, blk, 0, s, g); \
            hipLaunchKernelGGL((splitk_reduce_kernel<CT>), rgrid, rblk, 0, s, g.ws, splits, nb, Mp, Np, g.c, g.c1, \
                               g.ldc, g.M, g.N);                                                                   \
        } else if (vec) {                                                                                          \
            hipLaunchKernelGGL((gemm_bf16f4_tile_kernel<CT, false, WM, WN, TM, TN, S, LA, true>), grid, blk, 0, s, g);  \
        } else {                                                                                                   \
            hipLaunchKernelGGL((gemm_bf16f4_tile_kernel<CT, false, WM, WN, TM, TN, S, LA, false>), grid, blk, 0, s, g); \
        }                                                                                                          \
    } while (0)
    if (g.c_dtype == LSMX_F32) LSMX_T(LSMX_F32);
    else if (g.c_dtype == LSMX_BF16) LSMX_T(LSMX_BF16);
    else LSMX_T(LSMX_F16);
#undef LSMX_T
    return hipGetLastError();
}

// E8M0 scale rows that start at multiples of 4 bytes (the kernel loads 16
// bytes of a row at a time), and operand panels within 32-bit load offsets
static bool tile_ok(const GemmArgs &g) {
    return g.scale_fmt == LSMX_SCALE_E8M0 && g.ld_sb % 4 == 0 && (reinterpret_cast<uintptr_t>(g.sb) & 3) == 0 &&
           g.lda < ((int64_t)1 << 22) && g.ldb < ((int64_t)1 << 22);
}

hipError_t launch_gemm_bf16f4(const GemmArgs &g, hipStream_t s) {
    // the same M picks the same kernel for the single and the dual form
    // GEMV when the dual form's 2M activation rows of K bf16 fit in LDS (the
    // test depends on M and K only, so single and dual launches agree)
    if (g.M <= kGemvMaxM && 2 * g.M * g.K * 2 <= kGemvMaxLds) return launch_gemv(g, s);
    const bool tiles = tile_ok(g);
    // 2 .. 16 rows: the decode kernel while one pass covers K (M = 16, 4096 x
    // 4096: 9.9 us against 9.1 - 9.7 in slices; M = 16, 14336 x 4096: 11.8
    // against 12.4), past that K slices (M = 4, 4096 x 14336: 23.1 against 12.7)
    const int splits = tiles && g.ws ? g.splits : 1;
    if (g.M <= kDecodeMaxM && decode_ok(g) && (g.K <= dk::PASS_K || splits == 1)) return launch_decode(g, s);
    if (tiles ? route_of(g.M, g.N, g.K).skinny : g.M <= kSkinnyMaxM) return launch_skinny(g, s);
    if (!tiles) return g.a1 ? launch_w4_any<2>(g, s) : launch_w4_any<1>(g, s);
    const Plan p = best_plan(g.M, g.N, g.K, g.a1 ? 2 : 1, splits, splits > 1 ? split_budget(g.M, g.N, g.K) : 0, ring_ok(g));
    switch (p.tile) {
    case 0: return launch_tile<1, 4, 1, 1, 4, 4>(g, p.splits, s);
    case 1: return launch_tile<1, 4, 2, 1, 3, 2>(g, p.splits, s);
    case 2: return launch_tile<1, 4, 4, 1, 3, 2>(g, p.splits, s);
    case 3: return launch_tile<2, 4, 2, 2, 3, 2>(g, p.splits, s);
    case 4: return launch_tile<2, 4, 3, 2, 2, 1>(g, p.splits, s);
    default: return g.a1 ? launch_ring<2>(g, s) : launch_ring<1>(g, s);
    }
}

}  // namespace lsmx
