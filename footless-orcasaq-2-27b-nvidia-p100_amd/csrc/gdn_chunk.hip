// Chunked (WY / UT transform) Gated DeltaNet prefill on gfx950.
//
// Not in the reference: it runs the delta rule sequentially over a prefill
// (gdn_scan_rows, kernels.cu:2809-2914) and names the chunked scan as the
// undone optimisation (kernels.cu:1788-1791). This computes the same
// recurrence (S *= decay; delta = beta (v - S k); S += delta k^T; o = S q)
// chunk by chunk. For a chunk of C = 64 tokens with start state S0 [V][K] and
// g_i the in-chunk prefix sum of log(decay):
//   A[i][j] = beta_i e^{g_i - g_j} (k_i . k_j), j < i          (strictly lower)
//   T = (I + A)^-1                                              (unit lower)
//   X = K S0^T,  Y = diag(beta) (V - diag(e^g) X)               (C x V)
//   Delta = T Y
//   O   = diag(e^g) Q S0^T + (M o Q K^T) Delta,  M[i][j] = e^{g_i - g_j}, j <= i
//   S_C = e^{g_C} S0 + Delta^T diag(e^{g_C - g}) K
// (Delta = U - W S0^T with W = T diag(beta e^g) K and U = T diag(beta) V is
// the same product grouped otherwise; this grouping keeps only T and M o QK^T
// in the workspace and feeds K, Q and V, exact in fp16, straight to the
// matrix cores.) The decay ratios are formed as e^{g_i - g_j} with j <= i
// (never 1 / gamma_j, which overflows over a chunk of strong decay).
//
// Two launches. chunk_prep_kernel, every (chunk, v head) in parallel: K K^T
// and Q K^T of the v head's k head on MFMA (the three v heads of a k head
// each form them: one workgroup walking the three in turn measured 5 us
// slower at 8k), then the prefix sums, A, T in fp32 by blocks of 16 (the
// diagonal blocks by forward substitution, the others on fp32 MFMA), the
// gates, and T and M o QK^T written as fp16 MFMA operands.
// chunk_state_kernel: a state wavefront per 16 state rows (v) of a v head,
// all 128 k columns of them in fp32 registers, sequential over the chunks; a
// paired output wavefront takes its split S0 and Delta through LDS a chunk
// later, forms Q S0^T and O and stores y; a copy wavefront issues the HBM ->
// LDS copies of the operands one chunk ahead, so the state chain carries only
// its own products.
//
// Precision. Every product runs on v_mfma_f32_16x16x32_f16 (fp16 inputs,
// fp32 accumulate: the product of two fp16 values is exact in fp32). K, Q and
// V are fp16 data. An fp32 operand x of the recurrence's products (the state,
// Y, T, the decayed Delta) is scaled by a power of two 2^s chosen from its
// block's maximum (max |x| 2^s in [128, 256); a block is T or M o QK^T whole,
// and one state row, i.e. one column of a B operand, for the state, Y and
// Delta) and split x 2^s = hi + lo, both fp16: two MFMAs (hi, lo) against an
// exact operand, three (hi.hi, hi.lo, lo.hi) between two split operands, which
// leaves an error of ~2^-22 of the block's maximum, fp32's order. The output's products need it too: one fp16
// pass leaves y within its own tolerance, but its two terms cancel in places
// and the gated norm that follows divides each head's row by its RMS (7e-3 of
// the row's RMS against 2e-3 for fp32 products). Emulated in numpy before the
// kernels were written, on the test's inputs: the state within 1.2e-6 of the
// sequential recurrence after 8192 tokens and y as close as with all-fp32
// products.
//
// MFMA operand layout (v_mfma_f32_16x16x32_f16, lane l = 16 g + i): the A
// operand of rows r0 .. r0 + 15 and a 32-wide k-step at k0 holds, in lane l,
// row r0 + i at k = k0 + kap(g, e), e = 0..7, kap(g, e) = 4 g + e (e < 4) or
// 16 + 4 g + (e - 4); the B operand holds column c0 + i at the same k. The
// result holds, in lane l, rows 4 g + r (r = 0..3) of column i. The matrix
// core pairs A and B by (lane group, slot), so any k order the two share is
// the same product; with kap, the results of two consecutive 16-row blocks
// are, as they stand in the registers, the B operand of the next product
// over those 32 rows: the state, X, Y and Delta never move between lanes.
#include "fl_common.hpp"

#include <mutex>
#include <type_traits>

#pragma clang fp contract(off)

#include "gdn_gates.hpp"

namespace {

constexpr int CK_C = 64;       // tokens a chunk
constexpr int CK_K = 128;      // key dim
constexpr int CK_V = 128;      // value dim

// Workspace block of one (chunk, v head), bytes: T and M o QK^T, each as hi
// and lo fp16 A operands [6 blocks][64 lanes][8] (6 KiB each; block f is row
// block mb = f, k-step 0 for f < 4, and mb = f - 2, k-step 1 for f = 4, 5: both
// matrices are lower triangular, so rows 0..31 take nothing from k-step 1),
// then beta, e^{g} and e^{g_C - g} [64] f32 (beta 0 past the chunk's last
// token), then e^{g_C}, 2^-tau and 2^-kappa (T's and M o QK^T's scales).
constexpr int CK_NF = 6;
__host__ __device__ constexpr int f_mb(int f) { return f < 4 ? f : f - 2; }
__host__ __device__ constexpr int f_kq(int f) { return f < 4 ? 0 : 1; }
constexpr int WS_OP = CK_NF * 1024;
constexpr int WS_T_HI = 0, WS_T_LO = WS_OP, WS_Q_HI = 2 * WS_OP, WS_Q_LO = 3 * WS_OP,
              WS_BETA = 4 * WS_OP, WS_EG = WS_BETA + 256, WS_DK = WS_BETA + 512,
              WS_SC = WS_BETA + 768;
constexpr int CK_BLK = WS_BETA + 1024;

typedef __attribute__((address_space(3))) const f16x4 lds_f16x4;
typedef __attribute__((address_space(3))) const f16x8 lds_f16x8;
typedef __attribute__((address_space(3))) const f32x4 lds_f32x4;

__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// max over the 64 lanes, on every lane: quad exchanges and row rotations by
// 4 and 8 (DPP), then v_permlane16_swap and v_permlane32_swap
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_xor1(v));
    v = fmaxf(v, dpp_xor2(v));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xF, 0xF, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)));
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                    false);
    return pair32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

// max over the lanes l, l ^ 16, l ^ 32 and l ^ 48, the four lane groups that
// hold one column of an MFMA B operand (or result): v_permlane16_swap with
// both operands v returns v of the lane pair (l, l ^ 16), then
// v_permlane32_swap the pair (l, l ^ 32)
__device__ __forceinline__ float col_max(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                    false);
    return pair32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

// The power of two s with m s in [2^P, 2^(P+1)) for a block maximum m >= 0
// (from m's exponent field; at most 2^126, so 1 / s stays normal); inv = 1 / s.
template <int P>
__device__ __forceinline__ float pow2_scale(float m, float& inv) {
    const int e = (int)((__float_as_uint(m) >> 23) & 0xff);
    const int se = min(254 + P - e, 253);
    inv = __uint_as_float((uint32_t)(254 - se) << 23);
    return __uint_as_float((uint32_t)se << 23);
}

// 1 / x for a power of two x = 2^e with -126 <= e <= 126, exactly
__device__ __forceinline__ float pow2_inv(float x) {
    return __uint_as_float((254u - (__float_as_uint(x) >> 23)) << 23);
}

// x s = hi + lo, both fp16 (round to nearest), for two values into packed
// halves: v_fma_mix rounds x s (exact: s is a power of two) and x s - hi
// (exact in fp32: hi is x s to 11 bits) to fp16 once each, reading hi back as
// an fp16 source, so a value costs two instructions
__device__ __forceinline__ void split2(float x0, float x1, float s, uint32_t& hi, uint32_t& lo) {
    uint32_t h, e;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(h) : "v"(x0), "v"(s));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(h) : "v"(x1), "v"(s));
    asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(e) : "v"(x0), "v"(s), "v"(h));
    asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "+v"(e) : "v"(x1), "v"(s), "v"(h));
    hi = h;
    lo = e;
}

// the B operand of a k-step from the accumulators a (slots 0..3) and b
// (slots 4..7), scaled by s and split
__device__ __forceinline__ void split8(f32x4 a, f32x4 b, float s, f16x8& hi, f16x8& lo) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    uint32_t h0, h1, h2, h3, l0, l1, l2, l3;
    split2(a[0], a[1], s, h0, l0);
    split2(a[2], a[3], s, h1, l1);
    split2(b[0], b[1], s, h2, l2);
    split2(b[2], b[3], s, h3, l3);
    hi = __builtin_bit_cast(f16x8, (u32x4){h0, h1, h2, h3});
    lo = __builtin_bit_cast(f16x8, (u32x4){l0, l1, l2, l3});
}

// ---------------------------------------------------------------------------
// chunk_prep_kernel: one workgroup of 4 waves a (chunk, v head)
// ---------------------------------------------------------------------------
constexpr int PK_P = CK_K + 8;   // f16 pitch of staged K / Q rows
constexpr int PA_P = CK_C + 4;   // f32 pitch of the A / T and M o QK^T rows
static_assert(CK_C * PA_P * 4 == CK_C * PK_P * 2, "A / QKm reuse the K / Q storage");

__device__ __forceinline__ float safe_log(float d) { return logf(fmaxf(d, 1.17549435e-38f)); }

// an empty use: the value is loaded unconditionally (every address read is in
// bounds), instead of the load being moved under the select that keeps it
__device__ __forceinline__ void keep(float& v) { asm volatile("" : "+v"(v)); }

// v_mfma_f32_16x16x4_f32, lane l = 16 g + i: A holds X[i][g], B holds Y[g][i],
// the result Z[4 g + r][i] in slot r
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// T's block (bi, bj), bi = bj + LV, from the blocks of T already in sA (kept
// transposed above the diagonal, the diagonal blocks D with their zeros):
// S = sum_k A_{bi,k} T_{k,bj} (k-step s takes k = 16 k + 4 s + g), then
// T_{bi,bj} = -D_bi S with S's result slots as the B operand as they stand
// (k-step s pairs lane group g with S's row 4 g + s, so D is read at column
// 4 g + s); returns -T_{bi,bj}'s values of this lane
// Every operand is read before the first product (in turn with them each pair
// waited out an LDS round trip).
template <int LV>
__device__ __forceinline__ f32x4 t_block(float (*sA)[CK_C + 4], int bj, int lane) {
    const int g = lane >> 4, i = lane & 15, bi = bj + LV;
    float a[LV][4], t[LV][4], d[4];
#pragma unroll
    for (int m = 0; m < LV; ++m)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int kk = 16 * (bj + m) + 4 * s + g;
            a[m][s] = sA[16 * bi + i][kk];
            // T_{kb,bj}[kk][i]: transposed at sA[16 bj + i][kk] (D's zeros above
            // its diagonal are stored)
            t[m][s] = sA[16 * bj + i][kk];
        }
#pragma unroll
    for (int s = 0; s < 4; ++s) d[s] = sA[16 * bi + 4 * g + s][16 * bi + i];   // D_bi[i][kk], transposed
    f32x4 sm = (f32x4)(0.f), r = (f32x4)(0.f);
#pragma unroll
    for (int m = 0; m < LV; ++m)
#pragma unroll
        for (int s = 0; s < 4; ++s) sm = mfma4(a[m][s], t[m][s], sm);
#pragma unroll
    for (int s = 0; s < 4; ++s) r = mfma4(d[s], sm[s], r);
    *(f32x4*)&sA[16 * bj + i][16 * bi + 4 * g] = -r;
    return r;
}


// inclusive prefix sum over the 64 lanes of a wavefront: DPP row shifts by 1,
// 2, 4 and 8 (zero fill at the row start), then the row totals carried by
// row_bcast:15 and row_bcast:31
__device__ __forceinline__ float wave_prefix_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xA, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xC, 0xF, false));
    return v;
}

// The gates the prep reads: beta and decay [T][n_vheads] (gdn_scalars'
// output), or, LOGITS, the logits a and b [T][ab_stride] with A_log and
// dt_bias, from which a lane forms its token's beta and decay itself (the
// gates kernel's functions: the same values).
struct PrepGates {
    const float* beta;     // or a
    const float* decay;    // or b
    const float* A_log;
    const float* dt_bias;
    int stride;            // n_vheads, or ab_stride
};

// v of lane I of this lane's row of 16 (DPP row broadcast)
template <int I>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + I, 0xF, 0xF, true));
}

// Rows I .. 15 of column j of D = (I + A)^-1 for each 16-lane row's own 16 x 16
// A: na is row (lane % 16) of -A, x[i] = [i == j] + sum_{m < i} -A[i][m] x[m],
// even and odd m in two chains.
template <int I>
__device__ __forceinline__ void solve_rows(const float (&na)[16], float (&x)[16], int j) {
    if constexpr (I < 16) {
        float a0 = I == j ? 1.f : 0.f, a1 = 0.f;
#pragma unroll
        for (int m = 0; m < I; ++m) {
            if (m & 1)
                a1 = fmaf(row_bcast<I>(na[m]), x[m], a1);
            else
                a0 = fmaf(row_bcast<I>(na[m]), x[m], a0);
        }
        x[I] = a0 + a1;
        solve_rows<I + 1>(na, x, j);
    }
}

// A v head's part of a chunk's prep, on a team of 4 waves (w = 0..3, tid = 64 w
// + lane): K K^T and Q K^T from the staged rows (wave w the 32 x 32 block (w /
// 2, w % 2)), then A, T and M o QK^T with the head's gates (this lane's token's
// dec and bet; n tokens in the chunk), into the head's block of the workspace.
// sA / sM may lie over sK / sQ. The parts that take less than the four waves
// start at wave `rot`: teams of one workgroup pass different ones, or they
// would all fall to the same SIMD (a wave's place is its number modulo 4). mid() runs between the products and the first
// barrier, its vector instructions under the products' MFMAs.
template <class Mid>
__device__ __forceinline__ void prep_head(f16 (*sK)[PK_P], f16 (*sQ)[PK_P], float (*sA)[PA_P],
                                          float (*sM)[PA_P], float* sG, float* sB, float* sRed,
                                          int tid, int n, float dec, float bet, char* blk,
                                          int rot, Mid mid) {
    const int lane = tid & 63, w = tid >> 6, wr = (w - rot) & 3;
    const int ql = lane & 31, hh = lane >> 5;
    // K K^T and Q K^T: wave w the 32 x 32 block (bi, bj), kept in registers
    const int bi = w >> 1, bj = w & 1;
    f32x16 kk = (f32x16)(0.f), qk = (f32x16)(0.f);
#pragma unroll
    for (int ks = 0; ks < CK_K / 16; ++ks) {
        const f16x8 bk = *(const f16x8*)&sK[32 * bj + ql][16 * ks + 8 * hh];
        const f16x8 ak = *(const f16x8*)&sK[32 * bi + ql][16 * ks + 8 * hh];
        const f16x8 aq = *(const f16x8*)&sQ[32 * bi + ql][16 * ks + 8 * hh];
        kk = __builtin_amdgcn_mfma_f32_32x32x16_f16(ak, bk, kk, 0, 0, 0);
        qk = __builtin_amdgcn_mfma_f32_32x32x16_f16(aq, bk, qk, 0, 0, 0);
    }

    // this head's gates (decay 1 and beta 0 past the end: g stays at the last
    // token's), the in-chunk prefix sums of log decay on one wave
    if (wr == 0) {
        const float gs = wave_prefix_sum(lane < n ? safe_log(dec) : 0.f);
        sG[lane] = gs;
        sB[lane] = lane < n ? bet : 0.f;
    }
    mid();
    {
        __syncthreads();   // the gates in; every K / Q read done

        // A = strictly lower beta_i e^{g_i - g_j} k_i.k_j and M o QK^T, rows i =
        // 32 bi + 8 q + 4 hh + e of column j. The 32 x 32 block above the
        // diagonal (wave 1) is left alone: nothing reads M there, and T's
        // blocks below the diagonal are written there (transposed) before
        // anything reads it. mt, mq: the running maxima of |T| and |M o QK^T|
        // over their lower triangles (their operands' scales), kept as the
        // values are formed. The rows' gates are read four at a time ahead of
        // the stores: read one by one between them (the compiler has to
        // assume that they alias) this part took 4.4 k clocks instead of 2 k
        // with 12 waves on the LDS.
        float mt = 0.f, mq = 0.f;
        if (bi >= bj) {
            const int j = 32 * bj + ql;
            const float gj = sG[j];
            f32x4 gi[4], be[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                gi[q] = *(const f32x4*)&sG[32 * bi + 8 * q + 4 * hh];
                be[q] = *(const f32x4*)&sB[32 * bi + 8 * q + 4 * hh];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = 32 * bi + 8 * (r >> 2) + 4 * hh + (r & 3);
                // e^{g_i - g_j}, taken for every pair (above the diagonal it may
                // be inf, and is not selected)
                const float ratio = fast_exp2((gi[r >> 2][r & 3] - gj) * FL_LOG2E);
                const float m = j <= i ? ratio * qk[r] : 0.f;
                sA[i][j] = j < i ? be[r >> 2][r & 3] * ratio * kk[r] : 0.f;
                sM[i][j] = m;
                mq = fmaxf(mq, fabsf(m));
            }
        }
        __syncthreads();

        // T = (I + A)^-1 by blocks of 16, in fp32: T_ii = D_i = (I + A_ii)^-1
        // by forward substitution, then, a block diagonal at a time, T_ij = -D_i
        // sum_{k = j .. i-1} A_ik T_kj on fp32 MFMA. T is kept transposed in
        // sA's upper triangle (T_ij[a][b] at sA[16 j + b][16 i + a]), clear of A
        // below the diagonal. The substitution is one wave's: lane 16 i + j holds
        // row j of -A_ii and solves column j, row r's elements reaching the 16
        // lanes of their block by DPP row broadcasts. (A wave a block, the
        // elements read from LDS where they are used, kept the LDS busy for
        // 8 k clocks with three teams at it.)
        if (wr == 0) {
            const int o = lane & 48, j = lane & 15;
            float na[16];
#pragma unroll
            for (int m = 0; m < 16; m += 4) {
                const f32x4 v = *(const f32x4*)&sA[lane][o + m];
#pragma unroll
                for (int e = 0; e < 4; ++e) na[m + e] = -v[e];
            }
            float xd[16];
            solve_rows<0>(na, xd, j);
#pragma unroll
            for (int i = 0; i < 16; ++i) mt = fmaxf(mt, fabsf(xd[i]));
            // every element, the zeros above D's diagonal included: they land on
            // A_ii, which the remaining steps do not read
#pragma unroll
            for (int i = 0; i < 16; i += 4)
                *(f32x4*)&sA[lane][o + i] = (f32x4){xd[i], xd[i + 1], xd[i + 2], xd[i + 3]};
        }
        __syncthreads();
        auto level = [&](auto lv) {
            constexpr int LV = decltype(lv)::value;
            if (wr < 4 - LV) {
                const f32x4 t = t_block<LV>(sA, wr, lane);
#pragma unroll
                for (int r = 0; r < 4; ++r) mt = fmaxf(mt, fabsf(t[r]));
            }
        };
        level(std::integral_constant<int, 1>());
        __syncthreads();
        level(std::integral_constant<int, 2>());
        __syncthreads();
        level(std::integral_constant<int, 3>());
        mt = wave_max(mt);
        mq = wave_max(mq);
        if (lane == 0) {
            sRed[w] = mt;
            sRed[4 + w] = mq;
        }
        __syncthreads();
        mt = fmaxf(fmaxf(sRed[0], sRed[1]), fmaxf(sRed[2], sRed[3]));
        mq = fmaxf(fmaxf(sRed[4], sRed[5]), fmaxf(sRed[6], sRed[7]));
        float t_inv, q_inv;
        const float t_sc = pow2_scale<7>(mt, t_inv);
        const float q_sc = pow2_scale<7>(mq, q_inv);

        // the operands: slot (T or M o QK^T; block f, lane l = 16 g + i) holds
        // row 16 mb + i at columns 32 kq + kap(g, e), its hi and lo halves
        // 6 KiB apart
        // (which matrix a pass takes is the same for a whole wave: 6 blocks x
        // 64 lanes of T, then 6 of M o QK^T, over 3 passes of 256 threads)
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const int s = tid + 256 * m;
            const bool isq = s >= CK_NF * 64;
            const int f = (s % (CK_NF * 64)) >> 6, l = s & 63;
            const int g = l >> 4, row = 16 * f_mb(f) + (l & 15), kq = f_kq(f);
            float xs[8];
            if (isq) {   // M o QK^T[row][32 kq + kap(g, e)]: two row segments of 4
                const f32x4 a = *(const f32x4*)&sM[row][32 * kq + 4 * g];
                const f32x4 b = *(const f32x4*)&sM[row][32 * kq + 16 + 4 * g];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xs[e] = a[e] * q_sc;
                    xs[4 + e] = b[e] * q_sc;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int col = 32 * kq + (e < 4 ? 4 * g + e : 12 + 4 * g + e);
                    float ta = sA[col][row];   // T[row][col], transposed
                    keep(ta);
                    xs[e] = (row >= col ? ta : 0.f) * t_sc;
                }
            }
            f16x8 hi, lo;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const f16 h = (f16)xs[e];
                hi[e] = h;
                lo[e] = (f16)(xs[e] - (float)h);
            }
            char* dst = blk + (isq ? WS_Q_HI : WS_T_HI) + (f * 64 + l) * 16;
            *(f16x8*)dst = hi;
            *(f16x8*)(dst + WS_OP) = lo;
        }
        if (tid < CK_C) {
            const float gC = sG[CK_C - 1];
            ((float*)(blk + WS_BETA))[tid] = sB[tid];
            ((float*)(blk + WS_EG))[tid] = expf(sG[tid]);
            ((float*)(blk + WS_DK))[tid] = expf(gC - sG[tid]);
            if (tid < 4)
                ((float*)(blk + WS_SC))[tid] =
                    tid == 0 ? expf(gC) : tid == 1 ? t_inv : tid == 2 ? q_inv : 0.f;
        }
    }
}

// One workgroup of 4 waves a (chunk, v head), a grid of chunks x v heads: it
// loads its k head's K and Q rows of the chunk, then prep_head.
template <bool LOGITS>
__global__ void __launch_bounds__(256)
chunk_prep_kernel(const f16* __restrict__ q, const f16* __restrict__ k, const PrepGates gates,
                  int T, int n_vheads, int qk_stride, int group, char* __restrict__ work) {
    __shared__ __attribute__((aligned(16))) char smem[2 * CK_C * PK_P * 2];
    __shared__ __attribute__((aligned(16))) float sG[CK_C], sB[CK_C];
    __shared__ float sRed[8];
    f16(*sK)[PK_P] = (f16(*)[PK_P])smem;
    f16(*sQ)[PK_P] = (f16(*)[PK_P])(smem + CK_C * PK_P * 2);
    float(*sA)[PA_P] = (float(*)[PA_P])smem;                     // after the products
    float(*sM)[PA_P] = (float(*)[PA_P])(smem + CK_C * PA_P * 4);

    const int c = blockIdx.x, hv0 = blockIdx.y, hk = hv0 / group;
    const int tid = threadIdx.x, lane = tid & 63;
    const int t0 = c * CK_C;
    const int n = min(CK_C, T - t0);

    // Every global load issued up front and unconditionally, rows clamped to
    // the chunk's last token, past-the-end rows zeroed by a select: K and Q
    // (4 rows x 16 B a thread), the first v head's beta and decay.
    f16x8 kv8[4], qv8[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int idx = tid + 256 * m, i = idx >> 4, c8 = (idx & 15) * 8;
        const size_t off = (size_t)(t0 + min(i, n - 1)) * qk_stride + (size_t)hk * CK_K + c8;
        kv8[m] = *(const f16x8*)(k + off);
        qv8[m] = *(const f16x8*)(q + off);
    }
    const size_t gt = (size_t)(t0 + min(lane, n - 1)) * gates.stride + hv0;
    float dec, bet;
    if constexpr (LOGITS) {
        const float av = gates.beta[gt], bv = gates.decay[gt];
        const float dtb = gates.dt_bias[hv0], A = gates.A_log[hv0];
        dec = gdn_decay(av + dtb, A);
        bet = gdn_beta(bv);
    } else {
        dec = gates.decay[gt];
        bet = gates.beta[gt];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int idx = tid + 256 * m, i = idx >> 4, c8 = (idx & 15) * 8;
        *(f16x8*)&sK[i][c8] = i < n ? kv8[m] : (f16x8)(0);
        *(f16x8*)&sQ[i][c8] = i < n ? qv8[m] : (f16x8)(0);
    }
    __syncthreads();
    prep_head(sK, sQ, sA, sM, sG, sB, sRed, tid, n, dec, bet,
              work + ((size_t)c * n_vheads + hv0) * CK_BLK, 0, [] {});
}

// ---------------------------------------------------------------------------
// gdn_front_kernel: everything of a GDN prefill layer ahead of the state pass,
// a workgroup of 12 waves a (chunk, k head): the causal conv (width 4) of the
// k head's q and k channels and of its FG v heads' channels over the chunk's
// 64 tokens, the L2 norm of the q and k rows, and then a team of 4 waves a v
// head the prep (prep_head) on the rows still in LDS. Separately (conv, norm
// and prep kernels, the q / k rows through HBM between them and read by every
// v head) the three took 18 + 5.7 + 15 us of a 1024-token layer's 89; here
// 16 chunks x 16 k heads are one workgroup a CU and 23 us (kernel traces).
// Bound by the conv's vector instructions (of 43 k clocks ~18 k, most of them
// the silu), then the chain from A to T's operands (~13 k) that one workgroup
// a CU leaves exposed. 138 KiB of LDS.
//
// Conv: a 16-lane group takes one head's 128 channels (8 a lane) of 4
// consecutive tokens, all 7 rows requested at once; the chunk's 5 heads x 16
// token blocks are 20 wave tasks: waves 0-3 q, 4-7 k, 8-11 the first v head,
// then waves 0-7 the other two under the products' MFMAs, 5 tasks a SIMD. Same
// taps order, silu and roundings as conv_window_kernel; the norm's sums in the
// order of l2norm_rows_kernel.
// ---------------------------------------------------------------------------
constexpr int FG = 3;                        // v heads a k head
constexpr int FR_THREADS = 256 * FG;
constexpr int FR_TB = 4;                     // tokens a conv task
// The front kernel from this many workgroups up: two chunks at 16 k heads. One
// takes its ~20 us however few there are (a workgroup's own chain), while the three
// launches that it replaces spread a short call over more of the chip. Same box,
// GPU time of four layers of 16 k heads, us, front / separate: 1 chunk 108 / 82, 2
// (32 workgroups) 128 / 114, 3 142 / 131, 5 (80) 166 / 163, 6 (96) 173 / 177, 8 186 /
// 201, 16 259 / 306; the line lies at 96 workgroups for 4, 8 and 32 k heads too. But
// two launches more a layer cost an eager caller ~5 us of host time a layer (a
// 65-token prompt through three of them and an attention layer, nothing else
// running: 120 / 132), which only one chunk saves on the GPU.
constexpr int FR_MIN_WGS = 32;
constexpr int FR_TILE = CK_C * PK_P * 2;     // staged K or Q rows; A or M o QK^T of a team
constexpr int FR_LDS = 2 * FR_TILE + FG * 2 * FR_TILE + FG * (2 * CK_C + 8) * 4;
static_assert(FR_LDS <= 160 * 1024, "the front kernel's LDS fits 160 KiB");

// v of the lane 4 or 8 further round its 16-lane row (DPP row rotations)
template <int D>
__device__ __forceinline__ float row_ror(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + D, 0xF, 0xF, true));
}

// One 16-lane group's conv rows in flight: E[j] = row (tb - 3 + j) of its 8
// channels, the taps [channel][tap].
struct FrontRows {
    f16x8 e[FR_TB + 3];
    f16x8 w[4];
};

// Task of the group: head `ch0` (its first channel + 8 times this lane's place)
// and the call's tokens tb .. tb + 3. Rows are clamped to [0, T): those before
// the call are replaced by the stored frames (zeros at pos0 == 0), those after
// it are not used.
__device__ __forceinline__ FrontRows front_load(const f16* __restrict__ x,
                                                const f16* __restrict__ conv_w,
                                                const f16* __restrict__ st_in, int ch, int tb,
                                                int T, int pos0, int x_stride) {
    FrontRows r;
#pragma unroll
    for (int j = 0; j < FR_TB + 3; ++j)
        r.e[j] = *(const f16x8*)(x + (size_t)min(max(tb - 3 + j, 0), T - 1) * x_stride + ch);
#pragma unroll
    for (int m = 0; m < 4; ++m) r.w[m] = *(const f16x8*)(conv_w + (size_t)ch * 4 + 8 * m);
    if (tb == 0) {
        f16x8 h[3];   // [channel][frame]
#pragma unroll
        for (int m = 0; m < 3; ++m)
            h[m] = pos0 > 0 ? *(const f16x8*)(st_in + (size_t)ch * 3 + 8 * m) : (f16x8)(f16)0.f;
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int c = 0; c < 8; ++c) r.e[j][c] = h[(3 * c + j) >> 3][(3 * c + j) & 7];
    }
    return r;
}

// acc + a[A] * b[B] of two packed fp16 pairs, fp32 (v_fma_mix reads the halves
// as they stand: no conversions)
template <int A, int B>
__device__ __forceinline__ float fma_half(uint32_t a, uint32_t b, float acc) {
    float r;
    if constexpr (A == 0 && B == 0)
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "v"(acc));
    else if constexpr (A == 1 && B == 0)
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,1,0]"
            : "=v"(r) : "v"(a), "v"(b), "v"(acc));
    else if constexpr (A == 0)
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[1,1,0]"
            : "=v"(r) : "v"(a), "v"(b), "v"(acc));
    else
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,1,0] op_sel_hi:[1,1,0]"
            : "=v"(r) : "v"(a), "v"(b), "v"(acc));
    return r;
}

// The conv of channels c and c + 1 (one word of a row) at token row i of the task
__device__ __forceinline__ void conv_pair(const FrontRows& r, int i, int c, float& y0, float& y1) {
    const u32x4 w = __builtin_bit_cast(u32x4, r.w[c >> 1]);   // channel c: words 0, 1; c + 1: 2, 3
    uint32_t e[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) e[j] = __builtin_bit_cast(u32x4, r.e[i + j])[c >> 1];
    y0 = fma_half<0, 0>(w[0], e[0], 0.f);
    y1 = fma_half<0, 1>(w[2], e[0], 0.f);
    y0 = fma_half<1, 0>(w[0], e[1], y0);
    y1 = fma_half<1, 1>(w[2], e[1], y1);
    y0 = fma_half<0, 0>(w[1], e[2], y0);
    y1 = fma_half<0, 1>(w[3], e[2], y1);
    y0 = fma_half<1, 0>(w[1], e[3], y0);
    y1 = fma_half<1, 1>(w[3], e[3], y1);
}

// The task's outputs into cx (global, the conv'd and, NORM, normed rows) and,
// NORM, into the staged rows `stage` at this lane's place (row tb - t0, zeros
// past the call); the lane of the call's last token stores the new frames.
template <bool NORM>
__device__ __forceinline__ void front_conv(const FrontRows& r, f16* __restrict__ cx,
                                           f16* __restrict__ st_out, f16 (*stage)[PK_P], int ch,
                                           int c8, int t0, int tb, int T, int x_stride,
                                           float l2eps) {
    const int nt = T - tb;   // tokens of the task inside the call (may be <= 0)
#pragma unroll
    for (int i = 0; i < FR_TB; ++i) {
        float yf[8];
#pragma unroll
        for (int c = 0; c < 8; c += 2) conv_pair(r, i, c, yf[c], yf[c + 1]);
#pragma unroll
        for (int c = 0; c < 8; ++c) yf[c] = silu_f(yf[c]);
        f16x8 out = f16_sat8(yf);
        if constexpr (NORM) {
            float xf[8], sq[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                xf[c] = (float)out[c];
                sq[c] = xf[c] * xf[c];
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) sq[c] += dpp_xor2(sq[c]);
#pragma unroll
            for (int c = 0; c < 8; ++c) sq[c] += dpp_xor1(sq[c]);
            const float ss4 = ((sq[0] + sq[4]) + (sq[2] + sq[6])) + ((sq[1] + sq[5]) + (sq[3] + sq[7]));
            // quads q and q + 2, then the two pairs: rotations by 8 and 4
            float ss = ss4 + row_ror<8>(ss4);
            ss += row_ror<4>(ss);
            const float den = sqrtf(ss + l2eps);
            float rd = __builtin_amdgcn_rcpf(den);
            rd = fmaf(fmaf(-den, rd, 1.f), rd, rd);
#pragma unroll
            for (int c = 0; c < 8; ++c) {   // xf / den, rounded once (as div_big; den is normal)
                const float q = xf[c] * rd;
                yf[c] = fmaf(fmaf(-den, q, xf[c]), rd, q);
            }
            out = f16_sat8(yf);
            if (i >= nt) out = (f16x8)(f16)0.f;
            *(f16x8*)&stage[tb - t0 + i][c8] = out;
        }
        // (an opaque use: only the store is conditional, not the row's arithmetic)
        asm volatile("" : "+v"(out));
        if (i < nt) *(f16x8*)(cx + (size_t)(tb + i) * x_stride + ch) = out;
    }
    if (nt >= 1 && nt <= FR_TB) {   // the call's last token is here: the last three frames
        f16x8 f[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            f[j] = r.e[1 + j];
#pragma unroll
            for (int i = 1; i < FR_TB; ++i)
                if (i == nt - 1) f[j] = r.e[i + 1 + j];
            f[j] = __builtin_elementwise_maximum(   // f16_sat of an fp16: inf to the largest
                __builtin_elementwise_minimum(f[j], (f16x8)(f16)65504.f), (f16x8)(f16)-65504.f);
        }
        f16x8 h[3];   // [channel][frame]
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int c = 0; c < 8; ++c) h[(3 * c + j) >> 3][(3 * c + j) & 7] = f[j][c];
#pragma unroll
        for (int m = 0; m < 3; ++m) *(f16x8*)(st_out + (size_t)ch * 3 + 8 * m) = h[m];
    }
}

__global__ void __launch_bounds__(FR_THREADS)
gdn_front_kernel(const f16* __restrict__ x, const f16* __restrict__ conv_w,
                 const f16* __restrict__ st_in, f16* __restrict__ st_out, f16* __restrict__ cx,
                 const PrepGates gates, int T, int pos0, int n_kheads, int x_stride, float l2eps,
                 char* __restrict__ work) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    f16(*sK)[PK_P] = (f16(*)[PK_P])smem;
    f16(*sQ)[PK_P] = (f16(*)[PK_P])(smem + FR_TILE);
    const int c = blockIdx.x, hk = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // 0 .. 11
    const int team = wv >> 2;                                          // v head hk FG + team
    const int t0 = c * CK_C;
    const int n = min(CK_C, T - t0);
    const int c8 = 8 * (lane & 15);
    const int kdim = n_kheads * CK_K;
    // wave task wt: head wt / 4 (q, k, then the v heads), token blocks 4 (wt % 4) + lane / 16
    auto first_ch = [&](int wt) {
        const int head = wt >> 2;
        return (head == 0 ? hk * CK_K
                : head == 1 ? kdim + hk * CK_K
                            : 2 * kdim + (hk * FG + head - 2) * CK_V) + c8;
    };
    const int tb = t0 + FR_TB * (4 * (wv & 3) + (lane >> 4));   // the same for both tasks of a wave
    const int ch1 = first_ch(wv), ch2 = first_ch(wv + 4 * FG);
    const FrontRows r1 = front_load(x, conv_w, st_in, ch1, tb, T, pos0, x_stride);
    const int hv = hk * FG + team;
    const size_t gt = (size_t)(t0 + min(lane, n - 1)) * gates.stride + hv;
    const float av = gates.beta[gt], bv = gates.decay[gt];
    const float dtb = gates.dt_bias[hv], A = gates.A_log[hv];
    if (wv < 8)
        front_conv<true>(r1, cx, st_out, wv < 4 ? sQ : sK, ch1, c8, t0, tb, T, x_stride, l2eps);
    else
        front_conv<false>(r1, cx, st_out, nullptr, ch1, c8, t0, tb, T, x_stride, l2eps);
    // the second task's rows, on their way under the barrier and the products
    FrontRows r2;
    if (wv < 8) r2 = front_load(x, conv_w, st_in, ch2, tb, T, pos0, x_stride);
    const float dec = gdn_decay(av + dtb, A), bet = gdn_beta(bv);
    __syncthreads();   // the chunk's normed q and k rows staged
    char* own = smem + 2 * FR_TILE + team * 2 * FR_TILE;
    float* sml = (float*)(smem + 2 * FR_TILE + FG * 2 * FR_TILE) + team * (2 * CK_C + 8);
    prep_head(sK, sQ, (float(*)[PA_P])own, (float(*)[PA_P])(own + FR_TILE), sml, sml + CK_C,
              sml + 2 * CK_C, threadIdx.x & 255, n, dec, bet,
              work + ((size_t)c * (n_kheads * FG) + hv) * CK_BLK, team, [&] {
                  if (wv < 8)
                      front_conv<false>(r2, cx, st_out, nullptr, ch2, c8, t0, tb, T, x_stride,
                                        l2eps);
              });
}

// ---------------------------------------------------------------------------
// chunk_state_kernel: 32 state rows (v) of a v head a workgroup. Waves 0 and 1
// (state waves) each hold 16 rows of S and run the recurrence's chain: X = K
// S^T, Y, Delta = T Y, the state update. Waves 2 and 3 (output waves) each take
// a state wave's split S and Delta a chunk later, form Q S^T and O and store y.
// Waves 6 and 7 (copy waves) issue every HBM -> LDS copy, a chunk ahead and
// more. (A wave's SIMD is its number modulo 4: waves 4 and 5, which would share
// the state waves', leave at once.) The state waves' chain is what the kernel
// takes, so what is not part of it lies elsewhere, and within it the VALU work
// that a product does not wait for lies between the MFMAs of another: 42 -> 37.5
// us for 1024 tokens of 48 heads, with the output waves issuing the copies and
// the state waves forming Q S^T -> as here. (Measured and slower by 1 us: the
// hand-over written between X's MFMAs, or behind Delta, with M before it. Its
// 25 KB then meet the K reads and the y tiles in the LDS.)
// ---------------------------------------------------------------------------
constexpr int CS_ROWS = 32;   // state rows (v) a workgroup
// A stage (the state waves' operands of a chunk): K rows [64][256 B] (16-byte
// chunk c of row r at c ^ row_swz(r)), V columns [64][CS_ROWS] fp16, T's hi / lo
// operands and the gates KiB (as in the workspace)
constexpr int SA_K = 0, SA_V = 16384, SA_T = SA_V + CK_C * CS_ROWS * 2,
              SA_G = SA_T + 2 * WS_OP, SA_BYTES = SA_G + 1024;
// B stage (the output waves'): Q rows as K's, M o QK^T's hi / lo operands and
// the gates KiB
constexpr int SB_Q = 0, SB_M = 16384, SB_G = SB_M + 2 * WS_OP, SB_BYTES = SB_G + 1024;
// offsets in the gates KiB: beta, e^g, e^{g_C - g} [64] f32, then e^{g_C},
// 2^-tau, 2^-kappa
constexpr int G_BETA = WS_BETA - WS_BETA, G_EG = WS_EG - WS_BETA, G_DK = WS_DK - WS_BETA,
              G_SC = WS_SC - WS_BETA;
static_assert(WS_T_LO == WS_T_HI + WS_OP && WS_Q_HI == WS_T_LO + WS_OP &&
                  WS_Q_LO == WS_Q_HI + WS_OP && WS_BETA == WS_Q_LO + WS_OP &&
                  CK_BLK == WS_BETA + 1024 && WS_OP % 2048 == 0,
              "workspace block: T, then M o QK^T, then the gates KiB, whole copy pairs");
// LDS: two A stages, two B stages, the hand-over (each state wave's S as its
// hi and lo B operands and Delta, [12][64 lanes] 16 bytes, then the lanes' 1 / s
// and Delta's scale) and each output wave's y tile [64 tokens][16 rows] fp16
constexpr int X_SL = 4 * 1024, X_DL = 8 * 1024, X_SC = 12 * 1024, X_WAVE = X_SC + 1024;
constexpr int L_A = 0, L_B = 2 * SA_BYTES, L_X = L_B + 2 * SB_BYTES,
              L_Y = L_X + 2 * X_WAVE, CS_LDS = L_Y + 2 * CK_C * 16 * 2;
static_assert(CS_LDS <= 160 * 1024, "the state pass's LDS fits 160 KiB");
constexpr int CS_THREADS = 512;

typedef __attribute__((address_space(3))) f32x4 lds_f32x4w;
typedef __attribute__((address_space(3))) f16x8 lds_f16x8w;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f32x2 lds_f32x2w;
typedef __attribute__((address_space(3))) float lds_f32w;
typedef __attribute__((address_space(3))) f16 lds_f16w;

// The 16-byte chunk swizzle of staged K and Q rows: rows 4 g .. 4 g + 3 and
// chunks 4 js .. 4 js + 3 fall on 16 different chunks (the transposed reads), as
// do the rows 0 .. 15 of any one chunk (the row reads)
__device__ __forceinline__ int row_swz(int r) { return 4 * (r & 3) + ((r >> 2) & 3); }

// Per-lane source offsets of copy wave wb's copies of a 64-token chunk (the
// base is scalar): K / Q copy n (n = 2 j + wb) brings rows 4 n .. 4 n + 3,
// lane -> row 8 j + rr, rr = 4 wb + lane / 16, and 16-byte chunk
// (lane % 16) ^ row_swz(row), row & 15 = rr + 8 (j & 1); V copy n rows
// 16 n + lane / 4, 16 bytes (lane % 4) of the workgroup's 64-byte slice; a
// workspace copy 16 bytes a lane.
struct CsOff {
    uint32_t kq[2], v, w;
};
__device__ __forceinline__ CsOff cs_offsets(int qk_bytes, int v_bytes, int wb, int lane) {
    const int rr = 4 * wb + (lane >> 4), p = lane & 15;
    return {{(uint32_t)(rr * qk_bytes + 16 * (p ^ row_swz(rr))),
             (uint32_t)(rr * qk_bytes + 16 * (p ^ row_swz(rr + 8)))},
            (uint32_t)((lane >> 2) * v_bytes + 16 * (lane & 3)), (uint32_t)(16 * lane)};
}

// Copy wave wb's half of the 64 rows of K or Q of a chunk at t0 into dst: 8
// copies. Rows past the last token repeat it (beta is 0 there).
__device__ __forceinline__ void cs_copy_rows(uint32_t dst, const char* base, int t0, int T,
                                             int qk_bytes, int wb, int lane, const CsOff& o) {
    if (T - t0 >= CK_C) {
        const char* at = base + (size_t)t0 * qk_bytes;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            copy16(at + (size_t)(8 * j) * qk_bytes, o.kq[j & 1], dst + 1024 * (2 * j + wb));
    } else {
        const int last = T - t0 - 1;
        const int rr = 4 * wb + (lane >> 4), p = lane & 15;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int r = 8 * j + rr;
            copy16_v(base + (size_t)(t0 + min(r, last)) * qk_bytes + 16 * (p ^ row_swz(r)),
                     __builtin_amdgcn_readfirstlane(dst + 1024 * (2 * j + wb)));
        }
    }
}

// Copy wave wb's half of the copies of chunk c's A stage into dst: 8 K, 2 V and
// 6 T copies, and (wb = 0) the gates KiB.
__device__ __forceinline__ void cs_copy_a(uint32_t dst, const char* kb, const char* vb,
                                          const char* wk, int t0, int T, int qk_bytes, int v_bytes,
                                          int wb, int lane, const CsOff& o) {
    cs_copy_rows(dst + SA_K, kb, t0, T, qk_bytes, wb, lane, o);
    if (T - t0 >= CK_C) {
        const char* vt = vb + (size_t)t0 * v_bytes;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = 2 * j + wb;
            copy16(vt + (size_t)(16 * n) * v_bytes, o.v, dst + SA_V + 1024 * n);
        }
    } else {
        const int last = T - t0 - 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = 2 * j + wb, r = 16 * n + (lane >> 2);
            copy16_v(vb + (size_t)(t0 + min(r, last)) * v_bytes + 16 * (lane & 3),
                     __builtin_amdgcn_readfirstlane(dst + SA_V + 1024 * n));
        }
    }
#pragma unroll
    for (int j = 0; j < WS_OP / 1024; ++j) {
        const int n = 2 * j + wb;
        copy16(wk + WS_T_HI + 1024 * n, o.w, dst + SA_T + 1024 * n);
    }
    if (wb == 0) copy16(wk + WS_BETA, o.w, dst + SA_G);
}

// Copy wave wb's half of the copies of chunk c's B stage: 8 Q and 6 M o QK^T
// copies and (wb = 1) the gates KiB.
__device__ __forceinline__ void cs_copy_b(uint32_t dst, const char* qb, const char* wk, int t0,
                                          int T, int qk_bytes, int wb, int lane, const CsOff& o) {
    cs_copy_rows(dst + SB_Q, qb, t0, T, qk_bytes, wb, lane, o);
#pragma unroll
    for (int j = 0; j < WS_OP / 1024; ++j) {
        const int n = 2 * j + wb;
        copy16(wk + WS_Q_HI + 1024 * n, o.w, dst + SB_M + 1024 * n);
    }
    if (wb == 1) copy16(wk + WS_BETA, o.w, dst + SB_G);
}

// The state's k axis is held in another order than the tokens': block 2 js + h
// holds, in its row 4 g + r, k = 32 js + 8 g + 4 h + r. A k-step's B operand
// (blocks 2 js and 2 js + 1) then pairs with eight consecutive k of a K or Q
// row, one 16-byte read where kap's order takes two of 8 bytes (the LDS is a
// bound beside the chain: a chunk moves 280 KB through it). 37.5 -> 36 us for
// 1024 tokens of 48 heads.
//
// The lane's part of the swizzled K / Q row addresses, fixed for the kernel:
// the A operand of X = K S^T (or Q S^T) for row block mb, k-step js holds row
// 16 mb + i's 16-byte chunk 4 js + g (mb adds 16 rows = 4096 bytes): this is
// chunk g's, the others' differ from it by an exclusive or with 64 js
__device__ __forceinline__ uint32_t row_offset(int g, int i) {
    return i * 256 + 16 * (g ^ row_swz(i));
}
// Stage base (scalar) + lane part, once a chunk: opaque, so the constant parts
// of each read (row block, k step, operand) stay in the LDS instruction's
// offset field instead of each read forming its own address
__device__ __forceinline__ uint32_t lane_addr(uint32_t sbase, uint32_t lane_part) {
    uint32_t r;
    asm("v_add_u32 %0, %1, %2" : "=v"(r) : "s"(sbase), "v"(lane_part));
    return r;
}
// the four k-steps' addresses of a row or column offset (sbase a multiple of
// 256): the loop holds one register of them, not four
__device__ __forceinline__ void lane_addrs(uint32_t sbase, uint32_t lane_part, uint32_t (&ra)[4]) {
    ra[0] = lane_addr(sbase, lane_part);
#pragma unroll
    for (int j = 1; j < 4; ++j)
        asm("v_xor_b32 %0, %1, %2" : "=v"(ra[j]) : "i"(64 * j), "v"(ra[0]));
}
__device__ __forceinline__ f16x8 row_frag(const uint32_t (&ra)[4], uint32_t off, int mb, int js) {
    return *(lds_f16x8*)(uintptr_t)(ra[js] + off + 4096 * mb);
}

// A operand of K^T Delta' for block kb = 2 js + h of k rows, token step kq:
// lane 16 g + i gets K[32 kq + kap(g, e)][the block's row i] by two transposed
// reads (each: the group's 16 lanes read 4 rows x 16 columns, lane i addressing
// row r = 32 kq + 4 g + i / 4 (+ 16), columns 32 js + 8 (i % 4) + 4 h .. + 3,
// and receiving the block's column i of the four rows). r & 15 = 4 g + i / 4
// for both reads and every kq, so the swizzled column part is fixed for the
// lane; kq and the second read add 8192 and 4096 bytes.
__device__ __forceinline__ uint32_t col_offset(int g, int i) {
    const int rr = 4 * g + (i >> 2);
    return rr * 256 + 16 * ((i & 3) ^ row_swz(rr));
}
__device__ __forceinline__ f16x8 col_frag(const uint32_t (&ca)[4], int kb, int kq) {
    const uint32_t a0 = ca[kb >> 1] + SA_K + 8 * (kb & 1) + 8192 * kq;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)a0);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(a0 + 4096));
    const f16x4 ah = __builtin_bit_cast(f16x4, a), bh = __builtin_bit_cast(f16x4, b);
    return (f16x8){ah[0], ah[1], ah[2], ah[3], bh[0], bh[1], bh[2], bh[3]};
}

// A scheduling region's order: an LDS read behind each of the first R of its M
// MFMAs (left alone, the reads gather at one end of the region, where they are
// waited for or hold the MFMAs back)
template <int R, int M>
__device__ __forceinline__ void between_mfmas() {
#pragma unroll
    for (int j = 0; j < R; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if constexpr (M > R) __builtin_amdgcn_sched_group_barrier(0x8, M - R, 0);
}

// A state wave: 16 rows v0 .. v0 + 15 of the state, chunk after chunk.
// Barriers (every wave of the workgroup passes the same sequence): E(-1),
// then per chunk c: M(c-1) (the output wave has read the hand-over of c-1; the
// copies of A stage c + 1 and B stage c have landed), E(c) (the hand-over of c
// written; A stage c free for the copies of c + 2).
__device__ __forceinline__ void cs_state_wave(float* __restrict__ S, uint32_t lds0, int hv, int v0,
                                              int wa, int g, int i, int l, int n_chunks) {
    const uint32_t ro = row_offset(g, i), co = col_offset(g, i);
    const uint32_t vo = (4 * g + (i >> 2)) * (CS_ROWS * 2) + 32 * wa + 8 * (i & 3);
    // the state, st[2 js + h][r] = S[v0 + i][32 js + 8 g + 4 h + r]: the result
    // layout of the 16 x 16 blocks of S^T
    float* Sv = S + ((size_t)hv * CK_V + v0 + i) * CK_K + 8 * g;
    f32x4 st[8];
#pragma unroll
    for (int kb8 = 0; kb8 < 8; ++kb8)
        st[kb8] = *(const f32x4*)(Sv + 32 * (kb8 >> 1) + 4 * (kb8 & 1));
    tile_done();   // E(-1): stages 0 and 1 landed
    // Each phase's LDS operands are read a phase ahead, behind a scheduling
    // fence, so no phase waits on LDS latency; X's K fragments, which do not
    // wait for the state, ahead of the hand-over of the chunk before.
    f16x8 kx[4][4];
    auto read_k = [&](int c) {
        const uint32_t sb = lds0 + L_A + (c & 1) * SA_BYTES;
        uint32_t ra[4];
        lane_addrs(sb, ro, ra);
#pragma unroll
        for (int js = 0; js < 4; ++js)
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) kx[js][mb] = row_frag(ra, SA_K, mb, js);
    };
    read_k(0);
    float ms = 0.f;   // the lane's part of max |S| of row v0 + i
#pragma unroll
    for (int kb8 = 0; kb8 < 8; ++kb8)
#pragma unroll
        for (int r = 0; r < 4; ++r) ms = fmaxf(ms, fabsf(st[kb8][r]));
    for (int c = 0; c < n_chunks; ++c) {
        const uint32_t sb = lds0 + L_A + (c & 1) * SA_BYTES;
        // e^{g_C} and 2^-tau
        const float eg_c = *(const lds_f32w*)(uintptr_t)(sb + SA_G + G_SC);
        const float t_un = *(const lds_f32w*)(uintptr_t)(sb + SA_G + G_SC + 4);
        __builtin_amdgcn_sched_barrier(0);

        // the state, scaled and split: B operands of the four k-steps
        float s_inv;
        const float s_sc = pow2_scale<7>(col_max(ms), s_inv);
        f16x8 sh[4], sl[4];
        split8(st[0], st[1], s_sc, sh[0], sl[0]);
        __builtin_amdgcn_sched_barrier(0);

        // Y's inputs, then X = K S^T (two passes), 64 tokens x 16 rows, on four
        // accumulators
        const uint32_t va = lane_addr(sb, vo), ga = lane_addr(sb, 16 * g);
        f16x4 vv[4];
        f32x4 be[4], eg[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            vv[mb] = __builtin_bit_cast(
                f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(
                           va + SA_V + 16 * CS_ROWS * 2 * mb)));
            be[mb] = *(lds_f32x4*)(uintptr_t)(ga + SA_G + G_BETA + 64 * mb);
            eg[mb] = *(lds_f32x4*)(uintptr_t)(ga + SA_G + G_EG + 64 * mb);
        }
        f32x4 x[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) x[mb] = (f32x4)(0.f);
        auto x_mfmas = [&](int js) {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) x[mb] = mfma16(kx[js][mb], sh[js], x[mb]);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) x[mb] = mfma16(kx[js][mb], sl[js], x[mb]);
        };
#pragma unroll
        for (int js = 0; js < 3; ++js) {
            split8(st[2 * js + 2], st[2 * js + 3], s_sc, sh[js + 1], sl[js + 1]);
            x_mfmas(js);
        }
#pragma unroll
        for (int j = 0; j < 24; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (j < 12) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        x_mfmas(3);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) eg[mb] *= -s_inv;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);

        // T's operands for Delta; then Y = beta (V - e^g X) (tokens 16 mb + 4 g
        // + r, column v0 + i)
        const uint32_t ta = lane_addr(sb, 16 * l);
        f16x8 th[CK_NF], tl[CK_NF];
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) {
            th[f] = *(lds_f16x8*)(uintptr_t)(ta + SA_T + 1024 * f);
            tl[f] = *(lds_f16x8*)(uintptr_t)(ta + SA_T + WS_OP + 1024 * f);
        }
        f32x4 yv[4];
        float my = 0.f;
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                yv[mb][r] = be[mb][r] * fmaf(eg[mb][r], x[mb][r], (float)vv[mb][r]);
                my = fmaxf(my, fabsf(yv[mb][r]));
            }
        }
        float y_inv;
        const float y_sc = pow2_scale<7>(col_max(my), y_inv);
        f16x8 yh[2], yl[2];
#pragma unroll
        for (int kq = 0; kq < 2; ++kq) split8(yv[2 * kq], yv[2 * kq + 1], y_sc, yh[kq], yl[kq]);
        __builtin_amdgcn_sched_barrier(0);

        // the state update's first K^T fragments and the decays; then
        // Delta = T Y (three passes; T is zero above the diagonal, so rows
        // 0..31 take no columns 32..63)
        uint32_t ca[4];
        lane_addrs(sb, co, ca);
        f16x8 kt[2][2][4];
#pragma unroll
        for (int kq = 0; kq < 2; ++kq)
#pragma unroll
            for (int b = 0; b < 4; ++b) kt[0][kq][b] = col_frag(ca, b, kq);
        f32x4 dk[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
            dk[mb] = *(lds_f32x4*)(uintptr_t)(ga + SA_G + G_DK + 64 * mb);
        f32x4 dl[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) dl[mb] = (f32x4)(0.f);
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) {
            const int mb = f_mb(f), kq = f_kq(f);
            dl[mb] = mfma16(th[f], yh[kq], dl[mb]);
        }
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) {
            const int mb = f_mb(f), kq = f_kq(f);
            dl[mb] = mfma16(th[f], yl[kq], dl[mb]);
        }
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) {
            const int mb = f_mb(f), kq = f_kq(f);
            dl[mb] = mfma16(tl[f], yh[kq], dl[mb]);
        }
        between_mfmas<18, 18>();
        __builtin_amdgcn_sched_barrier(0);

        // the second half's K^T fragments; Delta' = e^{g_C - g} Delta for
        // the state update, scaled and split
#pragma unroll
        for (int kq = 0; kq < 2; ++kq)
#pragma unroll
            for (int b = 0; b < 4; ++b) kt[1][kq][b] = col_frag(ca, 4 + b, kq);
        __builtin_amdgcn_sched_barrier(0);
        // (dl is Delta in T's and Y's scales, powers of two: 1 / d_un of it)
        const float d_un = t_un * y_inv;
        float md = 0.f;
        f32x4 dp[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                dp[mb][r] = dk[mb][r] * dl[mb][r];
                md = fmaxf(md, fabsf(dp[mb][r]));
            }
        }
        float p_inv;
        const float p_sc = pow2_scale<7>(col_max(md), p_inv);
        f16x8 ph[2], pl[2];
#pragma unroll
        for (int kq = 0; kq < 2; ++kq) split8(dp[2 * kq], dp[2 * kq + 1], p_sc, ph[kq], pl[kq]);
        const float p_un = p_inv * d_un;

        // S^T = e^{g_C} S^T + K^T Delta' (K exact: two passes), in two halves
        // of 4 k blocks, the first's sums formed between the second's MFMAs;
        // the rows' next maximum with it
        f32x4 u[2][4];
        auto update_mfmas = [&](int h) {
#pragma unroll
            for (int b = 0; b < 4; ++b) u[h][b] = (f32x4)(0.f);
#pragma unroll
            for (int kq = 0; kq < 2; ++kq) {
#pragma unroll
                for (int b = 0; b < 4; ++b) u[h][b] = mfma16(kt[h][kq][b], ph[kq], u[h][b]);
#pragma unroll
                for (int b = 0; b < 4; ++b) u[h][b] = mfma16(kt[h][kq][b], pl[kq], u[h][b]);
            }
        };
        ms = 0.f;
        auto update_sums = [&](int h) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st[4 * h + b][r] = fmaf(u[h][b][r], p_un, st[4 * h + b][r]);
                    ms = fmaxf(ms, fabsf(st[4 * h + b][r]));
                }
                // here, not past the barriers on the way to the next chunk
                asm volatile("" : "+v"(st[4 * h + b]));
            }
        };
#pragma unroll
        for (int kb8 = 0; kb8 < 8; ++kb8) st[kb8] *= eg_c;
        update_mfmas(0);
        __builtin_amdgcn_sched_barrier(0);
        update_mfmas(1);
        update_sums(0);
#pragma unroll
        for (int j = 0; j < 12; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);
        __builtin_amdgcn_sched_barrier(0);
        update_sums(1);
        asm volatile("" : "+v"(ms));
        __builtin_amdgcn_sched_barrier(0);

        // hand S0 and Delta to the output wave (after it has read the previous
        // chunk's), the next chunk's K fragments on their way
        tile_done();   // M(c-1)
        const uint32_t xo = lane_addr(lds0 + L_X + wa * X_WAVE, 16 * l);
#pragma unroll
        for (int js = 0; js < 4; ++js) {
            *(lds_f16x8w*)(uintptr_t)(xo + 1024 * js) = sh[js];
            *(lds_f16x8w*)(uintptr_t)(xo + X_SL + 1024 * js) = sl[js];
            *(lds_f32x4w*)(uintptr_t)(xo + X_DL + 1024 * js) = dl[js];
        }
        *(lds_f32x2w*)(uintptr_t)(xo + X_SC) = (f32x2){s_inv, d_un};
        asm volatile("" ::: "memory");
        // LDS operations end in order: with 15 of the 16 reads left, the
        // hand-over is written (a stage's reads are waited for ahead of M)
        if (c + 1 < n_chunks) {
            read_k(c + 1);
            asm volatile("s_waitcnt lgkmcnt(15)\n\ts_barrier" ::: "memory");   // E(c)
        } else {
            tile_done();   // E(c)
        }
    }
    // (the lane's part anew: the loop has no register left for it)
    const int le = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    float* Se = S + ((size_t)hv * CK_V + v0) * CK_K + (le & 15) * CK_K + 8 * (le >> 4);
#pragma unroll
    for (int kb8 = 0; kb8 < 8; ++kb8)
        *(f32x4*)(Se + 32 * (kb8 >> 1) + 4 * (kb8 & 1)) = st[kb8];
}

// A copy wave. Barriers as the state waves'; every copy of an iteration has
// landed before its M.
__device__ __forceinline__ void cs_copy_wave(const f16* q, const f16* k, const f16* v,
                                             const char* work, uint32_t lds0, int T, int n_vheads,
                                             int hv, int hk, int vw0, int wb, int l, int n_chunks,
                                             int qk_bytes, int v_bytes) {
    const char* kb = uniform_ptr((const char*)(k + (size_t)hk * CK_K));
    const char* qb = uniform_ptr((const char*)(q + (size_t)hk * CK_K));
    const char* vb = uniform_ptr((const char*)(v + (size_t)hv * CK_V + vw0));
    auto wblock = [&](int c) {
        return uniform_ptr(work + ((size_t)c * n_vheads + hv) * CK_BLK);
    };
    const CsOff off = cs_offsets(qk_bytes, v_bytes, wb, l);
    auto copy_a = [&](int c) {
        cs_copy_a(lds0 + L_A + (c & 1) * SA_BYTES, kb, vb, wblock(c), c * CK_C, T, qk_bytes,
                  v_bytes, wb, l, off);
    };
    auto copy_b = [&](int c) {
        cs_copy_b(lds0 + L_B + (c & 1) * SB_BYTES, qb, wblock(c), c * CK_C, T, qk_bytes, wb, l, off);
    };
    copy_a(0);
    copy_b(0);
    if (n_chunks > 1) copy_a(1);
    WAIT_VMCNT(0);
    tile_done();   // E(-1)
    tile_done();   // M(-1)
    for (int c = 0; c < n_chunks; ++c) {
        tile_done();   // E(c): A stage c and B stage c - 1 are free
        if (c + 2 < n_chunks) copy_a(c + 2);
        if (c + 1 < n_chunks) {
            copy_b(c + 1);
            WAIT_VMCNT(0);
            tile_done();   // M(c)
        }
    }
}

// An output wave: the paired state wave's rows, a chunk behind it. y at token
// t = 16 mb + 4 g + r, row v0 + i: O = e^g Q S0^T (two passes, S split as the
// state wave did) + (M o QK^T) Delta (three passes), accumulated scaled by
// 2^(kappa + eps). Barriers: E(-1), M(-1), then per chunk c: E(c), and M(c) but
// for the last chunk.
__device__ __forceinline__ void cs_output_wave(f16* __restrict__ y, uint32_t lds0, int T, int hv,
                                               int v0, int wb, int g, int i, int l, int n_chunks,
                                               int y_stride, float out_scale) {
    const uint32_t ro = row_offset(g, i);
    tile_done();   // E(-1)
    tile_done();   // M(-1)
    const uint32_t yt = lds0 + L_Y + wb * (CK_C * 32);
    for (int c = 0; c < n_chunks; ++c) {
        tile_done();   // E(c)
        const uint32_t xo = lds0 + L_X + wb * X_WAVE + l * 16;
        const uint32_t sbb = lds0 + L_B + (c & 1) * SB_BYTES;
        f16x8 sh[4], sl[4];
        f32x4 qs[4], dl[4];
#pragma unroll
        for (int js = 0; js < 4; ++js) {
            sh[js] = *(lds_f16x8*)(uintptr_t)(xo + 1024 * js);
            sl[js] = *(lds_f16x8*)(uintptr_t)(xo + X_SL + 1024 * js);
            dl[js] = *(lds_f32x4*)(uintptr_t)(xo + X_DL + 1024 * js);
            qs[js] = (f32x4)(0.f);
        }
        const f32x2 un = *(const lds_f32x2w*)(uintptr_t)(xo + X_SC);
        uint32_t ra[4];
        lane_addrs(sbb, ro, ra);
#pragma unroll
        for (int js = 0; js < 4; ++js) {
            f16x8 qa[4];
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) qa[mb] = row_frag(ra, SB_Q, mb, js);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) qs[mb] = mfma16(qa[mb], sh[js], qs[mb]);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) qs[mb] = mfma16(qa[mb], sl[js], qs[mb]);
        }
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            qs[mb] *= un[0];
            dl[mb] *= un[1];
        }
        const f32x4 sc = *(lds_f32x4*)(uintptr_t)(sbb + SB_G + G_SC);
        float mo = 0.f;
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int r = 0; r < 4; ++r) mo = fmaxf(mo, fabsf(dl[mb][r]));
        float o_inv;
        float o_sc = pow2_scale<7>(col_max(mo), o_inv);
        // o_up below brings e^g Q S0^T into the accumulator's scale. Chosen
        // from Delta alone, that scale overflows it for a zero (or nearly
        // zero) Delta row -- a chunk with beta = 0 throughout -- or a zero M o
        // QK^T block (2^-kappa = 2^-126): at most 2^64 2^-kappa, where
        // Delta's own term is below 2^-40 of y
        const float o_cap = 0x1p64f * sc[2];
        if (o_sc > o_cap) {
            o_sc = o_cap;
            o_inv = pow2_inv(o_cap);
        }
        f16x8 oh[2], ol[2];
#pragma unroll
        for (int kq = 0; kq < 2; ++kq) split8(dl[2 * kq], dl[2 * kq + 1], o_sc, oh[kq], ol[kq]);
        const float o_un = sc[2] * o_inv;
        const float o_up = o_sc * __builtin_amdgcn_rcpf(sc[2]);   // 1 / o_un: powers of two, exact
        f32x4 o[4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            const f32x4 eg = *(lds_f32x4*)(uintptr_t)(sbb + SB_G + G_EG + 4 * (16 * mb + 4 * g));
#pragma unroll
            for (int r = 0; r < 4; ++r) o[mb][r] = eg[r] * qs[mb][r] * o_up;
        }
        f16x8 qh[CK_NF], ql[CK_NF];
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) {
            const uint32_t fo = (f * 64 + l) * 16;
            qh[f] = *(lds_f16x8*)(uintptr_t)(sbb + SB_M + fo);
            ql[f] = *(lds_f16x8*)(uintptr_t)(sbb + SB_M + WS_OP + fo);
        }
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) o[f_mb(f)] = mfma16(qh[f], oh[f_kq(f)], o[f_mb(f)]);
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) o[f_mb(f)] = mfma16(qh[f], ol[f_kq(f)], o[f_mb(f)]);
#pragma unroll
        for (int f = 0; f < CK_NF; ++f) o[f_mb(f)] = mfma16(ql[f], oh[f_kq(f)], o[f_mb(f)]);
        // y through this wave's LDS tile: element (token 16 mb + 4 g + r, row
        // i) in, then lane l stores token l's 16 rows (32 bytes) with two
        // 16-byte stores
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *(lds_f16w*)(uintptr_t)(yt + (16 * mb + 4 * g + r) * 32 + 2 * i) =
                    f16_sat(o[mb][r] * o_un * out_scale);
        const f16x8 y0 = *(lds_f16x8*)(uintptr_t)(yt + l * 32);
        const f16x8 y1 = *(lds_f16x8*)(uintptr_t)(yt + l * 32 + 16);
        const int t0 = c * CK_C;
        if (T - t0 >= CK_C || l < T - t0) {
            f16* yo = y + (size_t)(t0 + l) * y_stride + (size_t)hv * CK_V + v0;
            *(f16x8*)yo = y0;
            *(f16x8*)(yo + 8) = y1;
        }
        if (c + 1 < n_chunks) tile_done();   // M(c)
    }
}

__global__ void __launch_bounds__(CS_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
chunk_state_kernel(const f16* __restrict__ q, const f16* __restrict__ k,
                   const f16* __restrict__ v, float* __restrict__ S, f16* __restrict__ y, int T,
                   int n_vheads, int qk_stride, int v_stride, int y_stride, float out_scale,
                   int group, const char* __restrict__ work) {
    extern __shared__ __attribute__((aligned(256))) char cs_smem[];
    // a v head's workgroups are n_vheads apart in the flat id, so with
    // n_vheads a multiple of 8 (48 here) they land on one XCD (dispatch goes
    // round robin over the 8) and share its L2
    const int hv = blockIdx.x % n_vheads, part = blockIdx.x / n_vheads, hk = hv / group;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = l >> 4, i = l & 15;
    const int vw0 = part * CS_ROWS;
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) char*)cs_smem);
    const int n_chunks = (T + CK_C - 1) / CK_C;
    if (w < 2)
        cs_state_wave(S, lds0, hv, vw0 + 16 * w, w, g, i, l, n_chunks);
    else if (w < 4)
        cs_output_wave(y, lds0, T, hv, vw0 + 16 * (w - 2), w - 2, g, i, l, n_chunks, y_stride,
                       out_scale);
    else if (w >= 6)
        cs_copy_wave(q, k, v, work, lds0, T, n_vheads, hv, hk, vw0, w - 6, l, n_chunks,
                     2 * qk_stride, 2 * v_stride);
}

// The front kernel's and the state pass's dynamic LDS is above the 64 KiB
// default: raised once per device (a mutex: callers may come from several threads).
std::mutex g_cs_mu;
constexpr int CS_MAX_DEVICES = 64;
bool g_cs_done[CS_MAX_DEVICES];

int raise_lds_limit() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= CS_MAX_DEVICES) {
        fl::set_error("gdn_chunk_state: no current device below index %d", CS_MAX_DEVICES);
        return FL_ELAUNCH;
    }
    std::lock_guard<std::mutex> lock(g_cs_mu);
    if (g_cs_done[dev]) return FL_OK;
    if (hipFuncSetAttribute((const void*)chunk_state_kernel,
                            hipFuncAttributeMaxDynamicSharedMemorySize, CS_LDS) != hipSuccess ||
        hipFuncSetAttribute((const void*)gdn_front_kernel,
                            hipFuncAttributeMaxDynamicSharedMemorySize, FR_LDS) != hipSuccess) {
        fl::set_error("gdn_chunk: cannot raise the dynamic LDS limit to %d bytes",
                      CS_LDS > FR_LDS ? CS_LDS : FR_LDS);
        return FL_ELAUNCH;
    }
    g_cs_done[dev] = true;
    return FL_OK;
}

}  // namespace

extern "C" {

size_t fl_gdn_chunked_work_bytes(int T, int n_vheads, int K, int V, int chunk) {
    if (T < 1 || n_vheads < 1 || K != CK_K || V != CK_V || chunk != CK_C) return 0;
    const size_t n_chunks = (size_t)(T + CK_C - 1) / CK_C;
    return n_chunks * n_vheads * CK_BLK;
}

}  // extern "C"

namespace {

int launch_state(const void* q, const void* k, const void* v, float* S, void* y, int T,
                 int n_vheads, int qk_stride, int v_stride, int y_stride, float out_scale,
                 int group, const void* work, fl_stream_t stream) {
    const int rc = raise_lds_limit();
    if (rc) return rc;
    hipLaunchKernelGGL(chunk_state_kernel, dim3(n_vheads * (CK_V / CS_ROWS)), dim3(CS_THREADS),
                       CS_LDS, (hipStream_t)stream, (const f16*)q, (const f16*)k, (const f16*)v, S,
                       (f16*)y, T, n_vheads, qk_stride, v_stride, y_stride, out_scale, group,
                       (const char*)work);
    return fl::check_launch("gdn_chunk_state");
}

int prefill_chunked(const void* q, const void* k, const void* v, const PrepGates& gates,
                    bool logits, float* S, void* y, int T, int n_kheads, int n_vheads, int K,
                    int V, int qk_stride, int v_stride, int y_stride, float out_scale, int group,
                    int chunk, void* work, size_t work_bytes, fl_stream_t stream) {
    FL_REQUIRE(q && k && v && gates.beta && gates.decay && S && y && work, "null pointer");
    FL_REQUIRE(!logits || (gates.A_log && gates.dt_bias && gates.stride >= n_vheads),
               "A_log, dt_bias; ab_stride >= n_vheads");
    FL_REQUIRE(K == CK_K && V == CK_V, "K == V == 128");
    FL_REQUIRE(chunk == CK_C, "chunk == 64");
    FL_REQUIRE(T >= 1, "T >= 1");
    FL_REQUIRE(group >= 1 && (n_vheads - 1) / group < n_kheads, "n_vheads / group <= n_kheads");
    FL_REQUIRE(qk_stride % 8 == 0 && v_stride % 8 == 0 && ((uintptr_t)q & 15u) == 0 &&
                   ((uintptr_t)k & 15u) == 0 && ((uintptr_t)v & 15u) == 0,
               "16-byte aligned q / k / v rows");
    FL_REQUIRE(((uintptr_t)S & 15u) == 0 && ((uintptr_t)work & 15u) == 0 &&
                   ((uintptr_t)y & 15u) == 0 && y_stride % 8 == 0,
               "16-byte aligned S, work and y rows");
    const size_t need = fl_gdn_chunked_work_bytes(T, n_vheads, K, V, chunk);
    if (work_bytes < need) {
        fl::set_error("work: %zu bytes, fl_gdn_chunked_work_bytes asks %zu", work_bytes, need);
        return FL_ESCRATCH;
    }
    const int n_chunks = (T + CK_C - 1) / CK_C;
    if (logits)
        hipLaunchKernelGGL(chunk_prep_kernel<true>, dim3(n_chunks, n_vheads), dim3(256), 0,
                           (hipStream_t)stream, (const f16*)q, (const f16*)k, gates, T, n_vheads,
                           qk_stride, group, (char*)work);
    else
        hipLaunchKernelGGL(chunk_prep_kernel<false>, dim3(n_chunks, n_vheads), dim3(256), 0,
                           (hipStream_t)stream, (const f16*)q, (const f16*)k, gates, T, n_vheads,
                           qk_stride, group, (char*)work);
    int rc = fl::check_launch("gdn_chunk_prep");
    if (rc) return rc;
    return launch_state(q, k, v, S, y, T, n_vheads, qk_stride, v_stride, y_stride, out_scale, group,
                        work, stream);
}

}  // namespace

extern "C" {

int fl_gdn_prefill_chunked(const void* q, const void* k, const void* v, const float* beta,
                           const float* decay, float* S, void* y, int T, int n_kheads,
                           int n_vheads, int K, int V, int qk_stride, int v_stride, int y_stride,
                           float out_scale, int group, int chunk, void* work, size_t work_bytes,
                           fl_stream_t stream) {
    return prefill_chunked(q, k, v, PrepGates{beta, decay, nullptr, nullptr, n_vheads}, false, S,
                           y, T, n_kheads, n_vheads, K, V, qk_stride, v_stride, y_stride,
                           out_scale, group, chunk, work, work_bytes, stream);
}

int fl_gdn_prefill_chunked_logits(const void* q, const void* k, const void* v, const float* a,
                                  const float* b, int ab_stride, const float* A_log,
                                  const float* dt_bias, float* S, void* y, int T, int n_kheads,
                                  int n_vheads, int K, int V, int qk_stride, int v_stride,
                                  int y_stride, float out_scale, int group, int chunk, void* work,
                                  size_t work_bytes, fl_stream_t stream) {
    return prefill_chunked(q, k, v, PrepGates{a, b, A_log, dt_bias, ab_stride}, true, S, y, T,
                           n_kheads, n_vheads, K, V, qk_stride, v_stride, y_stride, out_scale,
                           group, chunk, work, work_bytes, stream);
}

size_t fl_gdn_prefill_layer_work_bytes(int T, int x_stride, int n_vheads, int K, int V) {
    const size_t chunks = fl_gdn_chunked_work_bytes(T, n_vheads, K, V, CK_C);
    if (chunks == 0 || x_stride < 1) return 0;
    // the chunks' blocks, the conv'd (normed) rows, the unnormed outputs
    return chunks + ((size_t)T * x_stride * 2 + 15) / 16 * 16 + (size_t)T * n_vheads * V * 2;
}

int fl_gdn_prefill_layer(const void* x, int x_stride, const void* conv_w, const void* st_in,
                         void* st_out, int pos0, const float* a, const float* b, int ab_stride,
                         const float* A_log, const float* dt_bias, float* S, const void* z,
                         const float* norm_w, void* y, int T, int n_kheads, int n_vheads, int K,
                         int V, float out_scale, float l2eps, float norm_eps, void* work,
                         size_t work_bytes, fl_stream_t stream) {
    FL_REQUIRE(x && conv_w && st_in && st_out && a && b && A_log && dt_bias && S && z && norm_w &&
                   y && work,
               "null pointer");
    FL_REQUIRE(K == CK_K && V == CK_V, "K == V == 128");
    FL_REQUIRE(T >= 1 && pos0 >= 0, "T >= 1, pos0 >= 0");
    FL_REQUIRE(n_kheads >= 1 && n_vheads >= 1 && n_vheads % n_kheads == 0, "n_vheads % n_kheads");
    const int dim = 2 * n_kheads * K + n_vheads * V;
    FL_REQUIRE(x_stride >= dim && x_stride % 8 == 0, "x_stride covers q|k|v, a multiple of 8");
    FL_REQUIRE(ab_stride >= n_vheads, "ab_stride >= n_vheads");
    FL_REQUIRE(st_in != st_out, "st_in and st_out must be distinct buffers");
    FL_REQUIRE(((uintptr_t)S & 15u) == 0 && ((uintptr_t)work & 15u) == 0, "16-byte aligned S, work");
    // (the output norm's conditions, before anything is written)
    FL_REQUIRE(((uintptr_t)z & 3u) == 0 && ((uintptr_t)y & 3u) == 0 &&
                   ((uintptr_t)norm_w & 7u) == 0 && norm_eps >= 0.f,
               "aligned z, y, norm_w; norm_eps >= 0");
    const size_t need = fl_gdn_prefill_layer_work_bytes(T, x_stride, n_vheads, K, V);
    if (work_bytes < need) {
        fl::set_error("work: %zu bytes, fl_gdn_prefill_layer_work_bytes asks %zu", work_bytes, need);
        return FL_ESCRATCH;
    }
    char* blocks = (char*)work;
    f16* cx = (f16*)(blocks + fl_gdn_chunked_work_bytes(T, n_vheads, K, V, CK_C));
    f16* yr = (f16*)((char*)cx + ((size_t)T * x_stride * 2 + 15) / 16 * 16);
    const f16* q = cx;
    const f16* k = cx + n_kheads * K;
    const f16* v = cx + 2 * n_kheads * K;
    const PrepGates gates = {a, b, A_log, dt_bias, ab_stride};
    const int group = n_vheads / n_kheads;
    auto al16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    int rc;
    // the one-launch front takes the model's three v heads a k head with 16-byte
    // rows and enough chunks; anything else the conv and norm kernels, then the
    // chunked scan's own prep
    const int n_chunks = (T + CK_C - 1) / CK_C;
    if (group == FG && (long long)n_chunks * n_kheads >= FR_MIN_WGS && al16(x) && al16(conv_w) &&
        al16(st_in) && al16(st_out)) {
        rc = raise_lds_limit();
        if (rc) return rc;
        hipLaunchKernelGGL(gdn_front_kernel, dim3(n_chunks, n_kheads), dim3(FR_THREADS), FR_LDS,
                           (hipStream_t)stream, (const f16*)x, (const f16*)conv_w,
                           (const f16*)st_in, (f16*)st_out, cx, gates, T, pos0, n_kheads, x_stride,
                           l2eps, blocks);
        rc = fl::check_launch("gdn_front");
        if (rc) return rc;
        rc = launch_state(q, k, v, S, yr, T, n_vheads, x_stride, x_stride, n_vheads * V, out_scale,
                          group, blocks, stream);
    } else {
        rc = fl_conv1d_causal(x, conv_w, st_in, cx, st_out, dim, T, pos0, x_stride, 4, stream);
        if (rc) return rc;
        rc = fl_l2norm_scaled_strided(cx, cx, 2 * n_kheads, K, x_stride, l2eps, 1.f, T, stream);
        if (rc) return rc;
        rc = prefill_chunked(q, k, v, gates, true, S, yr, T, n_kheads, n_vheads, K, V, x_stride,
                             x_stride, n_vheads * V, out_scale, group, CK_C, blocks,
                             fl_gdn_chunked_work_bytes(T, n_vheads, K, V, CK_C), stream);
    }
    if (rc) return rc;
    return fl_rmsnorm_gated(yr, z, norm_w, y, V, n_vheads, V, T, norm_eps, stream);
}

}  // extern "C"
