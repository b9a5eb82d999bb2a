// k_mfma.hip -- the grouped int4 expert GEMMs of prefill on the matrix cores,
// bit-identical to the dot8 kernels of k_dot8.hip.
//
// For a weight row and a group of 32 inputs, dot8 forms the exact integer
// acc = sum_k w_k D_k (w_k = n_k - 8 in [-8, 7], D_k the 7-limb integer of
// input k, |D_k| < 2^21.2) and the term (float)acc * (s * xf).  Here every D
// is cut into two 12-bit digits, D = E1 2^12 + E0 with E0 the residue of D
// mod 4096 in [-2048, 2048) and |E1| <= 585.  The weights and both digits are
// integers that f16 holds exactly, and every product (|w E| <= 2^14) and
// every partial sum of 32 of them (< 2^19) is an integer that f32 holds
// exactly, so two v_mfma_f32_16x16x32_f16 return R0 = sum_k w_k E0_k and
// R1 = sum_k w_k E1_k exactly, whatever order the hardware adds in; then
// fma(R1, 4096, R0) rounds the exact acc = 4096 R1 + R0 once, to nearest even,
// which is (float)acc, dot8's conversion of its int32, bit for bit.  The
// terms and the canonical row sum (pairwise trees over runs of 16 groups,
// padded with +0 terms, the runs added left to right) follow dot8's
// operations one for one, so a token's output has the same bits whichever
// kernel ran its group.
//
// Digits in memory: per (input row, group) 128 bytes, E0 of the 32 inputs as f16, then E1: the
// A operands of the two MFMAs (A rows: tokens; B columns: weight rows).  Lane l of an MFMA
// (token, resp. weight row, l % 16; k quarter q = l / 16) reads the 16 bytes of inputs 8q ..
// 8q+7 of its token (in the slot order of mf_expand), and its B operand holds the same inputs
// of its weight row as f16, expanded from packed dword q of the row's group.
//
// Block: 256 weight rows x a tile of up to 16 NT tokens (NT columns of 16) of one group, 8
// waves.  A wave owns two 16-row tiles (for gate_up the gate and the up rows of the same 16
// outputs) and runs them against every column.  Per quad of 4 input groups it loads 64 bytes
// of each of its rows straight into registers -- a lane the whole packed group kq of its row,
// transposed within the lanes by permlane swaps -- expands each weight once for all the
// tile's columns, and reads the columns' digits and factors from LDS, where the block stages
// them in two buffers, a chunk of quads ahead.  A lane's four results are of one weight row,
// whose scale is a plain register, and of four tokens.  Loads of a quad are
// issued a quad ahead, a step's two MFMAs one step (column, group, row tile) ahead of its
// sums.  A group's tokens are split into equal tiles of whole columns (sw_mf_tile), and a
// tile runs the loop of its own column count.
//
// What bounds it: no one unit.  A step is 2 MFMAs, 4 conversions (one fma each), 4 products of
// scale and factor, 4 terms, 4 sums on average, and its share of the expansion (9 operations
// per 8 weights): a quad of 4, 3, 2 or 1 columns has 599, 479, 359 or 243 VALU instructions
// beside 64, 48, 32 or 16 MFMAs.  VALU issue is the largest part, but 12 % more instructions
// in the loop took 3 % longer at 64 tokens and 7 % more 0.6-1.5 % at 16; at 64 tokens the
// waves, two per SIMD, spend 26 % of their time waiting (LDS reads, 1 KB per step for two
// row tiles, and a barrier per chunk).  (Those instructions round every term before it is
// added.  Acc times s, with the power of two applied by the fma of the add, had 8 fewer per
// quad, row tile and column, but left dot8's bits where s * xf is no normal number, acc * s
// overflows or a term does.)  A run's four quads stand in a line: as two loops of two, every
// pair began with an add to -0, and at 64 tokens a register reloaded in each quad made its
// wait drain the loads in flight (a step of C2, S = 2048, 4.5 % longer, S = 181 2.4 %, of C1, S
// = 333, 5.5 %).  16 tokens (NT = 1) fit 128 registers, four waves per SIMD; 64 take 256, two,
// and spill 13 (gate_up) and 47 (down, group scales of 32), reloaded once or a few times a run.
// Expanding in every wave from registers replaced weights expanded once per block into LDS,
// whose reads (1 KB per row tile and group) and barriers (one per chunk over 16 waves) bounded
// the loop: C2 S = 2048 gate_up 1,754 -> 1,425 us, down 963 -> 786; S = 181 568 -> 400 and 313
// -> 224; C1 S = 333 147 -> 131 and 78 -> 76.
#include "sw_hip.h"
#include "sw_gate.h"

#define MF_DW 32           // digit dwords per (input row, group)
#define MF_ROWS 256        // weight rows per block: 32 per wave
#define MF_NTH 512         // threads per block: 8 waves
// the (column, group) pairs of a staged chunk: 4 groups of up to four token columns, 8 of
// two, or 8 of one (fewer staging registers where a wave has 128)
#define MF_PAIRS(NT) ((NT) == 1 ? 8 : 16)
// the two chunk buffers in LDS: digits [g][column][op 2][quarter 4][token 16] x 16 B, and
// token factors [g][column][token]
#define MF_B_SZ(NT) (MF_PAIRS(NT) * 2048)
#define MF_X_SZ(NT) (MF_PAIRS(NT) * 64)
#define MF_X_OFF(NT) (2 * MF_B_SZ(NT))
#define MF_HLD 129         // floats per token row of h in the gate_up epilogue (64 rows within the buffers)

template <int N>
struct MfIc { static constexpr int v = N; };

// ------------------------------------------------------------ digits ----
// one group by the 32 lanes of a half-wave (i = lane in the half): the same
// exponent and 7 limbs as limbs_group, written as the MFMA digits above (E0
// then E1 of the 32 inputs as f16, each quarter of 8 inputs in the operand
// order of mf_expand); the factor 2^(e - 21) (NaN for a group holding a NaN or
// an infinity, whose digits are 0) is limbs_group's
__device__ __forceinline__ void digits_group(float v, int i, uint32_t *__restrict__ dst, float *__restrict__ fdst) {
    bool bad;
    const int e = limbs_exp(v, bad);
    float y = ldexpf(v, -e);
    int D = 0;
#pragma unroll
    for (int l = 0; l < SW_ND; l++) D = D * 8 + (int)limb_digit(y);
    if (bad) D = 0;
    const int E0 = ((D + 2048) & 4095) - 2048, E1 = (D - E0) >> 12;
    // the odd inputs of a quarter meet weights 16 w: their digits are E / 16 (exact:
    // at most 11 significant bits, none below 2^-4)
    const float sc = (i & 1) ? 0.0625f : 1.0f;
    const uint32_t h0 = __builtin_bit_cast(uint16_t, (_Float16)((float)E0 * sc));
    const uint32_t h1 = __builtin_bit_cast(uint16_t, (_Float16)((float)E1 * sc));
    // dword d of quarter q = i >> 3 holds inputs d (low half) and d + 4 (mf_expand's order)
    const uint32_t o0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h0, 0x104, 0xF, 0xF, true);   // row_shl 4: lane i + 4
    const uint32_t o1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h1, 0x104, 0xF, 0xF, true);
    if ((i & 4) == 0) {
        const int dw = (i >> 3) * 4 + (i & 3);
        dst[dw] = h0 | (o0 << 16);
        dst[16 + dw] = h1 | (o1 << 16);
    }
    if (i == 0) *fdst = bad ? __builtin_nanf("") : ldexpf(1.0f, e - 3 * SW_ND);
}

// rows x[r, K] f32 -> digits dg[r][K/32][32 dwords], factors xs[r][K/32]
__global__ __launch_bounds__(256) void k_digits(const float *__restrict__ x, int K, int rows, uint32_t *__restrict__ dg,
                                                float *__restrict__ xs) {
    const int G = K / SW_RG;
    const int tid = threadIdx.x, g = blockIdx.x * 8 + (tid >> 5), r = blockIdx.y;
    if (r >= rows || g >= G) return;                  // whole half-waves leave together
    digits_group(x[(int64_t)r * K + g * SW_RG + (tid & 31)], tid & 31, dg + ((int64_t)r * G + g) * MF_DW,
                 xs + (int64_t)r * G + g);
}

int sw_launch_digits(hipStream_t st, const float *x, int rows, int K, uint32_t *dg, float *xs) {
    if (K % SW_RG || rows <= 0) return -1;
    const int G = K / SW_RG;
    SW_LAUNCH(k_digits, dim3((unsigned)((G + 7) / 8), (unsigned)rows), dim3(256), 0, st, x, K, rows, dg, xs);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ------------------------------------------------------------ GEMM ----
struct MfArgs {
    SwQ4 W;
    int gsh;
    const uint32_t *dg;     // input digits [rows][G][MF_DW]
    const float *xs;        // input factors [rows][G]
    int dg_rows;            // rows of dg and xs (dg_rows * K * 4 < 2^32)
    SwGroups grp;           // tiles: items of up to 16 NT tokens, P live
    int I;                  // GLU: the intermediate size (W.O == 2 I)
    int nrb;                // row blocks
    int rbper;              // row blocks per block (dividing nrb)
    uint32_t *hdg;          // GLU: h of every packed row as digits [T][I/32][MF_DW]
    float *hxs;             //      and factors [T][I/32]
    float *Y;               // rows: [T][O]
    const SwTab *tab;       // per-group tensors (the _tab launches) or null
};

// the weight operand of packed dword w (nibble n_r = w_r + 8 of input r of the quarter at
// bits 4r) as f16 pairs (w0, w4), (16 w1, 16 w5), (w2, w6), (16 w3, 16 w7), the order of
// digits_group.  Nibbles r and r + 4 sit 16 bits apart: masked out in place and ORed into
// the mantissas of the f16 pair (1024, 1024) they give 1024 + n (bits 0-3) or 1024 + 16 n
// (bits 4-7); adding -1032, resp. -1152, leaves w, resp. 16 w, exactly.  9 operations per
// 8 weights, 4 of them on the packed f16 unit (which, like byte permutes and DPP, issues at
// about 4.6 cycles against 2.7 for plain 32-bit operations, two or more waves per SIMD)
__device__ __forceinline__ sw_half8 mf_expand(uint32_t w) {
    const uint32_t lo = 0x000F000Fu, hi = 0x00F000F0u, magic = 0x64006400u, v = w >> 8;
    const sw_half2 off_lo = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    const sw_half2 off_hi = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    sw_i32x4 a;
    a[0] = __builtin_bit_cast(int, __builtin_bit_cast(sw_half2, (w & lo) | magic) + off_lo);
    a[1] = __builtin_bit_cast(int, __builtin_bit_cast(sw_half2, (w & hi) | magic) + off_hi);
    a[2] = __builtin_bit_cast(int, __builtin_bit_cast(sw_half2, (v & lo) | magic) + off_lo);
    a[3] = __builtin_bit_cast(int, __builtin_bit_cast(sw_half2, (v & hi) | magic) + off_hi);
    return __builtin_bit_cast(sw_half8, a);
}

// A lane loads 16 bytes of its row: the whole packed group kq = lane / 16 of a quad.
// An MFMA of group g wants dword kq of group g in lane quarter kq, the transpose of
// the 4 x 4 (lane quarter, dword) block: two swaps of lane halves, two of 16-lane rows
__device__ __forceinline__ void mf_transpose(const sw_u32x4 &r, uint32_t (&o)[4]) {
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const u2 a = __builtin_amdgcn_permlane32_swap(r.x, r.z, false, false);
    const u2 b = __builtin_amdgcn_permlane32_swap(r.y, r.w, false, false);
    const u2 c = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false);
    const u2 d = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
    o[0] = c.x; o[1] = c.y; o[2] = d.x; o[3] = d.y;
}

// NT: the tile's most 16-token columns; SM: the weight scales, 0 one per row (after the
// sum), 1 one per 32 inputs, 2 one per 64, 3 one per 128 or more (one a quad)
template <int GLU, int NT, int SM, int PT>
__global__ __launch_bounds__(MF_NTH, NT == 1 ? 4 : 2) void k_mf(MfArgs A) {
    constexpr int CG = MF_PAIRS(NT) / NT, QPC = CG / 4;    // groups and quads per staged chunk
    constexpr int PV = MF_PAIRS(NT) / 4;                   // digit units per staging thread and chunk
    constexpr int B_SZ = MF_B_SZ(NT), X_SZ = MF_X_SZ(NT), X_OFF = MF_X_OFF(NT);
    constexpr int RPB = GLU ? MF_ROWS / 2 : MF_ROWS;       // output rows a row block moves on by
    static_assert(MF_NTH == 512, "staging map");
    extern __shared__ __align__(16) uint8_t mf_lds[];
    const SwQ4 W = A.W;
    const SwGroups grp = A.grp;
    const int K = W.K, G = K / SW_RG, O = W.O;
    const int NC = G / 4;                                  // quads of 4 groups
    const int NCH = (NC + QPC - 1) / QPC;                  // staged chunks of a row block
    const int NQ = G > 8 ? 4 : NC;                         // quads per run (G = 4, 8: one short run)
    // (the wave index in a scalar register: what derives from it is uniform to the compiler)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 15,
              kq = lane >> 4;

    // block -> (tile, run of rbper row blocks), XCD-aware over the live blocks; the chunk
    // pipeline runs on from one row block to the next
    const int rbper = GLU ? 1 : A.rbper;
    const int nrg = A.nrb / rbper;
    const int nlive = *grp.P * nrg;
    if ((int)blockIdx.x >= nlive) return;
    const int wk = sw_xcd_work((int)blockIdx.x, nlive);
    const int tile = wk / nrg, rbf = (wk - tile * nrg) * rbper;     // the block's first row block
    int e, beg, t0, tend;
    if (!grp_work(grp, tile, 16 * NT, e, beg, t0, tend)) return;
    const int nt = tend - t0, nact = (nt + 15) >> 4;       // tokens, token columns with tokens
    auto token = [&](int t) -> uint32_t {                  // input row of tile token t (past the tile: its last)
        const int pr = beg + t0 + min(t, nt - 1);
        return (uint32_t)(grp.grow ? grp.grow[pr] : pr);
    };
    const int ng = W.gs > 0 ? K / W.gs : 1;
    const uint32_t rbytes = (uint32_t)K / 2, sbytes = (uint32_t)ng * 4;
    sw_rsrc rq[2], rs[2];                                  // row tile t's tensor
    if constexpr (PT) {
        const SwTab tb_ = A.tab[e];
        const uint32_t rows = (uint32_t)(GLU ? A.I : O);
        rq[0] = sw_make_rsrc(GLU ? tb_.g : tb_.d, rows * rbytes);
        rq[1] = sw_make_rsrc(GLU ? tb_.u : tb_.d, rows * rbytes);
        rs[0] = sw_make_rsrc(GLU ? tb_.gs : tb_.ds, rows * sbytes);
        rs[1] = sw_make_rsrc(GLU ? tb_.us : tb_.ds, rows * sbytes);
    } else {
        rq[0] = rq[1] = sw_q4_rq(W);
        rs[0] = rs[1] = sw_q4_rs(W);
    }
    // ---- the wave's weight rows: row tile 0 and 1 start at tensor rows wr0, wr1.  gate_up:
    // the gate and the up rows of the same 16 outputs; down: 32 rows in a line (a wave past
    // O, where O is an odd number of half blocks, reads the last rows and stores nothing)
    const int lr = (GLU ? 16 : 32) * wave;                 // the wave's rows in a row block
    const uint32_t eo = PT ? 0u : (uint32_t)e * (uint32_t)O;
    auto wrow = [&](int t, int rb) -> uint32_t {
        if constexpr (GLU) return eo + (uint32_t)(rb * RPB + lr + (t && !PT ? A.I : 0));
        return eo + (uint32_t)(min(rb * RPB + lr, O - 32) + 16 * t);
    };
    struct Raw { sw_u32x4 q[2]; sw_f32x4 s[2]; };
    // quad c of row block rb: 64 bytes of each of the tile's 16 rows, 16 per lane, and the quad's
    // four scales of the lane's own row col (the same in the row's four lanes)
    auto load_w = [&](Raw &R, int rb, int c) {
        const uint32_t cu = (uint32_t)__builtin_amdgcn_readfirstlane(c);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t r0 = wrow(t, rb);
            R.q[t] = sw_ld16(rq[t], (r0 + (uint32_t)col) * rbytes + (uint32_t)kq * 16, cu * 64);
            const uint32_t vs = (r0 + (uint32_t)col) * sbytes;
            if constexpr (SM == 1) R.s[t] = __builtin_bit_cast(sw_f32x4, sw_ld16(rs[t], vs, cu * 16));
            if constexpr (SM == 2) {
                const uint2 v = sw_ld8(rs[t], vs, cu * 8);
                R.s[t][0] = R.s[t][1] = __builtin_bit_cast(float, v.x);
                R.s[t][2] = R.s[t][3] = __builtin_bit_cast(float, v.y);
            }
            if constexpr (SM == 3) {
                const float v = sw_ld4f(rs[t], vs, ((cu * 128) >> A.gsh) * 4);
                R.s[t] = sw_f32x4{v, v, v, v};
            }
        }
    };
    // ---- staging a chunk of CG groups: the digits in 16-byte units [g][column][op][quarter]
    // [token], PV per thread (unit v * 512 + tid: one wave load is 64 bytes of 16 tokens, one
    // wave store 1 KB in a line), and the token factors [g][column][token], one each by the
    // first threads.  Columns with no tokens are not staged.
    const int dtok = tid & 15, dpart = ((tid >> 6) & 1) * 64 + ((tid >> 4) & 3) * 16, drc = tid >> 7;
    const int dcol = __builtin_amdgcn_readfirstlane(drc % NT), dg0 = drc / NT;      // uniform per wave
    const int xg = NT == 1 ? (tid >> 4) & 7 : ((tid >> 4) & 3) + (NT == 2 ? 4 * ((tid >> 6) & 1) : 0);
    const int xcol = __builtin_amdgcn_readfirstlane(NT == 1 ? 0 : NT == 2 ? (tid >> 7) & 1 : (tid >> 6) & 3);
    const bool dact = dcol < nact, xact = wave < MF_PAIRS(NT) / 4 && xcol < nact;
    const sw_rsrc rd = sw_make_rsrc(A.dg, (uint32_t)A.dg_rows * (uint32_t)G * MF_DW * 4);
    const sw_rsrc rx = sw_make_rsrc(A.xs, (uint32_t)A.dg_rows * (uint32_t)G * 4);
    // (every load is unconditional -- an empty column's of column 0, from cache -- so that the
    // compiler's wait counts stay exact; only the stores are skipped)
    const uint32_t vd = token(16 * (dact ? dcol : 0) + dtok) * (uint32_t)G * (MF_DW * 4) + (uint32_t)dpart;
    const uint32_t vx = token(16 * (xcol < nact ? xcol : 0) + dtok) * (uint32_t)G * 4;
    sw_u32x4 pkb[PV];
    float pxf = 0.f;
    auto stage_load = [&](int ch) {                        // chunk ch % NCH of a row block (groups past G: the last)
        const int g0 = __builtin_amdgcn_readfirstlane((GLU ? ch : ch % NCH) * CG);
        if constexpr (QPC == 1) {                          // (never past G)
#pragma unroll
            for (int v = 0; v < PV; v++) pkb[v] = sw_ld16(rd, vd, (uint32_t)(g0 + v) * (MF_DW * 4));
            pxf = sw_ld4f(rx, vx + (uint32_t)xg * 4, (uint32_t)g0 * 4);
        } else {
#pragma unroll
            for (int v = 0; v < PV; v++) pkb[v] = sw_ld16(rd, vd + (uint32_t)min(g0 + dg0 + v * (4 / NT), G - 1) * (MF_DW * 4), 0);
            pxf = sw_ld4f(rx, vx + (uint32_t)min(g0 + xg, G - 1) * 4, 0);
        }
    };
    auto stage_store = [&](int buf) {
        sw_u32x4 *Bl = (sw_u32x4 *)(mf_lds + buf * B_SZ);
        if (dact)
#pragma unroll
            for (int v = 0; v < PV; v++) Bl[v * MF_NTH + tid] = pkb[v];
        if (xact) ((float *)(mf_lds + X_OFF + buf * X_SZ))[(xg * NT + xcol) * 16 + dtok] = pxf;
    };

    // a row block's sums out: gate_up, h = silu(gate) * up through LDS to its digits (four
    // groups of the down's input per token); down, the rows of each token
    auto epilogue = [&](auto NAC, int rb, const sw_f32x4 (&y)[2][decltype(NAC)::v]) {
        constexpr int NA = decltype(NAC)::v;
        if constexpr (GLU) {
            const int I = A.I, ib = rb * RPB;
            float *el = (float *)mf_lds;                   // (the chunk buffers: every wave is past its last read)
            const int i = lr + col;                        // the lane's output, of tokens 4 kq .. + 3
            float gsc = 1.f, usc = 1.f;
            if constexpr (SM == 0) {                       // per-row scales after the sum
                gsc = PT ? A.tab[e].gs[ib + i] : W.s[(int64_t)e * O + ib + i];
                usc = PT ? A.tab[e].us[ib + i] : W.s[(int64_t)e * O + I + ib + i];
            }
#pragma unroll
            for (int c = 0; c < NA; c++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float yg = y[0][c][j], yu = y[1][c][j];
                    if constexpr (SM == 0) {
                        yg = yg * gsc;
                        yu = yu * usc;
                    }
                    el[(16 * c + 4 * kq + j) * MF_HLD + i] = (yg / (1.0f + expf(-yg))) * yu;
                }
            __syncthreads();
            const int GI = I / SW_RG, hw = tid >> 5, ih = tid & 31;
            for (int job = hw; job < 4 * nt; job += MF_NTH / 32) {
                const int t = job >> 2, q = job & 3, gi = ib / SW_RG + q;
                const int64_t prow = beg + t0 + t;
                digits_group(el[t * MF_HLD + 32 * q + ih], ih, A.hdg + (prow * GI + gi) * MF_DW, A.hxs + prow * GI + gi);
            }
        } else {
            const int row0 = rb * RPB + lr;
            if (row0 >= O) return;                         // uniform per wave
#pragma unroll
            for (int rt = 0; rt < 2; rt++) {
                const int row = row0 + 16 * rt + col;      // the lane's row, of tokens 4 kq .. + 3
                const float ds = SM ? 1.f : PT ? A.tab[e].ds[row] : W.s[(int64_t)e * O + row];
#pragma unroll
                for (int c = 0; c < NA; c++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int t = 16 * c + 4 * kq + j;
                        if (t < nt) A.Y[(int64_t)(beg + t0 + t) * O + row] = SM ? y[rt][c][j] : y[rt][c][j] * ds;
                    }
            }
        }
    };

    auto main_loop = [&](auto NAC) {
        constexpr int NA = decltype(NAC)::v;               // the tile's token columns
        Raw raw;
        load_w(raw, rbf, 0);
        stage_load(0);
        stage_store(0);
        const int QT = rbper * NCH;                        // the block's chunks
        stage_load(min(1, QT - 1));
        int ch = 0;                                        // the chunk in LDS buffer ch & 1
        __syncthreads();
        // quad qc of row block rb into acc.  All loads -- the next quad's weights, the next
        // chunk's digits -- are issued at its top and waited for at the next one's or at the
        // chunk's end, a whole quad's work later: issued at its end, the next top's wait for
        // the (older) weights would drain them too
        auto quad = [&](auto FIRST, int rb, int qc, sw_f32x4 (&acc)[2][NA]) {   // FIRST: acc starts here
            // the quad's operands: 4 groups of both row tiles, then the next quad's loads
            // (expanded once for several columns; for a single one group by group, in registers)
            sw_half8 a[2][NA > 1 ? 4 : 1];
            uint32_t w[2][4];
            sw_f32x4 sc[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                mf_transpose(raw.q[t], w[t]);
                if constexpr (NA > 1)
#pragma unroll
                    for (int g = 0; g < 4; g++) a[t][g] = mf_expand(w[t][g]);
                if constexpr (SM) sc[t] = raw.s[t];
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                const bool more = qc + 1 < NC;
                load_w(raw, more ? rb : min(rb + 1, rbf + rbper - 1), more ? qc + 1 : 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            const int gl = qc % QPC * 4;               // the quad's first group in its chunk
            const uint8_t *pb = mf_lds + (ch & 1) * B_SZ + gl * NT * 2048 + lane * 16;
            const uint8_t *px = mf_lds + X_OFF + (ch & 1) * X_SZ + (gl * NT * 16 + 4 * kq) * 4;
            // steps (column c, group g, row tile t), t fastest: a (c, g)'s digits are read two
            // (c, g) ahead, a step's two MFMAs issued one step ahead of its sums
            struct Op { sw_half8 b0, b1; sw_f32x4 xf; } op[2];
            sw_f32x4 R[2][2];
            auto fetch = [&](int k, Op &o) {
                const int c = k >> 2, g = k & 3;
                o.b0 = *(const sw_half8 *)(pb + (g * NT + c) * 2048);
                o.b1 = *(const sw_half8 *)(pb + (g * NT + c) * 2048 + 1024);
                o.xf = *(const sw_f32x4 *)(px + (g * NT + c) * 64);
            };
            auto mul = [&](int i, const Op &o, sw_f32x4 (&r_)[2]) {
                const sw_f32x4 z = {0.f, 0.f, 0.f, 0.f};
                const int t = i & 1, g = (i >> 1) & 3;
                const sw_half8 av = NA > 1 ? a[t][NA > 1 ? g : 0] : mf_expand(w[t][g]);
                r_[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.b0, av, z, 0, 0, 0);
                r_[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.b1, av, z, 0, 0, 0);
            };
            constexpr int NS = 8 * NA;
            fetch(0, op[0]);
            fetch(1, op[1]);
            mul(0, op[0], R[0]);
            sw_f32x4 h[2], q[2];
#pragma unroll
            for (int i = 0; i < NS; i++) {
                const int c = i >> 3, g = (i >> 1) & 3, t = i & 1;
                const sw_f32x4 xf = op[(i >> 1) & 1].xf;
                if (i + 1 < NS) mul(i + 1, op[((i + 1) >> 1) & 1], R[(i + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                // dot8's terms and sums: (float)acc, exact, times the product of s and the
                // token's power of two
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float a_ = __builtin_fmaf(R[i & 1][1][j], 4096.0f, R[i & 1][0][j]);
                    const float p = a_ * (SM ? sc[t][g] * xf[j] : xf[j]);
                    if (g == 0 || g == 2) h[t][j] = p;
                    else if (g == 1) q[t][j] = h[t][j] + p;
                    else q[t][j] = q[t][j] + (h[t][j] + p);
                }
                // (formed here: the compiler would sink the sums to their last use, with every
                // product live until then)
                if (g == 0 || g == 2) asm volatile("" : "+v"(h[t]));
                else asm volatile("" : "+v"(q[t]));
                if (t == 1 && (i >> 1) + 2 < NS / 2) fetch((i >> 1) + 2, op[(i >> 1) & 1]);
                if (g == 3) acc[t][c] = decltype(FIRST)::v ? q[t] : acc[t][c] + q[t];
                __builtin_amdgcn_sched_barrier(0);
            }
            // the chunk's last quad: the next chunk into the other buffer (read by no wave since
            // the last barrier)
            if (qc % QPC == QPC - 1 || qc == NC - 1) {
                if (ch + 1 < QT) stage_store((ch + 1) & 1);
                stage_load(min(ch + 2, QT - 1));
                ch++;
                __syncthreads();
            }
        };
        auto fill = [&](sw_f32x4 (&v)[2][NA], float x) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int c = 0; c < NA; c++) v[t][c] = sw_f32x4{x, x, x, x};
        };
        // (y starts from -0, the identity of f32 addition: the first run's bits as they are)
        for (int rbi = 0; rbi < rbper; rbi++) {
            const int rb = rbf + rbi;
            sw_f32x4 y[2][NA];
            fill(y, -0.f);
#pragma unroll 1
            for (int r0 = 0; r0 < NC; r0 += 4) {
                // a run: (q0 + q1) + (q2 + q3), a short last run padded with +0 terms
                sw_f32x4 ra[2][NA], rv[2][NA];
                quad(MfIc<1>{}, rb, r0, ra);
                if (r0 + 1 < NC) quad(MfIc<0>{}, rb, r0 + 1, ra);
                if (NQ == 4) {
                    if (r0 + 2 < NC) {
                        quad(MfIc<1>{}, rb, r0 + 2, rv);
                        if (r0 + 3 < NC) quad(MfIc<0>{}, rb, r0 + 3, rv);
                    } else fill(rv, 0.f);
                    if (r0 + 4 > NC) {
#pragma unroll
                        for (int t = 0; t < 2; t++)
#pragma unroll
                            for (int c = 0; c < NA; c++) {
                                if (r0 + 1 == NC) ra[t][c] = ra[t][c] + 0.f;
                                rv[t][c] = rv[t][c] + 0.f;
                            }
                    }
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int c = 0; c < NA; c++) ra[t][c] = ra[t][c] + rv[t][c];
                }
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int c = 0; c < NA; c++) y[t][c] = y[t][c] + ra[t][c];
            }
            epilogue(NAC, rb, y);
        }
    };
    if constexpr (NT == 1) main_loop(MfIc<1>{});
    else if constexpr (NT == 2) {
        if (nact == 1) main_loop(MfIc<1>{});
        else main_loop(MfIc<2>{});
    } else {
        if (nact == 1) main_loop(MfIc<1>{});
        else if (nact == 2) main_loop(MfIc<2>{});
        else if (nact == 3) main_loop(MfIc<3>{});
        else main_loop(MfIc<4>{});
    }
}

// ------------------------------------------------------------ launch ----
// the chunk buffers; the gate_up epilogue's h lies over them
template <int NT>
static size_t mf_lds_bytes() {
    const size_t b = MF_X_OFF(NT) + 2 * MF_X_SZ(NT), h = (size_t)16 * NT * MF_HLD * 4;
    return b > h ? b : h;
}
// dynamic LDS above 64 KB, raised once per kernel, outside any stream work
template <int GLU, int NT, int SM, int PT>
static int mf_go(hipStream_t st, unsigned nblocks, const MfArgs &A) {
    static size_t raised = 0;
    const size_t lds = mf_lds_bytes<NT>();
    if (lds > raised) {
        if (hipFuncSetAttribute((const void *)k_mf<GLU, NT, SM, PT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess) return -1;
        raised = lds;
    }
    SW_LAUNCH((k_mf<GLU, NT, SM, PT>), dim3(nblocks), dim3(MF_NTH), lds, st, A);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <int GLU, int PT = 0>
static int mf_dispatch(hipStream_t st, unsigned nblocks, const MfArgs &A) {
    const int tt = A.grp.tt;
#define SW_MF_SM(N_) \
    (A.W.gs <= 0 ? mf_go<GLU, N_, 0, PT>(st, nblocks, A) \
     : A.W.gs == SW_RG ? mf_go<GLU, N_, 1, PT>(st, nblocks, A) \
     : A.W.gs == 2 * SW_RG ? mf_go<GLU, N_, 2, PT>(st, nblocks, A) : mf_go<GLU, N_, 3, PT>(st, nblocks, A))
    if (tt == 16) return SW_MF_SM(1);
    if (tt == 32) return SW_MF_SM(2);
    if (tt == 64) return SW_MF_SM(4);
#undef SW_MF_SM
    return -1;
}
// row blocks per block: the down's short row blocks (K = I) up to four at a time, one start
// and one drain for all, while that leaves at least 1024 blocks (four per CU) by the launch's
// bound on its tiles; the gate_up's long ones one at a time
#define MF_RBPER_ROWS 4
static int mf_rbper(int nrb, int tiles) {
    for (int r = MF_RBPER_ROWS; r > 1; r >>= 1)
        if (nrb % r == 0 && (int64_t)tiles * (nrb / r) >= 1024) return r;
    return 1;
}
// shapes: K a multiple of 128 (whole chunks of 4 input groups), tiles listed (items, P),
// the digits addressed by 32-bit offsets
static int mf_check(const SwQ4 &W, const SwGroups &g, int &gsh, int dg_rows) {
    if (W.K % (SW_RG * 4) || !g.items || !g.P || g.ngroups_max <= 0 || !sw_q4_extent_ok(W)) return -1;
    if (dg_rows <= 0 || (uint64_t)dg_rows * (uint64_t)W.K * 4 > 0xFFFFFFFFull) return -1;
    return sw_q4_gsh(W, gsh);
}

int sw_launch_mf_glu(hipStream_t st, SwQ4 W, const uint32_t *dg, const float *xs, int dg_rows, SwGroups g, int I,
                     uint32_t *hdg, float *hxs) {
    int gsh;
    if (mf_check(W, g, gsh, dg_rows) || I % 128 || W.O != 2 * I) return -1;
    const int nrb = I / 128;
    const MfArgs A = {W, gsh, dg, xs, dg_rows, g, I, nrb, 1, hdg, hxs, nullptr};
    return mf_dispatch<1>(st, (unsigned)(g.ngroups_max * nrb), A);
}

int sw_launch_mf_rows(hipStream_t st, SwQ4 W, const uint32_t *dg, const float *xs, int dg_rows, SwGroups g, float *Y) {
    int gsh;
    if (mf_check(W, g, gsh, dg_rows) || W.O % 32) return -1;
    const int nrb = (W.O + MF_ROWS - 1) / MF_ROWS;
    const int rp = mf_rbper(nrb, g.ngroups_max);
    const MfArgs A = {W, gsh, dg, xs, dg_rows, g, 0, nrb, rp, nullptr, nullptr, Y};
    return mf_dispatch<0>(st, (unsigned)(g.ngroups_max * (nrb / rp)), A);
}

// the same two GEMMs over per-group tensors: group c's gate/up/down are tab[gexp[c]]
// (W gives O, K and gs; each tensor holds one expert)
int sw_launch_mf_glu_tab(hipStream_t st, SwQ4 W, const SwTab *tab, const uint32_t *dg, const float *xs, int dg_rows,
                         SwGroups g, int I, uint32_t *hdg, float *hxs) {
    int gsh;
    W.E = 1;
    if (!tab || !hdg || !hxs || mf_check(W, g, gsh, dg_rows) || I % 128 || W.O != 2 * I) return -1;
    const int nrb = I / 128;
    const MfArgs A = {W, gsh, dg, xs, dg_rows, g, I, nrb, 1, hdg, hxs, nullptr, tab};
    return mf_dispatch<1, 1>(st, (unsigned)(g.ngroups_max * nrb), A);
}
int sw_launch_mf_rows_tab(hipStream_t st, SwQ4 W, const SwTab *tab, const uint32_t *dg, const float *xs, int dg_rows,
                          SwGroups g, float *Y) {
    int gsh;
    W.E = 1;
    if (!tab || !Y || mf_check(W, g, gsh, dg_rows) || W.O % 32) return -1;
    const int nrb = (W.O + MF_ROWS - 1) / MF_ROWS;
    const int rp = mf_rbper(nrb, g.ngroups_max);
    const MfArgs A = {W, gsh, dg, xs, dg_rows, g, 0, nrb, rp, nullptr, nullptr, Y, tab};
    return mf_dispatch<0, 1>(st, (unsigned)(g.ngroups_max * (nrb / rp)), A);
}
