// k_shared.hip -- the shared expert for batches (S > 1) on the bf16 MFMA: the
// three bf16 parts of the inputs, gate_up + SiLU-GLU (writing the parts of h),
// and down.  Per (row, token) the arithmetic is that of the single-token jobs
// of the decode stages (sw_shared.h), so a token's shared expert output does
// not depend on the batch it came in.
//
#include "sw_hip.h"
#include "sw_shared.h"

// parts of the rows of x [S, K] f32 -> [S][K/32][3][32] bf16, 8 inputs per thread
__global__ __launch_bounds__(256) void k_sh_parts(const float *__restrict__ x, int64_t n8, int K,
                                                  uint16_t *__restrict__ parts) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= n8) return;
    const int k8 = K / 8;
    const int64_t tok = c / k8;
    const int cc = (int)(c - tok * k8);
    const sw_f32x4 *xv = (const sw_f32x4 *)(x + tok * K + 8 * cc);
    sw_u32x4 p0, p1, p2;
    sh_split8(xv[0], xv[1], p0, p1, p2);
    uint16_t *dst = parts + tok * K * 3 + (cc >> 2) * 3 * SH_RG + (cc & 3) * 8;
    *(sw_u32x4 *)dst = p0;
    *(sw_u32x4 *)(dst + SH_RG) = p1;
    *(sw_u32x4 *)(dst + 2 * SH_RG) = p2;
}

// Prefill-sized batches.  Block: 4 waves, 128 rows x 64 tokens; wave w takes rows
// 32 w .. +31 (two 16-row tiles) against the four 16-token column tiles.  The
// tokens' part words of a step go through LDS (two buffers: the next step's
// loads are in flight in registers while the waves read this one, issued
// before each step's barrier), each token's 192 bytes a group at a padded stride;
// the waves' weight words come from global memory a step ahead.  All loads are
// unconditional (past the end they read the last step again): a load under a branch
// made the waits before it drain everything in flight.  What bounds it: up to ~1000
// tokens the serial chain of K / 64 steps (a barrier and a load's latency each, with
// a block or less per CU), beyond that LDS and the MFMAs.  Two groups of 32 inputs per
// barrier, C2 (D = 4096, Is = 1024), gate_up / down us, one group with branches ->
// now: 112 / 33 -> 78 / 24 at 181 tokens, 120 / 78 -> 114 / 67 at 2048; four groups:
// 78 / 26 and 142 / 93 (one block per CU by LDS).  Blocks are dealt so that an XCD runs whole
// token tiles (all their row blocks), whose part words then come from its L2.
// The fold starts from -0.0, the identity of
// f32 addition (-0 + y == y bit for bit), so every segment is added the same way.
#define SHB_TOK 64             // tokens per block
#define SHB_TS 208             // LDS bytes per token and group: 192 + 16 of padding
#define SHB_STAGE (SHB_TOK * SHB_TS)
#define SHB_CH (SHB_TOK * 12 / 256)   // 16-byte chunks staged per thread and group
#define SHB_NG 2               // groups of 32 inputs per step: K a multiple of 64
template <class RowPtr>
__device__ __forceinline__ void sh_block_tiles(RowPtr rowp, const uint16_t *__restrict__ xp, int S, int K, int tok0,
                                               uint8_t *lds, sw_f32x4 tot[2][4]) {
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kq = lane >> 4;
    const int G = K / SH_RG, GS = G / sh_nseg(G), NS = G / SHB_NG;
    const uint16_t *wr[2];
#pragma unroll
    for (int t = 0; t < 2; t++) wr[t] = rowp(t, m) + 8 * kq;
    // staging: chunk q = u * 256 + tid of a group -> token q / 12, chunk q % 12
    const uint16_t *sp[SHB_CH];
    int so[SHB_CH];
#pragma unroll
    for (int u = 0; u < SHB_CH; u++) {
        const int q = u * 256 + tid, tk = q / 12, ch = q - tk * 12;
        sp[u] = xp + (int64_t)min(tok0 + tk, S - 1) * G * 3 * SH_RG + ch * 8;
        so[u] = tk * SHB_TS + ch * 16;
    }
    // (unconditional: a step past the end re-reads the last)
    auto stage_load = [&](int s, sw_u32x4 (&r)[SHB_NG][SHB_CH]) {
        const int g0 = min(s, NS - 1) * SHB_NG;
#pragma unroll
        for (int n = 0; n < SHB_NG; n++)
#pragma unroll
            for (int u = 0; u < SHB_CH; u++) r[n][u] = *(const sw_u32x4 *)(sp[u] + (int64_t)(g0 + n) * 3 * SH_RG);
    };
    auto stage_store = [&](int buf, const sw_u32x4 (&r)[SHB_NG][SHB_CH]) {
#pragma unroll
        for (int n = 0; n < SHB_NG; n++)
#pragma unroll
            for (int u = 0; u < SHB_CH; u++) *(sw_u32x4 *)(lds + (buf * SHB_NG + n) * SHB_STAGE + so[u]) = r[n][u];
    };
    auto ald = [&](int s, sw_u32x4 (&a)[SHB_NG][2]) {
        const int g0 = min(s, NS - 1) * SHB_NG;
#pragma unroll
        for (int n = 0; n < SHB_NG; n++)
#pragma unroll
            for (int t = 0; t < 2; t++) a[n][t] = *(const sw_u32x4 *)(wr[t] + (int64_t)(g0 + n) * SH_RG);
    };
    sw_f32x4 acc[2][4];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            acc[t][c] = sw_f32x4{0.f, 0.f, 0.f, 0.f};
            tot[t][c] = sw_f32x4{-0.f, -0.f, -0.f, -0.f};
        }
    sw_u32x4 an[SHB_NG][2], sr[SHB_NG][SHB_CH];
    ald(0, an);
    stage_load(0, sr);
    stage_store(0, sr);
    stage_load(1, sr);
    __syncthreads();
    for (int s = 0; s < NS; s++) {
        sw_u32x4 a[SHB_NG][2];
#pragma unroll
        for (int n = 0; n < SHB_NG; n++) { a[n][0] = an[n][0]; a[n][1] = an[n][1]; }
        ald(s + 1, an);
#pragma unroll
        for (int n = 0; n < SHB_NG; n++) {
            const uint8_t *base = lds + ((s & 1) * SHB_NG + n) * SHB_STAGE + m * SHB_TS + kq * 16;
            // column tile c's part words from LDS, tile c + 1's read while c's MFMAs run
            sw_u32x4 b[2][3];
            auto bld = [&](int c, sw_u32x4 *bb) {
#pragma unroll
                for (int p = 0; p < 3; p++) bb[p] = *(const sw_u32x4 *)(base + 16 * c * SHB_TS + 64 * p);
            };
            bld(0, b[0]);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (c + 1 < 4) bld(c + 1, b[(c + 1) & 1]);
                acc[0][c] = sh_mfma3(a[n][0], b[c & 1][0], b[c & 1][1], b[c & 1][2], acc[0][c]);
                acc[1][c] = sh_mfma3(a[n][1], b[c & 1][0], b[c & 1][1], b[c & 1][2], acc[1][c]);
            }
            if ((s * SHB_NG + n + 1) % GS == 0) {          // a segment ends: fold it in
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        tot[t][c] = tot[t][c] + acc[t][c];
                        acc[t][c] = sw_f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
        stage_store((s + 1) & 1, sr);                  // read by no wave since the last barrier
        stage_load(s + 2, sr);                         // registers only: issued before the barrier's wait
        __syncthreads();
    }
}

// block (64 outputs i0 = 64 bx.., 64 tokens): wave w's tile t holds gate rows i0 + 16 w + 8 t
// + 0..7 (tile rows 0-7) and the same up rows (8-15); h's parts [S][Is/32][3][32]
__global__ __launch_bounds__(256) void k_sh_glu_mf(const uint16_t *__restrict__ Wg, const uint16_t *__restrict__ Wu,
                                                   const uint16_t *__restrict__ xp, int S, int D, int Is,
                                                   uint16_t *__restrict__ hp) {
    __shared__ __align__(16) uint8_t lds[2 * SHB_NG * SHB_STAGE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
    const int nrb = Is / 64, w = sw_xcd_work((int)blockIdx.x, (int)gridDim.x);   // an XCD's blocks: whole token tiles
    const int ib = (w % nrb) * 64 + 16 * wave, tok0 = (w / nrb) * SHB_TOK;
    sw_f32x4 tot[2][4];
    sh_block_tiles([&](int t, int r) {
        const int i = ib + 8 * t + (r & 7);
        return (r < 8 ? Wg : Wu) + (int64_t)i * D;
    }, xp, S, D, tok0, lds, tot);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            // lanes kq < 2 hold gate rows 4 kq + r; lane + 32 holds the up rows of the same outputs
            float hv[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float yg = tot[t][c][r], yu = __shfl_xor(tot[t][c][r], 32);
                hv[r] = (yg / (1.0f + expf(-yg))) * yu;
            }
            const int tok = tok0 + 16 * c + m;
            if (kq < 2 && tok < S) {
                const int i = ib + 8 * t + 4 * kq;      // four consecutive outputs of one group
                uint32_t pa[4], pb[4], pc[4];
#pragma unroll
                for (int r = 0; r < 4; r++) sh_split3(hv[r], pa[r], pb[r], pc[r]);
                uint16_t *dst = hp + (int64_t)tok * Is * 3 + (i >> 5) * 3 * SH_RG + (i & 31);
                *(uint2 *)dst = make_uint2(pa[0] | (pa[1] << 16), pa[2] | (pa[3] << 16));
                *(uint2 *)(dst + SH_RG) = make_uint2(pb[0] | (pb[1] << 16), pb[2] | (pb[3] << 16));
                *(uint2 *)(dst + 2 * SH_RG) = make_uint2(pc[0] | (pc[1] << 16), pc[2] | (pc[3] << 16));
            }
        }
}

// block (128 rows d0 = 128 bx.., 64 tokens): out[tok][d] f32
__global__ __launch_bounds__(256) void k_sh_down_mf(const uint16_t *__restrict__ Wd, const uint16_t *__restrict__ hp, int S,
                                                    int Is, int D, float *__restrict__ out) {
    __shared__ __align__(16) uint8_t lds[2 * SHB_NG * SHB_STAGE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
    const int nrb = D / 128, w = sw_xcd_work((int)blockIdx.x, (int)gridDim.x);
    const int db = (w % nrb) * 128 + 32 * wave, tok0 = (w / nrb) * SHB_TOK;
    sw_f32x4 tot[2][4];
    sh_block_tiles([&](int t, int r) { return Wd + (int64_t)(db + 16 * t + r) * Is; }, hp, S, Is, tok0, lds, tot);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int tok = tok0 + 16 * c + m;
            if (tok < S) *(sw_f32x4 *)(out + (int64_t)tok * D + db + 16 * t + 4 * kq) = tot[t][c];
        }
}

// ---- decode-sized batches: K split over the waves (sh_sk_block, sw_shared.h) ----
template <int GLU, int NC>
__global__ __launch_bounds__(SH_SK_NT) void k_sh_sk(ShSkArgs A) {
    __shared__ float red[8 * 16 * 16 * NC];                // [segment][row][token]
    sh_sk_block<GLU, NC, 0>(A, blockIdx.x, blockIdx.y, red);
}
// The shared expert's down fused with the rank-order combine of a decode-sized batch:
// block (bx, by) runs the down of rows 16 bx .. +15 for the 32 tokens of column tile
// by (sh_sk_block, written to shared [S][D]), then combines those outputs of those
// tokens (combine4, the combine launch's arithmetic) into out.  A block's 16 outputs
// are half of each 128-byte line of the slot rows it reads: the row blocks go to the
// XCDs in contiguous ranges, so both halves of a line are read through one L2.
__global__ __launch_bounds__(SH_SK_NT) void k_sh_combine(ShSkArgs A, const float *__restrict__ slots,
                                                        const int *__restrict__ rowof, const float *__restrict__ w, int K,
                                                        float route_scale, float *__restrict__ out) {
    __shared__ float red[8 * 16 * 16 * 2];
    const int rb = sw_xcd_work((int)blockIdx.x, (int)gridDim.x);
    sh_sk_block<0, 2, 0>(A, rb, blockIdx.y, red);
    __syncthreads();                                    // the tile's shared outputs are written
    const int tid = threadIdx.x;
    if (tid < 32 * 4) {
        const int64_t s = (int64_t)blockIdx.y * 32 + (tid >> 2);
        if (s < A.S) combine4(slots, rowof, w, s, K, A.O, rb * 16 + 4 * (tid & 3), route_scale,
                              (const float *)A.out, out, 1, nullptr, 0);
    }
}

// ---- batches between: the gate_up's K split over the waves, 32 rows x 16 NC tokens per block ----
// Wave w runs segment w of the K inputs (the chains of sh_sk_block, 2 row tiles instead of
// one), the results folded left to right in LDS.  No two waves share an input, so weights and
// parts come straight from global memory (the parts mostly from L2), the next step's in flight
// behind this one's MFMAs.  What bounds it: those reads, 2 KB of weights and 3 KB of parts per
// column tile and step for 4 or more MFMA triples; with one row tile (k_sh_sk) the parts are
// read twice as often, with k_sh_glu_mf's LDS tiles K is one serial chain in D/32 steps.
// C2 (D = 4096, Is = 1024), us per launch at 125 / 181 / 256 tokens: k_sh_sk 66 / 89 / 113,
// NC = 2 here 40 / 73 / 67, NC = 4 69 / 64 / 62, k_sh_glu_mf 82 / 78 / 74.
template <int NC>
__global__ __launch_bounds__(SH_SK_NT, 2) void k_sh_glu_skr(ShSkArgs A) {
    extern __shared__ __align__(16) float red[];       // [segment][row][token]
    constexpr int RT = 2, R = 16 * RT, T = 16 * NC;    // R / 2 outputs
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
    const int S = A.S, K = A.K, O = A.O, G = K / SH_RG, nseg = sh_nseg(G), GS = G / nseg;
    const int nrb = O / (R / 2), w = sw_xcd_work((int)blockIdx.x, (int)gridDim.x);
    const int r0 = (w % nrb) * (R / 2), tok0 = (w / nrb) * T;
    if (wave < nseg) {
        const int g0 = wave * GS;
        const uint16_t *wr[RT], *br[NC];
#pragma unroll
        for (int t = 0; t < RT; t++)
            wr[t] = (m < 8 ? A.W0 : A.W1) + (int64_t)(r0 + 8 * t + (m & 7)) * K + 8 * kq + (int64_t)g0 * SH_RG;
#pragma unroll
        for (int c = 0; c < NC; c++)
            br[c] = A.xp + (int64_t)min(tok0 + 16 * c + m, S - 1) * K * 3 + 8 * kq + (int64_t)g0 * 3 * SH_RG;
        struct Step { sw_u32x4 a[RT], b[NC][3]; };
        auto load = [&](int s, Step &st) {             // (past the segment: its last step again)
            const int g = min(s, GS - 1);
#pragma unroll
            for (int t = 0; t < RT; t++) st.a[t] = *(const sw_u32x4 *)(wr[t] + (int64_t)g * SH_RG);
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int p = 0; p < 3; p++) st.b[c][p] = *(const sw_u32x4 *)(br[c] + (int64_t)(g * 3 + p) * SH_RG);
        };
        sw_f32x4 acc[RT][NC];
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int c = 0; c < NC; c++) acc[t][c] = sw_f32x4{0.f, 0.f, 0.f, 0.f};
        auto use = [&](const Step &st) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int t = 0; t < RT; t++) acc[t][c] = sh_mfma3(st.a[t], st.b[c][0], st.b[c][1], st.b[c][2], acc[t][c]);
        };
        Step ring[2];
        load(0, ring[0]);
        load(1, ring[1]);
        int s0 = 0;
        for (; s0 + 2 < GS; s0 += 2) {
            use(ring[0]);
            load(s0 + 2, ring[0]);
            use(ring[1]);
            load(s0 + 3, ring[1]);
        }
        use(ring[0]);
        if (s0 + 1 < GS) use(ring[1]);
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) red[(wave * R + 16 * t + 4 * kq + r) * T + 16 * c + m] = acc[t][c][r];
    }
    __syncthreads();
    const int tid = threadIdx.x;
    // output i of the block: tile i / 8, gate row i % 8, up row 8 + i % 8 (outputs fastest, so a
    // token's parts are written side by side)
    for (int it = tid; it < R / 2 * T; it += SH_SK_NT) {
        const int i = it % (R / 2), t = it / (R / 2), tok = tok0 + t, row = (i >> 3) * 16 + (i & 7);
        float yg = -0.0f, yu = -0.0f;
        for (int sg = 0; sg < nseg; sg++) {
            yg = yg + red[(sg * R + row) * T + t];
            yu = yu + red[(sg * R + row + 8) * T + t];
        }
        if (tok < S) {
            const int oi = r0 + i;
            uint32_t pa, pb, pc;
            sh_split3((yg / (1.0f + expf(-yg))) * yu, pa, pb, pc);
            uint16_t *dst = (uint16_t *)A.out + (int64_t)tok * O * 3 + (oi >> 5) * 3 * SH_RG + (oi & 31);
            dst[0] = (uint16_t)pa;
            dst[SH_RG] = (uint16_t)pb;
            dst[2 * SH_RG] = (uint16_t)pc;
        }
    }
}
template <int NC>
static int launch_glu_skr(hipStream_t st, const ShSkArgs &A) {
    SW_LAUNCH((k_sh_glu_skr<NC>), dim3((unsigned)(A.O / 16 * sh_sk_cols(A.S, NC))), dim3(SH_SK_NT), 8 * 32 * 16 * NC * 4, st, A);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// decode-sized batches take the split-K blocks: the gate_up 16-token column tiles up to
// 32 tokens (the grid then fills the chip), else 32-token tiles
template <int GLU>
static int launch_sk(hipStream_t st, const uint16_t *W0, const uint16_t *W1, const uint16_t *xp, int S, int K, int O,
                     void *out) {
    const int nc = sh_sk_nc(GLU, S);
    const dim3 grid((unsigned)sh_sk_rows(GLU, O), (unsigned)sh_sk_cols(S, nc));
    const ShSkArgs A = {W0, W1, xp, nullptr, S, K, O, out};
    if (nc == 1) SW_LAUNCH((k_sh_sk<GLU, 1>), grid, dim3(SH_SK_NT), 0, st, A);
    else SW_LAUNCH((k_sh_sk<GLU, 2>), grid, dim3(SH_SK_NT), 0, st, A);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int sw_launch_sh_parts(hipStream_t st, const float *x, int S, int K, uint16_t *parts) {
    if (S <= 0 || !sh_shape_ok(K)) return -1;
    const int64_t n8 = (int64_t)S * (K / 8);
    SW_LAUNCH(k_sh_parts, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, x, n8, K, parts);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The gate_up of a batch on its own (beside the MFMA experts, or with the router over token
// tiles): the narrowest blocks with which the grid is at most a block per CU, as a second
// round costs as much as the first (figures at k_sh_glu_skr; C2 at 40 / 64 tokens: k_sh_sk 34
// / 37 us, NC = 2 41 / 40).  Up to 128 tokens a K split pays also beyond that.
int sw_launch_sh_glu(hipStream_t st, const uint16_t *Wg, const uint16_t *Wu, const uint16_t *xp, int S, int D, int Is,
                     uint16_t *hp) {
    if (S <= 0 || Is % 64 || D % (SHB_NG * SH_RG) || !sh_shape_ok(D)) return -1;
    const ShSkArgs A = {Wg, Wu, xp, nullptr, S, D, Is, hp};
    const int64_t cus = 256;
    if (S <= 32 || (S <= SH_SK_MAX_S && (int64_t)sh_sk_rows(1, Is) * sh_sk_cols(S, 2) <= cus))
        return launch_sk<1>(st, Wg, Wu, xp, S, D, Is, hp);
    if (S <= SH_SK_MAX_S || (int64_t)(Is / 16) * sh_sk_cols(S, 2) <= cus) return launch_glu_skr<2>(st, A);
    if ((int64_t)(Is / 16) * sh_sk_cols(S, 4) <= cus) return launch_glu_skr<4>(st, A);
    const dim3 grid((unsigned)(Is / 64 * ((S + SHB_TOK - 1) / SHB_TOK)));
    SW_LAUNCH(k_sh_glu_mf, grid, dim3(256), 0, st, Wg, Wu, xp, S, D, Is, hp);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The down on its own: the split-K blocks while the batch is one tile of k_sh_down_mf's, and
// up to 128 tokens while they run in one round on the CUs, or in two where K is long (a tile's
// time is its serial loop over K; D / 16 x S / 32 split blocks against D / 128 x 2 tiles).  us
// split / tiles, 128 tokens: D = 1024 (256 blocks) Is = 512 8.2 / 11.6, 2048 14 / 32; D = 2048
// (512) Is = 512 15 / 11.5, 1024 15 / 18, 2048 27 / 32; D = 4096 (1024) Is = 1024 30 / 18.6
int sw_launch_sh_down(hipStream_t st, const uint16_t *Wd, const uint16_t *hp, int S, int Is, int D, float *out) {
    if (S <= 0 || D % 128 || Is % (SHB_NG * SH_RG) || !sh_shape_ok(Is)) return -1;
    const int64_t blocks = (int64_t)sh_sk_rows(0, D) * sh_sk_cols(S, sh_sk_nc(0, S));
    if (S <= SHB_TOK || (S <= SH_SK_MAX_S && blocks <= (Is >= 1024 ? 512 : 256)))
        return launch_sk<0>(st, Wd, nullptr, hp, S, Is, D, out);
    const dim3 grid((unsigned)(D / 128 * ((S + SHB_TOK - 1) / SHB_TOK)));
    SW_LAUNCH(k_sh_down_mf, grid, dim3(256), 0, st, Wd, hp, S, Is, D, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int sw_launch_sh_combine(hipStream_t st, const uint16_t *Wd, const uint16_t *hp, int S, int Is, int D, float *shared,
                         const float *slots, const int *rowof, const float *w, int K, float route_scale, float *out) {
    if (S <= 0 || S > SH_SK_MAX_S || D % 16 || K <= 0 || !sh_shape_ok(Is)) return -1;
    const ShSkArgs A = {Wd, nullptr, hp, nullptr, S, Is, D, shared};
    const dim3 grid((unsigned)sh_sk_rows(0, D), (unsigned)sh_sk_cols(S, 2));
    SW_LAUNCH(k_sh_combine, grid, dim3(SH_SK_NT), 0, st, A, slots, rowof, w, K, route_scale, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
