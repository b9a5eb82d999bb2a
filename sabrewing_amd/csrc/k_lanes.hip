// k_lanes.hip -- the reference CPU's 16-lane GEMV contracts on gfx950, bit for
// bit: y[s, o] of a row-major weight matrix W [O, I] against rows of x.
//
// The reference's SIMD matmuls reduce each output in a fixed order that is
// part of their result.  Lane j of 16 keeps one f32 chain; the chains are
// then added by GCC's _mm512_reduce_add_ps tree (t8[j] = a[j] + a[j+8],
// t4[j] = t8[j] + t8[j+4], (t4[0] + t4[2]) + (t4[1] + t4[3])).  Two chain
// shapes cover the contracts this file serves:
//   F32X  lane j: acc = fma(x[i], w[i], acc) for i = j, j+16, j+32, ... while
//         a whole 16 (32 for int4) remain, then a scalar tail fused into the
//         sum.  Weights widen exactly: bf16 (c/moe_matmul.h:92-110, round_x =
//         0), int8 (matmul_q8_k F32, c/moe_quant.h:378-391), int4 nibble - 8
//         (matmul_q4_k F32, c/moe_quant.h:85-109); the int ones end in * scale.
//   DP    vdpbf16ps (round_x = 1, c/moe_matmul.h:66-89; inkling's matmul_h):
//         x rounded to bf16 (RNE, NaN quieted, a denormal input to a signed
//         zero), lane j takes the bf16 pair (2j, 2j+1) of every 32 columns,
//         two FMAs in a row -- the odd column first -- with denormal inputs
//         read as zero and a denormal result flushed to a signed zero.
//   I4G   matmul_i4_grouped (c/quant.h:168-203, its AVX2 body): per scale group
//         of gs columns 8 lanes, lane j: fma over columns i + j then i + 8 + j
//         for every 16 of the group, hsum8 ((v0+v4)+(v2+v6)) + ((v1+v5)+(v3+v7)),
//         then a = fma(h, scale[o][g], a) over the groups in order.  The 16
//         lanes of a row take two groups at a time (lanes 0-7 the even, 8-15
//         the odd one); the group sums go through LDS to the row's lane 0,
//         which runs the ordered scale chain.  A group wider than a tile (gs a
//         multiple of 256) is taken by lanes 0-7 alone, their chains carried
//         across its tiles.
// Each (row, token) is one lane chain, so a result never depends on the
// shape of the launch that computed it.
//
// k_lanes_w streams rows of whole 16-byte pieces (below).  k_lanes16 takes the rest -- the
// group-scaled int4, odd row lengths, odd addresses, short rows of many blocks: 256 threads = 16 rows x 16 lanes; tiles
// of CC columns of the 16 rows (coalesced 16-byte loads) and of up to TS tokens go through
// LDS, and each token's chains stay in registers across tiles.
#include "sw_hip.h"
#include "sw_libm.h"

#define LN_ROWS 16
#define LN_CC 256                  // columns per LDS tile

enum { WK_BF16 = 0, WK_I8 = 1, WK_I4 = 2, WK_I4G = 3 };

__device__ __forceinline__ float bf16_widen(uint32_t h) { return __builtin_bit_cast(float, h << 16); }
// a denormal to a signed zero (the DAZ / FTZ of vdpbf16ps)
__device__ __forceinline__ float flush_dn(float v) {
    // (one class test: 0x90 are the two subnormal classes)
    return __builtin_amdgcn_classf(v, 0x90) ? __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0x80000000u) : v;
}
// vcvtne2ps2bf16 of one float, widened back to f32
__device__ __forceinline__ float round_bf16_ne(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return bf16_widen((u >> 16) | 0x40);
    if ((u & 0x7F800000u) == 0) return bf16_widen((u >> 16) & 0x8000);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return bf16_widen(u >> 16);
}

template <int WK> struct WElem { static constexpr int bits = WK == WK_BF16 ? 16 : WK == WK_I8 ? 8 : 4; };
// wave-local LDS ordering (the 16 lanes of a row are in one wave)
__device__ __forceinline__ void lanes_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// element i of an LDS row tile, widened exactly
template <int WK>
__device__ __forceinline__ float w_at(const uint8_t *row, int i) {
    if constexpr (WK == WK_BF16) return bf16_widen(((const uint16_t *)row)[i]);
    else if constexpr (WK == WK_I8) return (float)((const int8_t *)row)[i];
    else {
        const uint8_t b = row[i >> 1];
        return (float)((int)((i & 1) ? (b >> 4) : (b & 15)) - 8);
    }
}

struct LanesArgs {
    const void *W;          // [O, I]
    const float *scale;     // [O] (int weights), [O][I/gs] (I4G) or null
    const float *x;         // [S, I]
    float *y;               // [S, O]
    int S, I, O;
    int gs;                 // I4G: columns per scale group (16..256, dividing I)
    int ldx, ldy;           // row strides of x and y
};

// reduce16 over the 16 lanes of a row (xor partners stay inside the row)
__device__ __forceinline__ float reduce16_lanes(float v) {
    v = v + __shfl_xor(v, 8, 16);
    v = v + __shfl_xor(v, 4, 16);
    v = v + __shfl_xor(v, 2, 16);
    return v + __shfl_xor(v, 1, 16);
}

// row o of token s out: the scalar tail of the columns past imain, then the row scale
template <int WK, int DP>
__device__ __forceinline__ void lanes_out(const LanesArgs &A, float sm, int s, int o, int imain) {
    const float *xs = A.x + (size_t)s * A.ldx;
    const uint8_t *wr = (const uint8_t *)A.W + (size_t)o * ((size_t)A.I * WElem<WK == WK_I4G ? WK_I4 : WK>::bits / 8);
    if constexpr (WK == WK_I4) {                       // the byte tail of c/moe_quant.h:105-108
        for (int i = imain; i + 1 < A.I; i += 2) {
            const uint8_t b = wr[i >> 1];
            const float lo = (float)((int)(b & 15) - 8), hi = (float)((int)(b >> 4) - 8);
            sm = sm + __builtin_fmaf(xs[i], lo, xs[i + 1] * hi);
        }
    } else if constexpr (!DP) {
        for (int i = imain; i < A.I; i++) {
            const float w = WK == WK_BF16 ? bf16_widen(((const uint16_t *)wr)[i]) : (float)((const int8_t *)wr)[i];
            sm = __builtin_fmaf(xs[i], w, sm);
        }
    }
    if (WK != WK_I4G && A.scale) sm = sm * A.scale[o];
    A.y[(size_t)s * A.ldy + o] = sm;
}

template <int WK, int DP, int TS>
__global__ __launch_bounds__(256) void k_lanes16(LanesArgs A) {
    constexpr int EB = WElem<WK == WK_I4G ? WK_I4 : WK>::bits;
    constexpr int RB = LN_CC * EB / 8;                 // bytes of one row tile
    constexpr int RS = RB + 32;                        // its LDS stride (+8 banks per row)
    __shared__ __align__(16) uint8_t wt[LN_ROWS * RS];
    __shared__ __align__(16) float xt[TS * LN_CC];
    __shared__ float hg[WK == WK_I4G ? LN_ROWS * TS * (LN_CC / 16) : 1];   // I4G: group sums of a tile
    const int tid = threadIdx.x, r = tid >> 4, j = tid & 15;
    const int o0 = blockIdx.x * LN_ROWS, s0 = blockIdx.y * TS;
    const int I = A.I, O = A.O, S = A.S;
    const int ns = min(TS, S - s0);
    // columns of the lane chains; the rest is the scalar tail (F32X) -- DP needs I % 32 == 0
    const int imain = DP || WK == WK_I4G ? I : (WK == WK_I4 ? I & ~31 : I & ~15);
    const uint8_t *W = (const uint8_t *)A.W;
    const size_t rowb = (size_t)I * EB / 8;
    float acc[TS], lg[TS];                             // lg: the lane chains of a group wider than a tile
#pragma unroll
    for (int t = 0; t < TS; t++) { acc[t] = 0.f; lg[t] = 0.f; }
    for (int c0 = 0; c0 < imain; c0 += LN_CC) {
        const int cn = min(LN_CC, imain - c0);         // a multiple of 16 (32 for DP and int4)
        // the 16 rows' tile: cn * EB / 8 bytes each, in 16-byte pieces (rows past O: zeros)
        const int rb = cn * EB / 8, pieces = (rb + 15) / 16;
        for (int p = tid; p < LN_ROWS * pieces; p += 256) {
            const int rr = p / pieces, q = p - rr * pieces;
            sw_u32x4 v = {0u, 0u, 0u, 0u};
            if (o0 + rr < O) {
                const uint8_t *src = W + (size_t)(o0 + rr) * rowb + (size_t)c0 * EB / 8 + 16 * q;
                if (16 * q + 16 <= rb && (((uintptr_t)src) & 15) == 0) v = *(const sw_u32x4 *)src;
                else {
                    uint8_t tmp[16] = {0};
                    for (int b = 0; b < 16 && 16 * q + b < rb; b++) tmp[b] = src[b];
                    v = *(const sw_u32x4 *)tmp;
                }
            }
            *(sw_u32x4 *)(wt + rr * RS + 16 * q) = v;
        }
        for (int p = tid; p < TS * cn; p += 256) {
            const int t = p / cn, cc = p - t * cn;
            float v = t < ns ? A.x[(size_t)(s0 + t) * A.ldx + c0 + cc] : 0.f;
            xt[t * LN_CC + cc] = DP ? round_bf16_ne(v) : v;
        }
        __syncthreads();
        const uint8_t *row = wt + r * RS;
        if constexpr (DP) {
            for (int k = 0; k < cn; k += 32) {
                const float wo = flush_dn(w_at<WK>(row, k + 2 * j + 1)), we = flush_dn(w_at<WK>(row, k + 2 * j));
#pragma unroll
                for (int t = 0; t < TS; t++) {
                    // the converted activations are never denormal; the accumulator is always a flushed result
                    acc[t] = flush_dn(__builtin_fmaf(xt[t * LN_CC + k + 2 * j + 1], wo, acc[t]));
                    acc[t] = flush_dn(__builtin_fmaf(xt[t * LN_CC + k + 2 * j], we, acc[t]));
                }
            }
        } else if constexpr (WK == WK_I4G) {
            const int gs = A.gs, ngt = cn / gs, half = j >> 3, jj = j & 7;
            float *hrow = hg + r * TS * (LN_CC / 16);
            if (gs > LN_CC) {
                // a group spans gs / LN_CC whole tiles: lanes 0-7 carry its chains across them,
                // and its hsum8 and scale fma follow its last tile
                if (half == 0) {
                    for (int i = 0; i < cn; i += 16) {
                        const float w0 = w_at<WK_I4>(row, i + jj), w1 = w_at<WK_I4>(row, i + 8 + jj);
#pragma unroll
                        for (int t = 0; t < TS; t++) {
                            lg[t] = __builtin_fmaf(xt[t * LN_CC + i + jj], w0, lg[t]);
                            lg[t] = __builtin_fmaf(xt[t * LN_CC + i + 8 + jj], w1, lg[t]);
                        }
                    }
                }
                if ((c0 + cn) % gs == 0) {                 // uniform
                    const int o = o0 + r;
                    const float sg = A.scale[(size_t)(o < O ? o : 0) * (I / gs) + (c0 + cn) / gs - 1];
#pragma unroll
                    for (int t = 0; t < TS; t++) {
                        float v = lg[t] + __shfl_xor(lg[t], 4, 8);
                        v = v + __shfl_xor(v, 2, 8);
                        v = v + __shfl_xor(v, 1, 8);
                        if (j == 0) acc[t] = __builtin_fmaf(v, sg, acc[t]);
                        lg[t] = 0.f;
                    }
                }
            }
            for (int g = half; g < ngt; g += 2) {          // this half's groups of the tile
                float ln[TS];
#pragma unroll
                for (int t = 0; t < TS; t++) ln[t] = 0.f;
                for (int i = g * gs; i < g * gs + gs; i += 16) {
                    const float w0 = w_at<WK_I4>(row, i + jj), w1 = w_at<WK_I4>(row, i + 8 + jj);
#pragma unroll
                    for (int t = 0; t < TS; t++) {
                        ln[t] = __builtin_fmaf(xt[t * LN_CC + i + jj], w0, ln[t]);
                        ln[t] = __builtin_fmaf(xt[t * LN_CC + i + 8 + jj], w1, ln[t]);
                    }
                }
#pragma unroll
                for (int t = 0; t < TS; t++) {             // hsum8 inside the 8 lanes of the half
                    float v = ln[t] + __shfl_xor(ln[t], 4, 8);
                    v = v + __shfl_xor(v, 2, 8);
                    v = v + __shfl_xor(v, 1, 8);
                    if (jj == 0) hrow[t * (LN_CC / 16) + g] = v;
                }
            }
            lanes_wave_sync();
            if (j == 0) {                                  // the ordered scale chain of the row
                const int o = o0 + r;
                const float *sc = A.scale + (size_t)(o < O ? o : 0) * (I / gs) + c0 / gs;
                for (int g = 0; g < ngt; g++) {
                    const float sg = sc[g];
#pragma unroll
                    for (int t = 0; t < TS; t++) acc[t] = __builtin_fmaf(hrow[t * (LN_CC / 16) + g], sg, acc[t]);
                }
            }
            lanes_wave_sync();
        } else {
            for (int k = 0; k < cn; k += 16) {
                const float w = w_at<WK>(row, k + j);
#pragma unroll
                for (int t = 0; t < TS; t++) acc[t] = __builtin_fmaf(xt[t * LN_CC + k + j], w, acc[t]);
            }
        }
        __syncthreads();
    }
    const int o = o0 + r;
#pragma unroll
    for (int t = 0; t < TS; t++) {
        float sm = WK == WK_I4G ? acc[t] : reduce16_lanes(acc[t]);    // I4G: lane 0 holds the row's sum
        if (j == 0 && t < ns && o < O) {
            lanes_out<WK, DP>(A, sm, s0 + t, o, imain);
        }
    }
}

// ---- rows in 16-byte pieces, streamed by waves (every contract but I4G) ----
// A wave owns 4 rows; lane 16 r + j runs chain j of row r for up to TS tokens.  Per step it
// loads 16 bytes per lane -- 16 EPL consecutive columns of each row, one contiguous KB, PF
// steps in flight -- and turns them through its own LDS into the chains' order (one b128
// write, then per element one 2-byte (bf16), 1-byte (int) or, for DP, per pair one 4-byte
// read).  The tokens' x goes through LDS for the whole block, LW_XC columns at a time in two
// buffers, stored by chain (xt[t][j][m], so a lane reads four of its chain's values at once);
// one barrier per LW_XC columns.  What bounds it: HBM latency at one token (1 KB x PF per
// wave in flight), LDS reads of x at 8 (8 values of 16 bytes per 8 weights and 32 fmas).
// k_lanes16, which every shape took before, walked 256-column tiles with two barriers each,
// nothing in flight across them and one LDS read of x per fma: bf16 4096 x 4096, 16 tokens
// 151 -> 35 us a launch; the gated shared experts at 4 tokens (DP, gate and up of 4096 x 4096
// each, two downs of 4096 x 2048) 64 -> 30 and 33 -> 14 us a launch.
#define LW_XC 512
#define LW_XM (LW_XC / 16)         // chain elements of an x chunk
#define LW_XS (LW_XM + 4)          // floats per (token, chain) in LDS
#define LW_WS 288                  // bytes per row of a wave's weight step in LDS
#define LW_WAVES 4
template <int WK, int DP, int TS>
__global__ __launch_bounds__(64 * LW_WAVES) void k_lanes_w(LanesArgs A) {
    constexpr int EPL = 128 / WElem<WK>::bits;         // elements of a lane's 16 bytes
    constexpr int CS = 16 * EPL, SPC = LW_XC / CS;     // columns per step, steps per x chunk
    constexpr int RC = WK == WK_BF16 ? 2 : 4;          // x chunks whose weight steps are in flight
    constexpr int PF = RC * SPC;
    constexpr int NTH = 64 * LW_WAVES, XR = (TS * LW_XC / 4 + NTH - 1) / NTH;
    extern __shared__ __align__(16) uint8_t lw_lds[];
    float *xt = (float *)lw_lds;                       // [2][TS][16][LW_XS]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane >> 4, j = lane & 15;
    uint8_t *wl = lw_lds + 2 * TS * 16 * LW_XS * 4 + wave * 2 * 4 * LW_WS;   // [2][4][LW_WS]
    const int I = A.I, O = A.O, S = A.S;
    const int o = (blockIdx.x * LW_WAVES + wave) * 4 + r, s0 = blockIdx.y * TS, ns = min(TS, S - s0);
    const int imain = WK == WK_I4 ? I & ~31 : I & ~15;
    const int nst = (imain + CS - 1) / CS, nch = (imain + LW_XC - 1) / LW_XC;
    const size_t rowb = (size_t)I * WElem<WK>::bits / 8;
    const uint8_t *wr = (const uint8_t *)A.W + (size_t)min(o, O - 1) * rowb;
    const int lastp = imain * WElem<WK>::bits / 128 - 1;    // the row's last whole 16-byte piece
    // (unconditional: a piece past the end re-reads the last one, whose elements are not used)
    auto wld = [&](int st) { return *(const sw_u32x4 *)(wr + 16 * (size_t)max(min(st * 16 + j, lastp), 0)); };
    sw_f32x4 xr[XR];
    auto xload = [&](int c) {                          // float4 f of a chunk: token f / 128, columns 4 (f % 128)
#pragma unroll
        for (int u = 0; u < XR; u++) {
            const int f = u * NTH + tid, t = min(f / (LW_XC / 4), TS - 1), k = c * LW_XC + 4 * (f % (LW_XC / 4));
            xr[u] = *(const sw_f32x4 *)(A.x + (size_t)(s0 + min(t, ns - 1)) * A.ldx + min(k, imain - 4));
        }
    };
    auto xstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < XR; u++) {
            const int f = u * NTH + tid, t = f / (LW_XC / 4), k4 = 4 * (f % (LW_XC / 4));
            if (TS * LW_XC / 4 % NTH == 0 || t < TS)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int k = k4 + i;
                    const int ch = DP ? (k & 31) >> 1 : k & 15, m = DP ? 2 * (k >> 5) + (k & 1) : k >> 4;
                    xt[((buf * TS + t) * 16 + ch) * LW_XS + m] = DP ? round_bf16_ne(xr[u][i]) : xr[u][i];
                }
        }
    };
    float acc[TS];
#pragma unroll
    for (int t = 0; t < TS; t++) acc[t] = 0.f;
    sw_u32x4 ring[PF];
#pragma unroll
    for (int u = 0; u < PF; u++) ring[u] = wld(u);
    xload(0);
    xstore(0);
    __syncthreads();
    // elements m .. m + 3 of the step (chain elements m0 + m .. of the x chunk in buffer buf)
    auto four = [&](const uint8_t *row, int m, const float *xc) {
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (DP) {                        // pair q = (m + i) / 2 of columns 32 q + 2 j: slot 0 even, 1 odd
                const uint32_t v = *(const uint32_t *)(row + ((m + i) >> 1) * 64 + 4 * j);
                w[i] = flush_dn((i & 1) ? __builtin_bit_cast(float, v & 0xFFFF0000u) : bf16_widen(v & 0xFFFFu));
            } else {
                w[i] = w_at<WK>(row, 16 * (m + i) + j);
            }
        }
#pragma unroll
        for (int t = 0; t < TS; t++) {
            const sw_f32x4 xv = *(const sw_f32x4 *)(xc + t * 16 * LW_XS + m);
            if constexpr (DP) {                        // the odd column first
                acc[t] = flush_dn(__builtin_fmaf(xv[1], w[1], acc[t]));
                acc[t] = flush_dn(__builtin_fmaf(xv[0], w[0], acc[t]));
                acc[t] = flush_dn(__builtin_fmaf(xv[3], w[3], acc[t]));
                acc[t] = flush_dn(__builtin_fmaf(xv[2], w[2], acc[t]));
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t] = __builtin_fmaf(xv[i], w[i], acc[t]);
            }
        }
    };
    for (int c0 = 0; c0 < nch; c0 += RC) {
#pragma unroll
        for (int h = 0; h < RC; h++) {
            const int c = c0 + h;
            if (c >= nch) break;                       // uniform
            xload(min(c + 1, nch - 1));
            const float *xc = xt + (((c & 1) * TS) * 16 + j) * LW_XS;
#pragma unroll
            for (int p = 0; p < SPC; p++) {
                const int st = c * SPC + p, u = h * SPC + p;
                if (st >= nst) break;                  // uniform
                uint8_t *row = wl + ((p & 1) * 4 + r) * LW_WS;
                *(sw_u32x4 *)(row + 16 * j) = ring[u];
                ring[u] = wld(st + PF);
                __builtin_amdgcn_sched_barrier(0);
                lanes_wave_sync();
                const int mc = min(EPL, (imain - st * CS) / 16);
                if (mc == EPL) {
#pragma unroll
                    for (int m = 0; m < EPL; m += 4) four(row, m, xc + p * EPL);
                } else {                               // the row's last columns: one (DP: two) at a time
                    for (int m = 0; m < mc; m += DP ? 2 : 1)
#pragma unroll
                        for (int t = 0; t < TS; t++) {
                            const float *xm = xc + p * EPL + t * 16 * LW_XS + m;
                            if constexpr (DP) {
                                const uint32_t v = *(const uint32_t *)(row + (m >> 1) * 64 + 4 * j);
                                acc[t] = flush_dn(__builtin_fmaf(xm[1], flush_dn(__builtin_bit_cast(float, v & 0xFFFF0000u)), acc[t]));
                                acc[t] = flush_dn(__builtin_fmaf(xm[0], flush_dn(bf16_widen(v & 0xFFFFu)), acc[t]));
                            } else {
                                acc[t] = __builtin_fmaf(xm[0], w_at<WK>(row, 16 * m + j), acc[t]);
                            }
                        }
                }
                lanes_wave_sync();                     // read before the buffer's next write
            }
            xstore((c + 1) & 1);                       // (read by no wave since the last barrier)
            __syncthreads();
        }
    }
#pragma unroll
    for (int t = 0; t < TS; t++) {
        const float sm = reduce16_lanes(acc[t]);
        if (j == 0 && t < ns && o < O) lanes_out<WK, DP>(A, sm, s0 + t, o, imain);
    }
}

template <int WK, int DP, int TS>
static void launch_lanes_w(hipStream_t st, const LanesArgs &A) {
    const size_t lds = (size_t)2 * TS * 16 * LW_XS * 4 + LW_WAVES * 2 * 4 * LW_WS;
    SW_LAUNCH((k_lanes_w<WK, DP, TS>), dim3((A.O + 4 * LW_WAVES - 1) / (4 * LW_WAVES), (A.S + TS - 1) / TS), dim3(64 * LW_WAVES),
              lds, st, A);
}
// whole 16-byte pieces: rows of W and of x at 16-byte strides and addresses, at least one
// chain step in a row; passes of 8 tokens within a grid's second dimension (k_lanes16's of 16
// reach twice as far)
#define LN_GRID_Y 65535
static bool lanes_w_ok(const LanesArgs &A, int bits) {
    return A.S <= 8 * LN_GRID_Y && (size_t)A.I * bits / 8 % 16 == 0 && (size_t)A.I * bits % 8 == 0 &&
           ((uintptr_t)A.W & 15) == 0 && ((uintptr_t)A.x & 15) == 0 && A.ldx % 4 == 0 && A.I >= 32;
}
// Short rows on many blocks stay with k_lanes16 (nb of its blocks): a block of k_lanes_w fills
// its pipeline and stages a whole x chunk for a few steps.  The line by k_lanes16 / k_lanes_w,
// bf16, us a launch: 1024 outputs, 128 tokens (512 blocks) I = 64 8.6 / 9.3, 160 12.2 / 10.8;
// 4096 outputs, 64 tokens (1024) I = 64 9.8 / 13.9, 256 19.1 / 17.4; 12288 outputs, 128 tokens
// (6144) I = 64 31 / 59, 320 69 / 85, 384 89 / 87.  On fewer blocks k_lanes16 is behind at any
// length (64 outputs, 64 tokens, I = 64: 9.0 / 4.8).
static bool lanes_short(const LanesArgs &A, int64_t nb) {
    return nb >= 512 && A.I <= (nb / 6 < 224 + nb / 40 ? nb / 6 : 224 + nb / 40);
}

template <int WK, int DP>
static void launch_lanes(hipStream_t st, const LanesArgs &A) {
    const int ts16 = A.S >= 16 ? 16 : A.S >= 8 ? 8 : A.S >= 4 ? 4 : 1;
    if constexpr (WK != WK_I4G) {
        if (lanes_w_ok(A, WElem<WK>::bits) && !lanes_short(A, (int64_t)((A.O + 15) / 16) * ((A.S + ts16 - 1) / ts16))) {
            // tokens per pass: the most (each weight turned once for all of them) that still give
            // 512 blocks, two waves per SIMD -- one alone issues at half rate (bf16 4096 x 4096 at 8
            // tokens, whole call: 66 us with 256 blocks, 58 with 512, 57 with 1024; 24 tokens at
            // 6144 rows no difference, 4 tokens there 55 / 52 / 56)
            int ts = A.S >= 8 ? 8 : A.S >= 3 ? 4 : A.S;
            while (ts > 1 && (int64_t)((A.O + 4 * LW_WAVES - 1) / (4 * LW_WAVES)) * ((A.S + ts - 1) / ts) < 512) ts >>= 1;
            if (ts == 8) launch_lanes_w<WK, DP, 8>(st, A);
            else if (ts == 4) launch_lanes_w<WK, DP, 4>(st, A);
            else if (ts == 2) launch_lanes_w<WK, DP, 2>(st, A);
            else launch_lanes_w<WK, DP, 1>(st, A);
            return;
        }
    }
    const dim3 block(256);
    if (ts16 == 16) SW_LAUNCH((k_lanes16<WK, DP, 16>), dim3((A.O + 15) / 16, (A.S + 15) / 16), block, 0, st, A);
    else if (ts16 == 8) SW_LAUNCH((k_lanes16<WK, DP, 8>), dim3((A.O + 15) / 16, (A.S + 7) / 8), block, 0, st, A);
    else if (ts16 == 4) SW_LAUNCH((k_lanes16<WK, DP, 4>), dim3((A.O + 15) / 16, (A.S + 3) / 4), block, 0, st, A);
    else SW_LAUNCH((k_lanes16<WK, DP, 1>), dim3((A.O + 15) / 16, A.S), block, 0, st, A);
}

// wkind 0 bf16, 1 int8 (+ scale), 2 per-row int4 (+ scale), 3 group-scaled int4
// (+ scale [O][I/gs]; gs dividing I, a multiple of 16 dividing 256 or a multiple of
// 256); dp: the vdpbf16ps
// contract (bf16 weights, I % 32 == 0)
int sw_launch_lanes16(hipStream_t st, const void *W, int wkind, int dp, const float *scale, const float *x, int S,
                      int I, int O, float *y, int gs) {
    return sw_launch_lanes16_ld(st, W, wkind, dp, scale, x, I, S, I, O, y, O, gs);
}

int sw_launch_lanes16_ld(hipStream_t st, const void *W, int wkind, int dp, const float *scale, const float *x, int ldx,
                         int S, int I, int O, float *y, int ldy, int gs) {
    if (!W || !x || !y || S <= 0 || I <= 0 || O <= 0 || ldx < I || ldy < O) return -1;
    if (dp && (wkind != WK_BF16 || I % 32)) return -1;
    if ((wkind == WK_I4 || wkind == WK_I4G) && (I & 1)) return -1;
    if (wkind == WK_I4G && (gs < 16 || gs % 16 || (gs <= LN_CC ? LN_CC % gs : gs % LN_CC) || I % gs)) return -1;
    if (wkind != WK_BF16 && !scale) return -1;
    const LanesArgs A = {W, wkind == WK_BF16 ? nullptr : scale, x, y, S, I, O, gs, ldx, ldy};
    if (dp) launch_lanes<WK_BF16, 1>(st, A);
    else if (wkind == WK_BF16) launch_lanes<WK_BF16, 0>(st, A);
    else if (wkind == WK_I8) launch_lanes<WK_I8, 0>(st, A);
    else if (wkind == WK_I4) launch_lanes<WK_I4, 0>(st, A);
    else if (wkind == WK_I4G) launch_lanes<WK_I4G, 0>(st, A);
    else return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ------------------------------------------------------------ SiLU-GLU ----
// h = siluf(g) * u elementwise, siluf(x) = x / (1 + expf(-x)) with the glibc-exact
// expf (c/moe_math.h:53): the bits of the CPU's `g[i] = siluf(g[i]) * u[i]`
__global__ void k_silu_mul(const float *__restrict__ g, const float *__restrict__ u, int64_t n, float *__restrict__ h) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float v = g[i];
        h[i] = (v / (1.0f + sw_expf(-v))) * u[i];
    }
}

int sw_launch_silu_mul(hipStream_t st, const float *g, const float *u, int64_t n, float *h) {
    if (!g || !u || !h || n <= 0) return -1;
    SW_LAUNCH(k_silu_mul, dim3((unsigned)sw_imin64((n + 255) / 256, 4096)), dim3(256), 0, st, g, u, n, h);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
