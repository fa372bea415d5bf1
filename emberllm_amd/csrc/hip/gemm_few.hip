// gemm_few.hip — the products of a pass of a few tokens (a short prompt, the
// next message of a conversation) for gfx950.
//
// Replaces ember_matmul_batch -> mmb_rows (src/kernels.c:223-264) with the
// RMSNorm, RoPE, KV store and SwiGLU around it (src/model.c:305-351), as
// gemm.hip does, where a pass has so few tokens that its products are bound by
// their launches and memory round trips and not by the matrix cores: the
// Qwen3-0.6B shape at 16 tokens spent 58 us per layer in seven kernels whose
// weights alone take 4.
//
// A workgroup takes 16 tokens and has 16 waves.  A wave owns 16 weight rows and
// a part of K: all its weights are requested at the start with whole 128-byte
// row pieces per load instruction, pass through an LDS buffer of the wave's
// own into v_mfma_i32_16x16x32_i8 fragments (no workgroup barrier), and the
// parts' sums meet once at the end, added in order.  Against the staged
// pipelines of k_gemm_small / k_gemm_qkv / k_gemm_swq (a barrier per 4
// blocks): one memory round trip and at most 16 blocks of serial work.
// The products that follow an RMSNorm normalize and quantize the workgroup's
// 16 rows themselves while their weights are in flight, a wave per row, so
// those rows need no launch of their own.
//
// Fragments of the 16 x 16 x 32 product: lane l holds A[l % 16][8 (l / 16) ..
// +7] of a weight block, B[8 (l / 16) .. +7][l % 16] of a token's codes, and
// outputs D[4 (l / 16) + r][l % 16].  Each block is applied as sum =
// fma((float)isum, dw * dx, sum), its scale products taken from the fp16
// matrix cores (exact: both are fp16 values).
#include "kernels.h"
#include "flimg.h"
#include "gemm_epi.h"

namespace ehip {

constexpr int FEW_T = 16;              // tokens per tile; a workgroup takes TN tiles
constexpr int FEW_CB = 4;              // quant blocks per chunk (a wave's unit of K)
constexpr int FEW_NW = 16;             // waves per workgroup
constexpr int FEW_K = 1024;            // inputs at most of a product that normalizes its rows
constexpr int FEW_XP = FEW_K + 16;     // LDS pitch of a quantized row

template <int DT> struct FewChunk {
    static constexpr int WB = DT == DT_Q8 ? 32 : 16;      // weight bytes per block
    static constexpr int ROW = FEW_CB * WB;                // bytes per row
    static constexpr int NL = 16 * ROW / 1024;             // 16-byte loads per lane
    static constexpr int PITCH = ROW + 16;                 // LDS row pitch
    static constexpr int BYTES = 16 * PITCH;
};

// Orders a wave's LDS stores before its own later reads of other lanes' data
// (the LDS executes a wave's instructions in order; this keeps the compiler's
// order the program's).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A wave's weights: 16 rows from row0, chunks c0 .. c0 + NCK - 1 of those
// below c1.  Past the end the last block is loaded again, with scale 0.
template <int DT, int NCK> struct FewWeights {
    using C = FewChunk<DT>;
    i32x4 q[NCK][C::NL];
    uint16_t d[NCK];   // lane l: row l % 16, block l / 16 of the chunk
    __device__ __forceinline__ void load(const DMat &W, int row0, int c0, int c1, int lane) {
        const int nb = W.cols / QB;
        constexpr int LPR = C::ROW / 16;                   // lanes per row
#pragma unroll
        for (int c = 0; c < NCK; c++) {
            const int b0 = (c0 + c) * FEW_CB;
            const int pb = (lane % LPR) * 16;
            const int blk = min(b0 + pb / C::WB, nb - 1);
#pragma unroll
            for (int i = 0; i < C::NL; i++) {
                const int row = row0 + lane / LPR + i * (64 / LPR);
                q[c][i] = *reinterpret_cast<const i32x4 *>(W.q + (size_t)row * (nb * C::WB) + (size_t)blk * C::WB + pb % C::WB);
            }
            const int sb = b0 + (lane >> 4);
            const uint16_t s = W.d[(size_t)(row0 + (lane & 15)) * nb + min(sb, nb - 1)];
            d[c] = c0 + c < c1 && sb < nb ? s : 0;
        }
    }
};

// One chunk: its weights through the wave's LDS buffer, then four blocks into
// acc.  xp(n, kb): this lane's eight codes of block kb (token l % 16 of tile
// n); sx: the scale bits of those tokens and block l / 16 (0 where there is no
// such block); xsum(n, kb): the code sum (Q4_0).
template <int DT, int TN, class XP, class XS>
__device__ __forceinline__ void few_chunk(f32x4 (&acc)[TN], const i32x4 (&wq)[FewChunk<DT>::NL], uint16_t dw, uint8_t *wbuf,
                                          XP xp, const uint16_t (&sx)[TN], XS xsum, int lane) {
    using C = FewChunk<DT>;
    constexpr int LPR = C::ROW / 16;
    const int fr = lane & 15, fg = lane >> 4;
#pragma unroll
    for (int i = 0; i < C::NL; i++)
        *reinterpret_cast<i32x4 *>(wbuf + (lane / LPR + i * (64 / LPR)) * C::PITCH + (lane % LPR) * 16) = wq[i];
    wave_lds_fence();
    long af[FEW_CB];
#pragma unroll
    for (int kb = 0; kb < FEW_CB; kb++) {
        const uint8_t *wp = wbuf + fr * C::PITCH + kb * C::WB;
        if (DT == DT_Q8) {
            af[kb] = *reinterpret_cast<const long *>(wp + 8 * fg);
        } else {   // nibbles: low = weights 0..15, high = 16..31 of the block
            const unsigned long long raw = *reinterpret_cast<const unsigned long long *>(wp + 8 * (fg & 1));
            af[kb] = (long)((raw >> (4 * (fg >> 1))) & 0x0f0f0f0f0f0f0f0full);
        }
    }
    // A: every lane's scale at k = 4 (l / 16); B: only block kb's lanes, so the
    // product of row i and token j is dw[i][kb] * dx[j][kb]
    f16x4 sa{}, sb{};
    sa[0] = __builtin_bit_cast(_Float16, dw);
#pragma unroll
    for (int n = 0; n < TN; n++) {
        long bf[FEW_CB];
        int xs[FEW_CB];
#pragma unroll
        for (int kb = 0; kb < FEW_CB; kb++) {
            bf[kb] = xp(n, kb);
            xs[kb] = DT == DT_Q4 ? xsum(n, kb) : 0;
        }
        i32x4 d[FEW_CB];
#pragma unroll
        for (int kb = 0; kb < FEW_CB; kb++)
            d[kb] = __builtin_amdgcn_mfma_i32_16x16x32_i8(af[kb], bf[kb], i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int kb = 0; kb < FEW_CB; kb++) {
            sb[0] = __builtin_bit_cast(_Float16, (uint16_t)(fg == kb ? sx[n] : 0));
            const f32x4 sc = __builtin_amdgcn_mfma_f32_16x16x16f16(sa, sb, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int isum = DT == DT_Q4 ? d[kb][r] - 8 * xs[kb] : d[kb][r];
                acc[n][r] = fmaf((float)isum, sc[r], acc[n][r]);
            }
        }
    }
    wave_lds_fence();   // the next chunk's stores stay behind these reads
}

// --------------------------------------------------------------- wo, w2 --
// out[token][row] += W . x over rows quantized before (grid: 16-row tiles,
// 16-token tiles).  Wave w takes chunks w NCK .. of K; each also loads its own
// part of the tokens' codes.  23 tokens of the Qwen3-0.6B shape: wo 4.5-5.0 us,
// w2 5.1 (k_gemm_small 9.0 each); 64 workgroups of 35 and 52 KB of weights.
template <int DT, int NCK, int TN>
__global__ __launch_bounds__(64 * FEW_NW) void k_few_resid(GemmArgs a) {
    using C = FewChunk<DT>;
    constexpr int XP = FEW_CB * 32 + 16;   // LDS pitch of a token's codes of a chunk
    __shared__ __align__(16) uint8_t wbuf[FEW_NW][C::BYTES];
    __shared__ __align__(16) uint8_t xbuf[FEW_NW][TN * FEW_T * XP];
    __shared__ f32x4 red[FEW_NW][TN][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, fg = lane >> 4;
    const int u0 = blockIdx.x * 16, t0 = blockIdx.y * (TN * FEW_T);
    const int K = a.W.cols, nb = K / QB, nc = (nb + FEW_CB - 1) / FEW_CB;
    const int c0 = wave * NCK;
    FewWeights<DT, NCK> w;
    i32x4 xq[NCK][2 * TN];
    float dx[NCK][TN];
    int xs[NCK][TN];
    // the outputs' old values, for the waves that store them (wave n tile n)
    const int to = t0 + FEW_T * min(wave, TN - 1) + fr;
    f32x4 *const op = reinterpret_cast<f32x4 *>(a.out + (size_t)min(to, a.n - 1) * a.out_stride + u0 + 4 * fg);
    const f32x4 pre = wave < TN ? *op : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < NCK; c++) {
        const int b0 = (c0 + c) * FEW_CB;
#pragma unroll
        for (int i = 0; i < 2 * TN; i++) {
            const int t = min(t0 + (lane >> 3) + 8 * i, a.n - 1), pb = (lane & 7) * 16;
            xq[c][i] = *reinterpret_cast<const i32x4 *>(a.qx + (size_t)t * K + (size_t)min(b0 + pb / 32, nb - 1) * 32 + pb % 32);
        }
#pragma unroll
        for (int n = 0; n < TN; n++) {
            const size_t so = (size_t)min(t0 + FEW_T * n + fr, a.n - 1) * nb + min(b0 + fg, nb - 1);
            dx[c][n] = a.dx[so];
            xs[c][n] = DT == DT_Q4 ? a.xs[so] : 0;
        }
    }
    w.load(a.W, u0, c0, nc, lane);
    f32x4 acc[TN] = {};
    uint8_t *xb = xbuf[wave];
    if (c0 < nc) {
#pragma unroll
        for (int c = 0; c < NCK; c++) {
#pragma unroll
            for (int i = 0; i < 2 * TN; i++)
                *reinterpret_cast<i32x4 *>(xb + ((lane >> 3) + 8 * i) * XP + (lane & 7) * 16) = xq[c][i];
            const bool have = (c0 + c) * FEW_CB + fg < nb;
            uint16_t sx[TN];
#pragma unroll
            for (int n = 0; n < TN; n++) sx[n] = have ? f2h(dx[c][n]) : (uint16_t)0;
            few_chunk<DT, TN>(
                acc, w.q[c], w.d[c], wbuf[wave],
                [&](int n, int kb) { return *reinterpret_cast<const long *>(xb + (FEW_T * n + fr) * XP + kb * 32 + 8 * fg); },
                sx, [&](int n, int kb) { return __shfl(xs[c][n], fr + 16 * kb); }, lane);
        }
    }
#pragma unroll
    for (int n = 0; n < TN; n++) red[wave][n][lane] = acc[n];
    __syncthreads();
    if (wave >= TN) return;
    const int np = (nc + NCK - 1) / NCK;   // waves with a part of K
    f32x4 v = red[0][wave][lane];
    for (int p = 1; p < np; p++) v += red[p][wave][lane];
    if (to < a.n) *op = pre + v;
}

// ------------------------------------------------- normalized products --
// The RMSNorm (model.c:50-55) and Q8_0 codes (kernels.c:73-92) of row t of x
// by one wave: lane l holds elements 4 (l + 64 s) .. + 3, eight lanes a block.
struct FewRow { f32x4 x[4], w[4]; };
__device__ __forceinline__ void few_row_load(FewRow &r, const NormIn &in, int K, int t, int lane) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int i = min(lane + 64 * s, K / 4 - 1);
        r.x[s] = reinterpret_cast<const f32x4 *>(in.x + (size_t)t * K)[i];
        r.w[s] = reinterpret_cast<const f32x4 *>(in.norm_w)[i];
    }
}
template <int DT>
__device__ __forceinline__ void few_row_quant(const FewRow &r, float eps, int K, int lane, uint8_t *xq, uint16_t *dx, int *xs) {
    float ss = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; s++)
        if (lane + 64 * s < K / 4)
            ss += (r.x[s].x * r.x[s].x + r.x[s].y * r.x[s].y) + (r.x[s].z * r.x[s].z + r.x[s].w * r.x[s].w);
    const float scale = 1.0f / sqrtf(wave_sum(ss) / (float)K + eps);
    f32x4 v[4];
    float mx[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[s][e] = r.x[s][e] * scale * r.w[s][e];
        mx[s] = max8(fmaxf(fmaxf(fabsf(v[s].x), fabsf(v[s].y)), fmaxf(fabsf(v[s].z), fabsf(v[s].w))));
    }
    // the eight lanes' four blocks: lane j of each four takes the divisions of
    // block j, and the inverses are passed back by quad broadcasts
    const int j = lane & 3;
    const float m = j < 2 ? (j == 0 ? mx[0] : mx[1]) : (j == 2 ? mx[2] : mx[3]);
    const float d = m / 127.0f;
    const int id4 = __float_as_int(d > 0.0f ? 1.0f / d : 0.0f);
    const float id[4] = {__int_as_float(__builtin_amdgcn_mov_dpp(id4, 0x00, 0xf, 0xf, false)),
                         __int_as_float(__builtin_amdgcn_mov_dpp(id4, 0x55, 0xf, 0xf, false)),
                         __int_as_float(__builtin_amdgcn_mov_dpp(id4, 0xaa, 0xf, 0xf, false)),
                         __int_as_float(__builtin_amdgcn_mov_dpp(id4, 0xff, 0xf, 0xf, false))};
    if ((lane & 4) == 0 && lane + 64 * j < K / 4) dx[(lane >> 3) + 8 * j] = f2h(d);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        int c[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            // round half away from zero: the float below 1/2, added to the
            // magnitude, carries exactly the values from k + 1/2 up
            const float x = fminf(fmaxf(v[s][e] * id[s], -127.0f), 127.0f);
            c[e] = (int)(x + copysignf(0.49999997f, x));
        }
        const int i = lane + 64 * s;
        int cs = 0;
        if (DT == DT_Q4) cs = sum8(c[0] + c[1] + c[2] + c[3]);
        if (i >= K / 4) continue;
        *reinterpret_cast<uint32_t *>(xq + 4 * i) = ((uint32_t)c[0] & 0xffu) | (((uint32_t)c[1] & 0xffu) << 8) |
                                                    (((uint32_t)c[2] & 0xffu) << 16) | (((uint32_t)c[3] & 0xffu) << 24);
        if (DT == DT_Q4 && (lane & 7) == 0) xs[i >> 3] = cs;
    }
}

template <int TN> struct FewRows {   // the workgroup's quantized rows, in LDS
    __align__(16) uint8_t q[TN * FEW_T][FEW_XP];
    uint16_t d[TN * FEW_T][FEW_K / QB + 2];
    int s[TN * FEW_T][FEW_K / QB + 1];
};

// A wave's sums over chunks c0 .. c0 + NCK - 1 (below nc) of its 16 rows.
template <int DT, int NCK, int TN>
__device__ __forceinline__ void few_product(f32x4 (&acc)[TN], const FewWeights<DT, NCK> &w, const FewRows<TN> &x, int c0, int nc,
                                            int nb, uint8_t *wbuf, int lane) {
    const int fr = lane & 15, fg = lane >> 4;
#pragma unroll
    for (int n = 0; n < TN; n++) acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < NCK; c++) {
        if (c0 + c >= nc) break;   // uniform over the wave
        const int b0 = (c0 + c) * FEW_CB, sb = b0 + fg;
        uint16_t sx[TN];
#pragma unroll
        for (int n = 0; n < TN; n++) sx[n] = sb < nb ? x.d[FEW_T * n + fr][sb] : (uint16_t)0;
        few_chunk<DT, TN>(
            acc, w.q[c], w.d[c], wbuf,
            [&](int n, int kb) { return *reinterpret_cast<const long *>(x.q[FEW_T * n + fr] + (size_t)min(b0 + kb, nb - 1) * 32 + 8 * fg); },
            sx, [&](int n, int kb) { return x.s[FEW_T * n + fr][min(b0 + kb, nb - 1)]; }, lane);
    }
}

// q|k|v with k_qkpost's work in the epilogue (qkv_finish): a head vector per
// workgroup, HD / 16 row tiles, the other waves splitting K.  raw, when set,
// receives the product with its bias.  23 tokens of the Qwen3-0.6B shape 12.0 us
// (k_quant_rows and k_gemm_qkv 16.4): 130 KB of weights per workgroup, of which
// a CU keeps 30-40 KB in flight.
template <int DT, int HD, bool F16>
__global__ __launch_bounds__(64 * FEW_NW) void k_few_qkv(GemmArgs a, NormIn in, QkPostArgs p, float *raw) {
    constexpr int NT = HD / 16, NP = FEW_NW / NT, NCK = FEW_K / (32 * FEW_CB) / NP;   // row tiles, K parts, chunks
    __shared__ FewRows<1> x;
    __shared__ __align__(16) uint8_t wbuf[FEW_NW][FewChunk<DT>::BYTES];
    __shared__ f32x4 red[NP - 1][NT][64];
    __shared__ float hs[QV_T][HD + 1];
    __shared__ int exs[QV_T];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, fg = lane >> 4;
    const int tile = wave % NT, part = wave / NT;
    const int vh = blockIdx.x, u0 = vh * HD + tile * 16, t0 = blockIdx.y * QV_T;
    const int K = a.W.cols, nb = K / QB, nc = (nb + FEW_CB - 1) / FEW_CB, c0 = part * NCK;
    FewRow row;
    few_row_load(row, in, K, min(t0 + wave, a.n - 1), lane);
    FewWeights<DT, NCK> w;
    w.load(a.W, u0, c0, nc, lane);
    float nwv[HD / 64];
    float2 cs[1][HD / 64];
    qkv_preload<HD, 1>(p, vh, t0, a.n, wave, lane, nwv, cs);
    float bias[4];
#pragma unroll
    for (int r = 0; r < 4; r++) bias[r] = a.bias ? a.bias[u0 + 4 * fg + r] : 0.0f;
    if (t0 + wave < a.n) few_row_quant<DT>(row, in.eps, K, lane, x.q[wave], x.d[wave], x.s[wave]);
    __syncthreads();
    f32x4 accs[1];
    few_product<DT, NCK, 1>(accs, w, x, c0, nc, nb, wbuf[wave], lane);
    f32x4 acc = accs[0];
    if (part > 0) red[part - 1][tile][lane] = acc;
    __syncthreads();
    if (part == 0) {
#pragma unroll
        for (int s = 0; s < NP - 1; s++)
            if ((s + 1) * NCK < nc) acc += red[s][tile][lane];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float v = a.bias ? acc[r] + bias[r] : acc[r];
            hs[fr][tile * 16 + 4 * fg + r] = v;
            if (raw && t0 + fr < a.n) raw[(size_t)(t0 + fr) * p.stride + u0 + 4 * fg + r] = v;
        }
    }
    __syncthreads();
    qkv_finish<HD, F16, FEW_NW, 64 * FEW_NW>(p, hs, exs, nwv, cs, vh, t0, a.n, wave, lane, true);
}

// out = W . x (+ bias): 16-row tiles, eight waves over K, two of the rows per
// wave to normalize.  16 tokens of the Qwen3-0.6B shape 6.8 us on 256
// workgroups of 16 KB of weights (k_few_qkv 12.5 on 32), of which the
// attention's QK-norm, RoPE and KV store take 3 back.
constexpr int FEW_SW = 8;
template <int DT>
__global__ __launch_bounds__(64 * FEW_SW) void k_few_store(GemmArgs a, NormIn in) {
    constexpr int NCK = FEW_K / (32 * FEW_CB) / FEW_SW, NR = FEW_T / FEW_SW;
    __shared__ FewRows<1> x;
    __shared__ __align__(16) uint8_t wbuf[FEW_SW][FewChunk<DT>::BYTES];
    __shared__ f32x4 red[FEW_SW][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, fg = lane >> 4;
    const int u0 = blockIdx.x * 16, t0 = blockIdx.y * FEW_T;
    const int K = a.W.cols, nb = K / QB, nc = (nb + FEW_CB - 1) / FEW_CB, c0 = wave * NCK;
    FewRow row[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) few_row_load(row[j], in, K, min(t0 + wave + FEW_SW * j, a.n - 1), lane);
    FewWeights<DT, NCK> w;
    w.load(a.W, u0, c0, nc, lane);
    f32x4 bias{0.0f, 0.0f, 0.0f, 0.0f};
    if (a.bias && wave == 0) bias = *reinterpret_cast<const f32x4 *>(a.bias + u0 + 4 * fg);
#pragma unroll
    for (int j = 0; j < NR; j++) {
        const int t = wave + FEW_SW * j;
        if (t0 + t < a.n) few_row_quant<DT>(row[j], in.eps, K, lane, x.q[t], x.d[t], x.s[t]);
    }
    __syncthreads();
    f32x4 accs[1];
    few_product<DT, NCK, 1>(accs, w, x, c0, nc, nb, wbuf[wave], lane);
    red[wave][lane] = accs[0];
    __syncthreads();
    if (wave > 0) return;
    f32x4 acc = red[0][lane];
    for (int p = 1; p * NCK < nc; p++) acc += red[p][lane];
    if (t0 + fr < a.n) *reinterpret_cast<f32x4 *>(a.out + (size_t)(t0 + fr) * a.out_stride + u0 + 4 * fg) = a.bias ? acc + bias : acc;
}

// w1|w3 with the SwiGLU and its Q8_0 rows in the epilogue (swiglu_rows): 32
// hidden units per workgroup, four row tiles (gate, gate, up, up), four waves
// each over K.  23 tokens of the Qwen3-0.6B shape 9 us (k_quant_rows and
// k_gemm_swq 11.9): 68 KB of weights per workgroup, then the rows' codes.
template <int DT, int TN>
__global__ __launch_bounds__(64 * FEW_NW) void k_few_swiglu(GemmArgs a, NormIn in) {
    constexpr int NT = 2 * SW_U / 16, NP = FEW_NW / NT, NCK = FEW_K / (32 * FEW_CB) / NP;
    static_assert(SW_T == FEW_T, "tokens per tile");
    __shared__ FewRows<TN> x;
    __shared__ __align__(16) uint8_t wbuf[FEW_NW][FewChunk<DT>::BYTES];
    __shared__ f32x4 red[NP - 1][NT][TN][64];
    __shared__ float hs[TN][SW_T][2 * SW_U + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fr = lane & 15, fg = lane >> 4;
    const int tile = wave % NT, part = wave / NT;
    const int u0 = blockIdx.x * SW_U, t0 = blockIdx.y * (TN * SW_T);
    const int K = a.W.cols, nb = K / QB, nc = (nb + FEW_CB - 1) / FEW_CB, c0 = part * NCK;
    const int half = tile >> 1, ut = (tile & 1) * 16;   // up rows or gate rows, first unit of the tile
    FewRow row[TN];
#pragma unroll
    for (int n = 0; n < TN; n++) few_row_load(row[n], in, K, min(t0 + FEW_NW * n + wave, a.n - 1), lane);
    FewWeights<DT, NCK> w;
    w.load(a.W, half * a.pair_off + u0 + ut, c0, nc, lane);
#pragma unroll
    for (int n = 0; n < TN; n++) {
        const int t = FEW_NW * n + wave;
        if (t0 + t < a.n) few_row_quant<DT>(row[n], in.eps, K, lane, x.q[t], x.d[t], x.s[t]);
    }
    __syncthreads();
    f32x4 acc[TN];
    few_product<DT, NCK, TN>(acc, w, x, c0, nc, nb, wbuf[wave], lane);
#pragma unroll
    for (int n = 0; n < TN; n++)
        if (part > 0) red[part - 1][tile][n][lane] = acc[n];
    __syncthreads();
    if (part == 0) {
#pragma unroll
        for (int n = 0; n < TN; n++) {
#pragma unroll
            for (int s = 0; s < NP - 1; s++)
                if ((s + 1) * NCK < nc) acc[n] += red[s][tile][n][lane];
            const int t = t0 + SW_T * n + fr;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                hs[n][fr][half * SW_U + ut + 4 * fg + r] = acc[n][r];
                if (a.out && t < a.n)   // the gate | up products themselves, where asked for
                    a.out[(size_t)t * a.out_stride + half * a.pair_off + u0 + ut + 4 * fg + r] = acc[n][r];
            }
        }
    }
    __syncthreads();
    if (threadIdx.x >= TN * SW_T * 8) return;
    const int n = threadIdx.x / (SW_T * 8);
    swiglu_rows(a, hs[n], u0, t0 + SW_T * n, threadIdx.x % (SW_T * 8));
}

// -------------------------------------------------------------- launches --
static bool few_quantized(const DMat &W) { return (W.dtype == DT_Q8 || W.dtype == DT_Q4) && W.cols > 0 && W.cols % QB == 0; }

// Up to 128 tokens (Qwen3-0.6B shape: 64 tokens 1.69 -> 1.32 ms, 128 tokens
// 1.79 -> 1.67, 144 tokens 2.24 -> 2.28; stories110M 64 tokens 0.52 -> 0.36 ms,
// 128 0.57 -> 0.53, 176 0.63 -> 0.64), or 256 where K is no whole number of the
// staged kernels' 4-block stages and those clamp every load (SmolLM2-135M:
// 144 tokens 1.42 -> 1.13, 256 1.52 -> 1.39): every 16 tokens read the weights
// and, in each workgroup, quantize their rows again.
bool gemm_few_fits(const FewShape &s) {
    if (s.n <= 0 || s.n > (s.qkv.cols / QB % FEW_CB == 0 ? 128 : 256)) return false;
    if (!few_quantized(s.qkv) || !few_quantized(s.wo) || !few_quantized(s.w13) || !few_quantized(s.w2)) return false;
    if (s.qkv.cols > FEW_K || s.w13.cols > FEW_K || (s.hd != 64 && s.hd != 128)) return false;
    if (s.qkv.rows % s.hd != 0 || s.w13.rows % (2 * SW_U) != 0 || s.wo.rows % 16 != 0 || s.w2.rows % 16 != 0) return false;
    const int most = FEW_NW * FEW_CB * QB * 4;   // four chunks per wave
    return s.wo.cols <= most && s.w2.cols <= most;
}

// Two token tiles per workgroup, whose weights and LDS trips then serve 32
// tokens, once single tiles give more workgroups than fit the GPU's CUs `per`
// to a CU at a time, or more than one per CU where the pairs still fit:
// Qwen3-0.6B shape 64 tokens 1343 -> 1269 us, SmolLM2-135M 128 tokens 1085 ->
// 961, stories110M 128 tokens 535 -> 477 (below that line the halved grid
// loses: Qwen2.5-0.5B, w1|w3 456 workgroups at 48 tokens, 355 -> 373).
static bool few_two(int tiles, int n, int per) {
    const long g1 = (long)tiles * ((n + FEW_T - 1) / FEW_T), g2 = (long)tiles * ((n + 2 * FEW_T - 1) / (2 * FEW_T));
    return g1 > 256 && (g2 <= 256 || g1 > 256 * per);
}

int launch_few_resid(hipStream_t st, const GemmArgs &a) {
    const int nc = (a.W.cols / QB + FEW_CB - 1) / FEW_CB, nck = (nc + FEW_NW - 1) / FEW_NW;
    if (!few_quantized(a.W) || a.units % 16 != 0 || a.out_stride % 4 != 0 || a.n <= 0 || nck > 4) return -1;
    const bool two = nck < 4 && few_two(a.units / 16, a.n, 1);
    const dim3 g(a.units / 16, (a.n + FEW_T * (two ? 2 : 1) - 1) / (FEW_T * (two ? 2 : 1))), b(64 * FEW_NW);
#define FR(N, TN)                                                                                   \
    if (nck == N && two == (TN == 2)) {                                                             \
        if (a.W.dtype == DT_Q8) hipLaunchKernelGGL((k_few_resid<DT_Q8, N, TN>), g, b, 0, st, a);    \
        else hipLaunchKernelGGL((k_few_resid<DT_Q4, N, TN>), g, b, 0, st, a);                       \
        return 0;                                                                                   \
    }
    FR(1, 1) FR(2, 1) FR(3, 1) FR(4, 1) FR(1, 2) FR(2, 2) FR(3, 2)
#undef FR
    return -1;
}

int launch_few_qkv(hipStream_t st, bool f16kv, const GemmArgs &a, const NormIn &in, const QkPostArgs &p, float *raw) {
    if (!few_quantized(a.W) || a.W.cols > FEW_K || a.n <= 0 || p.n_tok != a.n || a.units != (p.n_heads + 2 * p.n_kv) * p.hd) return -1;
    const dim3 g(p.n_heads + 2 * p.n_kv, (a.n + QV_T - 1) / QV_T), b(64 * FEW_NW);
#define FQ(DT, H)                                                                                         \
    if (a.W.dtype == DT && p.hd == H) {                                                                   \
        if (f16kv) hipLaunchKernelGGL((k_few_qkv<DT, H, true>), g, b, 0, st, a, in, p, raw);              \
        else hipLaunchKernelGGL((k_few_qkv<DT, H, false>), g, b, 0, st, a, in, p, raw);                   \
        return 0;                                                                                         \
    }
    FQ(DT_Q8, 64) FQ(DT_Q8, 128) FQ(DT_Q4, 64) FQ(DT_Q4, 128)
#undef FQ
    return -1;
}

int launch_few_store(hipStream_t st, const GemmArgs &a, const NormIn &in) {
    if (!few_quantized(a.W) || a.W.cols > FEW_K || a.n <= 0 || a.units % 16 != 0 || a.out_stride % 4 != 0) return -1;
    const dim3 g(a.units / 16, (a.n + FEW_T - 1) / FEW_T), b(64 * FEW_SW);
    if (a.W.dtype == DT_Q8) hipLaunchKernelGGL((k_few_store<DT_Q8>), g, b, 0, st, a, in);
    else hipLaunchKernelGGL((k_few_store<DT_Q4>), g, b, 0, st, a, in);
    return 0;
}

int launch_few_swiglu(hipStream_t st, const GemmArgs &a, const NormIn &in) {
    if (!few_quantized(a.W) || a.W.cols > FEW_K || a.n <= 0 || a.units % SW_U != 0 || a.pair_off < a.units) return -1;
    if (!a.oq || !a.odx || !a.oxs) return -1;
    const int tn = few_two(a.units / SW_U, a.n, 2) ? 2 : 1;
    const dim3 g(a.units / SW_U, (a.n + SW_T * tn - 1) / (SW_T * tn)), b(64 * FEW_NW);
#define FS(DT)                                                                                  \
    if (tn == 2) hipLaunchKernelGGL((k_few_swiglu<DT, 2>), g, b, 0, st, a, in);                 \
    else hipLaunchKernelGGL((k_few_swiglu<DT, 1>), g, b, 0, st, a, in);
    if (a.W.dtype == DT_Q8) { FS(DT_Q8) } else { FS(DT_Q4) }
#undef FS
    return 0;
}

}  // namespace ehip
