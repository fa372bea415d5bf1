// gemm_epi.h — epilogues shared by the short prompts' products (gemm.hip,
// gemm_few.hip): QK-norm, RoPE, KV store and the K/V tile images of a q|k|v
// tile, SwiGLU and Q8_0 quantization of a w1|w3 tile.
#pragma once
#include "kernels.h"
#include "flimg.h"

namespace ehip {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int SW_U = 32, SW_T = 16;   // hidden units, tokens of a w1|w3 tile
constexpr int QV_T = 16;              // tokens of a q|k|v tile

// SwiGLU (model.c:403-406) and Q8_0 rows of a w1|w3 tile in LDS, hs[token]
// [gate 0..31 | up 32..63], by the first SW_T * 8 threads: eight lanes per
// token, k_quant_rows's arithmetic.
__device__ __forceinline__ void swiglu_rows(const GemmArgs &a, float (&hs)[SW_T][2 * SW_U + 1], int u0, int t0, int tid) {
    // token tid / 8, hidden units 4 (tid % 8) .. + 3 of the tile
    const int tt = tid >> 3, hp = (tid & 7) * 4;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float g = hs[tt][hp + i], u = hs[tt][SW_U + hp + i];
        v[i] = g / (1.0f + expf(-g)) * u;
    }
    const float mx = max8(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    const float dq = mx / 127.0f;
    const float id = dq > 0.0f ? 1.0f / dq : 0.0f;
    int c[4];
#pragma unroll
    for (int i = 0; i < 4; i++) c[i] = (int)fminf(fmaxf(roundf(v[i] * id), -127.0f), 127.0f);
    const int cs = sum8(c[0] + c[1] + c[2] + c[3]);
    const int t = t0 + tt;
    if (t >= a.n || u0 + hp >= a.units) return;
    const int nbo = a.units / QB;
    *reinterpret_cast<uint32_t *>(a.oq + (size_t)t * a.units + u0 + hp) =
        ((uint32_t)c[0] & 0xffu) | (((uint32_t)c[1] & 0xffu) << 8) | (((uint32_t)c[2] & 0xffu) << 16) |
        (((uint32_t)c[3] & 0xffu) << 24);
    if (hp == 0) {
        a.odx[(size_t)t * nbo + u0 / QB] = h2f(f2h(dq));
        a.oxs[(size_t)t * nbo + u0 / QB] = cs;
    }
}


// One key's K rows in its 64-key tile image for k_pf_flash16 (k_pf_kvsplit's
// layout, flimg.h), for k_gemm_qkv's wave-per-token epilogue: lane l holds
// dims l + 64 k of the key's cache values v[k]; ex is the key's power-of-two
// scale (fp32 cache: from its largest |value|).
template <int HD, bool F16>
__device__ __forceinline__ void qkv_key_image(uint8_t *im, const float *v, int kl, int ex, int lane) {
    using I = FlImg<HD, F16>;
    const int rk = fl_krow(kl);
#pragma unroll
    for (int k = 0; k < HD / 64; k++) {
        const int d = lane + 64 * k;
        const float x = F16 ? v[k] : __builtin_amdgcn_ldexpf(v[k], ex);
        const _Float16 hi = (_Float16)x, lo = (_Float16)(x - (float)hi);
        *reinterpret_cast<uint16_t *>(im + I::k_at(rk, d >> 3) + 2 * (d & 7)) = __builtin_bit_cast(uint16_t, hi);
        if constexpr (!F16)
            *reinterpret_cast<uint16_t *>(im + I::k_at(FL_BK + rk, d >> 3) + 2 * (d & 7)) = __builtin_bit_cast(uint16_t, lo);
    }
    if (!F16 && lane == 0) reinterpret_cast<int *>(im + I::KBYTES)[kl] = ex;
}
// A k head's key at position pos.  The image's K rows past the pass's last
// key stay as they are: the attention masks a key it may not see after its
// score product, whatever that product was.
template <int HD, bool F16>
__device__ __forceinline__ void qkv_tile_image(const QkPostArgs &p, int g, const float *v, int pos, int lane) {
    using I = FlImg<HD, F16>;
    uint8_t *im = p.kvimg + ((size_t)g * p.kvimg_tiles + pos / FL_BK) * I::HBYTES;
    int ex = 0;
    if constexpr (!F16) {
        float m = 0.0f;
#pragma unroll
        for (int k = 0; k < HD / 64; k++) m = fmaxf(m, fabsf(v[k]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        ex = fl_exp(m);
    }
    qkv_key_image<HD, F16>(im, v, pos % FL_BK, ex, lane);
}

// The inputs of a q|k|v tile's epilogue that a wave loads ahead of the
// product: the head's norm weights and the RoPE rows of its TPW tokens.
template <int HD, int TPW>
__device__ __forceinline__ void qkv_preload(const QkPostArgs &p, int vh, int t0, int n, int wave, int lane,
                                            float (&nwv)[HD / 64], float2 (&cs)[TPW][HD / 64]) {
    const bool isq = vh < p.n_heads, isk = !isq && vh < p.n_heads + p.n_kv;
    const bool neox = p.rope_style == ROPE_NEOX;
    const float *nwp = isq ? p.q_norm : p.k_norm;
#pragma unroll
    for (int k = 0; k < HD / 64; k++) {
        const int d = lane + 64 * k, i = neox ? d % (HD / 2) : d / 2;
        nwv[k] = p.q_norm && (isq || isk) ? nwp[d] : 1.0f;
#pragma unroll
        for (int j = 0; j < TPW; j++) {
            const int t = min(t0 + wave * TPW + j, n - 1);
            cs[j][k] = p.rope[(size_t)(p.pos_base + t) * (HD / 2) + i];
        }
    }
}

// The epilogue of a head vector's tile hs[token][HD] in LDS (complete, behind
// a barrier): a wave per token (NWV working waves, QV_T / NWV tokens each;
// NT threads in the workgroup) does k_qkpost's work for it, with the same
// lane layout (lane l holds elements l, l + 64) and so the same sums: the
// RMSNorm of q and k heads (model.c:386-389), RoPE from the host table
// (model.c:66-80), q back into its q|k|v row, k and v into the cache
// (model.c:39-48); with p.kvimg also the keys' bytes in the K/V tile images
// of the matrix-core attention.
template <int HD, bool F16, int NWV, int NT>
__device__ __forceinline__ void qkv_finish(const QkPostArgs &p, float (&hs)[QV_T][HD + 1], int (&exs)[QV_T],
                                           const float (&nwv)[HD / 64], const float2 (&cs)[QV_T / NWV][HD / 64],
                                           int vh, int t0, int n, int wave, int lane, bool work) {
    constexpr int ND = HD / 64, TPW = QV_T / NWV;
    const int u0 = vh * HD;
    const bool isq = vh < p.n_heads, isk = !isq && vh < p.n_heads + p.n_kv;
    const int g = vh - p.n_heads - (isk || isq ? 0 : p.n_kv);  // kv head of a k or v head
    const bool neox = p.rope_style == ROPE_NEOX;
    // a v head writing the tile image keeps every wave for the transposed
    // V rows at the end (a barrier)
    const bool vimg = p.kvimg && !isq && !isk;
    if (!work && !vimg) return;
#pragma unroll
    for (int j = 0; j < TPW; j++) {
        if (!work) break;
        const int tt = wave * TPW + j, t = t0 + tt;              // uniform over the wave
        if (t >= n) break;
        const int pos = p.pos_base + t;
        float x[ND];
#pragma unroll
        for (int k = 0; k < ND; k++) x[k] = hs[tt][lane + 64 * k];
        if (!isq && !isk) {   // a v head: to the cache as it is
            const size_t off = (size_t)pos * p.kv_dim + (size_t)g * HD;
#pragma unroll
            for (int k = 0; k < ND; k++) {
                if (F16) reinterpret_cast<uint16_t *>(p.vc)[off + lane + 64 * k] = f2h(x[k]);
                else reinterpret_cast<float *>(p.vc)[off + lane + 64 * k] = x[k];
            }
            if (vimg && !F16) {   // the key's scale from its largest |value|
                float m = 0.0f;
#pragma unroll
                for (int k = 0; k < ND; k++) m = fmaxf(m, fabsf(x[k]));
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
                if (lane == 0) exs[tt] = fl_exp(m);
            }
            continue;
        }
        if (p.q_norm) {   // RMSNorm of the head vector (model.c:50-55)
            float ss = 0.0f;
#pragma unroll
            for (int k = 0; k < ND; k++) ss += x[k] * x[k];
            ss = wave_sum(ss);
            const float scale = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
            for (int k = 0; k < ND; k++) x[k] = x[k] * scale * nwv[k];
        }
        // RoPE: the first element of a pair becomes v0 * cos - v1 * sin, the
        // second v0 * sin + v1 * cos
        float y[ND];
#pragma unroll
        for (int k = 0; k < ND; k++) {
            const int d = lane + 64 * k;
            const bool first = neox ? d < HD / 2 : (d & 1) == 0;
            float xp;
            if (HD == 128 && neox) xp = x[k ^ 1];
            else xp = __shfl(x[k], (neox ? (d < HD / 2 ? d + HD / 2 : d - HD / 2) : d ^ 1) % 64);
            y[k] = first ? x[k] * cs[j][k].x - xp * cs[j][k].y : xp * cs[j][k].y + x[k] * cs[j][k].x;
        }
        if (isq) {
#pragma unroll
            for (int k = 0; k < ND; k++) p.qkv[(size_t)t * p.stride + u0 + lane + 64 * k] = y[k];
        } else {
            const size_t off = (size_t)pos * p.kv_dim + (size_t)g * HD;
#pragma unroll
            for (int k = 0; k < ND; k++) {
                if (F16) reinterpret_cast<uint16_t *>(p.kc)[off + lane + 64 * k] = f2h(y[k]);
                else reinterpret_cast<float *>(p.kc)[off + lane + 64 * k] = y[k];
            }
            if (p.kvimg) qkv_tile_image<HD, F16>(p, g, y, pos, lane);
        }
    }
    if (vimg) {
        // V^T rows of the image (k_pf_kvsplit's bytes): 16-byte pieces of 8
        // keys for every dim, the workgroup's 16 keys and, in the workgroup
        // of the pass's last token, the rest of its tile (the last key
        // repeated), from the tile in LDS
        using I = FlImg<HD, F16>;
        __syncthreads();   // every key's scale in exs
        const int n_t = min(QV_T, n - t0), kl0 = (p.pos_base + t0) % FL_BK;
        const int pc0 = kl0 / 8, pc1 = t0 + QV_T >= n ? FL_BK / 8 : (kl0 + QV_T) / 8;
        uint8_t *im = p.kvimg + ((size_t)g * p.kvimg_tiles + (p.pos_base + t0) / FL_BK) * I::HBYTES;
        for (int w = threadIdx.x; w < HD * (pc1 - pc0); w += NT) {
            const int d = w % HD, pc = pc0 + w / HD;
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                _Float16 hi[2], lo[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int tt = min(8 * pc + e + u - kl0, n_t - 1);
                    const float x = F16 ? hs[tt][d] : __builtin_amdgcn_ldexpf(hs[tt][d], exs[tt]);
                    hi[u] = (_Float16)x;
                    lo[u] = (_Float16)(x - (float)hi[u]);
                }
                hw[e / 2] = fl_pack(hi[0], hi[1]);
                lw[e / 2] = fl_pack(lo[0], lo[1]);
            }
            *reinterpret_cast<u32x4 *>(im + I::KE + I::v_at(d, pc)) = u32x4{hw[0], hw[1], hw[2], hw[3]};
            if constexpr (!F16) {
                *reinterpret_cast<u32x4 *>(im + I::KE + I::v_at(HD + d, pc)) = u32x4{lw[0], lw[1], lw[2], lw[3]};
                if (d == 0)
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        reinterpret_cast<int *>(im + I::KBYTES)[FL_BK + 8 * pc + e] = exs[min(8 * pc + e - kl0, n_t - 1)];
            }
        }
    }
}


}  // namespace ehip
