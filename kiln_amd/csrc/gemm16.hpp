// Pieces shared by the fp16 GEMM kernels (gemm16.hip: the large tiles, gemm16s.hip: the small ones): the launch
// parameters, the epilogues and the prepared weight layout's constants.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace kiln {

constexpr int GBN = 256;             // weight rows (n) of a prepared column tile (and of a large workgroup tile)
constexpr int GBK = 32;              // k per tile: one 64-byte LDS row segment
constexpr int NBW = 4;               // 16-row W blocks per wave (64 n)
constexpr int W_REG_H = GBN * GBK;   // halves of one k tile of a prepared column tile (16 KB)

typedef __attribute__((address_space(3))) half8 lds_half8;
typedef float f2v __attribute__((ext_vector_type(2)));

// s_waitcnt vmcnt(N) (lgkmcnt and expcnt left alone). A device function, so that the host pass never checks
// the builtin's constant argument inside a kernel template (where it depends on the tile height).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}

#define GEMM_RSRC(base, bytes)                                                                             \
    __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(base), (short)0, (int)min((size_t)(bytes), (size_t)0x7fffffff), \
                                      0x00020000 /* raw, CDNA */)

struct GemmParams {
    const _Float16* a;
    const _Float16* w;
    const _Float16* a2;
    const _Float16* w2;
    int K, K2, M, N;
    void* c;
    int ldc;
    const float* gate;
    float beta;
    int tiles_m, tiles_n, total, per;
    int pairs;  // output rows or base not 16-byte (fp32) / 8-byte (fp16) aligned: store element pairs
    int wprep;  // w is in the prepared tile layout (kiln_linear16_prepare_weight), not [N, K] rows
    // EPI_QKV (the DiT self-attention projection with its QK-RMSNorm, RoPE and fp16 K/V preparation fused):
    // columns [0, D) are Q, [D, 2D) K, [2D, 3D) V of H heads; row r is token r % T of item r / T
    _Float16* q16;      // [M, D]: fp16(rope(rmsnorm(q)) * qscale)
    uint16_t* kvp[MAX_JOBS];  // prepared K/V per item (common.hpp layout), K = rope(rmsnorm(k))
    int T, H;
    const uint16_t* qw;  // bf16 [128] norm weights
    const uint16_t* kw;
    float eps, qscale;
    const float* rcos;  // [T, 64]
    const float* rsin;
};
__device__ __forceinline__ floatx4 mfma16(half8 a, half8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// GELU(v) = v Phi(v) = v (1 + erf(v / sqrt 2)) / 2, with Phi from erfc, which keeps its relative accuracy in the
// negative tail: Phi(v) = erfc(z) / 2 for v < 0 and 1 - erfc(z) / 2 for v >= 0, z = |v| / sqrt 2. erfc(z) for
// z >= 0 is the Chebyshev approximation "erfcc" of Numerical Recipes in C (Press et al., 2nd ed., section 6.2),
// fractional error below 1.2e-7 everywhere: ~17 VALU operations and no branches, about half of a library erff,
// and far below the fp16 output's rounding.
__device__ __forceinline__ float gelu_erf(float v) {
    const float z = fabsf(v) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(1.f + 0.5f * z);
    float r = 0.17087277f;
    r = fmaf(t, r, -0.82215223f);
    r = fmaf(t, r, 1.48851587f);
    r = fmaf(t, r, -1.13520398f);
    r = fmaf(t, r, 0.27886807f);
    r = fmaf(t, r, -0.18628806f);
    r = fmaf(t, r, 0.09678418f);
    r = fmaf(t, r, 0.37409196f);
    r = fmaf(t, r, 1.00002368f);
    r = fmaf(t, r, -1.26551223f);
    const float half_erfc = 0.5f * t * __expf(r - z * z);
    return v * (v >= 0.f ? 1.f - half_erfc : half_erfc);
}


// Small tiles (gemm16s.hip, linear_f32.hip): consecutive workgroups of an XCD share a weight tile in its L2. Tile i of an
// XCD-contiguous range lies in a raster group of `group` row tiles, column by column.
__device__ __forceinline__ void raster_tile(int i, int group, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int per_group = group * tiles_n, g0 = (i / per_group) * group, gsz = min(group, tiles_m - g0);
    tm = g0 + (i % per_group) % gsz, tn = (i % per_group) / gsz;
}
// The accumulators of a workgroup's KG groups of MN waves meet in LDS (every wave's blocks, any stage's memory), in the
// groups' order; group kg ends with row blocks kg, kg + KG, .. of its wave position.
template <int MN, int MB, int KG>
__device__ __forceinline__ void merge_k_groups(const floatx4 (&acc)[NBW][MB], floatx4 (&out)[NBW][(MB + KG - 1) / KG],
                                               floatx4* red, int wv, int kg, int lane) {
    constexpr int MBO = (MB + KG - 1) / KG;
    if constexpr (KG == 1) {
#pragma unroll
        for (int nb = 0; nb < NBW; nb++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++) out[nb][mb] = acc[nb][mb];
    } else {
        __syncthreads();  // every wave is done with the stages
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NBW; nb++) red[((wv * MB + mb) * NBW + nb) * 64 + lane] = acc[nb][mb];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < MBO; j++) {
            const int mb = min(kg + KG * j, MB - 1);
#pragma unroll
            for (int nb = 0; nb < NBW; nb++) {
                floatx4 t = red[(((wv % MN) * MB + mb) * NBW + nb) * 64 + lane];
#pragma unroll
                for (int k = 1; k < KG; k++) t += red[(((k * MN + wv % MN) * MB + mb) * NBW + nb) * 64 + lane];
                out[nb][j] = t;
            }
        }
    }
}

// Plain epilogues: 4 consecutive columns n .. n + 3 of row m
template <int EPI>
__device__ __forceinline__ void store_out(const GemmParams& p, int m, int n, floatx4 v, floatx4 gv) {
    const size_t off = (size_t)m * p.ldc + n;
    if constexpr (EPI == KILN_EPI_F32 || EPI == KILN_EPI_RESID) {
        float* dst = static_cast<float*>(p.c) + off;
        floatx4 o;
        const bool need_old = EPI == KILN_EPI_RESID || p.beta != 0.f;
        if (need_old) {
            if (!p.pairs) {
                o = *reinterpret_cast<const floatx4*>(dst);
            } else {
                const f2v o0 = reinterpret_cast<const f2v*>(dst)[0], o1 = reinterpret_cast<const f2v*>(dst)[1];
                o = floatx4{o0[0], o0[1], o1[0], o1[1]};
            }
        }
        floatx4 r;
        if constexpr (EPI == KILN_EPI_RESID) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = o[e] + gv[e] * v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = need_old ? v[e] + p.beta * o[e] : v[e];
        }
        if (!p.pairs) {
            *reinterpret_cast<floatx4*>(dst) = r;
        } else {
            reinterpret_cast<f2v*>(dst)[0] = f2v{r[0], r[1]};
            reinterpret_cast<f2v*>(dst)[1] = f2v{r[2], r[3]};
        }
    } else {
        _Float16* dst = static_cast<_Float16*>(p.c) + off;
        floatx4 r = v;
        if constexpr (EPI == KILN_EPI_GELU16) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = gelu_erf(v[e]);
        }
        if (!p.pairs) {
            *reinterpret_cast<half4*>(dst) = half4{(_Float16)r[0], (_Float16)r[1], (_Float16)r[2], (_Float16)r[3]};
        } else {
            reinterpret_cast<half2v*>(dst)[0] = half2v{(_Float16)r[0], (_Float16)r[1]};
            reinterpret_cast<half2v*>(dst)[1] = half2v{(_Float16)r[2], (_Float16)r[3]};
        }
    }
}
// the gate of columns n .. n + 3
template <int EPI>
__device__ __forceinline__ floatx4 gate_of(const GemmParams& p, int n) {
    if (EPI != KILN_EPI_RESID || !p.gate) return floatx4{1.f, 1.f, 1.f, 1.f};
    const float* g = p.gate + n;
    return floatx4{g[0], g[1], g[2], g[3]};
}

// EPI_QKV epilogue. The workgroup's WN*64 columns are WN/2 heads of one region (Q, K or V: D is a multiple of 256).
// A wave holds 64 columns = half a head; its partner wave (wn ^ 1, the same rows) holds the other half. In the Q and
// K regions the k loop read the wave's W blocks so that block nb holds head dims dq(nb) + 0..15, dq(nb) =
// 32*(wn & 1) + 16*(nb & 1) + 64*(nb >> 1): each RoPE pair (i, i + 64) is element (nb, e) and (nb + 2, e) of one
// lane. Q/K: per-row sum of squares over the head (own half + partner's, through LDS), scale by rsqrt(mean + eps)
// and the bf16 weight, then RoPE in registers. Q is stored as fp16(q * qscale) rows, K and V in the prepared K/V
// layout of their item (kv_k_el / kv_v_el).
// The wave's 16-row block j is block mb = kg + KG*j of its MB (KG k groups share them out; MBO = ceil(MB / KG)).
// Every thread of the workgroup (THREADS) calls it; LDS_HALVES bounds the staged V tile.
template <int WN, int WM, int MB, int KG, int LDS_HALVES>
__device__ __forceinline__ void qkv_epilogue(const GemmParams& p, floatx4 (&acc)[NBW][(MB + KG - 1) / KG], _Float16* lds,
                                             int m0, int n0, int wv, int wn, int wm, int kg, int lane) {
    constexpr int MBO = (MB + KG - 1) / KG, BM = 16 * MB * WM, WAVES = WN * WM * KG;
    const int D = p.H * HD;
    const int region = n0 / D, c0 = n0 - region * D;
    const int hd = (c0 + (wn >> 1) * HD) / HD, half = wn & 1;
    const int rl = lane & 15, cq = 4 * (lane >> 4);  // column within a 16-column block: cq + e
    auto trow = [&](int j) { return (wm * MB + kg + KG * j) * 16 + rl; };  // row within the tile
    auto has = [&](int j) { return KG == 1 || kg + KG * j < MB; };
    auto dq = [&](int nb) { return 32 * half + 16 * (nb & 1) + 64 * (nb >> 1); };  // Q/K head dim of block nb
    float* lf = reinterpret_cast<float*>(lds);
    __syncthreads();  // every wave is done with the k loop's LDS stages
    if (region < 2) {
        const uint16_t* w = region == 0 ? p.qw : p.kw;
        float wt[NBW][4];
#pragma unroll
        for (int nb = 0; nb < NBW; nb++)
#pragma unroll
            for (int e = 0; e < 4; e++) wt[nb][e] = bf16_to_f32(w[dq(nb) + cq + e]);  // any alignment of w
        float r[MBO];
#pragma unroll
        for (int j = 0; j < MBO; j++) {
            float ss = 0.f;
#pragma unroll
            for (int nb = 0; nb < NBW; nb++)
#pragma unroll
                for (int e = 0; e < 4; e++) ss += acc[nb][j][e] * acc[nb][j][e];
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            if (lane < 16) lf[(wv * MBO + j) * 16 + rl] = ss;
            r[j] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < MBO; j++) r[j] = rsqrtf((r[j] + lf[((wv ^ WM) * MBO + j) * 16 + rl]) * (1.0f / HD) + p.eps);
#pragma unroll
        for (int j = 0; j < MBO; j++)
#pragma unroll
            for (int nb = 0; nb < NBW; nb++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[nb][j][e] *= r[j] * wt[nb][e];
        if (p.rcos) {  // RoPE (none for the cross-attention Q projection)
#pragma unroll
            for (int j = 0; j < MBO; j++) {
                const int row = m0 + trow(j);
                const int t = (row < p.M ? row : 0) % p.T;
#pragma unroll
                for (int nb = 0; nb < 2; nb++) {
                    const floatx4 cs = *reinterpret_cast<const floatx4*>(p.rcos + (size_t)t * 64 + dq(nb) + cq);
                    const floatx4 sn = *reinterpret_cast<const floatx4*>(p.rsin + (size_t)t * 64 + dq(nb) + cq);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float a = acc[nb][j][e], b = acc[nb + 2][j][e];
                        acc[nb][j][e] = a * cs[e] - b * sn[e];
                        acc[nb + 2][j][e] = b * cs[e] + a * sn[e];
                    }
                }
            }
        }
    }
    if (region == 2 && p.T % 32 == 0) {
        // V through LDS, one head (128 columns) per pass: the wave pairs of that head write their fp16 values
        // row-major (rows padded to 288 bytes), then every wave assembles whole 16-byte V^T operand units (8 keys of
        // one d) with transposing reads, as the K/V prepare pass does, instead of 2-byte scatters. With T a
        // multiple of 32 (and the tile's first row one too) no 32-key half tile straddles two items.
        constexpr int VRS = HD + 16;
        static_assert(BM % 32 == 0 && BM * VRS <= LDS_HALVES, "the staged V tile fits in the ring's LDS");
        const int i = lane & 15, gq = lane >> 4;
        typedef short s4 __attribute__((ext_vector_type(4)));
        typedef short s8 __attribute__((ext_vector_type(8)));
        typedef __attribute__((address_space(3))) s4 lds_s4;
#pragma unroll
        for (int pass = 0; pass < WN / 2; pass++) {
            if ((wn >> 1) == pass) {
#pragma unroll
                for (int j = 0; j < MBO; j++)
                    if (has(j))
#pragma unroll
                        for (int nb = 0; nb < NBW; nb++) {
                            const floatx4 v = acc[nb][j];
                            *reinterpret_cast<half4*>(lds + trow(j) * VRS + half * 64 + nb * 16 + cq) =
                                half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                        }
            }
            __syncthreads();
            const int hdp = (c0 + pass * HD) / HD;
            for (int op = wv; op < (BM / 32) * 8; op += WAVES) {
                const int ht = op >> 3, db = op & 7, row0 = m0 + ht * 32;
                if (row0 >= p.M) break;  // ops ascend with ht: every later one is past the matrix too
                const int b = row0 / p.T, key0 = row0 - b * p.T;
                const _Float16* src = lds + (ht * 32 + 4 * gq + (i >> 2)) * VRS + 16 * db + 4 * (i & 3);
                const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)src);
                const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(src + 16 * VRS));
                _Float16* kv = reinterpret_cast<_Float16*>(p.kvp[b]) + (size_t)hdp * kv_head_stride(p.T) +
                               (size_t)(key0 / KT) * KV_TILE_H;
                *reinterpret_cast<s8*>(kv + kv_v_off((key0 % KT) / 32, db, lane)) =
                    s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
            __syncthreads();  // every read of this head's values precedes the next pass's writes
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < MBO; j++) {
        const int row = m0 + trow(j);
        if (row >= p.M || !has(j)) continue;
        const int b = row / p.T, key = row - b * p.T;
        _Float16* kv = reinterpret_cast<_Float16*>(p.kvp[b]) + (size_t)hd * kv_head_stride(p.T) +
                       (size_t)(key / KT) * KV_TILE_H;
        const int kc = (key % KT) / 32, k32 = key % 32;
#pragma unroll
        for (int nb = 0; nb < NBW; nb++) {
            // 4 consecutive d, inside one 8-element chunk (Q/K: the permuted head dims; V: the plain ones)
            const int d = (region < 2 ? dq(nb) : half * 64 + nb * 16) + cq;
            const floatx4 v = acc[nb][j];
            if (region == 0) {
                *reinterpret_cast<half4*>(p.q16 + (size_t)row * D + hd * HD + d) =
                    half4{(_Float16)(v[0] * p.qscale), (_Float16)(v[1] * p.qscale), (_Float16)(v[2] * p.qscale),
                          (_Float16)(v[3] * p.qscale)};
            } else if (region == 1) {
                *reinterpret_cast<half4*>(kv + kv_k_el(kc, k32, d)) =
                    half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) kv[kv_v_el(kc, k32, d + e)] = (_Float16)v[e];
            }
        }
    }
}

// The small-tile kernels (gemm16s.hip): the one with the smallest modelled time for a product (K with the LoRA's
// k2), and its launch. The model serves the large tiles' choice too.
struct GemmCost {
    double launch, tile, slice, shared;
};
double gemm_cost(const GemmCost& c, long tiles, int slices, int cus);
struct SmallGemm {
    int cfg;
    double cost;
    int bn, bm;
};
SmallGemm gemm16s_choose(int M, int N, int K, int epi, int cus);
hipError_t launch_gemm16s(const GemmParams& p, int cfg, int epi, hipStream_t s);

}  // namespace kiln
