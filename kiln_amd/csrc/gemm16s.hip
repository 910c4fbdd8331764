// fp16 GEMM on small workgroup tiles (gfx950), for products whose 256-wide tiles (gemm16.hip) leave most of the
// chip idle: few activation rows (a preview picture, one item) against the DiT's weights.
//
// Same contract, operand layouts, epilogues and transposed product (C^T = W A^T) as k_gemm16. What differs:
//  * the workgroup tile is 64*WN weight rows x 16*MB*WM activation rows. With few rows the product is bound by the
//    stream of the weights (8 MB to 33 MB, each used for a few hundred flop per byte), so what counts is how many
//    CUs read at once and how many bytes each keeps in flight, not the operand reuse of one tile.
//  * the 8 waves of a workgroup are KG groups of WN x WM waves that share the k range: in a step of SL = KG*KS
//    32-wide k slices (SL*64 bytes of every row), group kg multiplies slices kg*KS .. kg*KS + KS - 1. All the
//    accumulators meet once, through LDS, after the k loop. A tile of 32 rows then still has 8 waves' loads in
//    flight, with no partial sums in memory and a fixed order of summation.
//  * a step's weights and activations stream global -> LDS by buffer-form DMA through NST stages of up to 48 KB,
//    NST - 1 steps ahead; one barrier per step.
//  * at M = 256 a CU takes in 40 (128 x 64) to 62 GB/s (64 x 32) of operands, a third to a half of what LDS DMA alone
//    takes from L2 (120 to 130): what bounds these products is the chain of a step (barrier, operand reads, MFMAs) in the
//    one workgroup of a CU, and where a product has fewer tiles than CUs (128 of 128 x 32 at 2048 x 2048, 192 of 128 x 64
//    at 6144 x 2048), the idle ones. Measured, us, one product of M rows, fp16 out, weights from memory, 256-wide tiles with
//    plain / prepared weights -> these (alike with both): 2048 x 2048 M = 64 44.6 / 35.6 -> 10.3, M = 256 47.1 / 39.5 -> 9.9,
//    M = 1024 54.3 / 44.4 -> 17.5, M = 3072 56.2 / 48.0 -> 33.6; 2048 x 8192 M = 256 155.5 / 128.5 -> 25.7; 8192 x 2048
//    M = 256 48.7 / 41.3 -> 18.9.
//  * row-major operands (activations, plain weights) lie in LDS as 128-byte rows of two k slices, 16-byte chunk c
//    of row r at position c ^ (r & 7): the DMA reads whole 128-byte lines, the operand reads are conflict free.
//    Prepared weights keep their 64-byte rows (one contiguous run per slice).
#include "gemm16.hpp"

namespace kiln {

constexpr int STHR = 512;

template <int WN_, int WM_, int MB_, int KG_, int KS_, int NST_>
struct SCfg {
    static constexpr int WN = WN_, WM = WM_, MB = MB_, KG = KG_, KS = KS_, NST = NST_;
    static constexpr int BN = 64 * WN, BM = 16 * MB * WM, SL = KG * KS;
    static constexpr int W_BYTES = SL * BN * 64, A_BYTES = SL * BM * 64, STAGE = W_BYTES + A_BYTES;
    static constexpr int W_DMA = W_BYTES / 16 / STHR, A_DMA = A_BYTES / 16 / STHR, DPS = W_DMA + A_DMA;
    static constexpr int RED = KG > 1 ? STHR / 64 * NBW * MB * 1024 : 0;  // the groups' accumulators
    static constexpr int LDS = NST * STAGE > RED ? NST * STAGE : RED;
    static_assert(WN * WM * KG * 64 == STHR && SL % 2 == 0, "8 waves, whole 128-byte rows");
    static_assert(W_DMA * 16 * STHR == W_BYTES && A_DMA * 16 * STHR == A_BYTES, "every thread copies whole pieces");
    static_assert((WM & (WM - 1)) == 0 && LDS <= 160 * 1024, "partner wave = wave ^ WM; LDS of a CU");
};

template <int EPI, class C, bool WPREP>
__global__ __launch_bounds__(STHR, 1) void k_gemm16s(const GemmParams p) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass only needs the kernel's handle (and rejects the DMA builtin's lambdas)
    constexpr int WN = C::WN, WM = C::WM, MB = C::MB, KG = C::KG, KS = C::KS, NST = C::NST, SL = C::SL;
    constexpr int BN = C::BN, BM = C::BM;
    extern __shared__ __attribute__((aligned(16))) _Float16 lds[];  // NST stages of [W slices | A slices]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wv / (WN * WM), wn = wv % (WN * WM) / WM, wm = wv % WM;

    const int i = (int)(blockIdx.x & 7) * p.per + (int)(blockIdx.x >> 3);  // XCD b % 8: a contiguous range of tiles
    if (i >= p.total) return;
    constexpr int S_GROUP_M = 16;  // row tiles per raster group
    int tm, tn;
    raster_tile(i, S_GROUP_M, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int mrows = min(BM, p.M - m0);  // N is a multiple of BN

    // DMA: 16-byte pieces q = tid + STHR*r of a region. Row-major form: pair of slices q / (8 R), row (q >> 3) % R,
    // LDS position q & 7 holding chunk (q & 7) ^ (row & 7). Prepared form: slice q / (4 BN), already in LDS order.
    // Rows past the matrix re-read its last row (results unused); slices past a product's last one (`have` of the
    // step's SL are real) re-read the step's first slice and are not multiplied.
    auto row_off = [&](int r, int R, int rows, int ld, int have) {
        const int q = tid + STHR * r, row = (q >> 3) % R, c = (q & 7) ^ (row & 7);
        const bool in = 2 * (q / (8 * R)) + (c >> 2) < have;
        return (uint32_t)(min(row, rows - 1) * ld * 2 + (in ? q / (8 * R) * 128 + c * 16 : (c & 3) * 16));
    };
    auto prep_off = [&](int r, int have) {
        const int q = tid + STHR * r, s = q / (BN * 4);
        return (uint32_t)((s < have ? s : 0) * (W_REG_H * 2) + q % (BN * 4) * 16);
    };
    uint32_t voff_w[C::W_DMA], voff_a[C::A_DMA];
#pragma unroll
    for (int r = 0; r < C::W_DMA; r++) voff_w[r] = WPREP ? prep_off(r, SL) : row_off(r, BN, BN, p.K, SL);
#pragma unroll
    for (int r = 0; r < C::A_DMA; r++) voff_a[r] = row_off(r, BM, mrows, p.K, SL);
    // prepared: the tile's rows of the 256-row column tile's first k block
    const __amdgpu_buffer_rsrc_t rw1 =
        WPREP ? GEMM_RSRC(p.w + (size_t)(n0 / GBN) * GBN * p.K + n0 % GBN * GBK,
                          (size_t)GBN * p.K * 2 - n0 % GBN * GBK * 2)
              : GEMM_RSRC(p.w + (size_t)n0 * p.K, (size_t)BN * p.K * 2);
    const __amdgpu_buffer_rsrc_t ra1 = GEMM_RSRC(p.a + (size_t)m0 * p.K, (size_t)mrows * p.K * 2);
    const __amdgpu_buffer_rsrc_t rw2 = GEMM_RSRC(p.w2 + (size_t)n0 * p.K2, (size_t)BN * p.K2 * 2);
    const __amdgpu_buffer_rsrc_t ra2 = GEMM_RSRC(p.a2 + (size_t)m0 * p.K2, (size_t)mrows * p.K2 * 2);
    const int KT1 = p.K / GBK, KT2 = p.K2 / GBK;
    const int S1 = (KT1 + SL - 1) / SL, S = S1 + (KT2 + SL - 1) / SL;  // steps of the main product; with the LoRA's
    typedef __attribute__((address_space(3))) void* lds_p;
    auto dma = [&](int st, int stage) {
        char* base = reinterpret_cast<char*>(lds) + stage * C::STAGE + wv * 1024;
        if ((st + 1) * SL <= KT1) {
            const int sa = st * SL * 64, sw = WPREP ? st * SL * W_REG_H * 2 : sa;
#pragma unroll
            for (int r = 0; r < C::W_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rw1, (lds_p)(base + STHR * 16 * r), 16, voff_w[r], sw, 0, 0);
#pragma unroll
            for (int r = 0; r < C::A_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra1, (lds_p)(base + C::W_BYTES + STHR * 16 * r), 16, voff_a[r],
                                                         sa, 0, 0);
        } else {  // a partial last step, or the LoRA product's (few): offsets recomputed
            const bool lora = st >= S1;
            const int s0 = (lora ? st - S1 : st) * SL, have = (lora ? KT2 : KT1) - s0, ld = lora ? p.K2 : p.K;
            const int sa = s0 * 64, sw = WPREP && !lora ? s0 * W_REG_H * 2 : sa;
#pragma unroll
            for (int r = 0; r < C::W_DMA; r++) {
                const uint32_t o = WPREP && !lora ? prep_off(r, have) : row_off(r, BN, BN, ld, have);
                const lds_p to = (lds_p)(base + STHR * 16 * r);
                if (lora) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw2, to, 16, o, sw, 0, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw1, to, 16, o, sw, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < C::A_DMA; r++) {
                const uint32_t o = row_off(r, BM, mrows, ld, have);
                const lds_p to = (lds_p)(base + C::W_BYTES + STHR * 16 * r);
                if (lora) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra2, to, 16, o, sa, 0, 0);
                else __builtin_amdgcn_raw_ptr_buffer_load_lds(ra1, to, 16, o, sa, 0, 0);
            }
        }
    };

    // operand reads: lane reads row lane & 15 of a 16-row block, k chunk lane >> 4 of a slice. EPI_QKV, Q and K
    // regions: the wave's W blocks are the head rows 32*(wn & 1) + {0, 16, 64, 80} (see qkv_epilogue).
    const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) _Float16*)lds;
    const int rl = lane & 15, g = lane >> 4;
    const bool qkperm = EPI == EPI_QKV && n0 / (p.H * HD) < 2;
    const int wrow = (wn >> 1) * 128 + (wn & 1) * (qkperm ? 32 : 64) + rl;
    const int wrow_hi = wrow + (qkperm ? 32 : 0);  // blocks nb >= 2
    auto read = [&](uint32_t a) { return *reinterpret_cast<const lds_half8*>((size_t)a); };
    auto pair_at = [&](int s, int R) {  // slice s of a row-major region: its pair's rows, this lane's chunk position
        return (uint32_t)((s >> 1) * R * 128 + (((4 * (s & 1) + g) ^ (rl & 7)) * 16));
    };
    floatx4 acc[NBW][MB];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[nb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};
    // slices s of a stage, s < have
    auto compute = [&](uint32_t st_base, auto prep_tag, int have, auto refill) {
        constexpr bool PREP = decltype(prep_tag)::value;
        half8 fw[KS][NBW], fa[KS][MB];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int s = kg * KS + ks;
            if (s >= have) break;
#pragma unroll
            for (int nb = 0; nb < NBW; nb++) {
                const int row = (nb < 2 ? wrow : wrow_hi) + 16 * nb;
                fw[ks][nb] = PREP ? read(st_base + s * BN * 64 + row * 64 + ((g ^ ((rl >> 1) & 3)) * 16))
                                  : read(st_base + pair_at(s, BN) + row * 128);
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
                fa[ks][mb] = read(st_base + C::W_BYTES + pair_at(s, BM) + (wm * MB * 16 + mb * 16 + rl) * 128);
        }
        __builtin_amdgcn_sched_barrier(0);  // every operand read in flight before the first MFMA waits for one
        // with k groups (few MFMAs per step) the refill goes behind the reads that the MFMAs wait for: 2048 x 8192, M = 256
        // 27.6 -> 25.3 us; the 128 x 192 tile keeps it ahead of them (6144 x 2048, M = 3072 95.0, behind them 98.8)
        if constexpr (KG > 1) {
            refill();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            if (kg * KS + ks >= have) break;
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int nb = 0; nb < NBW; nb++) acc[nb][mb] = mfma16(fw[ks][nb], fa[ks][mb], acc[nb][mb]);
        }
    };
    using Prep = std::integral_constant<bool, WPREP>;

#pragma unroll
    for (int s = 0; s < NST - 1; s++)
        if (s < S) dma(s, s);
    int stage = 0;
    auto step = [&](int st, bool steady) {
        // step st landed in every wave; every wave is done with step st - 1, whose stage is refilled
        const int ahead = S - 1 - st;
        if (steady || ahead >= NST - 2) wait_vmcnt<(NST - 2) * C::DPS>();
        else if (NST > 3 && ahead == 1) wait_vmcnt<C::DPS>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of the stage to refill are complete
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const int into = stage == 0 ? NST - 1 : stage - 1;
        auto refill = [&]() {
            if (steady || st + NST - 1 < S) dma(st + NST - 1, into);
        };
        if constexpr (KG == 1) refill();
        const uint32_t sb = lds_base + stage * C::STAGE;
        if (steady) compute(sb, Prep{}, SL, refill);
        else if (st < S1) compute(sb, Prep{}, KT1 - st * SL, refill);
        else compute(sb, std::false_type{}, KT2 - (st - S1) * SL, refill);
        __builtin_amdgcn_sched_barrier(0);
        stage = stage == NST - 1 ? 0 : stage + 1;
    };
    const int nsteady = min(KT1 / SL, S - (NST - 1));  // whole main-product steps with a refill to issue
    int st = 0;
    for (; st < nsteady; st++) step(st, true);
    for (; st < S; st++) step(st, false);

    // the groups' sums meet in LDS; group kg finishes row blocks kg, kg + KG, ..
    constexpr int MBO = (MB + KG - 1) / KG;
    floatx4 out[NBW][MBO];
    merge_k_groups<WN * WM, MB, KG>(acc, out, reinterpret_cast<floatx4*>(lds), wv, kg, lane);
    if constexpr (EPI == EPI_QKV) {
        qkv_epilogue<WN, WM, MB, KG, C::LDS / 2>(p, out, lds, m0, n0, wv, wn, wm, kg, lane);
    } else {
        const int n = n0 + wn * 64 + 4 * g;
        floatx4 gv[NBW];
#pragma unroll
        for (int nb = 0; nb < NBW; nb++) gv[nb] = gate_of<EPI>(p, n + nb * 16);
#pragma unroll
        for (int j = 0; j < MBO; j++) {
            const int mb = kg + KG * j, m = m0 + (wm * MB + mb) * 16 + rl;
            if (mb >= MB || m >= p.M) break;
#pragma unroll
            for (int nb = 0; nb < NBW; nb++) store_out<EPI>(p, m, n + nb * 16, out[nb][j], gv[nb]);
        }
    }
#endif
}

template <int EPI, class C>
static hipError_t launch_cfg(GemmParams p, hipStream_t s) {
    p.tiles_m = (p.M + C::BM - 1) / C::BM;
    p.tiles_n = p.N / C::BN;
    p.total = p.tiles_m * p.tiles_n;
    const int nb = (p.total + 7) / 8 * 8;
    p.per = nb / 8;
    auto kern = p.wprep ? k_gemm16s<EPI, C, true> : k_gemm16s<EPI, C, false>;
    hipLaunchKernelGGL(kern, dim3(nb), dim3(STHR), C::LDS, s, p);
    return hipGetLastError();
}

// The configurations: the tile shrinks (and the k groups multiply) as the rows get fewer.
//            WN WM MB KG KS NST    tile (n x m), k per step
using S0 = SCfg<2, 4, 3, 1, 2, 4>;  // 128 x 192, 64
using S1 = SCfg<2, 2, 4, 2, 1, 4>;  // 128 x 128, 64
using S2 = SCfg<2, 1, 4, 4, 1, 3>;  // 128 x 64, 128
using S3 = SCfg<2, 1, 2, 4, 1, 4>;  // 128 x 32, 128
using S4 = SCfg<1, 1, 2, 8, 1, 3>;  //  64 x 32, 256 (no whole head: not for EPI_QKV)

template <class C>
static hipError_t launch_epi(const GemmParams& p, int epi, hipStream_t s) {
    switch (epi) {
        case KILN_EPI_F32: return launch_cfg<KILN_EPI_F32, C>(p, s);
        case KILN_EPI_F16: return launch_cfg<KILN_EPI_F16, C>(p, s);
        case KILN_EPI_GELU16: return launch_cfg<KILN_EPI_GELU16, C>(p, s);
        case KILN_EPI_RESID: return launch_cfg<KILN_EPI_RESID, C>(p, s);
        case EPI_QKV:
            if constexpr (C::WN % 2 == 0) return launch_cfg<EPI_QKV, C>(p, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gemm16s(const GemmParams& p, int cfg, int epi, hipStream_t s) {
    switch (cfg) {
        case 0: return launch_epi<S0>(p, epi, s);
        case 1: return launch_epi<S1>(p, epi, s);
        case 2: return launch_epi<S2>(p, epi, s);
        case 3: return launch_epi<S3>(p, epi, s);
        case 4: return launch_epi<S4>(p, epi, s);
        default: return hipErrorInvalidValue;
    }
}

// Modelled time of a product in us: a launch, per round of the chip's CUs a tile's fixed cost and its k slices, and
// the contention of the tiles in flight for L2 and HBM. The coefficients are least-squares fits of measured times
// (M = 64 .. 6912 x {2048 x 2048, 8192 x 2048, 2048 x 8192, 6144 x 2048}, each configuration at every size, weights
// rotated through memory), 10 to 18% off at most; the 128 x 128 tile's contention is set above its fit (0.055), where two
// rounds of it meet the 256-wide tile (2048 x 8192, M = 4096 158 against 151). It does not depend on the weight's layout,
// so a prepared weight gives the bits of the row-major one, and where the two forms meet it is a compromise between the
// layouts: 2048 x 2048, 256 x 224 tiles -> 128 x 128, fp16 / fp32 / residual out, M = 3584 plain 47.3 / 47.2 / 52.6 -> 43.2 /
// 44.7 / 47.6, prepared 42.1 / 42.3 / 47.7 -> 41.9 / 43.8 / 47.7; M = 4096 plain 48.3 / 48.4 / 53.9 -> 44.2 / 46.5 / 50.4,
// prepared 43.7 / 43.4 / 49.3 -> 43.3 / 45.5 / 50.5: at most 5% over the better one. A DiT block there: T = 3584 718 ->
// 696, T = 4096 721 -> 727.
double gemm_cost(const GemmCost& c, long tiles, int slices, int cus) {
    const double rounds = (double)((tiles + cus - 1) / cus);
    return c.launch + rounds * (c.tile + c.slice * slices) + c.shared * tiles * slices / cus;
}

SmallGemm gemm16s_choose(int M, int N, int K, int epi, int cus) {
    static const struct {
        int bn, bm;
        GemmCost c;
    } cfg[] = {{128, 192, {2.55, 4.76, 0.270, 0.133}},
               {128, 128, {2.03, 4.75, 0.224, 0.080}},
               {128, 64, {2.06, 2.97, 0.142, 0.035}},
               {128, 32, {2.35, 2.09, 0.115, 0.016}},
               {64, 32, {2.46, 2.05, 0.074, 0.000}}};
    SmallGemm best{-1, 0.0, 0, 0};
    for (int i = 0; i < 5; i++) {
        if (epi == EPI_QKV && cfg[i].bn % 128) continue;
        const long tiles = (long)((M + cfg[i].bm - 1) / cfg[i].bm) * (N / cfg[i].bn);
        const double t = gemm_cost(cfg[i].c, tiles, K / GBK, cus);
        if (best.cfg < 0 || t < best.cost) best = {i, t, cfg[i].bn, cfg[i].bm};
    }
    return best;
}

}  // namespace kiln
