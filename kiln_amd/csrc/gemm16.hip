// fp16 GEMM with fused epilogues for the DiT's linear layers on gfx950 (CDNA4) MFMA, fp32 accumulation.
//
// Contract: the reference's linear16 / tc16::k_gemm16 (engine/src/kernels.cu:559-609,
// engine/src/tcgemm16.cuh:1-200):
//   acc = A[M,K] W[N,K]^T (+ A2[M,K2] W2[N,K2]^T, the folded LoRA product), all fp16, row-major, K innermost;
//   epilogue F32:    C (fp32)  = acc + beta*C
//            F16:    C (fp16)  = acc
//            GELU16: C (fp16)  = GELU(acc), GELU(v) = v/2 (1 + erf(v/sqrt 2))
//            RESID:  C (fp32) += gate[col] * acc   (gate null: 1)
// The reference accumulates each 32-wide k tile in fp16 and flushes it into fp32 (tcgemm16.cuh:6-7); here
// every product accumulates in fp32 (the MFMA's native accumulator): more accurate, same inputs.
//
// Design (gfx950, wave64):
//  * workgroup tile 256 weight rows (n) x 32*MB activation rows (m, MB = 8 or 7, whichever leaves the fewest
//    idle CUs in the last round), k tiles of 32; 8 waves in 4 (n) x 2 (m), each wave 64 n x 16*MB m =
//    4 x MB blocks of v_mfma_f32_16x16x32_f16 (the shape that sustains the higher rate on a power-limited
//    MI355X), up to 128 fp32 accumulators per lane, two waves per SIMD.
//  * the product is computed transposed, C^T = W A^T: the MFMA's A operand is a 16-row block of W, its B
//    operand a 16-row block of A, and each lane ends with 4 consecutive output columns of one output row
//    (one 16-byte fp32 / 8-byte fp16 store per block).
//  * both tiles stream global -> LDS through a 4-stage ring of buffer-form DMA (buffer_load ... lds), three
//    k tiles ahead; one barrier per k tile. LDS rows are 64 bytes (32 fp16 of k) holding four 16-byte
//    chunks, chunk c of row r at position c ^ ((r >> 1) & 3): the DMA reads whole row segments (coalesced)
//    and the MFMA operand reads (16 rows x one chunk per 16 lanes) are bank-conflict free.
//  * the operands of k tile t+1 are read from LDS while the MFMAs of k tile t run.
//  * products too small to fill the chip with these tiles run on gemm16s.hip's.
//  * 1-D grid, XCD-aware: workgroup b runs on XCD b % 8, and each XCD takes a contiguous range of tiles in
//    groups of 4 row tiles, so the workgroups resident on one XCD share A and W tiles in its L2.
#include "gemm16.hpp"

namespace kiln {

constexpr int GNS = 4;               // LDS ring stages
constexpr int WAVES_N = 4;                   // waves along n; 2 along m
constexpr int WAVES_M = 2;
static_assert(NBW == GBN / 16 / WAVES_N, "64 n per wave");
constexpr int GTHR = 64 * WAVES_N * WAVES_M;
constexpr int GROUP_M = 4;           // row tiles per raster group
constexpr int W_DMA = W_REG_H * 2 / (GTHR * 16);  // 16-byte W pieces per thread per k tile

// MB: 16-row activation blocks per wave; the workgroup's activation tile is 32*MB rows
template <int MB>
struct Tile {
    static constexpr int BM = 32 * MB;
    static constexpr int A_REG_H = BM * GBK;
    static constexpr int STAGE_H = W_REG_H + A_REG_H;
};
// 16-byte A pieces per thread per k tile (the same for every tile height used, so that no array size in the
// kernel depends on the template argument)
constexpr int A_DMA = Tile<8>::A_REG_H * 2 / (GTHR * 16);
constexpr int DMA_PER_TILE = W_DMA + A_DMA;
static_assert(Tile<8>::A_REG_H * 2 == A_DMA * GTHR * 16 && Tile<7>::A_REG_H * 2 > (A_DMA - 1) * GTHR * 16, "A pieces");

// LATE (prepared weights): in steady steps the refill DMA leaves the barrier's shadow and the two waves of a SIMD
// issue it at different points of the MFMA stream: waves 0-3 after the first activation block's MFMAs, waves 4-7
// after the fourth. Waves w and w + 4 share a SIMD; with both refills issued together right after the barrier,
// the DMA issue stalls of the two waves coincide and the matrix core idles through them. Measured on the DiT
// shapes (A/B on one box): the block's four GEMMs -1.4% with waves 4-7 moved, -1.0 to -1.9% more with waves 0-3
// moved as well; the split slows plain-weight launches (whose W rows arrive as 64-byte row pieces) by ~2%, which
// keep the refill after the barrier.
constexpr int EARLY_MB = 1, LATE_MB = 3;
template <int EPI, int MB, bool LATE>
__global__ __launch_bounds__(GTHR, 1) void k_gemm16(const GemmParams p) {
    using TL = Tile<MB>;
    constexpr int BM = TL::BM, STAGE_H = TL::STAGE_H;
    extern __shared__ __attribute__((aligned(16))) _Float16 lds[];  // GNS stages of [W 256 rows | A BM rows]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wv / WAVES_M, wm = wv % WAVES_M;

    // tile of this workgroup: XCD b % 8 takes the contiguous range [xcd * per, (xcd + 1) * per)
    const int i = (int)(blockIdx.x & 7) * p.per + (int)(blockIdx.x >> 3);
    if (i >= p.total) return;
    const int per_group = GROUP_M * p.tiles_n;
    const int g0 = (i / per_group) * GROUP_M;
    const int gsz = min(GROUP_M, p.tiles_m - g0);
    const int tm = g0 + (i % per_group) % gsz, tn = (i % per_group) / gsz;
    const int m0 = tm * BM, n0 = tn * GBN;
    const int mrows = min(BM, p.M - m0), nrows = min(GBN, p.N - n0);

    // DMA: this thread's 16-byte pieces q = tid + GTHR*r of a region: row q >> 2, LDS position q & 3 holding
    // k chunk (q & 3) ^ ((row >> 1) & 3). Rows past the matrix re-read its last row (results unused); pieces
    // past a region's end repeat the piece one round earlier (same source, same LDS bytes), so every wave
    // issues the same number of DMA operations. The k tile goes in the scalar offset.
    uint32_t voff_w[W_DMA], voff_a[A_DMA];
    auto voffs = [&](int ld, bool prep, uint32_t(&vw)[W_DMA], uint32_t(&va)[A_DMA]) {
#pragma unroll
        for (int r = 0; r < W_DMA; r++) {
            const int q = tid + GTHR * r, row = q >> 2, c = (q & 3) ^ ((row >> 1) & 3);
            // prepared W (main product only): the k tile's 16 KB block is already in LDS order
            vw[r] = prep ? (uint32_t)q * 16 : (uint32_t)(min(row, nrows - 1) * ld + c * 8) * 2;
        }
#pragma unroll
        for (int r = 0; r < A_DMA; r++) {
            int q = tid + GTHR * r;
            if (q >= BM * 4) q -= GTHR;
            const int row = q >> 2, c = (q & 3) ^ ((row >> 1) & 3);
            va[r] = (uint32_t)(min(row, mrows - 1) * ld + c * 8) * 2;
        }
    };
    voffs(p.K, p.wprep != 0, voff_w, voff_a);
    const __amdgpu_buffer_rsrc_t rw1 =
        p.wprep ? GEMM_RSRC(p.w + (size_t)tn * GBN * p.K, (size_t)GBN * p.K * 2)
                : GEMM_RSRC(p.w + (size_t)n0 * p.K, (size_t)nrows * p.K * 2);
    const __amdgpu_buffer_rsrc_t ra1 = GEMM_RSRC(p.a + (size_t)m0 * p.K, (size_t)mrows * p.K * 2);
    const __amdgpu_buffer_rsrc_t rw2 = GEMM_RSRC(p.w2 + (size_t)n0 * p.K2, (size_t)nrows * p.K2 * 2);
    const __amdgpu_buffer_rsrc_t ra2 = GEMM_RSRC(p.a2 + (size_t)m0 * p.K2, (size_t)mrows * p.K2 * 2);
    const int KT1 = p.K / GBK, KTT = KT1 + p.K2 / GBK;
    // the wave's 64 lanes write 1 KB of contiguous LDS at the wave-uniform base the DMA takes from M0
    auto dma = [&](int kt, int stage) {
        _Float16* base = lds + stage * STAGE_H;
        _Float16* aq0[A_DMA];
#pragma unroll
        for (int r = 0; r < A_DMA; r++) {
            int q0 = GTHR * r + wv * 64;
            if (q0 >= BM * 4) q0 -= GTHR;
            aq0[r] = base + W_REG_H + q0 * 8;
        }
        if (kt < KT1) {
            const int so = kt * GBK * 2;
            const int sow = p.wprep ? kt * W_REG_H * 2 : so;
#pragma unroll
            for (int r = 0; r < W_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rw1, (__attribute__((address_space(3))) void*)(base + (GTHR * r + wv * 64) * 8), 16, voff_w[r], sow, 0, 0);
#pragma unroll
            for (int r = 0; r < A_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra1, (__attribute__((address_space(3))) void*)aq0[r], 16,
                                                         voff_a[r], so, 0, 0);
        } else {
            const int so = (kt - KT1) * GBK * 2;
            uint32_t vw2[W_DMA], va2[A_DMA];  // the LoRA tiles (few): offsets recomputed
            voffs(p.K2, false, vw2, va2);
#pragma unroll
            for (int r = 0; r < W_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rw2, (__attribute__((address_space(3))) void*)(base + (GTHR * r + wv * 64) * 8), 16, vw2[r], so, 0, 0);
#pragma unroll
            for (int r = 0; r < A_DMA; r++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra2, (__attribute__((address_space(3))) void*)aq0[r], 16,
                                                         va2[r], so, 0, 0);
        }
    };

    // operand reads: lane reads row (lane & 15) of a 16-row block, k chunk lane >> 4; blocks of one wave are
    // 1 KB apart, so they fold into ds_read_b128 immediate offsets.
    const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) _Float16*)lds;
    const int rl = lane & 15;
    const uint32_t swz = (uint32_t)((((lane >> 4) ^ ((rl >> 1) & 3))) * 16);
    // EPI_QKV, Q and K regions: the wave's W blocks are the head rows 32*(wn & 1) + {0, 16, 64, 80} instead of
    // 64*(wn & 1) + {0, 16, 32, 48}, so that each RoPE pair (d, d + 64) lands in one lane (blocks nb and nb + 2)
    const bool qkperm = EPI == EPI_QKV && n0 / (p.H * HD) < 2;
    const uint32_t wbase = lds_base + (uint32_t)((((wn >> 1) * 128 + (wn & 1) * (qkperm ? 32 : 64)) + rl) * 64) + swz;
    const uint32_t wbase_hi = wbase + (qkperm ? 2048u : 0u);  // blocks nb >= 2
    const uint32_t abase = lds_base + (uint32_t)(W_REG_H * 2 + (wm * MB * 16 + rl) * 64) + swz;
    auto wfrag = [&](int stage, int nb) {
        return reinterpret_cast<const lds_half8*>((size_t)((nb < 2 ? wbase : wbase_hi) + stage * STAGE_H * 2))[nb * 64];
    };
    auto afrag = [&](int stage, int mb) {
        return reinterpret_cast<const lds_half8*>((size_t)(abase + stage * STAGE_H * 2))[mb * 64];
    };

    floatx4 acc[NBW][MB];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[nb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};

    // prologue: k tiles 0..3 in flight; wait for tile 0 and read its operands
#pragma unroll
    for (int s = 0; s < GNS; s++)
        if (s < KTT) dma(s, s);
    if (KTT >= GNS) wait_vmcnt<(GNS - 1) * DMA_PER_TILE>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    // Operands in registers: the activation blocks of the current k tile (each replaced by the next tile's
    // block as soon as its four MFMAs are issued) and the W blocks of the current and the next tile (the loop
    // alternates them).
    half8 fa[MB], fw[NBW], gw[NBW];
#pragma unroll
    for (int b = 0; b < MB; b++) fa[b] = afrag(0, b);
#pragma unroll
    for (int b = 0; b < NBW; b++) fw[b] = wfrag(0, b);
    __builtin_amdgcn_sched_barrier(0);

    // STEADY: kt + GNS < KTT (a refill to issue, the next tile's operands to read, GNS - 2 tiles in flight)
    auto step = [&](auto steady_tag, int kt, half8(&cw)[NBW], half8(&nw)[NBW]) {
        constexpr bool STEADY = decltype(steady_tag)::value;
        // tile kt+1 landed in every wave, and every wave has read tile kt's operands (stage kt is free):
        // refill it with tile kt+GNS. Only tiles kt+2 .. kt+GNS-1 may stay in flight.
        const int ahead = KTT - 1 - kt;
        static_assert(GNS == 4, "the waits below assume a 4-stage ring");
        if (STEADY || ahead >= 3) wait_vmcnt<2 * DMA_PER_TILE>();
        else if (ahead == 3) wait_vmcnt<2 * DMA_PER_TILE>();
        else if (ahead == 2) wait_vmcnt<DMA_PER_TILE>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of stage kt are complete
        __builtin_amdgcn_s_barrier();
        const bool split = LATE && STEADY;  // the refill moves into the MFMA stream (position by wave)
        if (!split && (STEADY || kt + GNS < KTT)) dma(kt + GNS, kt % GNS);
        __builtin_amdgcn_sched_barrier(0);
        const int nst = (kt + 1) % GNS;
        const bool more = STEADY || ahead >= 1;
        if (more) {
#pragma unroll
            for (int b = 0; b < NBW; b++) nw[b] = wfrag(nst, b);
        }
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
#pragma unroll
            for (int nb = 0; nb < NBW; nb++) acc[nb][mb] = mfma16(cw[nb], fa[mb], acc[nb][mb]);
            if (more) fa[mb] = afrag(nst, mb);
            if (split && mb == (wv >= 4 ? LATE_MB : EARLY_MB)) {
                __builtin_amdgcn_sched_barrier(0);
                dma(kt + GNS, kt % GNS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // steady steps: one operand read, then two MFMAs, in turn (the backend otherwise clusters the reads;
        // +1-1.5% on the DiT shapes)
        if constexpr (STEADY) {
#pragma unroll
            for (int i = 0; i < NBW + MB; i++) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // MFMA
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    using True = std::true_type;
    using False = std::false_type;
    int kt = 0;
    for (; kt + 1 + GNS < KTT; kt += 2) {
        step(True{}, kt, fw, gw);
        step(True{}, kt + 1, gw, fw);
    }
    for (; kt + 1 < KTT; kt += 2) {
        step(False{}, kt, fw, gw);
        step(False{}, kt + 1, gw, fw);
    }
    if (kt < KTT) step(False{}, kt, fw, gw);

    if constexpr (EPI == EPI_QKV) {
        qkv_epilogue<WAVES_N, WAVES_M, MB, 1, GNS * STAGE_H>(p, acc, lds, m0, n0, wv, wn, wm, 0, lane);
        return;
    }
    // epilogue: lane holds rows m0 + wm*16*MB + mb*16 + (lane & 15), columns n0 + wn*64 + nb*16 + 4*(lane >> 4) + e
    const int mrow = m0 + wm * 16 * MB + rl;
    const int ncol = n0 + wn * NBW * 16 + 4 * (lane >> 4);
    if (ncol >= p.N) return;  // a column range of the last tile past N (N % 256 == 128)
    floatx4 gv[NBW];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) gv[nb] = gate_of<EPI>(p, ncol + nb * 16);
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const int m = mrow + mb * 16;
        if (m >= p.M) break;
#pragma unroll
        for (int nb = 0; nb < NBW; nb++) store_out<EPI>(p, m, ncol + nb * 16, acc[nb][mb], gv[nb]);
    }
}

// Prepared weight layout: [ceil(N/256) column tiles][K/32 k tiles][16 KB block], the block holding the 256 rows
// x 32 k of the tile in the kernel's LDS order (16-byte piece q: row q >> 2, k chunk (q & 3) ^ ((row >> 1) & 3));
// rows past N are zero. The k loop's W DMA then reads one contiguous 16 KB block per k tile instead of 256 row
// segments 2 KB or more apart (measured 14-17% faster on the DiT shapes). The source is fp16 or bf16; bf16 is
// clamped to the fp16 range and rounded to nearest even (the reference's weight_to_f16, kernels.cu:531-544).
__global__ void k_gemm_wprep(_Float16* __restrict__ wp, const uint16_t* __restrict__ w, int N, int K, int src_bf16,
                             long total) {
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total) return;
    const int q = (int)(g & 1023);
    const long blk = g >> 10;
    const int KT = K / GBK;
    const int kt = (int)(blk % KT), tn = (int)(blk / KT);
    const int row = q >> 2, c = (q & 3) ^ ((row >> 1) & 3);
    const int n = tn * GBN + row;
    half8 v = {};
    if (n < N) {
        const uint16_t* src = w + (size_t)n * K + kt * GBK + c * 8;
        if (src_bf16) {
            const u32x4 raw = *reinterpret_cast<const u32x4*>(src);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint16_t b = (uint16_t)(raw[e / 2] >> (16 * (e & 1)));
                v[e] = (_Float16)fminf(fmaxf(bf16_to_f32(b), -65504.f), 65504.f);
            }
        } else {
            v = *reinterpret_cast<const half8*>(src);
        }
    }
    *reinterpret_cast<half8*>(wp + g * 8) = v;
}

size_t gemm16_prepped_bytes(int N, int K) { return (size_t)((N + GBN - 1) / GBN) * GBN * K * sizeof(_Float16); }

hipError_t launch_gemm_wprep(uint16_t* wp, const uint16_t* w, int N, int K, bool src_bf16, hipStream_t s) {
    const long total = (long)((N + GBN - 1) / GBN) * (K / GBK) * 1024;
    hipLaunchKernelGGL(k_gemm_wprep, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<_Float16*>(wp), w, N, K, src_bf16 ? 1 : 0, total);
    return hipGetLastError();
}

struct KvTailJobs {
    uint16_t* kvp[MAX_JOBS];
};
__global__ void k_kv_zero_tail(KvTailJobs j, size_t head_stride, size_t tail_off) {
    // block (item, head): 32 KB of the last tile, 16 bytes per thread and step
    _Float16* base = reinterpret_cast<_Float16*>(j.kvp[blockIdx.y]) + blockIdx.x * head_stride + tail_off;
    for (int i = threadIdx.x; i < KV_TILE_H / 8; i += blockDim.x) reinterpret_cast<half8*>(base)[i] = half8{};
}

hipError_t launch_kv_zero_tail(uint16_t* const* kvp, int njobs, int T, int H, hipStream_t s) {
    if (T % KT == 0 || njobs <= 0) return hipSuccess;
    KvTailJobs j{};
    for (int b = 0; b < njobs && b < MAX_JOBS; b++) j.kvp[b] = kvp[b];
    hipLaunchKernelGGL(k_kv_zero_tail, dim3(H, njobs), dim3(256), 0, s, j, kv_head_stride(T),
                       (size_t)(kv_tiles(T) - 1) * KV_TILE_H);
    return hipGetLastError();
}

int cu_count() {
    static int cus[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cus[dev] && hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cus[dev] = 256;
    return cus[dev];
}

template <int MB>
static hipError_t launch_mb(GemmParams p, int epi, hipStream_t s) {
    constexpr int BM = Tile<MB>::BM;
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + GBN - 1) / GBN;
    p.total = p.tiles_m * p.tiles_n;
    const int nb = (p.total + 7) / 8 * 8;
    p.per = nb / 8;
    const size_t lds = (size_t)GNS * Tile<MB>::STAGE_H * sizeof(_Float16);
    void (*kern)(GemmParams) = nullptr;
    const bool late = p.wprep != 0;
    switch (epi) {
        case KILN_EPI_F32: kern = late ? k_gemm16<KILN_EPI_F32, MB, true> : k_gemm16<KILN_EPI_F32, MB, false>; break;
        case KILN_EPI_F16: kern = late ? k_gemm16<KILN_EPI_F16, MB, true> : k_gemm16<KILN_EPI_F16, MB, false>; break;
        case KILN_EPI_GELU16:
            kern = late ? k_gemm16<KILN_EPI_GELU16, MB, true> : k_gemm16<KILN_EPI_GELU16, MB, false>;
            break;
        case KILN_EPI_RESID:
            kern = late ? k_gemm16<KILN_EPI_RESID, MB, true> : k_gemm16<KILN_EPI_RESID, MB, false>;
            break;
        case EPI_QKV: kern = late ? k_gemm16<EPI_QKV, MB, true> : k_gemm16<EPI_QKV, MB, false>; break;
        default: return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(kern, dim3(nb), dim3(GTHR), lds, s, p);
    return hipGetLastError();
}


// Activation tile height (32*MB rows, MB in {8, 7}): the one with the fewest CU rounds x rows per tile, one
// workgroup per CU. M = 6912 (the DiT's CFG batch) is 27 tiles of 256 rows, so every grid of 256-row tiles
// leaves 5/32 of the last round idle; 224-row tiles give 31 per column and fill 97%.
static int gemm16_mb(int M, int N, int cus, long* tiles) {
    const int tn = (N + GBN - 1) / GBN;
    int best = 8;
    long best_cost = -1;
    for (int mb : {8, 7}) {
        const long t = (long)((M + 32 * mb - 1) / (32 * mb)) * tn;
        const long cost = (t + cus - 1) / cus * mb;
        if (best_cost < 0 || cost < best_cost) {
            best = mb;
            best_cost = cost;
            *tiles = t;
        }
    }
    return best;
}

// Few rows leave most CUs without a 256-wide tile: M = 256 x 2048 x 2048 takes 47.1 us (39.5 with prepared weights) on this
// kernel's 8 tiles and 9.9 on 64 x 32 ones, M = 1024 54.3 (44.4) against 17.5 (128 x 64), M = 3072 56.2 (48.0) against 33.6
// (128 x 192); at M = 4608 it is 56.4 (47.3) against 58.8 (58.2). Weights from memory, fp16 out. The models meet near the
// size where the large tiles fill the chip (gemm_cost gives both sides there).
GemmTile gemm16_choose(int M, int N, int K, int epi) {
    const int cus = cu_count();
    long tiles = 0;
    const int mb = gemm16_mb(M, N, cus, &tiles);
    const SmallGemm small = gemm16s_choose(M, N, K, epi, cus);
    const double large = gemm_cost({1.54, 1.57 * mb, 0.0663 * mb, 0.0315 * mb}, tiles, K / GBK, cus);
    if (small.cost < large) return {small.cfg, small.bn, small.bm};
    return {-1, GBN, 32 * mb};
}

hipError_t launch_gemm16(const GemmLaunch& g, hipStream_t s) {
    GemmParams p;
    p.a = reinterpret_cast<const _Float16*>(g.a);
    p.w = reinterpret_cast<const _Float16*>(g.w);
    p.a2 = reinterpret_cast<const _Float16*>(g.K2 > 0 ? g.a2 : g.a);
    p.w2 = reinterpret_cast<const _Float16*>(g.K2 > 0 ? g.w2 : g.w);
    p.K = g.K;
    p.K2 = g.K2;
    p.M = g.M;
    p.N = g.N;
    p.c = g.c;
    p.ldc = g.ldc;
    p.gate = g.gate;
    p.beta = g.beta;
    const size_t esz = (g.epi == KILN_EPI_F32 || g.epi == KILN_EPI_RESID) ? 4 : 2;
    p.pairs = ((size_t)g.c % (4 * esz) != 0) || (g.ldc % 4 != 0);
    p.wprep = g.wprep ? 1 : 0;
    if (g.epi == EPI_QKV) {
        p.q16 = reinterpret_cast<_Float16*>(g.q16);
        for (int b = 0; b < MAX_JOBS; b++) p.kvp[b] = g.kvp[b];
        p.T = g.T;
        p.H = g.H;
        p.qw = g.qw;
        p.kw = g.kw;
        p.eps = g.eps;
        p.qscale = LOG2E / sqrtf((float)HD);
        p.rcos = g.rcos;
        p.rsin = g.rsin;
    }
    const GemmTile t = gemm16_choose(g.M, g.N, g.K + g.K2, g.epi);
    if (t.cfg >= 0) return launch_gemm16s(p, t.cfg, g.epi, s);
    if (t.bm == 224) return launch_mb<7>(p, g.epi, s);
    return launch_mb<8>(p, g.epi, s);
}

}  // namespace kiln
