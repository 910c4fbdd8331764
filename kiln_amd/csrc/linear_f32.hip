// fp32 linear layers with bf16 weights on the bf16 matrix cores (gfx950), as exact as on the fp32 ones.
//
// Contract: the reference's linear (engine/src/kernels.cu:508-529): y [T, rows] = x [T, cols] W^T, x and y fp32, W bf16
// [rows, cols]. An fp32 value is the sum of three bf16 values with no remainder (24 significand bits, 8 + 8 + 8, cut
// off by truncation), and a product of two bf16 values is exact in fp32, so x W^T = x1 W^T + x2 W^T + x3 W^T holds
// term by term: what is left is the rounding of fp32 sums, as in v_mfma_f32_16x16x4_f32, and there are fewer of
// them. Three v_mfma_f32_16x16x32_bf16 do the work of eight v_mfma_f32_16x16x4_f32 in 3/16 of their cycles.
// It is 2^24 x that is split, and the sums are scaled back: the last bit of any fp32 value (2^-149) then lies in
// bf16's normal range, where without the scale the third part of |x| < 2^-110 is cut. (1 to 3% of the time: T = 1024,
// 2048 x 2048 30.1 -> 30.6 us, x 8192 100.0 -> 102.9; T = 6912, 8192 x 2048 556 -> 560.)
//
//  * transposed product (C^T = W x^T): the MFMA's A operand is a 16-row block of W, its B operand 16 rows of x1, x2 or
//    x3; each lane ends with 4 consecutive output columns of one row.
//  * workgroup tile 64*WN weight rows x 16*MB*WM rows of x; 8 waves in KG groups of WN x WM that share the k range (a
//    step is SL = KG*KS slices of 32 k; the groups' sums meet in LDS after the loop), so that a context of a hundred
//    tokens or the 64-column final layer still keeps every wave busy.
//  * W goes global -> LDS by DMA; x through registers, where it is split once per tile, into three bf16 planes in LDS.
//    Two stages: step s + 1 is split and stored, and step s + 2 of x loaded, while step s is multiplied.
//  * an infinite or NaN sum is recomputed in plain fp32: 2^24 x or its sum past fp32's range (|x| >= 2^104), or 0 x inf
//    in a term that fp32 arithmetic would not have (a zero remainder against an infinite weight).
//  * a subnormal weight (below 2^-126) counts with 17 to 24 bits, as the matrix cores align its products.
#include "gemm16.hpp"

namespace kiln {

constexpr int XTHR = 512;
constexpr float X_UP = 0x1p24f, X_DOWN = 0x1p-24f;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

struct LinearParams {
    float* y;
    const float* x;
    const uint16_t* w;
    int ldy, ldx, T, rows, cols;
    int tiles_m, tiles_n, total, per;
    int vec;  // y rows and base 16-byte aligned
};

template <int WN_, int WM_, int MB_, int KG_, int KS_>
struct XCfg {
    static constexpr int WN = WN_, WM = WM_, MB = MB_, KG = KG_, KS = KS_;
    static constexpr int BN = 64 * WN, BM = 16 * MB * WM, SL = KG * KS;
    static constexpr int W_BYTES = SL * BN * 64, P_BYTES = SL * BM * 64, STAGE = W_BYTES + 3 * P_BYTES;
    static constexpr int W_DMA = W_BYTES / 16 / XTHR, X_LD = P_BYTES / 16 / XTHR;  // 16-byte pieces per thread
    static constexpr int RED = KG > 1 ? XTHR / 64 * NBW * MB * 1024 : 0;
    static constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
    static_assert(WN * WM * KG * 64 == XTHR && SL % 2 == 0 && LDS <= 160 * 1024, "8 waves, whole 128-byte W rows");
    static_assert(W_DMA * 16 * XTHR == W_BYTES && X_LD * 16 * XTHR == P_BYTES, "every thread copies whole pieces");
};

template <class C>
__global__ __launch_bounds__(XTHR, 1) void k_linear_x3(const LinearParams p) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass only needs the kernel's handle
    constexpr int WN = C::WN, WM = C::WM, MB = C::MB, KG = C::KG, KS = C::KS, SL = C::SL, BN = C::BN, BM = C::BM;
    constexpr int X_LD = C::X_LD;
    extern __shared__ __attribute__((aligned(16))) char smem[];  // 2 stages of [W slices | x1 | x2 | x3 slices]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wv / (WN * WM), wn = wv % (WN * WM) / WM, wm = wv % WM;
    const int i = (int)(blockIdx.x & 7) * p.per + (int)(blockIdx.x >> 3);  // XCD b % 8: a contiguous range of tiles
    if (i >= p.total) return;
    int tm, tn;
    raster_tile(i, 8, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int mrows = min(BM, p.T - m0), nrows = min(BN, p.rows - n0);
    const int KT = p.cols / 32, S = (KT + SL - 1) / SL;

    // W: 16-byte pieces q = tid + XTHR*r: pair of slices q / (8 BN), row (q >> 3) % BN, LDS position q & 7 holding
    // chunk (q & 7) ^ (row & 7). Rows past the matrix re-read its last one, slices past the last (`have` of the
    // step's are real) the step's first: neither is used.
    auto w_off = [&](int r, int have) {
        const int q = tid + XTHR * r, row = (q >> 3) % BN, c = (q & 7) ^ (row & 7);
        const bool in = 2 * (q / (8 * BN)) + (c >> 2) < have;
        return (uint32_t)(min(row, nrows - 1) * p.cols * 2 + (in ? q / (8 * BN) * 128 + c * 16 : (c & 3) * 16));
    };
    uint32_t voff_w[C::W_DMA];
#pragma unroll
    for (int r = 0; r < C::W_DMA; r++) voff_w[r] = w_off(r, SL);
    const __amdgpu_buffer_rsrc_t rw =
        GEMM_RSRC(reinterpret_cast<const _Float16*>(p.w) + (size_t)n0 * p.cols, (size_t)nrows * p.cols * 2);
    typedef __attribute__((address_space(3))) void* lds_p;
    auto dma_w = [&](int st, int stage) {
        char* base = smem + stage * C::STAGE + wv * 1024;
        const int so = st * SL * 64, have = KT - st * SL;
#pragma unroll
        for (int r = 0; r < C::W_DMA; r++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_p)(base + XTHR * 16 * r), 16,
                                                     have >= SL ? voff_w[r] : w_off(r, have), so, 0, 0);
    };
    // x: pieces of 8 floats, q = tid + XTHR*r: slice q / (4 BM), row (q >> 2) % BM, octet q & 3
    floatx4 xr[X_LD][2];
    auto load_x = [&](int st) {
#pragma unroll
        for (int r = 0; r < X_LD; r++) {
            const int q = tid + XTHR * r, row = min((q >> 2) % BM, mrows - 1);
            const int s = min(st * SL + q / (4 * BM), KT - 1);
            const float* src = p.x + (size_t)(m0 + row) * p.ldx + s * 32 + (q & 3) * 8;
            xr[r][0] = *reinterpret_cast<const floatx4*>(src);
            xr[r][1] = *reinterpret_cast<const floatx4*>(src + 4);
        }
    };
    const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)smem;
    // 2^24 x = x1 + x2 + x3, each the upper half of an fp32 word; 64-byte plane rows, octet c of row r at c ^ ((r >> 1) & 3)
    auto split_x = [&](int stage) {
#pragma unroll
        for (int r = 0; r < X_LD; r++) {
            const int q = tid + XTHR * r, row = (q >> 2) % BM, c = (q & 3) ^ ((row >> 1) & 3);
            u32x4 pl[3];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                uint32_t a[3], b[3];
                auto cut = [&](float v, uint32_t(&o)[3]) {
                    v *= X_UP;
#pragma unroll
                    for (int t = 0; t < 3; t++) {
                        o[t] = __float_as_uint(v);
                        v -= __uint_as_float(o[t] & 0xffff0000u);
                    }
                };
                cut(xr[r][e / 4][e % 4], a);
                cut(xr[r][e / 4][e % 4 + 1], b);
#pragma unroll
                for (int t = 0; t < 3; t++) pl[t][e / 2] = __builtin_amdgcn_perm(b[t], a[t], 0x07060302);  // the upper halves
            }
            const uint32_t at = lds_base + stage * C::STAGE + C::W_BYTES + q / (4 * BM) * BM * 64 + row * 64 + c * 16;
#pragma unroll
            for (int t = 0; t < 3; t++) *reinterpret_cast<lds_u32x4*>((size_t)(at + t * C::P_BYTES)) = pl[t];
        }
    };

    const int rl = lane & 15, g = lane >> 4;
    auto read = [&](uint32_t a) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const lds_u32x4*>((size_t)a)); };
    floatx4 acc[NBW][MB];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[nb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](uint32_t sb, int have) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int s = kg * KS + ks;
            if (s >= have) break;
            bf16x8 fw[NBW];
#pragma unroll
            for (int nb = 0; nb < NBW; nb++)
                fw[nb] = read(sb + (s >> 1) * BN * 128 + (wn * 64 + nb * 16 + rl) * 128 + (((4 * (s & 1) + g) ^ (rl & 7)) * 16));
            bf16x8 fx[MB][3];
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                const uint32_t at = sb + C::W_BYTES + s * BM * 64 + ((wm * MB + mb) * 16 + rl) * 64 + ((g ^ ((rl >> 1) & 3)) * 16);
#pragma unroll
                for (int t = 2; t >= 0; t--) fx[mb][t] = read(at + t * C::P_BYTES);
            }
            __builtin_amdgcn_sched_barrier(0);  // every operand read in flight before the first MFMA waits for one
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int t = 2; t >= 0; t--)  // the smallest terms first
#pragma unroll
                    for (int nb = 0; nb < NBW; nb++)
                        acc[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[nb], fx[mb][t], acc[nb][mb], 0, 0, 0);
        }
    };

    load_x(0);
    dma_w(0, 0);
    split_x(0);
    if (S > 1) load_x(1);
    for (int st = 0; st < S; st++) {
        // stage st & 1 is whole: this wave's W pieces (the X_LD*2 loads of x after them may be in flight) and plane
        // writes; the barrier extends that to every wave, and every wave is done with the other stage
        if (st + 1 < S) wait_vmcnt<2 * X_LD>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t sb = lds_base + (st & 1) * C::STAGE;
        const int have = KT - st * SL;
        if (st + 1 < S) {
            split_x((st + 1) & 1);
            dma_w(st + 1, (st + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (st + 2 < S) load_x(st + 2);
        }
        compute(sb, have);
        __builtin_amdgcn_sched_barrier(0);
    }

    constexpr int MBO = (MB + KG - 1) / KG;
    floatx4 out[NBW][MBO];
    merge_k_groups<WN * WM, MB, KG>(acc, out, reinterpret_cast<floatx4*>(smem), wv, kg, lane);
#pragma unroll
    for (int j = 0; j < MBO; j++) {
        const int mb = kg + KG * j, m = m0 + (wm * MB + mb) * 16 + rl;
        if (mb >= MB || m >= p.T) break;
#pragma unroll
        for (int nb = 0; nb < NBW; nb++) {
            const int n = n0 + wn * 64 + nb * 16 + 4 * g;
            floatx4 v = out[nb][j] * X_DOWN;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if ((__float_as_uint(v[e]) & 0x7fffffffu) >= 0x7f800000u && n + e < p.rows) {  // infinite or NaN
                    const float* xrow = p.x + (size_t)m * p.ldx;
                    const uint16_t* wrow = p.w + (size_t)(n + e) * p.cols;
                    float s = 0.f;  // a NaN stays one: no need to walk the rest of the row
                    // (unrolled in full, these loops make the code of 256 x 128 tiles 10% slower where no NaN is)
                    for (int k0 = 0; k0 < p.cols && (__float_as_uint(s) & 0x7fffffffu) <= 0x7f800000u; k0 += 32)
#pragma unroll 4
                        for (int k = k0; k < k0 + 32; k++) s = fmaf(xrow[k], bf16_to_f32(wrow[k]), s);
                    v[e] = s;
                }
            float* dst = p.y + (size_t)m * p.ldy + n;
            if (p.vec && n + 3 < p.rows) {
                *reinterpret_cast<floatx4*>(dst) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < p.rows) dst[e] = v[e];
            }
        }
    }
#endif
}

//            WN WM MB KG KS    tile (n x m), k per step
using X0 = XCfg<4, 2, 4, 1, 2>;  // 256 x 128, 64
using X1 = XCfg<2, 2, 4, 2, 1>;  // 128 x 128, 64
using X2 = XCfg<2, 1, 4, 4, 1>;  // 128 x 64, 128
using X3 = XCfg<2, 1, 2, 4, 1>;  // 128 x 32, 128
using X4 = XCfg<1, 1, 2, 8, 1>;  //  64 x 32, 256

template <class C>
static hipError_t launch_x3(LinearParams p, hipStream_t s) {
    p.tiles_m = (p.T + C::BM - 1) / C::BM;
    p.tiles_n = (p.rows + C::BN - 1) / C::BN;
    p.total = p.tiles_m * p.tiles_n;
    const int nb = (p.total + 7) / 8 * 8;
    p.per = nb / 8;
    hipLaunchKernelGGL(k_linear_x3<C>, dim3(nb), dim3(XTHR), C::LDS, s, p);
    return hipGetLastError();
}

// W's DMA has 32-bit offsets in a tile of up to 256 rows: 256 * cols * 2 bytes below 2 GiB.
// One or two slices of k are less than this form's own start and end (LDS, 8 waves, the k groups' merge): k_linear_f32
// takes them, us, here / there: T = 1, 64 x 32 4.06 / 2.61, 2048 x 32 4.24 / 3.08, 64 x 64 4.14 / 3.41, 2048 x 64 4.26 /
// 3.98; T = 1000, 64 x 32 4.47 / 3.40, 2048 x 32 6.48 / 5.15; T = 4096, 64 x 64 4.68 / 4.62. Past 2^21 outputs, or at 64
// columns from a few rows of both on, this form is as fast or faster: T = 2048, 2048 x 32 8.32 / 8.83; T = 16, 2048 x 64
// 4.25 / 4.39; T = 64, 128 x 64 4.31 / 4.36.
bool linear_x3_takes(const float* x, int ldx, const uint16_t* W, int T, int rows, int cols) {
    if (cols <= 64 && (size_t)T * rows <= (1 << 21) && (cols <= 32 || rows <= 64 || T <= 4)) return false;
    return cols % 32 == 0 && cols < (1 << 22) && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)W & 15) == 0;
}

// The tile with the smallest modelled time (gemm_cost; fitted to measured times of every tile at T = 8 .. 6912 and the
// DiT's widths, 6 to 12% off at most, its choice the measured best at all of them). us, v_mfma_f32_16x16x4_f32 ->
// here: T = 120, 2048 x 1024 44.9 -> 9.8; T = 1024, 2048 x 2048 92.0 -> 30.6; T = 6912, 8192 x 2048 1840 -> 560 (414
// TFLOP/s against the 154 of a large fp32 matrix product); T = 6912, 64 x 2048 61.2 -> 16.4. Error against 64 bits
// (2-norm, K = 2048): 8.1e-7 -> 1.7e-7 to 4.8e-7.
LinearTile linear_x3_choose(int T, int rows, int cols) {
    static const struct {
        int bn, bm;
        GemmCost c;
    } cfg[] = {{256, 128, {0.00, 5.24, 1.015, 0.213}},
               {128, 128, {1.78, 3.73, 0.616, 0.118}},
               {128, 64, {2.13, 2.70, 0.328, 0.070}},
               {128, 32, {1.97, 1.75, 0.200, 0.037}},
               {64, 32, {2.51, 1.90, 0.119, 0.029}}};
    LinearTile best{};
    double best_cost = 0;
    for (int i = 0; i < 5; i++) {
        const long tiles = (long)((T + cfg[i].bm - 1) / cfg[i].bm) * ((rows + cfg[i].bn - 1) / cfg[i].bn);
        const double t = gemm_cost(cfg[i].c, tiles, cols / 32, cu_count());
        if (i == 0 || t < best_cost) best = {i, cfg[i].bn, cfg[i].bm}, best_cost = t;
    }
    return best;
}

hipError_t launch_linear_x3(float* y, int ldy, const float* x, int ldx, const uint16_t* W, int T, int rows, int cols,
                            hipStream_t s) {
    LinearParams p{};
    p.y = y, p.x = x, p.w = W;
    p.ldy = ldy, p.ldx = ldx, p.T = T, p.rows = rows, p.cols = cols;
    p.vec = ldy % 4 == 0 && ((uintptr_t)y & 15) == 0;
    switch (linear_x3_choose(T, rows, cols).cfg) {
        case 0: return launch_x3<X0>(p, s);
        case 1: return launch_x3<X1>(p, s);
        case 2: return launch_x3<X2>(p, s);
        case 3: return launch_x3<X3>(p, s);
        default: return launch_x3<X4>(p, s);
    }
}

}  // namespace kiln
