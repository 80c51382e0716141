// The dense part in int8 (attention projections, shared experts, the LM head): one-token GEMV, the
// MFMA product of 2 to 256 tokens and the row-block dequantisation for more. Weights (O, K) int8, group scales (O, K/gs)
// fp16, symmetric (the store's int8 format).

#include "lanevec.hpp"

namespace moehip {

// ---------------------------------------------------------------------------------------
// y (O) = W x, one token. Lane groups of G = 2^lg lanes per row; a lane holds CPL chunks of 16
// int8 values (32 values) of a row segment of G * 32 values; NP row passes per wave, every
// weight and scale load of a segment issued before the first product; fp16 pairs and the
// 1024-offset dot (fp32 accumulation), the group scale per chunk. Rows and chunks past the end
// read valid memory and are dropped.
// ---------------------------------------------------------------------------------------
template <int XDT, int G8_NP>
__global__ __launch_bounds__(256) void k_gemv8(gbyte *q, gbyte *s, const void *x, void *y, int O, int K, int gs,
                                               int lg, int nseg) {
    constexpr int PREC = MOEHIP_PREC_INT8;
    constexpr int CPL = DlFmt<PREC>::CPL, VPC = DlFmt<PREC>::VPC;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int G = 1 << lg, RPW = 64 >> lg;
    const int slot = lane >> lg, cl = lane & (G - 1);
    const int C = K / VPC;                     // chunks per row
    const int CS = G * CPL;                    // chunks per segment
    const uint32_t RB = (uint32_t)K;           // bytes per row
    const int ng = K / gs;
    const int r0 = (blockIdx.x * 4 + wave) * RPW * G8_NP + slot;  // row of pass 0
    float acc[G8_NP];
#pragma unroll
    for (int p = 0; p < G8_NP; ++p) acc[p] = 0.f;
    for (int sg = 0; sg < nseg; ++sg) {
        const int c0 = sg * CS;  // first chunk of the segment
        uint4 qd[G8_NP][CPL];
        uint32_t sd[G8_NP][CPL];
        uint32_t okm = 0;
#pragma unroll
        for (int p = 0; p < G8_NP; ++p) {
            const int rr = r0 + p * RPW;
            const int r = min(rr, O - 1);
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const int cc = c0 + cl + i * G;
                const int c = min(cc, C - 1);
                okm |= (cc < C && rr < O ? 1u : 0u) << (p * CPL + i);
                qd[p][i] = gld16(q + (size_t)r * RB + (size_t)c * 16);
                sd[p][i] = gld2(s + 2 * ((size_t)r * ng + (c * VPC) / gs));
            }
        }
        LaneVec<PREC, XDT> lv;
        load_x<PREC, XDT>(reinterpret_cast<const uint8_t *>(x) + (size_t)c0 * VPC * (XDT == MOEHIP_DT_F32 ? 4 : 2),
                          cl, G, C - c0, lv);
#pragma unroll
        for (int p = 0; p < G8_NP; ++p)
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const float sc = ((okm >> (p * CPL + i)) & 1u) ? f16_to_f32(sd[p][i]) : 0.f;
                acc[p] = fmaf(sc * lv.p2e[i], lane_dot<PREC, XDT>(qd[p][i], lv, i), acc[p]);
            }
    }
    grp_total_n<G8_NP>(acc, lg);
    if (cl == G - 1)
#pragma unroll
        for (int p = 0; p < G8_NP; ++p) {
            const int r = r0 + p * RPW;
            if (r < O) st_act<XDT>(y, r, acc[p]);
        }
}

// ---------------------------------------------------------------------------------------
// y (T, O) = x W^T (+ bias) for a few tokens (a batched decode step's dense layers), straight from
// the int8 weights on MFMA: the integers are exact in fp16 and in bf16, so B = the integers in the
// activation dtype, A = the activations as they are, and each group's fp32 product sum is scaled by
// the group's scale into the fp32 accumulators (no rounding of a scaled weight).
//
// Bound by the weight stream: O * K bytes read once. One workgroup owns 32 SUB rows x 32 NM tokens;
// its 4 waves split K (pairs of 64-value groups, dealt round robin so that the four read whole
// cache lines of a row), so a small projection still gives O / 32 workgroups and no wave waits for
// another before the final sum through LDS; R groups per wave are in flight. 151936 x 2048 (311 MB,
// 61 us at 5.1 TB/s): 2 tokens 78 us, 32: 97, 64: 140 (the activations from L2 are then half of the
// bytes); dequantised into memory for a library product it took 560 at any of these. The passes of a row
// tile over the tokens run on one XCD, one after the other (its L2 serves the re-reads).
// v_mfma_f32_32x32x16: A lane (token i, half h) holds K h * 32 + 8 m .. + 7 of a group at step m,
// B lane (row j, half h) the same K; D: lane (row j, half), element r = token 8 (r / 4) + 4 half + r % 4.
// ---------------------------------------------------------------------------------------
typedef _Float16 d_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 d_bf16x8 __attribute__((ext_vector_type(8)));
typedef float d_f32x16 __attribute__((ext_vector_type(16)));

// 8 int8 values as 8 activation-dtype values, natural order
template <int XDT>
__device__ __forceinline__ uint4 i8_to_act(uint32_t lo, uint32_t hi) {
    uint32_t r[4];
    if constexpr (XDT == MOEHIP_DT_F16) {
        // bytes 2i, 2i + 1 into the low bytes of two halves, fp16 1024 + q + 128, - 1152 (exact)
        const half2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = __builtin_amdgcn_perm(0u, i < 2 ? lo : hi, (i & 1) ? 0x0C030C02u : 0x0C010C00u) ^ 0x64806480u;
            r[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, u) + off);
        }
    } else {
        // an integer of 8 bits is exact in bf16: the high halves of the fp32 values
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = i < 2 ? lo : hi;
            const float a = (float)(int8_t)(w >> (16 * (i & 1))), b = (float)(int8_t)(w >> (16 * (i & 1) + 8));
            r[i] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
        }
    }
    return make_uint4(r[0], r[1], r[2], r[3]);
}

template <int XDT>
__device__ __forceinline__ d_f32x16 d_mfma(uint4 a, uint4 b, d_f32x16 c) {
    if constexpr (XDT == MOEHIP_DT_F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(d_f16x8, a), __builtin_bit_cast(d_f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(d_bf16x8, a), __builtin_bit_cast(d_bf16x8, b), c, 0, 0, 0);
}

template <int XDT, int NM, int SUB, int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NM * SUB == 1 ? 3 : 2, NM * SUB == 1 ? 3 : 2))) void k_dense8(
    gbyte *q, gbyte *s, gbyte *x, const uint16_t *bias, uint16_t *y, int T, int O, int K, int npass) {
    __shared__ float red[4][SUB * NM * 1024];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
    const int b = blockIdx.x, tile = b / (8 * npass) * 8 + (b & 7), pass = (b >> 3) % npass;
    const int row0 = tile * 32 * SUB, t0 = pass * 32 * NM;
    if (row0 >= O) return;  // tiles are padded to a multiple of 8
    const int ng = K / 64;
    gbyte *qb = q + (size_t)row0 * K, *sb = s + (size_t)row0 * ng * 2;
    uint32_t qo[SUB], so[SUB];
    gbyte *xr[NM];
#pragma unroll
    for (int t = 0; t < SUB; ++t) {  // rows past the end repeat the last one and are not stored
        const uint32_t r = (uint32_t)min(32 * t + j, O - 1 - row0);
        qo[t] = r * (uint32_t)K + 32u * h;
        so[t] = r * (uint32_t)ng * 2u;
    }
#pragma unroll
    for (int m = 0; m < NM; ++m) xr[m] = x + ((size_t)min(t0 + 32 * m + j, T - 1) * K + 32 * h) * 2;
    uint4 wq[R][SUB][2], xa[R][NM][4];
    uint32_t ws[R][SUB];
    // the wave's n-th group; past the end the last group is loaded again and not used
    auto group = [&](int n) { return 8 * (n >> 1) + 2 * wave + (n & 1); };
    auto load = [&](int u, int n) {
        const int g = min(group(n), ng - 1);
#pragma unroll
        for (int t = 0; t < SUB; ++t) {
            wq[u][t][0] = gld16(qb + (size_t)g * 64 + qo[t]);
            wq[u][t][1] = gld16(qb + (size_t)g * 64 + qo[t] + 16);
            ws[u][t] = gld2(sb + (size_t)g * 2 + so[t]);
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int c = 0; c < 4; ++c) xa[u][m][c] = gld16(xr[m] + (size_t)g * 128 + 16 * c);
    };
    d_f32x16 acc[NM][SUB];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int t = 0; t < SUB; ++t) acc[m][t] = d_f32x16{};
    auto compute = [&](int u) {
#pragma unroll
        for (int t = 0; t < SUB; ++t) {
            uint4 bw[4];
            const uint4 w0 = wq[u][t][0], w1 = wq[u][t][1];
            bw[0] = i8_to_act<XDT>(w0.x, w0.y);
            bw[1] = i8_to_act<XDT>(w0.z, w0.w);
            bw[2] = i8_to_act<XDT>(w1.x, w1.y);
            bw[3] = i8_to_act<XDT>(w1.z, w1.w);
            const float sc = f16_to_f32(ws[u][t]);
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                d_f32x16 p = d_f32x16{};
#pragma unroll
                for (int c = 0; c < 4; ++c) p = d_mfma<XDT>(xa[u][m][c], bw[c], p);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[m][t][r] = fmaf(sc, p[r], acc[m][t][r]);
            }
        }
    };
    // groups of this wave: 2 per full round of 8, and what the last round leaves it
    const int N = ng / 8 * 2 + max(0, min(2, ng % 8 - 2 * wave));
#pragma unroll
    for (int u = 0; u < R; ++u) load(u, u);
    int n0 = 0;
#pragma unroll 1
    for (; n0 + R < N; n0 += R)
#pragma unroll
        for (int u = 0; u < R; ++u) {
            compute(u);
            load(u, n0 + u + R);
        }
#pragma unroll
    for (int u = 0; u < R; ++u)
        if (n0 + u < N) compute(u);
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int t = 0; t < SUB; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[wave][((m * SUB + t) * 16 + r) * 64 + lane] = acc[m][t][r];
    __syncthreads();
    for (int i = threadIdx.x; i < SUB * NM * 1024; i += 256) {
        const int l = i & 63, r = (i >> 6) & 15, mt = i >> 10;
        const int tok = t0 + 32 * (mt / SUB) + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), row = row0 + 32 * (mt % SUB) + (l & 31);
        if (tok >= T || row >= O) continue;
        float v = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
        if (bias != nullptr) v += ld_act<XDT>(bias, row);
        st_act<XDT>(y, (size_t)tok * O + row, v);
    }
}

// ---------------------------------------------------------------------------------------
// W (rows [r0, r0 + n), K) in the activation dtype: q * round(s), rounded once (as the store's
// dequantisation in that dtype); 16 values per thread, stored 16 bytes at a time
// ---------------------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(256) void k_dequant8(gbyte *q, gbyte *s, int n, int K, int gs, void *w) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t nchunk = (size_t)n * (K / 16);
    if (t >= nchunk) return;
    const size_t r = t / (size_t)(K / 16);
    const int c = (int)(t - r * (size_t)(K / 16));
    const uint4 v = gld16(q + t * 16);
    const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
    const int ng = K / gs;
    float out[16];
    const bool one = gs % 16 == 0;  // the 16 values are in one group
    float sc = f16_to_f32(gld2(s + 2 * (r * ng + c * 16 / gs)));
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (!one) sc = f16_to_f32(gld2(s + 2 * (r * ng + (c * 16 + j) / gs)));
        const int qv = (int)(int8_t)((wd[j >> 2] >> (8 * (j & 3))) & 0xffu);
        out[j] = (float)qv * (DT == MOEHIP_DT_BF16 ? rnd_act<MOEHIP_DT_BF16>(sc) : sc);
    }
    if (((uintptr_t)w & 15) != 0) {  // (a caller's unaligned buffer)
#pragma unroll
        for (int j = 0; j < 16; ++j) st_act<DT>(w, t * 16 + j, out[j]);
        return;
    }
    constexpr int NV = DT == MOEHIP_DT_F32 ? 4 : 2;  // 16-byte stores
    uint32_t d[4 * NV];
#pragma unroll
    for (int j = 0; j < 4 * NV; ++j) {
        if constexpr (DT == MOEHIP_DT_F32) d[j] = __float_as_uint(out[j]);
        else if constexpr (DT == MOEHIP_DT_F16) d[j] = pack_h2(out[2 * j], out[2 * j + 1]);
        else d[j] = (uint32_t)f32_to_bf16_rne(out[2 * j]) | ((uint32_t)f32_to_bf16_rne(out[2 * j + 1]) << 16);
    }
    uint4 *dst = reinterpret_cast<uint4 *>(w) + t * NV;
#pragma unroll
    for (int j = 0; j < NV; ++j) dst[j] = make_uint4(d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]);
}

}  // namespace moehip

using namespace moehip;

static bool dense_dt(int d) { return d >= MOEHIP_DT_F16 && d <= MOEHIP_DT_F32; }

extern "C" int moehip_dense_gemv_int8(const void *q, const void *s, const void *x, void *y, int O, int K, int gs,
                                      int dtype, void *stream) {
    MOEHIP_REQUIRE(q && s && x && y, "dense_gemv_int8: null pointer");
    MOEHIP_REQUIRE(dense_dt(dtype), "dense_gemv_int8: bad dtype %d", dtype);
    MOEHIP_REQUIRE(O > 0 && K > 0 && K % 32 == 0 && gs > 0 && gs % 16 == 0 && K % gs == 0,
                   "dense_gemv_int8: O=%d K=%d gs=%d (K a multiple of 32, gs of 16 dividing K)", O, K, gs);
    MOEHIP_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)x % 16) == 0,
                   "dense_gemv_int8: q and x must be 16-byte aligned");
    const int chunks = K / 16, cpl = 2;
    int G = 1, lg = 0;
    while (G < (chunks + cpl - 1) / cpl && G < 64) G <<= 1, ++lg;
    const int nseg = (chunks + G * cpl - 1) / (G * cpl);
    // row passes per wave: 4, unless the grid would then hold fewer than 2 workgroups per CU (a
    // small matrix: an attention projection, a shared expert), where 2 or 1 give more workgroups
    int cus = 256;
    {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            n > 0)
            cus = n;
    }
    int np = 1;
    for (int cand : {4, 2})
        if ((O + 4 * (64 >> lg) * cand - 1) / (4 * (64 >> lg) * cand) >= 2 * cus) {
            np = cand;
            break;
        }
    const int rows_per_block = 4 * (64 >> lg) * np;
    const dim3 grid((unsigned)((O + rows_per_block - 1) / rows_per_block));
    hipStream_t st = as_stream(stream);
    gbyte *qb = (gbyte *)(uintptr_t)q, *sb = (gbyte *)(uintptr_t)s;
#define G8_LAUNCH(DT, NP) hipLaunchKernelGGL((k_gemv8<DT, NP>), grid, dim3(256), 0, st, qb, sb, x, y, O, K, gs, lg, nseg)
#define G8_NPS(DT)           \
    if (np == 4)             \
        G8_LAUNCH(DT, 4);    \
    else if (np == 2)        \
        G8_LAUNCH(DT, 2);    \
    else                     \
        G8_LAUNCH(DT, 1)
    switch (dtype) {
        case MOEHIP_DT_F16: G8_NPS(MOEHIP_DT_F16); break;
        case MOEHIP_DT_BF16: G8_NPS(MOEHIP_DT_BF16); break;
        default: G8_NPS(MOEHIP_DT_F32); break;
    }
#undef G8_NPS
#undef G8_LAUNCH
    return check_launch("dense_gemv_int8");
}

extern "C" int moehip_dense_gemm_int8(const void *q, const void *s, const void *x, const void *bias, void *y, int T,
                                      int O, int K, int gs, int dtype, void *stream) {
    MOEHIP_REQUIRE(q && s && x && y, "dense_gemm_int8: null pointer");
    MOEHIP_REQUIRE(dtype == MOEHIP_DT_F16 || dtype == MOEHIP_DT_BF16, "dense_gemm_int8: dtype %d (fp16 or bf16)", dtype);
    MOEHIP_REQUIRE(T > 0 && O > 0 && K > 0 && K % 64 == 0 && gs == 64, "dense_gemm_int8: T=%d O=%d K=%d gs=%d (K a multiple of 64, gs = 64)",
                   T, O, K, gs);
    MOEHIP_REQUIRE((uint64_t)K < (1u << 25), "dense_gemm_int8: K=%d (a tile's row offsets are 32 bits)", K);
    MOEHIP_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)x % 16) == 0, "dense_gemm_int8: q and x must be 16-byte aligned");
    hipStream_t st = as_stream(stream);
    gbyte *qb = (gbyte *)(uintptr_t)q, *sb = (gbyte *)(uintptr_t)s, *xb = (gbyte *)(uintptr_t)x;
    const int nm = T <= 32 ? 1 : 2, npass = (T + 32 * nm - 1) / (32 * nm);
    // Rows per workgroup: as many as leave the chip full, since every workgroup reads the tokens'
    // activations once (32 tokens x 2048 values are as many bytes as 64 weight rows). Measured at
    // O x 2048 (us): 151936 rows, 2 / 16 / 32 tokens: 32 rows 85 / 113 / 129, 64 rows 78 / 92 / 105,
    // 128 rows 82 / 90 / 97; 50304 rows, 32 tokens: 47 / 45 / 41; 8192 rows: 13 / 14 / 22.
    int sub;
    if (nm == 1 && T > 16 && (O + 127) / 128 >= 256) sub = 4;
    else sub = (O + 63) / 64 * npass >= 512 ? 2 : 1;
    const int tiles = ((O + 32 * sub - 1) / (32 * sub) + 7) / 8 * 8;
    const dim3 grid((unsigned)(tiles * npass));
#define D8(DT, NM, SUB, R) hipLaunchKernelGGL((k_dense8<DT, NM, SUB, R>), grid, dim3(256), 0, st, qb, sb, xb, \
                                              reinterpret_cast<const uint16_t *>(bias), reinterpret_cast<uint16_t *>(y), T, O, K, npass)
#define D8_DT(DT)                                                     \
    if (nm == 1 && sub == 4) D8(DT, 1, 4, 2);                         \
    else if (nm == 1 && sub == 1) D8(DT, 1, 1, 4);                         \
    else if (nm == 1) D8(DT, 1, 2, 4);                                \
    else if (sub == 1) D8(DT, 2, 1, 2);                               \
    else D8(DT, 2, 2, 2)
    if (dtype == MOEHIP_DT_F16) {
        D8_DT(MOEHIP_DT_F16);
    } else {
        D8_DT(MOEHIP_DT_BF16);
    }
#undef D8_DT
#undef D8
    return check_launch("dense_gemm_int8");
}

extern "C" int moehip_dense_dequant_int8(const void *q, const void *s, int rows, int K, int gs, int dtype, void *w,
                                         void *stream) {
    MOEHIP_REQUIRE(q && s && w, "dense_dequant_int8: null pointer");
    MOEHIP_REQUIRE(dense_dt(dtype), "dense_dequant_int8: bad dtype %d", dtype);
    MOEHIP_REQUIRE(rows > 0 && K > 0 && K % 16 == 0 && gs > 0 && K % gs == 0,
                   "dense_dequant_int8: rows=%d K=%d gs=%d (K a multiple of 16)", rows, K, gs);
    MOEHIP_REQUIRE(((uintptr_t)q % 16) == 0, "dense_dequant_int8: q must be 16-byte aligned");
    const size_t nchunk = (size_t)rows * (K / 16);
    const dim3 grid((unsigned)((nchunk + 255) / 256));
    hipStream_t st = as_stream(stream);
    gbyte *qb = (gbyte *)(uintptr_t)q, *sb = (gbyte *)(uintptr_t)s;
    switch (dtype) {
        case MOEHIP_DT_F16: hipLaunchKernelGGL(k_dequant8<MOEHIP_DT_F16>, grid, dim3(256), 0, st, qb, sb, rows, K, gs, w); break;
        case MOEHIP_DT_BF16: hipLaunchKernelGGL(k_dequant8<MOEHIP_DT_BF16>, grid, dim3(256), 0, st, qb, sb, rows, K, gs, w); break;
        default: hipLaunchKernelGGL(k_dequant8<MOEHIP_DT_F32>, grid, dim3(256), 0, st, qb, sb, rows, K, gs, w); break;
    }
    return check_launch("dense_dequant_int8");
}
