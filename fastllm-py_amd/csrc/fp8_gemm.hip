// FP8-E4M3 128x128-block matmul above 16 rows (K % 64 == 0): decode batches of
// 17..64 rows and the prefill GEMM.
//
//   C[M, N] = A[M, K] @ (codes * block scale)^T (+ bias), A and C fp16 or bf16
#include "fp8_gemm.cuh"
#include "fp8_codec.cuh"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <bool BF16>
FL_DEV f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    if (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8>(a), bitcast<bf16x8>(b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(bitcast<f16x8>(a), bitcast<f16x8>(b), c, 0, 0, 0);
}

// One workgroup = KB k-groups on a tile of 32 MT WM rows x 32 NT WN columns.
// K-group g takes the 128-k blocks g, g + KB, ...; its WM x WN x KS waves
// share a two-stage LDS ring of the block's activations (32 MT WM x 256 B)
// and codes (32 NT WN x 128 B), KS of them splitting the block's k.
//
// Every copy brings whole 128-byte lines (4 activation rows or 8 code rows;
// the codes are row-major, so a wave's own fragment loads would touch 64
// sixteen-byte pieces per KB).  Activation chunk c of row r sits at c ^ (r %
// 16), code chunk c of row r at c ^ (r / 2 % 8): fragment reads hit all banks.
// Lane (column lc, half hi) reads 16 codes of k 32 p + 16 hi; they make two
// 32x32x16 MFMA operands (k + 0..7, + 8..15), converted exactly, and the
// block's fp32 partial takes the block scale.
//
// Bound at large M by LDS: the 128 x 256 tile of 64 x 64 waves reads 128 KB
// of activations and 64 KB of codes and writes 64 KB per block, about the
// time of its MFMAs (128 x 32 waves read twice the activations: N10944 K2048
// M2000 108 against 95 us).  The partial beside the accumulators keeps a wave
// from larger tiles, and a stage of 64 KB one workgroup per CU.
//
// Rows past M, columns past N and the second half of a trailing 64-wide block
// read zeros (offsets past the buffers), as do blocks past the end, which are
// not computed.
template <bool BF16, int MT, int NT, int WM, int WN, int KS, int KB>
__global__ __launch_bounds__(64 * WM * WN * KS * KB, (WM * WN * KS * KB <= 8 ? 2 : WM * WN * KS * KB / 4)) void fp8_gemm_wide(
    const uint16_t* __restrict__ A, const uint8_t* __restrict__ W, const float* __restrict__ Sc,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ C, int M, int N, int K) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, NT_W = WM * WN, NW = NT_W * KS, KG = KS * KB;
    constexpr int kStage = BM * 256 + BN * 128;
    constexpr int CA = (BM / 4 + NW - 1) / NW, CB = (BN / 8 + NW - 1) / NW;  // copies of a wave and block
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / NW, wg = wave % NW, ks = wg / NT_W, wt = wg % NT_W, wm = wt / WN, wn = wt % WN;
    const int lc = lane & 31, hi = lane >> 5;
    const int nkb = (K + 127) >> 7, nks = nkb;

    constexpr int gm = 4;  // tile order as in int4_gemm.hip: four row tiles by all column tiles, XCD by XCD
    const int mblk = (M + BM - 1) / BM, nblk = (N + BN - 1) / BN;
    const int total = mblk * nblk;
    int lin = blockIdx.x;
    if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
    const int grp = lin / (gm * nblk), first = grp * gm;
    const int rows = mblk - first < gm ? mblk - first : gm;
    const int in = lin - grp * gm * nblk;
    const int nb_i = in / rows, mb_i = first + in - nb_i * rows;
    const int m0 = mb_i * BM, nb0 = nb_i * BN, n0 = nb0 + wn * 32 * NT;

    const i32x4_t rA = raw_rsrc(A, (uint32_t)M * K * 2);
    const i32x4_t rW = raw_rsrc(W, (uint32_t)N * K);
    const __amdgpu_buffer_rsrc_t rS = buf_rsrc(Sc, (uint32_t)((N + 127) >> 7) * nks * 4);
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem + kg * 2 * kStage;
    constexpr uint32_t kOut = 0x80000000u;

    uint32_t ao[4], ah[4], bo[2], bh[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * (wg * CA + i) + (lane >> 4), c = (lane & 15) ^ (r & 15);
        ao[i] = 2u * ((uint32_t)(m0 + r) * K) + 16u * c;
        ah[i] = c >= 8 ? kOut : 0u;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 8 * (wg * CB + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        bo[i] = (uint32_t)(nb0 + r) * K + 16u * c;
        bh[i] = c >= 4 ? kOut : 0u;
    }
    uint32_t so[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        int n = n0 + 32 * t;
        n = n < N ? n : N - 1;
        so[t] = 4u * (uint32_t)(n >> 7) * nks;
    }
    auto copy = [&](int kb, int slot) {
        const uint32_t oob = kb < nkb ? 0u : kOut;
        const bool tail = (K & 127) && kb == nkb - 1;  // half a block: the second half reads zeros
        const int kc = kb < nkb ? kb : 0;
        const uint32_t st = lds0 + (uint32_t)slot * kStage;
#pragma unroll
        for (int i = 0; i < CA; ++i)
            if (BM / 4 % NW == 0 || wg * CA + i < BM / 4)
                lds_copy(rA, st + (wg * CA + i) * 1024,
                         (ao[i & 3] + (uint32_t)(i >> 2) * (32u * K)) | oob | (tail ? ah[i & 3] : 0u), kc * 256);
#pragma unroll
        for (int i = 0; i < CB; ++i)
            if (BN / 8 % NW == 0 || wg * CB + i < BN / 8)
                lds_copy(rW, st + BM * 256 + (wg * CB + i) * 1024,
                         (bo[i & 1] + (uint32_t)(i >> 1) * (16u * K)) | oob | (tail ? bh[i & 1] : 0u), kc * 128);
    };
    auto load_s = [&](uint32_t (&sv)[NT], int kb) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
            sv[t] = __builtin_amdgcn_raw_buffer_load_b32(rS, (int)so[t], (kb < nkb ? kb : 0) * 4, 0);
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mt][t][i] = 0.f;

    const unsigned char* sbase = smem + kg * 2 * kStage;
    const int arow = (wm * 32 * MT + lc) * 256, asw = lane & 15;
    const int brow = BM * 256 + (wn * 32 * NT + lc) * 128, bsw = (lc >> 1) & 7;
    const int its = (nkb + KB - 1) / KB;
    uint32_t sc[2][NT];
    load_s(sc[0], kg);
    copy(kg, 0);
    for (int it0 = 0; it0 < its; it0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int it = it0 + u;
            if (it >= its) break;
            const int kb = it * KB + kg;
            __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
            if (NW > 1) asm volatile("s_barrier" ::: "memory");
            if (it + 1 < its) {
                load_s(sc[u ^ 1], kb + KB);
                copy(kb + KB, u ^ 1);
            }
            if (KB > 1 && kb >= nkb) continue;
            const unsigned char* st = sbase + u * kStage;
            f32x16 part[MT][NT];
#pragma unroll
            for (int q = 0; q < 4 / KS; ++q) {
                const int p = ks * (4 / KS) + q;
                u32x4 w[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    w[t] = *reinterpret_cast<const u32x4*>(st + brow + t * 4096 + 16 * ((2 * p + hi) ^ bsw));
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 a[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        a[mt] = *reinterpret_cast<const u32x4*>(st + arow + mt * 8192 + 16 * ((4 * p + 2 * hi + h) ^ asw));
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const u32x4 b = fp8x8_to_16<BF16>(w[t][2 * h], w[t][2 * h + 1]);
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            const f32x16 z{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                            part[mt][t] = mfma32<BF16>(a[mt], b, q == 0 && h == 0 ? z : part[mt][t]);
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const float sv = __uint_as_float(__builtin_amdgcn_readfirstlane(sc[u][t]));
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[mt][t][i] = __builtin_fmaf(sv, part[mt][t][i], acc[mt][t][i]);
            }
        }
    }
    if constexpr (KG > 1) {
        __builtin_amdgcn_s_waitcnt(7 << 4);
        asm volatile("s_barrier" ::: "memory");
        constexpr int QT = MT * NT * 4;
        f32x4* red = reinterpret_cast<f32x4*>(smem);
        const int g0 = kg * KS + ks;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int t = (q >> 2) % NT, mt = (q >> 2) / NT, i = q & 3;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[mt][t][4 * i + e];
            red[((g0 * NT_W + wt) * QT + q) * 64 + lane] = v;
        }
        __syncthreads();
#pragma unroll
        for (int q0 = 0; q0 < QT; q0 += KG) {
            const int q = q0 + g0;
            if (q >= QT) break;
            f32x4 v = red[(wt * QT + q) * 64 + lane];
#pragma unroll
            for (int g = 1; g < KG; ++g) v += red[((g * NT_W + wt) * QT + q) * 64 + lane];
            const int t = (q >> 2) % NT, mt = (q >> 2) / NT, i = q & 3;
            const int n = n0 + 32 * t + lc;
            const float bv = bias && n < N ? act_to_f32<BF16>(bias[n]) : 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + wm * 32 * MT + 32 * mt + 8 * i + 4 * hi + e;
                if (m < M && n < N) C[(size_t)m * N + n] = f32_to_act<BF16>(v[e] + bv);
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n = n0 + 32 * t + lc;
            if (n >= N) continue;
            const float bv = bias ? act_to_f32<BF16>(bias[n]) : 0.f;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = m0 + wm * 32 * MT + 32 * mt + 8 * (i >> 2) + 4 * hi + (i & 3);
                    if (m < M) C[(size_t)m * N + n] = f32_to_act<BF16>(acc[mt][t][i] + bv);
                }
        }
    }
}

struct Args {
    const uint16_t* A;
    const uint8_t* W;
    const float* Sc;
    const uint16_t* bias;
    uint16_t* C;
    int M, N, K;
    hipStream_t stream;
};

template <bool BF16, int MT, int NT, int WM, int WN, int KS, int KB>
void launch(const Args& a) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
    constexpr int stages = 2 * KB * (BM * 256 + BN * 128), red = KS * KB > 1 ? KS * KB * BM * BN * 4 : 0;
    static_assert(stages <= 160 * 1024 && red <= 160 * 1024, "LDS");
    const int tiles = fl_ceil_div(a.M, BM) * fl_ceil_div(a.N, BN);
    hipLaunchKernelGGL((fp8_gemm_wide<BF16, MT, NT, WM, WN, KS, KB>), dim3(tiles), dim3(64 * WM * WN * KS * KB),
                       stages > red ? stages : red, a.stream, a.A, a.W, a.Sc, a.bias, a.C, a.M, a.N, a.K);
}

int tiles_of(const Args& a, int bm, int bn) { return fl_ceil_div(a.M, bm) * fl_ceil_div(a.N, bn); }

// Rounds of 256 workgroups (one per CU): a full one costs `full`, the last one
// between `few` and `full` by how many it holds.
float rounds1(int tiles, float few, float full) {
    const int rem = tiles % 256;
    return (tiles / 256) * full + (rem == 0 ? 0.f : few + (full - few) * rem / 256.f);
}

// 17..64 rows, with the times in us of the three tiles modelled from their
// rounds and steps along K (measured at N 1024..10944, K 1024..10944, M
// 17..64: within 1 % of the fastest).  2048 x 2048 / 10944 x 2048 / 2048 x
// 10944 at 48 rows, bf16: 22.4 / 33.6 / 57.1 us as three 16-row decode
// launches -> 5.2 / 9.3 / 13.6 us.
template <bool BF16>
void launch_small(const Args& a) {
    const int nkb = (a.K + 127) >> 7;
    const auto r = [](int tiles) { return (float)fl_ceil_div(tiles, 256); };
    const float t0 = 1.4f + r(tiles_of(a, 32, 32)) * (1.7f + 0.65f * ((nkb + 5) / 6));
    const float t1 = r(tiles_of(a, 32, 64)) * (3.9f + 0.85f * ((nkb + 3) / 4));
    const float t2 = r(tiles_of(a, 64, 64)) * (3.2f + 1.0f * ((nkb + 2) / 3));
    if (t0 <= t1 && t0 <= t2)
        launch<BF16, 1, 1, 1, 1, 1, 6>(a);
    else if (t1 <= t2)
        launch<BF16, 1, 1, 1, 2, 2, 4>(a);
    else
        launch<BF16, 2, 1, 1, 2, 2, 3>(a);
}

// Above 64 rows (the caller sends 1700 and more), likewise.  Against 64 x 128
// tiles of 16x16x32 MFMAs, 2000 rows, weights from HBM: 2048 x 2048 / 10944 x
// 2048 / 2048 x 10944 23.8 / 122 / 115 -> 22.7 / 107 / 113 us; 4096 rows 48 /
// 240 / 228 -> 38 / 205 / 172.
template <bool BF16>
void launch_large(const Args& a) {
    const float nkb = (float)((a.K + 127) >> 7);
    const float t0 = 1.5f + nkb * rounds1(tiles_of(a, 64, 256), 1.0f, 1.17f);
    const float t1 = 1.5f + nkb * rounds1(tiles_of(a, 128, 256), 1.55f, 1.95f);
    if (t0 <= t1)
        launch<BF16, 2, 1, 1, 8, 1, 1>(a);
    else
        launch<BF16, 2, 2, 2, 4, 1, 1>(a);
}

}  // namespace

int fp8_gemm_rows(int K) {
    // activation offsets, those of the last tile's rows past M among them,
    // stay below 2^31
    const long rows = ((1l << 31) - 1) / ((long)K * 2) - 128;
    return rows < 128 ? 0 : (int)(rows / 128 * 128);
}

hipError_t fp8_gemm_b128(const uint16_t* A, const uint8_t* W, const float* Sc, const uint16_t* bias, uint16_t* C,
                         int M, int N, int K, bool bf16, hipStream_t stream) {
    const Args a{A, W, Sc, bias, C, M, N, K, stream};
    if (M <= 64)
        bf16 ? launch_small<true>(a) : launch_small<false>(a);
    else
        bf16 ? launch_large<true>(a) : launch_large<false>(a);
    return hipGetLastError();
}
