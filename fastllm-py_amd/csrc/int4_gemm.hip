// INT4 group-128 matmul behind the Marlin C-ABI above 16 rows (K % 128 == 0):
// the decode batches of 17..64 rows and the prefill GEMM.
//
//   C[M, N] (fp16) = A[M, K] (fp16) @ dequant(W)^T, dequant = s (q - z)
//
// Weights, scales and zeros are in the layouts that int4_marlin.hip describes.
#include "int4_gemm.cuh"
#include "int4_common.cuh"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// One v_and_or_b32 per nibble pair: the masks stay in SGPRs and the exponent
// magics in VGPRs (the instruction takes one scalar operand and no literal).
// The empty asm hides the constants, or the compiler folds them into two
// instructions with a literal each; written as inline asm instead, the
// instruction could not be moved between the MFMAs (M4096 N24576 K4096 711
// -> 691 us).
struct Magic {
    uint32_t lo, hi, mlo, mhi;
};
FL_DEV Magic make_magic() {
    Magic m{0x64006400u, 0x54005400u, 0x000F000Fu, 0x00F000F0u};
    asm("" : "+v"(m.lo), "+v"(m.hi));
    asm("" : "+s"(m.mlo), "+s"(m.mhi));
    return m;
}

// q - z exactly, or (SCALED) s (q - z) rounded to fp16 as a Marlin kernel
// feeds its matrix cores, of the 8 nibbles of a tile-layout word.
template <bool SCALED>
FL_DEV f16x8 dequant(uint32_t w, uint32_t zlo, uint32_t zhi, f16x2 s2, const Magic& k) {
    const uint32_t w8 = w >> 8;
    f16x2 p0 = bitcast<f16x2>((w & k.mlo) | k.lo) + bitcast<f16x2>(zlo);
    f16x2 p1 = bitcast<f16x2>((w & k.mhi) | k.hi) + bitcast<f16x2>(zhi);
    f16x2 p2 = bitcast<f16x2>((w8 & k.mlo) | k.lo) + bitcast<f16x2>(zlo);
    f16x2 p3 = bitcast<f16x2>((w8 & k.mhi) | k.hi) + bitcast<f16x2>(zhi);
    if (SCALED) {
        p0 *= s2;
        p1 *= s2;
        p2 *= s2;
        p3 *= s2;
    }
    const u32x4 r{bitcast<uint32_t>(p0), bitcast<uint32_t>(p1), bitcast<uint32_t>(p2),
                  bitcast<uint32_t>(p3)};
    return bitcast<f16x8>(r);
}

// s_waitcnt vmcnt(V) lgkmcnt(0)
template <int V>
FL_DEV void wait_vm_lgkm() {
    static_assert(V < 16, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(V | (7 << 4));
}

// One workgroup = WK k-groups of WM x WN waves on a tile of 32 MT WM rows x
// 32 NT WN columns; a wave holds 32 MT x 32 NT of it in 32x32x16 MFMA
// accumulators, and k-group g takes the 128-k blocks g, g + WK, ...
//
// Why 32x32x16: an activation fragment read from LDS feeds twice the columns
// of a 16x16x32 one.  The tile layout holds a block in 16-column tiles (lane
// (c, q): column c, k 32 j + 8 q .. + 7 in word j); one v_permlane16_swap of
// word j of two neighbouring tiles gives both operands of 32 columns: lane l
// has column l % 32 and k 32 j + 16 (l / 32) + {0, 8} .. + 7, and the
// activations are read at the same k.
//
// Memory: each k-group copies its block's activation rows global -> LDS one
// step ahead (two stages; whole 256-byte rows, the 16-byte chunks of row r
// XOR-swizzled by r % 16 so that fragment reads hit all banks), each wave
// loads its own weights, scales and zeros into registers D steps ahead.  A
// step begins when the copies and the weights of its block have landed (the
// copies go out before the weights of the same step, so at D > 1 the 2 NT
// weight loads behind them may stay out), with one barrier -- none where the
// k-group is one wave, which then shares nothing until the end.
// The k-groups' partials are added through LDS in group order.
//
// EX: the MFMAs take q - z exactly and the fp32 partial of a block takes the
// group scale, as the decode GEMV does (up to 64 rows); otherwise B is
// s (q - z) rounded to fp16 (above 64 rows: fewer VALU operations per MFMA).
//
// Bound: above 500 rows by power -- M4096 N24576 K4096 runs at 76 % MFMA
// issue but 1.5 of 2.4 GHz -- so the tile that moves the fewest LDS bytes per
// MFMA wins there; below by the activation bytes each CU must pull from L2
// (M K 2 per column tile), so the tiles get narrow and K is split over waves.
//
// Rows at or past M read zeros (past the buffer), columns past N the last
// ones; neither is stored.  Blocks past the end load zeros from offsets past
// the buffers (the waits count loads, so none may be left out) and are not
// computed.
template <int NT>
struct WBlock {  // one 128-k block of a wave's 32 NT columns
    u32x4 w[2 * NT];
    uint16_t s[NT];
    uint32_t z[NT];
};

template <int MT, int NT, int WM, int WN, int WK, int D, bool EX>
__global__ __launch_bounds__(64 * WM * WN * WK, (WM * WN * WK <= 8 ? 2 : WM * WN * WK / 4)) void int4_gemm_wide(
    const f16* __restrict__ A, const uint32_t* __restrict__ Wq, const uint16_t* __restrict__ S,
    const uint32_t* __restrict__ Z, f16* __restrict__ C, int M, int N, int K) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, NW = WM * WN;
    constexpr int kStage = BM * 256, CPW = (BM / 4 + NW - 1) / NW;  // LDS stage, copies of a wave
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = wave / NW, wg = wave % NW, wm = wg / WN, wn = wg % WN;
    const int lc = lane & 31, hi = lane >> 5;
    const int nkb = K >> 7;

    // Tile order: the hardware deals workgroup b to XCD b % 8, so the tiles of
    // one XCD are made a contiguous run, in groups of four row tiles by all
    // column tiles: the tiles in flight on an XCD then share few activation
    // rows and weight columns (M4096 N24576 K4096: groups of 2 / 4 / 8 / 16
    // row tiles 697 / 670 / 673 / 682 us).
    constexpr int gm = 4;
    const int mblk = (M + BM - 1) / BM, nblk = (N + BN - 1) / BN;
    const int total = mblk * nblk;
    int lin = blockIdx.x;
    if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
    const int grp = lin / (gm * nblk), first = grp * gm;
    const int rows = mblk - first < gm ? mblk - first : gm;
    const int in = lin - grp * gm * nblk;
    const int nb_i = in / rows, mb_i = first + in - nb_i * rows;
    const int m0 = mb_i * BM, n0 = nb_i * BN + wn * 32 * NT;

    const i32x4_t rA = raw_rsrc(A, (uint32_t)M * K * 2);
    const __amdgpu_buffer_rsrc_t rW = buf_rsrc(Wq, (uint32_t)N * K / 2);
    const __amdgpu_buffer_rsrc_t rS = buf_rsrc(S, (uint32_t)nkb * N * 2);
    const __amdgpu_buffer_rsrc_t rZ = buf_rsrc(Z, (uint32_t)nkb * (N >> 3) * 4);
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem + wk * 2 * kStage;

    uint32_t ao[CPW < 4 ? CPW : 4];
#pragma unroll
    for (int i = 0; i < (CPW < 4 ? CPW : 4); ++i) {
        const int r = 4 * (wg * CPW + i) + (lane >> 4);
        ao[i] = 2u * ((uint32_t)(m0 + r) * K) + 16u * ((lane & 15) ^ (r & 15));
    }
    uint32_t bo[2 * NT], so[NT], zo[NT], zsh[NT];
#pragma unroll
    for (int t = 0; t < 2 * NT; ++t) {
        int nt = (n0 >> 4) + t;
        nt = nt < (N >> 4) ? nt : (N >> 4) - 1;
        bo[t] = (uint32_t)nt * (8u * K);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        int n = n0 + 32 * t + lc;
        n = n < N ? n : N - 1;
        const int cl = n & 63;
        so[t] = 2u * ((n & ~63) + 8 * (cl & 7) + (cl >> 3));
        zo[t] = 4u * (((n >> 6) << 3) + (cl & 7));
        zsh[t] = 4 * slot_of(cl >> 3);
    }
    // blocks at or past the end: lane offsets past every buffer
    auto copy_a = [&](int kb, int slot) {
        const uint32_t st = lds0 + (uint32_t)slot * kStage + wg * CPW * 1024;
        const uint32_t oob = kb < nkb ? 0u : 0x80000000u;
        const int kc = kb < nkb ? kb : 0;
#pragma unroll
        for (int i = 0; i < CPW; ++i)
            if (BM / 4 % NW == 0 || wg * CPW + i < BM / 4)
                lds_copy(rA, st + i * 1024, (ao[i & 3] + (uint32_t)(i >> 2) * (32u * K)) | oob, kc * 256);
    };
    auto load_sz = [&](WBlock<NT>& b, int kb) {
        const uint32_t oob = kb < nkb ? 0u : 0x80000000u;
        const int kc = kb < nkb ? kb : 0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            b.s[t] = __builtin_amdgcn_raw_buffer_load_b16(rS, (int)(so[t] | oob), kc * 2 * N, 0);
            b.z[t] = __builtin_amdgcn_raw_buffer_load_b32(rZ, (int)(zo[t] | oob), kc * (N >> 1), 0);
        }
    };
    auto load_w = [&](WBlock<NT>& b, int kb) {
        const uint32_t oob = kb < nkb ? 0u : 0x80000000u;
        const int kc = kb < nkb ? kb : 0;
#pragma unroll
        for (int t = 0; t < 2 * NT; ++t)
            b.w[t] = bitcast<u32x4>(__builtin_amdgcn_raw_buffer_load_b128(rW, (int)(lane * 16 | oob), (int)(bo[t] + kc * 1024), 0));
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mt][t][i] = 0.f;

    const unsigned char* abase = smem + wk * 2 * kStage + (wm * 32 * MT + lc) * 256;
    const int sw = lane & 15;
    auto read_a = [&](f16x8 (&a)[MT], const unsigned char* as, int c) {
        const unsigned char* p = as + 16 * ((c + 2 * hi) ^ sw);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[mt] = *reinterpret_cast<const f16x8*>(p + mt * 8192);
    };

    const Magic mg = make_magic();
    constexpr int R = D > 1 ? D : 2;  // ring slots
    WBlock<NT> ring[R];
    const int its = (nkb + WK - 1) / WK;
    if constexpr (D == 1) {
        load_sz(ring[0], wk);
        copy_a(wk, 0);
        load_w(ring[0], wk);
    } else {
#pragma unroll
        for (int d = 0; d < D - 1; ++d) {
            load_sz(ring[d], wk + d * WK);
            load_w(ring[d], wk + d * WK);
        }
        load_sz(ring[D - 1], wk + (D - 1) * WK);
        __builtin_amdgcn_sched_barrier(0);
        copy_a(wk, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(ring[D - 1], wk + (D - 1) * WK);
    }
    for (int it0 = 0; it0 < its; it0 += R) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int it = it0 + u;
            if (it >= its) break;
            const int kb = it * WK + wk;
            // this block's activations and weights have landed, and the LDS
            // reads of the stage that is refilled below are done
            constexpr int V = D == 1 ? 0 : 2 * NT;
            wait_vm_lgkm<V>();
            if (NW > 1) asm volatile("s_barrier" ::: "memory");
            if (D > 1) {  // named here, so that the compiler's own waits fall before the loads issued below
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    asm volatile("" : "+v"(ring[u].w[2 * t]), "+v"(ring[u].w[2 * t + 1]), "+v"(ring[u].s[t]), "+v"(ring[u].z[t]));
            }
            const int slot = it & 1;
            const WBlock<NT> b = ring[u];
            if constexpr (D == 1) {
                if (kb + WK < nkb) {
                    load_sz(ring[u ^ 1], kb + WK);
                    copy_a(kb + WK, slot ^ 1);
                    load_w(ring[u ^ 1], kb + WK);
                }
            } else {
                load_sz(ring[u], kb + D * WK);
                __builtin_amdgcn_sched_barrier(0);
                copy_a(kb + WK, slot ^ 1);
                __builtin_amdgcn_sched_barrier(0);
                load_w(ring[u], kb + D * WK);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (WK > 1 && kb >= nkb) continue;
            const unsigned char* as = abase + slot * kStage;
            uint32_t zl[NT], zh[NT];
            f16x2 s2[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                zero_bits((b.z[t] >> zsh[t]) & 0xFu, zl[t], zh[t]);
                const f16 s = bitcast<f16>(b.s[t]);
                s2[t] = f16x2{s, s};
            }
            f16x8 a[2][MT];
            read_a(a[0], as, 0);
            f32x16 part[EX ? MT : 1][EX ? NT : 1];
            if constexpr (EX)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int i = 0; i < 16; ++i) part[mt][t][i] = 0.f;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                if (s < 7) read_a(a[(s + 1) & 1], as, 4 * ((s + 1) >> 1) + ((s + 1) & 1));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const auto r = __builtin_amdgcn_permlane16_swap(b.w[2 * t][s >> 1], b.w[2 * t + 1][s >> 1], false, false);
                    const f16x8 bv = dequant<!EX>(r[s & 1], zl[t], zh[t], s2[t], mg);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        f32x16& d = EX ? part[mt][t] : acc[mt][t];
                        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s & 1][mt], bv, d, 0, 0, 0);
                    }
                }
            }
            if constexpr (EX)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const float sv = (float)s2[t][0];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[mt][t][i] = __builtin_fmaf(sv, part[mt][t][i], acc[mt][t][i]);
                }
        }
    }
    if constexpr (WK > 1) {
        // k-group g adds (in group order) and stores every WK-th quarter of
        // the 32x32 tiles
        wait_vm_lgkm<0>();
        asm volatile("s_barrier" ::: "memory");
        constexpr int QT = MT * NT * 4;  // f32x4 per lane
        f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int t = (q >> 2) % NT, mt = (q >> 2) / NT, i = q & 3;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[mt][t][4 * i + e];
            red[((wk * NW + wg) * QT + q) * 64 + lane] = v;
        }
        __syncthreads();
#pragma unroll
        for (int q0 = 0; q0 < QT; q0 += WK) {
            const int q = q0 + wk;
            if (q >= QT) break;
            f32x4 v = red[(wg * QT + q) * 64 + lane];
#pragma unroll
            for (int g = 1; g < WK; ++g) v += red[((g * NW + wg) * QT + q) * 64 + lane];
            const int t = (q >> 2) % NT, mt = (q >> 2) / NT, i = q & 3;
            const int n = n0 + 32 * t + lc;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + wm * 32 * MT + 32 * mt + 8 * i + 4 * hi + e;
                if (m < M && n < N) C[(size_t)m * N + n] = (f16)v[e];
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n = n0 + 32 * t + lc;
            if (n >= N) continue;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = m0 + wm * 32 * MT + 32 * mt + 8 * (i >> 2) + 4 * hi + (i & 3);
                    if (m < M) C[(size_t)m * N + n] = (f16)acc[mt][t][i];
                }
        }
    }
}

struct Args {
    const f16* A;
    const uint32_t* Wq;
    const uint16_t* S;
    const uint32_t* Z;
    f16* C;
    int M, N, K;
    hipStream_t stream;
};

template <int MT, int NT, int WM, int WN, int WK, int D, bool EX>
void launch(const Args& a) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
    constexpr int stages = 2 * WK * BM * 256, red = WK > 1 ? WK * BM * BN * 4 : 0;
    static_assert(stages <= 160 * 1024 && red <= 160 * 1024, "LDS");
    const int tiles = fl_ceil_div(a.M, BM) * fl_ceil_div(a.N, BN);
    hipLaunchKernelGGL((int4_gemm_wide<MT, NT, WM, WN, WK, D, EX>), dim3(tiles), dim3(64 * WM * WN * WK),
                       stages > red ? stages : red, a.stream, a.A, a.Wq, a.S, a.Z, a.C, a.M, a.N, a.K);
}

int tiles_of(const Args& a, int bm, int bn) { return fl_ceil_div(a.M, bm) * fl_ceil_div(a.N, bn); }

// Time of `tiles` workgroups where 512 fit the chip, two per CU: a round of
// up to 256 costs `half`, up to 512 `part` and a full one `full`.
float rounds2(int tiles, float half, float part, float full) {
    const int rem = tiles % 512;
    return (tiles / 512) * full + (rem == 0 ? 0.f : rem <= 256 ? half : part);
}

// 17..64 rows.  Each shape's time in us is modelled as its rounds of 256
// workgroups (one per CU) times its steps along K, with the constants
// measured at N 1024..24576, K 1024..12288, M 17..64: over those 40 sizes the
// choice is the fastest of the four every time.  Qwen3-8B at 48 rows: qkv /
// o / gate_up / down 25.8 / 14.6 / 86 / 36 us with one n-tile per workgroup
// and activations read as fragments -> 9.9 / 6.8 / 16.8 / 14.2 us.
void launch_small(const Args& a) {
    const int nkb = a.K >> 7, s4 = (nkb + 3) / 4, s8 = (nkb + 7) / 8;
    const auto r = [](int tiles) { return (float)fl_ceil_div(tiles, 256); };
    const float t0 = 1.5f + r(tiles_of(a, 32, 32)) * (1.1f + 0.95f * s8);
    const float t1 = 3.6f + s4 * rounds2(tiles_of(a, 32, 64), 0.68f, 1.3f, 1.3f);
    const float t2 = r(tiles_of(a, 32, 96)) * (3.4f + 0.98f * s4);
    const float t3 = r(tiles_of(a, 64, 96)) * (3.9f + 1.4f * s4);
    const float best = fminf(fminf(t0, t1), fminf(t2, t3));
    if (best == t0)
        launch<1, 1, 1, 1, 8, 1, true>(a);
    else if (best == t1)
        launch<1, 2, 1, 1, 4, 2, true>(a);
    else if (best == t2)
        launch<1, 1, 1, 3, 4, 2, true>(a);
    else
        launch<2, 1, 1, 3, 4, 1, true>(a);
}

// Above 64 rows.  The tiles trade activation bytes per MFMA against filling
// the last round of workgroups; each one's time in us per 128-k block is its
// rounds times a measured constant (M 65..4096 at ten N x K: the choice is
// within 0.2 % of the fastest of the five on average, 7 % at worst).
// Against 64 x 256 tiles for every shape: M4096 N24576 K4096 784 -> 667 us
// (1234 TFLOP/s), M500 N24576 K4096 96 -> 90, M500 N4096 K12288 96 -> 56,
// M100 N4096 K4096 34 -> 18.
void launch_large(const Args& a) {
    const float t0 = rounds2(tiles_of(a, 128, 256), 1.85f, 3.2f, 3.55f);
    const int w = tiles_of(a, 256, 192), rem = w % 256;
    const float t1 = (w / 256) * 2.75f +
                     (rem == 0 ? 0.f : rem <= 128 && w < 256 ? 2.0f : rem <= 200 ? 2.4f : 2.75f);
    const float t2 = rounds2(tiles_of(a, 128, 128), 1.08f, 1.75f, 1.93f);
    const float t3 = 1.05f * fl_ceil_div(tiles_of(a, 128, 128), 256);
    const float t4 = 0.64f * fl_ceil_div(tiles_of(a, 64, 128), 256);
    const float best = fminf(fminf(fminf(t0, t1), fminf(t2, t3)), t4);
    if (best == t0)
        launch<4, 2, 1, 4, 1, 1, false>(a);
    else if (best == t1)
        launch<4, 1, 2, 6, 1, 1, false>(a);
    else if (best == t2)
        launch<4, 1, 1, 4, 1, 1, false>(a);
    else if (best == t3)
        launch<4, 1, 1, 4, 2, 1, false>(a);
    else
        launch<2, 1, 1, 4, 4, 1, false>(a);
}

}  // namespace

int int4_gemm_rows(int K) {
    // rows of one launch: activation offsets, those of the last tile's rows
    // past M among them, stay below 2^31
    const long rows = ((1l << 31) - 1) / ((long)K * 2) - 256;
    return rows < 256 ? 0 : (int)(rows / 256 * 256);
}

hipError_t int4_gemm_g128(const f16* A, const uint32_t* Wq, const uint16_t* S, const uint32_t* Z, f16* C, int M,
                          int N, int K, hipStream_t stream) {
    const Args a{A, Wq, S, Z, C, M, N, K, stream};
    if (M <= 64)
        launch_small(a);
    else
        launch_large(a);
    return hipGetLastError();
}
