// Small-tile GEMM kernels: see gemm_mid.h for what they are for and how the tiles are staged.
#include <math.h>

#include "gemm_mid.h"

namespace fx {

// Item of workgroup b of `total`: contiguous runs of items per XCD (workgroups are dealt to
// the 8 XCDs round-robin), so the tiles that share operand panels share an L2.
__device__ __forceinline__ int mid_item(int b, int total) {
    const int x = b & 7, q = total >> 3, r = total & 7;
    return x * q + min(x, r) + (b >> 3);
}

// Tile t of an nm x nn grid: groups of four row panels, the column tiles outer inside a group.
__device__ __forceinline__ void mid_tile(int t, int nm, int nn, int& mt, int& nt) {
    const int grp = t / (4 * nn), w = t - grp * (4 * nn);
    const int rows = min(4, nm - 4 * grp);
    mt = 4 * grp + w % rows;
    nt = w / rows;
}

// 16 bytes of row r of `src` at column n (n < N), elementwise where a row start is not aligned
// or the chunk passes N
__device__ __forceinline__ void mid_put(uint16_t* o, int n, int N, bool vec, const uint4& u) {
    if (vec && n + 8 <= N) {
        st16(o, u);
    } else {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (n + e < N) o[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
}

// The fp32 accumulators of a wave's part of a tile into the slice's partial (M x N, N % 4 == 0),
// each 32-row block through the wave's LDS share as 16-byte row chunks.
template <int TI, int TJ>
__device__ __forceinline__ void mid_store_part(float* stg, float* part, int row, int col, int M, int N, int lane,
                                               const f32x16 (&acc)[TJ][TI]) {
    constexpr int LDF = 32 * TJ + 4;   // floats per staged row
    const int g = lane >> 5;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4*>(stg + (lane & 31) * LDF + 32 * j + 8 * q + 4 * g) =
                    make_float4(acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
        const int row0 = row + 32 * i;
#pragma unroll
        for (int k = 0; k < 4 * TJ; ++k) {
            const int v = lane + 64 * k, r = v / (8 * TJ), c = (v - r * (8 * TJ)) * 4;
            if (row0 + r < M && col + c < N)
                *reinterpret_cast<float4*>(part + (int64_t)(row0 + r) * N + col + c) =
                    *reinterpret_cast<const float4*>(stg + r * LDF + c);
        }
    }
}

// C = act(A B^T + bias) (forward, B rows along K) or C = (A B) [* gate] (input gradient, B's
// K down its rows).  EPI: bit 0 GELU, 1 H out, 2 bias, 4 H is the GELU derivative, 5 times the
// bf16 values of G, 6 times gelu'(G), 7 the fp32 products of a K slice; values are rounded as the 256-wide kernels round them.
// The accumulators hold C^T, so a lane has 4 consecutive columns of a row; each 32-row block
// leaves through the wave's LDS share as 16-byte row chunks.
template <int BM, int BN, int TI, int TJ, int NST, int AK, int BK, int EPI>
__global__ void __launch_bounds__(64 * (BM / (32 * TI)) * (BN / (32 * TJ)), BM == 256 ? 2 : (BN / (32 * TJ)) * (BM / (32 * TI)) / 2)
gemm_mid_kernel(MidArgs a) {
    constexpr bool kGelu = EPI & 1, kH = EPI & 2, kBias = EPI & 4, kDeriv = EPI & 16, kGate = EPI & 32, kGateH = EPI & 64,
                   kPart = EPI & 128;
    constexpr int kWaves = (BM / (32 * TI)) * (BN / (32 * TJ)), kWN = BN / (32 * TJ);
    constexpr int LDE = 32 * TJ + 8;
    constexpr int kStg = kPart ? 2 * 32 * (32 * TJ + 4)                // elements per wave
                               : 32 * LDE * (kH || kGate || kGateH ? 2 : 1);
    static_assert(kWaves * kStg <= NST * (BM + BN) * 64, "staging fits the stages");
    __shared__ __attribute__((aligned(16))) uint16_t lds[NST * (BM + BN) * 64];
    __shared__ __attribute__((aligned(16))) uint16_t sbias[kBias ? BN : 1];
    const int lane = threadIdx.x & 63, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave / kWN) * 32 * TI, wn = (wave % kWN) * 32 * TJ;
    const int nm = (a.M + BM - 1) / BM, nn = (a.N + BN - 1) / BN;
    const int item = mid_item(blockIdx.x, nm * nn * (kPart ? a.slices : 1));
    const int sl = kPart ? item / (nm * nn) : 0, nk = (a.K + 63) / 64;
    int mt, nt;
    mid_tile(item - sl * nm * nn, nm, nn, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;
    if constexpr (kBias) {
        if (threadIdx.x < BN) sbias[threadIdx.x] = n0 + (int)threadIdx.x < a.N ? a.bias[n0 + threadIdx.x] : (uint16_t)0;
    }
    // the gate's chunks, loaded before the K loop (older than its loads: its waits only get
    // stricter) in the layout of the stores below
    uint4 gate[TI][2 * TJ];
    if constexpr (kGate || kGateH) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int k = 0; k < 2 * TJ; ++k) {
                const int v = lane + 64 * k, r = v / (4 * TJ), c = (v - r * (4 * TJ)) * 8;
                const int m = min(m0 + wm + 32 * i + r, a.M - 1), n = min(n0 + wn + c, a.N - 8);
                gate[i][k] = ld16(a.G + (int64_t)m * a.ldg + n);   // N % 8 == 0: the host checks
            }
    }
    f32x16 acc[TJ][TI];
    mid_product<BM, BN, TI, TJ, AK, BK, NST, true>(
        a.A, a.B, m0, n0, a.K, kPart ? (int)((int64_t)nk * sl / a.slices) : 0,
        kPart ? (int)((int64_t)nk * (sl + 1) / a.slices) : nk, lds, wave, lane, wm, wn, acc, [&](int kt, const uint16_t* sa) {
            if constexpr (AK == kGather) {
                // gathered rows out, the K steps of a row panel dealt to its column tiles
                if (a.Xg == nullptr || kt % nn != nt) return;
                for (int v = threadIdx.x; v < BM * 8; v += 64 * kWaves) {
                    const int r = v >> 3, c = v & 7, m = m0 + r, k = kt * 64 + c * 8;
                    if (m < a.M && k < a.K)
                        st16(a.Xg + (int64_t)m * a.ldxg + k,
                             *reinterpret_cast<const uint4*>(sa + r * 64 + ((c ^ mid_swz(r)) << 3)));
                }
            }
        });
    if constexpr (kPart) {
        mid_store_part<TI, TJ>(reinterpret_cast<float*>(lds) + wave * 32 * (32 * TJ + 4), a.part + (int64_t)sl * a.M * a.N,
                               m0 + wm, n0 + wn, a.M, a.N, lane, acc);
        return;
    }
    uint16_t* stg = lds + wave * kStg;
    uint16_t* stg2 = stg + 32 * LDE;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        if constexpr (kGate || kGateH) {
#pragma unroll
            for (int k = 0; k < 2 * TJ; ++k) {
                const int v = lane + 64 * k, r = v / (4 * TJ), c = (v - r * (4 * TJ)) * 8;
                *reinterpret_cast<uint4*>(stg2 + r * LDE + c) = gate[i][k];
            }
        }
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int off = (lane & 31) * LDE + 32 * j + 8 * q + 4 * g;
                float v[4], d[4];
                uint2 hh = make_uint2(0u, 0u);
                if constexpr (kGate || kGateH) hh = *reinterpret_cast<const uint2*>(stg2 + off);
                const float hv[4] = {bf16_lo(hh.x), bf16_hi(hh.x), bf16_lo(hh.y), bf16_hi(hh.y)};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float h = acc[j][i][4 * q + e];
                    if constexpr (kBias) h += bf16_to_f32(sbias[wn + 32 * j + 8 * q + 4 * g + e]);
                    d[e] = h;
                    if constexpr (kDeriv) gelu_tanh_and_grad(h, v[e], d[e]);
                    else if constexpr (kGelu) v[e] = gelu_tanh(h);
                    else if constexpr (kGate) v[e] = bf16_to_f32(f32_to_bf16(h)) * hv[e];
                    else if constexpr (kGateH) v[e] = bf16_to_f32(f32_to_bf16(h)) * gelu_tanh_grad(hv[e]);
                    else v[e] = h;
                }
                *reinterpret_cast<uint2*>(stg + off) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                if constexpr (kH)
                    *reinterpret_cast<uint2*>(stg2 + off) = make_uint2(pack_bf16x2(d[0], d[1]), pack_bf16x2(d[2], d[3]));
            }
#pragma unroll
        for (int k = 0; k < 2 * TJ; ++k) {
            const int v = lane + 64 * k, r = v / (4 * TJ), c = (v - r * (4 * TJ)) * 8;
            const int m = m0 + wm + 32 * i + r, n = n0 + wn + c;
            if (m >= a.M || n >= a.N) continue;
            mid_put(a.C + (int64_t)m * a.ldc + n, n, a.N, a.vec_c, *reinterpret_cast<const uint4*>(stg + r * LDE + c));
            if constexpr (kH)
                mid_put(a.H + (int64_t)m * a.ldh + n, n, a.N, a.vec_h,
                        *reinterpret_cast<const uint4*>(stg2 + r * LDE + c));
        }
    }
}

// Weight gradient C (M x N) = A^T B over the tokens (K) of a slice, both operands' tokens down
// their rows, in the K order of the 256-wide kernels (bit-identical partials); the slices'
// token ranges are theirs too.
template <int BM, int BN, int TI, int TJ, int NST>
__global__ void __launch_bounds__(64 * (BM / (32 * TI)) * (BN / (32 * TJ)), BM == 256 ? 2 : 1) gemm_mid_wgrad_kernel(MidArgs a) {
    constexpr int kWaves = (BM / (32 * TI)) * (BN / (32 * TJ)), kWN = BN / (32 * TJ);
    constexpr int LDF = 32 * TJ + 4;   // floats per staged row
    static_assert(kWaves * 32 * LDF * 2 <= NST * (BM + BN) * 64, "staging fits the stages");
    __shared__ __attribute__((aligned(16))) uint16_t lds[NST * (BM + BN) * 64];
    const int lane = threadIdx.x & 63, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave / kWN) * 32 * TI, wn = (wave % kWN) * 32 * TJ;
    const int nm = (a.M + BM - 1) / BM, nn = (a.N + BN - 1) / BN, ntiles = nm * nn;
    const int item = mid_item(blockIdx.x, ntiles * a.slices);
    const int sl = item / ntiles;
    int mt, nt;
    mid_tile(item - sl * ntiles, nm, nn, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;
    const int nk = (a.K + 63) / 64;
    const int kb = (int)((int64_t)nk * sl / a.slices), ke = (int)((int64_t)nk * (sl + 1) / a.slices);
    f32x16 acc[TJ][TI];
    mid_product<BM, BN, TI, TJ, kColK, kColK, NST, false>(a.A, a.B, m0, n0, a.K, kb, ke, lds, wave, lane, wm, wn, acc,
                                                          [](int, const uint16_t*) {});
    float* stg = reinterpret_cast<float*>(lds) + wave * 32 * LDF;
    if (a.slices > 1) {
        mid_store_part<TI, TJ>(stg, a.part + (int64_t)sl * a.M * a.N, m0 + wm, n0 + wn, a.M, a.N, lane, acc);
        return;
    }
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<float4*>(stg + (lane & 31) * LDF + 32 * j + 8 * q + 4 * g) =
                    make_float4(acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
        const int row0 = m0 + wm + 32 * i;
#pragma unroll
        for (int k = 0; k < 2 * TJ; ++k) {
            const int v = lane + 64 * k, r = v / (4 * TJ), c = (v - r * (4 * TJ)) * 8;
            if (row0 + r < a.M && n0 + wn + c < a.N) {
                const float4 lo = *reinterpret_cast<const float4*>(stg + r * LDF + c);
                const float4 hi = *reinterpret_cast<const float4*>(stg + r * LDF + c + 4);
                st16(a.C + (int64_t)(row0 + r) * a.ldc + n0 + wn + c,
                     make_uint4(pack_bf16x2(lo.x, lo.y), pack_bf16x2(lo.z, lo.w), pack_bf16x2(hi.x, hi.y),
                                pack_bf16x2(hi.z, hi.w)));
            }
        }
    }
}

static unsigned tiles_of(const MidArgs& a, int bm, int bn) {
    return (unsigned)((((int64_t)a.M + bm - 1) / bm) * (((int64_t)a.N + bn - 1) / bn));
}

template <int AK, int EPI>
static void forward_launch(const MidArgs& a, int tile, hipStream_t s) {
    if (tile == kMidBig)
        hipLaunchKernelGGL((gemm_mid_kernel<256, 128, 2, 2, 3, AK, kRowK, EPI>), dim3(tiles_of(a, 256, 128)), dim3(512), 0, s, a);
    else
        hipLaunchKernelGGL((gemm_mid_kernel<64, 128, 1, 1, 3, AK, kRowK, EPI>), dim3(tiles_of(a, 64, 128)), dim3(512), 0, s, a);
}

template <int AK>
static int forward_epi(const MidArgs& a, int tile, int epi, hipStream_t s) {
    switch (epi) {
#define FX_MID(E) case E: forward_launch<AK, E>(a, tile, s); break;
        FX_MID(0) FX_MID(1) FX_MID(2) FX_MID(3) FX_MID(4) FX_MID(5) FX_MID(6) FX_MID(7) FX_MID(19) FX_MID(23)
#undef FX_MID
        default: return set_error(FX_EINVAL, "mid_forward: epilogue %d", epi);
    }
    return check_launch("gemm_mid");
}

int mid_forward(const MidArgs& a, int tile, int epi, hipStream_t s) {
    return a.A.idx ? forward_epi<kGather>(a, tile, epi, s) : forward_epi<kRowK>(a, tile, epi, s);
}

int mid_dgrad(const MidArgs& a, int tile, int gate, hipStream_t s) {
    if (a.slices > 1) {
        if (gate != 0 || tile != kMidBig) return set_error(FX_EINVAL, "mid_dgrad: slices with a gate or small tiles");
        hipLaunchKernelGGL((gemm_mid_kernel<256, 128, 2, 2, 3, kRowK, kColK, 128>), dim3(tiles_of(a, 256, 128) * a.slices),
                           dim3(512), 0, s, a);
        return check_launch("gemm_mid_dgrad");
    }
#define FX_MID(E)                                                                                                       \
    if (tile == kMidBig)                                                                                                \
        hipLaunchKernelGGL((gemm_mid_kernel<256, 128, 2, 2, 3, kRowK, kColK, E>), dim3(tiles_of(a, 256, 128)), dim3(512), 0, s, a); \
    else                                                                                                                \
        hipLaunchKernelGGL((gemm_mid_kernel<64, 128, 1, 1, 3, kRowK, kColK, E>), dim3(tiles_of(a, 64, 128)), dim3(512), 0, s, a);
    if (gate == 2) {
        FX_MID(32)
    } else if (gate == 1) {
        FX_MID(64)
    } else {
        FX_MID(0)
    }
#undef FX_MID
    return check_launch("gemm_mid_dgrad");
}

int mid_wgrad(const MidArgs& a, int tile, hipStream_t s) {
    if (tile == kMidBig)
        hipLaunchKernelGGL((gemm_mid_wgrad_kernel<256, 128, 2, 2, 3>), dim3(tiles_of(a, 256, 128) * a.slices), dim3(512), 0, s, a);
    else
        hipLaunchKernelGGL((gemm_mid_wgrad_kernel<128, 128, 2, 1, 4>), dim3(tiles_of(a, 128, 128) * a.slices), dim3(512), 0, s, a);
    return check_launch("gemm_mid_wgrad");
}

// Time of a product on each tile, in us: rounds of resident workgroups, each a first load and
// an epilogue plus its K steps of 64 (one 256 x 128 workgroup a CU; two 64 x 128 ones, faster
// per step alone).  Fitted to 35 layer shapes of 2,048 to 16,384 rows, K 256 to 3072 (most
// within 10 %).
float mid_cost(int64_t M, int64_t N, int64_t K, int* tile) {
    const float cus = (float)device_cus(), steps = (float)((K + 63) / 64);
    const float nb = (float)(((M + 255) / 256) * ((N + 127) / 128)), ns = (float)(((M + 63) / 64) * ((N + 127) / 128));
    const float big = ceilf(nb / cus) * (4.4f + 0.8f * steps);
    const float small = ns <= cus ? 2.5f + 0.45f * steps : ceilf(ns / (2 * cus)) * (3.5f + 0.63f * steps);
    *tile = small < big ? kMidSmall : kMidBig;
    return small < big ? small : big;
}

// The weight gradient's tile and K split: as above, plus the partials' way through memory
// (written by the product, read by the reduce) and the reduce's launch.  At least 4 K steps of
// 64 tokens a slice, at most 32 slices.
float mid_wgrad_cost(int64_t M, int64_t N, int64_t K, int* tile, int* slices) {
    const float cus = (float)device_cus();
    const int64_t nk = (K + 63) / 64;
    const float nb = (float)(((M + 255) / 256) * ((N + 127) / 128)), ns = (float)(((M + 127) / 128) * ((N + 127) / 128));
    float best = 0.f;
    for (int sl = 1; sl <= 32 && (sl == 1 || nk / sl >= 4); ++sl) {
        const float steps = (float)((nk + sl - 1) / sl);
        const float red = sl > 1 ? 3.f + (float)sl * (float)(M * N) * 8.f / 5e6f : 0.f;
        const float big = ceilf(nb * sl / cus) * (4.5f + 0.98f * steps) + red;
        const float small = ceilf(ns * sl / cus) * (3.f + 0.66f * steps) + red;
        const float t = small < big ? small : big;
        if (sl == 1 || t < best) {
            best = t;
            *slices = sl;
            *tile = small < big ? kMidSmall : kMidBig;
        }
    }
    return best;
}

}  // namespace fx
