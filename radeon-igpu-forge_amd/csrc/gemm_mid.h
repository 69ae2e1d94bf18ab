// Small-tile bf16 GEMM kernels (gemm_mid.hip): forward, input gradient and weight gradient
// for the products whose 256-wide whole tiles would leave most of the chip idle, and for the
// ragged and gathered ones.
//
// A 4096 x 512 output is 32 tiles of 256 x 256: one CU in eight works, each through the whole
// K loop and a 256 x 256 epilogue.  These kernels cut the output into 64 x 128, 128 x 128 or
// 256 x 128 tiles of 8 waves.  A K step is 64 values: an operand row is one 128-byte line
// in memory and in LDS, where its eight 16-byte chunks are permuted (mid_swz), so row reads
// (ds_read_b128) and transposed reads (ds_read_b64_tr_b16) are both free of bank conflicts
// without padding.  Stages are filled by direct global -> LDS loads two or three steps ahead;
// the loads are spread over the step's MFMAs, since a wave that issues them in a burst waits
// for the address unit before its first MFMA (4096 x 2048 x 4096: 78.6 -> 64.2 us).
//
// What bounds the K loop: tile loads alone run at 1.0 us and MFMAs alone at 1.2 us per 1.6 us
// of both together (256 x 128 tiles), so it is the overlap of the two inside a step; at the
// small sizes it is the ends: of 12.6 us at 4096 x 2048 x 512, 1.5 are the launch, 4.5 the
// first loads and the epilogue.
//
// The small tiles have 8 waves too, of 32 x 32 (64 x 128) or 64 x 32 (128 x 128) each: they read
// a third to a half more from LDS than 4 waves of twice the width, but two waves a SIMD cover
// each other's waits.  Input gradients 4096 x 512 x 1536 15.0 -> 13.7 us, 2048 x 768 x 3072
// 25.2 -> 22.6; weight gradients 4096 x 1536 x 512 21.0 -> 20.1, 2048 x 3072 x 768 25.1 -> 23.0;
// forwards 4096 x 512 x 2048 18.6 -> 16.3.
#pragma once

#include "fx_mfma.h"

namespace fx {

// s_waitcnt vmcnt(N) lgkmcnt(0), then the workgroup barrier, in one statement: this wave's
// tile loads older than its N youngest have landed and its LDS reads are done, so after the
// barrier the stage the loads filled may be read and the stage just read may be refilled.
template <int N>
__device__ __forceinline__ void mid_arrive() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ constexpr int mid_swz(int row) {
    return (((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1);
}

// How an operand lies in memory: K along its rows, K down its rows, or gathered windows
// (K along the rows, a row pointer per output row).
enum MidKind { kRowK = 0, kColK = 1, kGather = 2 };

struct MidOperand {
    const uint16_t* p;
    int64_t ld;
    int n;                // rows (kRowK, kGather) or columns (kColK) of the operand
    const int32_t* idx;   // kGather: window starts, row length F, rows R
    int64_t F, R;
};

// One operand's share of a stage: kR rows (or columns) x 64 K values.
template <int kR, int kind, int waves>
struct MidLoad {
    static constexpr int kIns = kR / 8;            // wave loads per stage: 64 16-byte slots each
    static constexpr int kPW = kIns / waves;
    static_assert(kIns % waves == 0, "loads divide over the waves");
    const uint16_t* src[kPW];
    int kpos[kPW];       // K offset of the lane's chunk inside a stage
    int64_t step;        // elements from one K step to the next
    uint32_t ok;         // kGather: bit k, the window lies inside X

    __device__ __forceinline__ void init(const MidOperand& o, int first, int K, int kt0, int wave, int lane) {
        step = kind == kColK ? 64 * o.ld : 64;
        ok = ~0u;
#pragma unroll
        for (int k = 0; k < kPW; ++k) {
            const int i = wave + waves * k;
            if constexpr (kind == kColK) {
                const int sub = i >> 3, kr = (i & 7) * 8 + (lane >> 3);
                int col = first + sub * 64 + (((lane & 7) ^ mid_swz(kr)) << 3);
                col = min(col, o.n - 8);           // columns past the end are never stored
                kpos[k] = kr;
                src[k] = o.p + ((int64_t)kt0 * 64 + kr) * o.ld + col;
            } else {
                const int r = i * 8 + (lane >> 3);
                const int c = ((lane & 7) ^ mid_swz(r)) << 3;
                const int m = min(first + r, o.n - 1);   // rows past the end are never stored
                kpos[k] = c;
                if constexpr (kind == kGather) {
                    const int64_t st = o.idx[m];
                    const bool in = st >= 0 && st * o.F + K <= o.R * o.F;
                    if (!in) ok &= ~(1u << k);
                    src[k] = o.p + (in ? st * o.F : 0) + c + kt0 * 64;
                } else {
                    src[k] = o.p + (int64_t)m * o.ld + c + kt0 * 64;
                }
            }
        }
    }
    // load k of the next stage into LDS at `dst` (bytes); left: the values of K from that stage on
    __device__ __forceinline__ void issue(int k, uint32_t dst, int left, int wave) {
        const void* p = src[k];
        bool in = true;
        if constexpr (kind == kGather) in = (ok >> k) & 1;
        if (left < 64) in = in && kpos[k] < left;
        if (kind == kGather || left < 64) p = in ? p : (const void*)g_zero_line;
        dma16(p, dst + (wave + waves * k) * 1024);
        src[k] += step;
    }
};

// MFMA operand reads from a stage (64 x kR, swizzled 128-byte rows)
template <int kind, bool natural>
struct MidRead {
    int o[4];
    __device__ __forceinline__ void init(int lane) {
        if constexpr (kind == kColK) {
            const int grp = lane >> 4, s = lane & 15;
            const int cl = 2 * (grp & 1) + ((s & 3) >> 1);
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int rb = natural ? 8 * (grp >> 1) + (s >> 2) + 4 * h : 4 * (grp >> 1) + (s >> 2) + 8 * h;
                    o[2 * m + h] = rb * 64 + (((4 * m + cl) ^ mid_swz(rb)) << 3) + 4 * (s & 1);
                }
        } else {
            const int l32 = lane & 31, p = (lane >> 5) ^ mid_swz(l32);
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = l32 * 64 + (((2 * c) ^ p) << 3);
        }
    }
    // rows (or columns) r0 .. r0 + 31 (r0 a multiple of 32), K chunk kc of 16
    __device__ __forceinline__ bf16x8 op(const uint16_t* tile, int r0, int kc) const {
        if constexpr (kind == kColK) {
            const uint16_t* t = tile + (r0 >> 6) * 4096 + kc * 1024;
            const int m = (r0 >> 5) & 1;
            // selected, not indexed: m differs between waves where a wave is 32 wide, and an array
            // indexed at run time goes to LDS (8 KB a workgroup: + 10 us a product)
            const int oa = m ? o[2] : o[0], ob = m ? o[3] : o[1];
            return cat8(lds_tr16(t + oa), lds_tr16(t + ob));
        } else {
            return *reinterpret_cast<const bf16x8*>(tile + r0 * 64 + o[kc]);
        }
    }
};

// acc[j][i]: C^T tiles (lane: row 32 i + l % 32, columns 32 j + 8 q + 4 (l / 32) + e) of the
// wave's (32 TI) x (32 TJ) part of a BM x BN tile over the K steps [kt0, kt1).  `stage_out`
// is called for every K step with the A stage (after its arrival).
template <int BM, int BN, int TI, int TJ, int AK, int BK, int NST, bool natural, class StageOut>
__device__ __forceinline__ void mid_product(const MidOperand& A, const MidOperand& B, int m0, int n0, int K, int kt0,
                                            int kt1, uint16_t* lds, int wave, int lane, int wm, int wn,
                                            f32x16 (&acc)[TJ][TI], StageOut&& stage_out) {
    constexpr int kWaves = (BM / (32 * TI)) * (BN / (32 * TJ));
    constexpr int kStage = (BM + BN) * 64;         // elements
    MidLoad<BM, AK, kWaves> la;
    MidLoad<BN, BK, kWaves> lb;
    constexpr int kPW = MidLoad<BM, AK, kWaves>::kPW + MidLoad<BN, BK, kWaves>::kPW;
    la.init(A, m0, K, kt0, wave, lane);
    lb.init(B, n0, K, kt0, wave, lane);
    MidRead<AK, natural> ra;
    MidRead<BK, natural> rb;
    ra.init(lane);
    rb.init(lane);
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    constexpr int kPA = MidLoad<BM, AK, kWaves>::kPW;
    auto issue = [&](int k, int kt, int st) {
        const uint32_t dst = base + st * (kStage * 2);
        if (k < kPA) la.issue(k, dst, K - 64 * kt, wave);
        else lb.issue(k - kPA, dst + BM * 128, K - 64 * kt, wave);
    };
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[j][i] = f32x16{};
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
        if (kt0 + s < kt1) {
#pragma unroll
            for (int k = 0; k < kPW; ++k) issue(k, kt0 + s, s);
        }
    int st = 0;
    for (int kt = kt0; kt < kt1; ++kt) {
        // stages kt + 1 .. kt + NST - 2 may stay in flight
        if (kt + 1 >= kt1) mid_arrive<0>();
        else if (NST > 3 && kt + 2 >= kt1) mid_arrive<kPW>();
        else mid_arrive<(NST - 2) * kPW>();
        const uint16_t* sa = lds + st * kStage;
        const uint16_t* sb = sa + BM * 64;
        const bool more = kt + NST - 1 < kt1;
        const int nst = st == 0 ? NST - 1 : st - 1;
        stage_out(kt, sa);
        bf16x8 av[2][TI], bv[2][TJ];
        auto read = [&](int kc) {
#pragma unroll
            for (int i = 0; i < TI; ++i) av[kc & 1][i] = ra.op(sa, wm + 32 * i, kc);
#pragma unroll
            for (int j = 0; j < TJ; ++j) bv[kc & 1][j] = rb.op(sb, wn + 32 * j, kc);
        };
        read(0);
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) {
            if (kc < 3) read(kc + 1);
#pragma unroll
            for (int ji = 0; ji < TJ * TI; ++ji) {
                const int j = ji / TI, i = ji - j * TI, slot = kc * TJ * TI + ji;
                // the next stage's loads, spread over the step's MFMAs
                if (more) {
#pragma unroll
                    for (int k = slot * kPW / (4 * TJ * TI); k < (slot + 1) * kPW / (4 * TJ * TI); ++k)
                        issue(k, kt + NST - 1, nst);
                }
                acc[j][i] = mfma32(bv[kc & 1][j], av[kc & 1][i], acc[j][i]);
            }
        }
        st = st + 1 == NST ? 0 : st + 1;
    }
    mid_arrive<0>();   // every wave is done with the stages: they become store scratch
}

struct MidArgs {
    MidOperand A, B;
    uint16_t* C;
    int64_t ldc;
    uint16_t* H;           // forward: the pre-activation, or the GELU derivative there
    int64_t ldh;
    const uint16_t* bias;
    const uint16_t* G;     // input gradient: the GELU derivative, or the pre-activation
    int64_t ldg;
    uint16_t* Xg;          // gathered rows out
    int64_t ldxg;
    float* part;           // weight gradient: slices x M x N fp32 partials (slices > 1)
    int M, N, K, slices;
    bool vec_c, vec_h;     // C / H rows start 16-byte aligned
};

enum MidTile { kMidNone = 0, kMidBig = 1, kMidSmall = 2 };   // 256 x 128; 64 x 128 (forward, input gradient) or 128 x 128

// launch (gemm_mid.hip); epi: bit 0 GELU, bit 1 H out, bit 2 bias, bit 4 (with 0 and 1) H is the
// GELU derivative
int mid_forward(const MidArgs& a, int tile, int epi, hipStream_t s);
// gate 0: dX = dY W (slices > 1: the slices' fp32 products, summed by the caller); 1: times
// gelu'(G); 2: times G
int mid_dgrad(const MidArgs& a, int tile, int gate, hipStream_t s);
// partials (slices > 1, summed by the caller) or C
int mid_wgrad(const MidArgs& a, int tile, hipStream_t s);
// modelled time of the forward / input gradient on the faster of the two tiles, in us
float mid_cost(int64_t M, int64_t N, int64_t K, int* tile);
float mid_wgrad_cost(int64_t M, int64_t N, int64_t K, int* tile, int* slices);

}  // namespace fx
