// w4_batch_kernels.hip - W4A16 linears of a decode batch for gfx950: more
// activation rows than the decode GEMVs take, fewer than fill the prefill
// GEMM's 128 x 256 tiles.
//
// y[m][n] = sum_k x[m][k] * (q[n][k] - z[n][g]) * s[n][g],  g = k / group.
//
// What bounds it: at these M the weights are read once (a few microseconds of
// HBM time) and the products are a few microseconds of matrix-core time if
// the chip is full, so the kernel is about filling it: 128 output columns per
// workgroup leave 14 to 224 workgroups for a whole K, and K is split, first
// over the wave groups of a workgroup (their sums meet in LDS), then over
// workgroups (their sums meet in memory, about 2.5 us).  What is left is
// latency more than any unit: the vector units are busy for 27 % of the
// cycles and the matrix cores for 10 at 16 rows (N = 4096, K = 14336), 26 and
// 36 at 96 (N = 6144, K = 4096); and a launch reads its code, 0.6 us per KB
// from a cold instruction cache.
// Measured (calls in a loop over eight sets of weights, before: 64-row slices
// of k_w4a16_gemv, k_w4a16_splitk and, with groups of 32 and 64,
// k_w4a16_generic):
//   N = 6144,  K = 4096:  M = 32 21.7 -> 10.9 us, 96 57.3 -> 18.0, 192 107 -> 25.5
//   N = 28672, K = 4096:  M = 32 79 -> 24.3 us, 96 195 -> 46
//   N = 4096,  K = 14336: M = 16 19.7 -> 16.6 us, 96 176 -> 30.3
//   N = 6144,  K = 4096, groups of 64: M = 16 459 -> 10.6 us, 96 2714 -> 18.5
#include <hip/hip_runtime.h>

#include <cstdint>

#include "codec.h"
#include "launch.h"
#include "../snx_internal.h"

using namespace snx;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

constexpr int BN = 128;         // output columns of a workgroup: 4 waves of 32
constexpr int BK = 128;         // columns of one step
constexpr int KW = 2;           // wave groups of a workgroup, each with a share of its K

// s_waitcnt of vmcnt `vm` and lgkmcnt 0 (expcnt not waited for)
constexpr int wait_imm(int vm) { return (vm & 15) | 0x70 | ((vm >> 4) << 14); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00020000);
}
// direct global -> LDS loads: lane l's bytes land at dst + 16 l (4 l)
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void lds_load4(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 4, voff, 0, 0, 0);
}

template <int MR> struct mfma_of;
template <> struct mfma_of<16> {
    typedef f32x4 acc_t;
    static __device__ __forceinline__ f32x4 mul(bf16x8 a, bf16x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct mfma_of<32> {
    typedef f32x16 acc_t;
    static __device__ __forceinline__ f32x16 mul(bf16x8 a, bf16x8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

// Eight nibbles of a packed word as bf16 16 + q, in column order: nibble 2r
// sits in byte r of w << 3 and nibble 2r + 1 in byte r of w >> 1, both at the
// top of the bf16 mantissa, so one v_perm and one v_and_or give a pair.
__device__ __forceinline__ bf16x8 nibbles16(uint32_t w, uint32_t mask, uint32_t bias) {
    const uint32_t even = w << 3, odd = w >> 1;
    u32x4 b;
    b[0] = (__builtin_amdgcn_perm(odd, even, 0x0c040c00u) & mask) | bias;
    b[1] = (__builtin_amdgcn_perm(odd, even, 0x0c050c01u) & mask) | bias;
    b[2] = (__builtin_amdgcn_perm(odd, even, 0x0c060c02u) & mask) | bias;
    b[3] = (__builtin_amdgcn_perm(odd, even, 0x0c070c03u) & mask) | bias;
    return __builtin_bit_cast(bf16x8, b);
}

// LDS of one stage of one wave group: MT * MR activation rows of 256 bytes
// (16-byte chunk c of row r at c ^ (r & 15)), 128 weight rows of 64 bytes
// (chunk c of row r at c ^ bsw(r)), 64 scale words and 64 zero words per wave.
__device__ __forceinline__ int bsw(int r) { return ((r >> 1) ^ (r >> 2)) & 3; }
constexpr int lds_a(int rows) { return rows * BK * 2; }
constexpr int OFF_S = BN * BK / 2, OFF_Z = OFF_S + 4 * 256, LDS_B = OFF_Z + 4 * 256;
constexpr int lds_stage(int rows) { return lds_a(rows) + LDS_B; }
constexpr int lds_bytes(int rows, int ring) { return KW * ring * lds_stage(rows); }

// (one argument: see k_q8_batch)
struct Args {
    const uint16_t* x;
    const uint32_t* qw;
    const uint16_t* scales;
    const uint32_t* qz;
    void* y;
    const float* bias;
    int y_f32, M, N, K, gshift, glu, per, extra;
    float* part;
    uint32_t* cnt;
};

// One workgroup: 4 KW waves.  Wave (nw, kw) computes output columns
// n0 + 32 nw .. + 31 for all MT * MR activation rows of the block over wave
// group kw's share of the workgroup's steps.  MR is the row count of the
// MFMA: 16 (16x16x32, for M <= 16) or 32 (32x32x16, twice its rate).
// GS columns (128, or the group when it is smaller) share a scale: per GS
// columns acc = sum x (16 + q) - sum x (16 + z), the two products of a word
// one after the other, and y += s acc.  The second product (a constant
// operand) doubles the matrix-core work, which is not what bounds the kernel,
// and keeps acc from growing to 16 times the sum of x: with 16 + q in place of
// the usual 128 + q (the nibble at the top of the bf16 mantissa instead of the
// bottom) the fp32 result is 9e-8 off at K = 4096, 1e-6 with the 128s.
// Every operand goes through LDS by direct loads, so the ring's depth costs
// no registers and each wait counts exactly the loads in flight.  A step's
// weight words, scales and first activation fragments are read from LDS
// before the last products of the step before it, so that their latency is
// covered.  The code is kept short on purpose: a launch runs it from a cold
// instruction cache.
// part / cnt (gridDim.y > 1 spans of K): the workgroups of a tile meet as in
// k_w4a16_gemm: results stored past the L2s, counted per wave, and summed in
// span order by the last wave to arrive; no wave waits for another.
template <int MR, int MT, int GS, int RING>
__global__ void __launch_bounds__(256 * KW) __attribute__((amdgpu_waves_per_eu(KW, KW))) k_w4a16_batch(
    const Args p) {
    const uint16_t *__restrict__ const x = p.x, *__restrict__ const scales = p.scales;
    const uint32_t *__restrict__ const qw = p.qw, *__restrict__ const qz = p.qz;
    void* __restrict__ const y = p.y;
    const float* __restrict__ const bias = p.bias;
    const int y_f32 = p.y_f32, M = p.M, N = p.N, K = p.K, gshift = p.gshift, glu = p.glu, per = p.per, extra = p.extra;
    float* __restrict__ const part = p.part;
    uint32_t* __restrict__ const cnt = p.cnt;
    typedef mfma_of<MR> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int ROWS = MT * MR, NS = 32 / MR, LQ = 64 / MR;   // NS column subtiles, LQ lane groups along k
    constexpr int UPS = BK / GS, WPU = GS / 8 / LQ, J = UPS * WPU;   // scale units per step, words per lane
    constexpr int SA = lds_a(ROWS), STAGE = lds_stage(ROWS);
    constexpr int AL = ROWS / 16;                               // activation loads per wave and stage
    constexpr int PER = AL + 4;
    constexpr int NE = MR == 32 ? 16 : 4;                       // results per lane and block
    constexpr int NP = NS * MT * NE / 4;                        // 16-byte result pieces per lane
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = wave & 3, kw = wave >> 2;
    const int r = lane & (MR - 1), q = lane / MR;
    const int tile = blockIdx.x, span = blockIdx.y, splits = gridDim.y;
    const int m0 = blockIdx.z * ROWS;
    // the wave's output columns c0 .. c0 + 31 of N, and the weight row of the
    // first (GLU: waves 2, 3 take the up rows N + .. of the columns whose gate
    // rows waves 0, 1 take)
    const int c0 = glu ? tile * (BN / 2) + 32 * (nw & 1) : tile * BN + 32 * nw;
    const int n0 = glu && nw >= 2 ? N : 0;

    // the workgroup's steps (per, one more in the first `extra` spans), and of
    // those this wave group's: [g0, g0 + ns)
    const int wg0 = span * per + (span < extra ? span : extra), wgn = per + (span < extra ? 1 : 0);
    const int g0 = wg0 + wgn * kw / KW, ns = wg0 + wgn * (kw + 1) / KW - g0;
    const int nmax = (wgn + KW - 1) / KW;                       // barriers of the loop: the same for all groups

    uint8_t* ring = lds + kw * (RING * STAGE);

    const uint32_t G = (uint32_t)K >> gshift, ZW = (G + 7) >> 3;
    const __amdgpu_buffer_rsrc_t rx = rsrc(x), rq = rsrc(qw), rs = rsrc(scales);
    const __amdgpu_buffer_rsrc_t rz = rsrc(qz ? (const void*)qz : (const void*)scales);
    // activations: load i of wave nw fills rows 4 (4 i + nw) .. + 3
    uint32_t ga[AL];
#pragma unroll
    for (int i = 0; i < AL; i++) {
        const int row = (4 * i + nw) * 4 + (lane >> 4);
        const int gr = m0 + row < M ? m0 + row : M - 1;
        ga[i] = (uint32_t)gr * (uint32_t)(K * 2) + (uint32_t)((lane & 15) ^ (row & 15)) * 16u;
    }
    // weights: load i fills rows 16 i .. + 15 of the wave's 32
    uint32_t gb[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = 16 * i + (lane >> 2), n = c0 + row;
        gb[i] = (uint32_t)(n0 + (n < N ? n : N - 1)) * (uint32_t)(K / 2) + (uint32_t)((lane & 3) ^ bsw(row)) * 16u;
    }
    const int ncol = c0 + (lane & 31), nc = n0 + (ncol < N ? ncol : N - 1);
    const uint32_t srow = (uint32_t)nc * G, zrow = (uint32_t)nc * ZW;
    // an odd number of scales has a last one that no aligned word within the
    // array holds: read by itself, by every wave (only groups of 128 and more
    // can leave an odd number)
    const uint32_t total = (uint32_t)(glu ? 2 * N : N) * G, lastw = (total & ~1u) - 2u;
    // (made scalar here, so that no wait for it sits among the loop's loads);
    // glast: its group, none where the number is even
    const uint32_t glast = total & 1u ? G - 1 : ~0u;
    const int last_row = (glu ? 2 * N : N) - 1;
    const float slast = GS == 128 && (total & 1u)
                            ? f16_dev((uint16_t)__builtin_amdgcn_readfirstlane(scales[total - 1])) : 0.0f;

    auto issue = [&](int slot, int t) {
        uint8_t* st = ring + slot * STAGE;
        const int kt = g0 + t;
#pragma unroll
        for (int i = 0; i < AL; i++) lds_load16(rx, st + (4 * i + nw) * 1024, ga[i], kt * (BK * 2));
#pragma unroll
        for (int i = 0; i < 2; i++) lds_load16(rq, st + SA + nw * 2048 + i * 1024, gb[i], kt * (BK / 2));
        // the aligned words that hold the step's scales (groups of 32: words
        // of units 0, 1 in lanes 0..31 and of units 2, 3 in lanes 32..63)
        const uint32_t g = ((uint32_t)kt * BK) >> gshift;
        const uint32_t si = srow + g + (GS == 32 ? 2u * (uint32_t)(lane >> 5) : 0u);
        lds_load4(rs, st + SA + OFF_S + nw * 256, ((si & ~1u) < lastw ? si & ~1u : lastw) * 2u);
        // without zero points the slot is filled and never read
        lds_load4(rz, st + SA + OFF_Z + nw * 256, qz ? (zrow + (g >> 3)) * 4u : 0u);
    };

    acc_t yv[NS][MT];
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int i = 0; i < MT; i++) yv[s][i] = acc_t{};
    uint32_t mask, biasw;
    asm volatile("s_mov_b32 %0, 0x780078" : "=s"(mask));
    asm volatile("v_mov_b32 %0, 0x41804180" : "=v"(biasw));

    // what a step reads from its stage ahead of its products
    uint32_t wd[NS][J], sw[NS][2], zw[NS];
    bf16x8 f0[MT];
    auto chunk = [&](int j) { return ((j / WPU) * (GS / 8) + q * WPU + j % WPU) ^ (r & 15); };
    const uint8_t* st;
    auto frag = [&](int i, int j) {
        return *reinterpret_cast<const bf16x8*>(st + (i * MR + r) * (BK * 2) + (chunk(j) << 4));
    };
    auto begin = [&](int slot) {
        st = ring + slot * STAGE;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int row = s * MR + r;
            const uint8_t* wrow = st + SA + nw * 2048 + row * 64;
#pragma unroll
            for (int u = 0; u < UPS; u++) {
                const int w0 = u * (GS / 8) + q * WPU;          // first word of this lane in the unit
                if constexpr (WPU >= 4) {
#pragma unroll
                    for (int c = 0; c < WPU / 4; c++) {
                        const u32x4 v = *reinterpret_cast<const u32x4*>(wrow + (((w0 / 4 + c) ^ bsw(row)) << 4));
#pragma unroll
                        for (int e = 0; e < 4; e++) wd[s][u * WPU + 4 * c + e] = v[e];
                    }
                } else {
                    const uint8_t* p = wrow + (((w0 >> 2) ^ bsw(row)) << 4) + (w0 & 3) * 4;
                    if constexpr (WPU == 2) {
                        const uint2 v = *reinterpret_cast<const uint2*>(p);
                        wd[s][u * WPU] = v.x;
                        wd[s][u * WPU + 1] = v.y;
                    } else {
                        wd[s][u] = *reinterpret_cast<const uint32_t*>(p);
                    }
                }
            }
            const uint32_t* sl = reinterpret_cast<const uint32_t*>(st + SA + OFF_S + nw * 256);
            sw[s][0] = sl[row];
            sw[s][1] = GS == 32 ? sl[32 + row] : 0u;
            zw[s] = reinterpret_cast<const uint32_t*>(st + SA + OFF_Z + nw * 256)[row];
        }
#pragma unroll
        for (int i = 0; i < MT; i++) f0[i] = frag(i, 0);
    };
    // s_waitcnt until at most `newer` stages of this wave's loads are in flight
    auto landed = [&](int newer) {
        if (RING > 4 && newer >= 4) __builtin_amdgcn_s_waitcnt(wait_imm(4 * PER));
        else if (RING > 3 && newer >= 3) __builtin_amdgcn_s_waitcnt(wait_imm(3 * PER));
        else if (RING > 2 && newer >= 2) __builtin_amdgcn_s_waitcnt(wait_imm(2 * PER));
        else if (newer >= 1) __builtin_amdgcn_s_waitcnt(wait_imm(PER));
        else __builtin_amdgcn_s_waitcnt(wait_imm(0));
    };

#pragma unroll 1
    for (int p = 0; p < RING && p < ns; p++) issue(p, p);
    landed(ns - 1 < RING - 1 ? ns - 1 : RING - 1);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    begin(0);
    int slot = 0;
#pragma unroll 1
    for (int t = 0; t < nmax; t++) {
        acc_t acc[NS][MT];
        float sc[UPS][NS];
        uint32_t zc[UPS][NS];
        const uint32_t gq = ((uint32_t)(g0 + t) * BK) >> gshift;   // the step's first group
        // products of word j (fragments in fa), then the unit's fold after its last word
        auto mul = [&](int j, const bf16x8 (&fa)[MT]) {
            const int u = j / WPU;
            if (j % WPU == 0) {
#pragma unroll
                for (int s = 0; s < NS; s++)
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[s][i] = acc_t{};
            }
            bf16x8 fb[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) fb[s] = nibbles16(wd[s][j], mask, biasw);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int s = 0; s < NS; s++) acc[s][i] = MF::mul(fa[i], fb[s], acc[s][i]);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const uint32_t nz = (zc[u][s] << 3 | 0xC180u) * 0x10001u;   // bf16 -(16 + z), twice
                const u32x4 nzv = {nz, nz, nz, nz};
#pragma unroll
                for (int i = 0; i < MT; i++) acc[s][i] = MF::mul(fa[i], __builtin_bit_cast(bf16x8, nzv), acc[s][i]);
            }
        };
        auto fold = [&](int u) {
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int e = 0; e < NE; e++) yv[s][i][e] = __builtin_fmaf(sc[u][s], acc[s][i][e], yv[s][i][e]);
        };
        const bool live = t < ns;
        bf16x8 fl[MT];                 // the fragments of the next word
#pragma unroll
        for (int i = 0; i < MT; i++) fl[i] = f0[i];
        if (live) {
            // scales of the step: groups of 128 and more take the half of the
            // word that the group's index picks, smaller ones start at a word
#pragma unroll
            for (int u = 0; u < UPS; u++)
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const int n = c0 + s * MR + r;
                    const uint32_t half = GS == 128 ? ((uint32_t)(n0 + (n < N ? n : N - 1)) * G + gq) & 1u : (uint32_t)(u & 1);
                    const uint32_t word = GS == 32 ? sw[s][u >> 1] : sw[s][0];
                    zc[u][s] = qz ? (zw[s] >> (4 * ((gq + (GS == 128 ? 0 : u)) & 7))) & 15u : 8u;
                    sc[u][s] = f16_dev((uint16_t)(word >> (16 * half)));
                    if (GS == 128 && gq == glast && n0 + n >= last_row) sc[u][s] = slast;
                }
#pragma unroll
            for (int j = 0; j < J - 1; j++) {
                bf16x8 fn[MT];
#pragma unroll
                for (int i = 0; i < MT; i++) fn[i] = frag(i, j + 1);
                mul(j, fl);
                if ((j + 1) % WPU == 0) fold(j / WPU);
#pragma unroll
                for (int i = 0; i < MT; i++) fl[i] = fn[i];
            }
        }
        uint32_t wlast[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) wlast[s] = wd[s][J - 1];
        // stage t + 1 landed (newer ones may fly); this wave is done reading stage t
        {
            const int newest = t + RING - 1 < ns - 1 ? t + RING - 1 : ns - 1;
            landed(newest - (t + 1));
        }
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t + RING < ns) issue(slot, t + RING);
        slot = slot + 1 == RING ? 0 : slot + 1;
        if (t + 1 < ns) begin(slot);
        if (live) {
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const uint32_t keep = wd[s][J - 1];
                wd[s][J - 1] = wlast[s];
                wlast[s] = keep;
            }
            mul(J - 1, fl);
#pragma unroll
            for (int s = 0; s < NS; s++) wd[s][J - 1] = wlast[s];
            fold(UPS - 1);
        }
    }
    __builtin_amdgcn_s_waitcnt(wait_imm(0));
    __builtin_amdgcn_s_barrier();

    // the wave groups' sums meet in LDS: [KW][4][NP][64] pieces; wave (nw, kw)
    // then owns pieces kw, kw + KW, ... of its columns
    constexpr int OWN = NP / KW;
    static_assert(NP % KW == 0 && KW * 4 * NP * 1024 <= KW * RING * STAGE, "the sums fit where the rings were");
    f32x4 res[OWN];
    f32x4* red = reinterpret_cast<f32x4*>(lds) + nw * NP * 64 + lane;
    {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int s = p % NS, i = (p / NS) % MT, v = p / (NS * MT);
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = yv[s][i][MR == 32 ? 4 * v + e : e];
            red[(kw * 4 * NP + p) * 64] = o;
        }
        __builtin_amdgcn_s_waitcnt(wait_imm(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int p = kw + o * KW;
            res[o] = red[p * 64];
#pragma unroll
            for (int k = 1; k < KW; k++) res[o] += red[(k * 4 * NP + p) * 64];
        }
    }

    // GLU: the wave that writes a column's output takes gate and up, from slots
    // (nw & 1) and (nw & 1) + 2 of the workgroup
    f32x4 up[OWN] = {};
    if (splits > 1) {
        constexpr int kSysCoherent = 1 | 16;            // buffer cache policy sc0 sc1
        constexpr uint32_t SLOTB = 4 * KW * OWN * 1024; // bytes of one workgroup's results
        const uint32_t tl = blockIdx.z * gridDim.x + tile;
        const __amdgpu_buffer_rsrc_t rp = rsrc(part);
        const uint32_t first = tl * (uint32_t)splits * SLOTB;
        auto slot_of = [&](int w) { return first + (uint32_t)(w * OWN) * 1024u; };
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const float e0 = res[o][0], e1 = res[o][1], e2 = res[o][2], e3 = res[o][3];
            const u32x4 v = {__builtin_bit_cast(uint32_t, e0), __builtin_bit_cast(uint32_t, e1),
                             __builtin_bit_cast(uint32_t, e2), __builtin_bit_cast(uint32_t, e3)};
            __builtin_amdgcn_raw_buffer_store_b128(v, rp, lane * 16, slot_of(wave) + (uint32_t)span * SLOTB + o * 1024, kSysCoherent);
        }
        // written before counted (see k_w4a16_gemm)
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0f70);             // vmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        const int first_wave = glu ? (wave & ~2) : wave, arrivals = glu ? 2 * splits : splits;
        uint32_t* mine = cnt + (size_t)tl * (4 * KW) + first_wave;
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(mine, 1u);
        if ((int)__builtin_amdgcn_readfirstlane(c) != arrivals - 1) return;
        __builtin_amdgcn_sched_barrier(0);
        if (lane == 0) atomicExch(mine, 0u);            // ready for the next call
        // the spans' results in span order, CH spans' loads in flight together
        // (a load past the last span repeats it and is not added)
        constexpr int CH = OWN >= 4 ? 4 : 8;
#pragma unroll 1
        for (int w = first_wave; w <= first_wave + (glu ? 2 : 0); w += 2) {
            f32x4 sum[OWN] = {};
#pragma unroll 1
            for (int s0 = 0; s0 < splits; s0 += CH) {
                u32x4 v[CH][OWN];
#pragma unroll
                for (int c2 = 0; c2 < CH; c2++)
#pragma unroll
                    for (int o = 0; o < OWN; o++)
                        v[c2][o] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                            rp, lane * 16, slot_of(w) + (uint32_t)(s0 + c2 < splits ? s0 + c2 : splits - 1) * SLOTB + o * 1024, kSysCoherent));
#pragma unroll
                for (int c2 = 0; c2 < CH; c2++)
                    if (s0 + c2 < splits)
#pragma unroll
                        for (int o = 0; o < OWN; o++)
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const uint32_t d = v[c2][o][e];
                                sum[o][e] += __builtin_bit_cast(float, d);
                            }
            }
#pragma unroll
            for (int o = 0; o < OWN; o++) {
                if (w == first_wave) res[o] = sum[o];
                else up[o] = sum[o];
            }
        }
    } else if (glu) {
        // a piece's place is read by its own wave alone: the up sums go back there
        if (nw >= 2)
#pragma unroll
            for (int o = 0; o < OWN; o++) red[(kw + o * KW) * 64] = res[o];
        __builtin_amdgcn_s_waitcnt(wait_imm(0));
        __builtin_amdgcn_s_barrier();
        if (nw >= 2) return;
#pragma unroll
        for (int o = 0; o < OWN; o++) up[o] = red[(2 * NP + kw + o * KW) * 64];
    }

    // rows past M lie past the buffer's records and are dropped there; lanes
    // of columns past N take an offset that is
    auto finish = [&] {
        const uint32_t eb = y_f32 ? 4 : 2;
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y, (short)0, (int)((uint32_t)M * (uint32_t)N * eb), 0x00020000);
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int p = kw + o * KW;
            const int s = p % NS, i = (p / NS) % MT, v = p / (NS * MT);
            const int n = c0 + s * MR + r, m = m0 + i * MR + (MR == 32 ? 8 * v + 4 * q : 4 * q);
            uint32_t off = n < N ? ((uint32_t)m * (uint32_t)N + (uint32_t)n) * eb : 0x80000000u;
            if (bias) res[o] += bias[n < N ? n : N - 1];
            if (glu) {
                if (bias) up[o] += bias[N + (n < N ? n : N - 1)];
#pragma unroll
                for (int e = 0; e < 4; e++) res[o][e] = silu_mul_fast(res[o][e], up[o][e]);
            }
            if (y_f32) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float f = res[o][e];
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, f), ry, off, 0, 0);
                    off += (uint32_t)N * 4u;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    __builtin_amdgcn_raw_buffer_store_b16(bf16_out(res[o][e]), ry, off, 0, 0);
                    off += (uint32_t)N * 2u;
                }
            }
        }
    };

    // An infinite activation (or one past 1e37) makes both products infinite and
    // their difference NaN where sum x (q - z) s is an infinity or a number.  A
    // wave with a result that is not finite computes its columns once more in
    // that form, straight from memory, and takes from it what was not finite:
    // codes as bf16 (q - z) 2^-16, whose products with any activation are finite,
    // 32 rows at a time, as K / GS round trips to memory whatever the number of
    // such results.  N = 6144, K = 4096, groups of 64, M = 96: 0.29 ms with one
    // row of them, 0.51 with 96 (k_w4a16_generic, which these groups ran before,
    // 2.7); N = 4096, K = 11008, groups of 128: 0.59 and 0.97 (7.6).  It stores
    // its results itself: calls without such results then pay for the test alone
    // (0.1 us at 96 rows; 0.8 where the two ways met before the stores).
    f32x4 odd = {};                 // NaN where a result is not finite
#pragma unroll
    for (int o = 0; o < OWN; o++)
#pragma unroll
        for (int e = 0; e < 4; e++) odd[e] = __builtin_fmaf(0.0f, res[o][e], odd[e]);
    if (glu) {
#pragma unroll
        for (int o = 0; o < OWN; o++)
#pragma unroll
            for (int e = 0; e < 4; e++) odd[e] = __builtin_fmaf(0.0f, up[o][e], odd[e]);
    }
    const float any = (odd[0] + odd[1]) + (odd[2] + odd[3]);
    if (__builtin_expect(__ballot(any != any) != 0, 0)) {
        constexpr int RB = MR / 16;             // blocks of 16 rows, by two of 16 columns
        const int c16 = lane & 15, q16 = lane >> 4;
#pragma unroll 1
        for (int half = 0; half <= glu; half++) {
            size_t row[2];
#pragma unroll
            for (int cb = 0; cb < 2; cb++) {
                const int n = c0 + 16 * cb + c16;
                row[cb] = (size_t)(n < N ? n : N - 1) + (half ? (size_t)N : 0);
            }
#pragma unroll 1
            for (int i = 0; i < MT; i++) {
                const uint16_t* xr[RB];
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    const int m = m0 + i * MR + 16 * rb + c16;
                    xr[rb] = x + (size_t)(m < M ? m : M - 1) * (size_t)K + 8 * q16;
                }
                f32x4 sum[RB][2] = {};
#pragma unroll 1
                for (int u = 0; u < K / GS; u++) {
                    const uint32_t g = (uint32_t)(u * GS) >> gshift;
                    f32x4 acc[RB][2] = {};
                    int z[2];
                    float sc[2];
#pragma unroll
                    for (int cb = 0; cb < 2; cb++) {
                        z[cb] = qz ? (int)((qz[row[cb] * ZW + (g >> 3)] >> (4 * (g & 7))) & 15u) : 8;
                        sc[cb] = f16_dev(scales[row[cb] * G + g]) * 65536.0f;
                    }
#pragma unroll
                    for (int j = 0; j < GS / 32; j++) {
                        bf16x8 a[RB];
#pragma unroll
                        for (int rb = 0; rb < RB; rb++) a[rb] = *reinterpret_cast<const bf16x8*>(xr[rb] + u * GS + 32 * j);
#pragma unroll
                        for (int cb = 0; cb < 2; cb++) {
                            const uint32_t word = qw[row[cb] * (size_t)(K / 8) + (u * GS / 8 + 4 * j + q16)];
                            u32x4 c;
#pragma unroll
                            for (int t = 0; t < 4; t++) {
                                const float lo = (float)((int)((word >> (8 * t)) & 15u) - z[cb]) * 0x1p-16f;
                                const float hi = (float)((int)((word >> (8 * t + 4)) & 15u) - z[cb]) * 0x1p-16f;
                                c[t] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
                            }
#pragma unroll
                            for (int rb = 0; rb < RB; rb++) acc[rb][cb] = mfma_of<16>::mul(a[rb], __builtin_bit_cast(bf16x8, c), acc[rb][cb]);
                        }
                    }
#pragma unroll
                    for (int rb = 0; rb < RB; rb++)
#pragma unroll
                        for (int cb = 0; cb < 2; cb++)
#pragma unroll
                            for (int e = 0; e < 4; e++) sum[rb][cb][e] = __builtin_fmaf(sc[cb], acc[rb][cb][e], sum[rb][cb][e]);
                }
                // rows 4 q16 .. + 3 of column c16 of a block, to the places in LDS of the
                // wave's own pieces (which no other wave reads) in the order of res
#pragma unroll
                for (int rb = 0; rb < RB; rb++)
#pragma unroll
                    for (int cb = 0; cb < 2; cb++) {
                        const int piece = MR == 32 ? MT * (2 * rb + (q16 >> 1)) + i : cb;
                        const int to = MR == 32 ? 32 * (q16 & 1) + 16 * cb + c16 : lane;
                        if (piece % KW == kw) red[piece * 64 + to - lane] = sum[rb][cb];
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int o = 0; o < OWN; o++) {
                const f32x4 f = red[(kw + o * KW) * 64];
                float a[4], b[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    a[e] = half || __builtin_isfinite(res[o][e]) ? res[o][e] : f[e];
                    b[e] = !half || __builtin_isfinite(up[o][e]) ? up[o][e] : f[e];
                }
                res[o] = f32x4{a[0], a[1], a[2], a[3]};
                up[o] = f32x4{b[0], b[1], b[2], b[3]};
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        finish();
        return;
    }
    finish();
}

struct Batch {
    const uint16_t* x;
    const uint32_t* qw;
    const uint16_t* scales;
    const uint32_t* qz;
    void* y;
    const float* bias;
    int y_f32, M, N, K, gshift, glu, splits;
    float* part;
    uint32_t* cnt;
    hipStream_t s;
};

template <int MR, int MT, int GS, int RING>
int launch(const Batch& a) {
    constexpr int bytes = lds_bytes(MT * MR, RING);
    static_assert(bytes <= 160 * 1024, "LDS of a workgroup");
    static std::atomic<uint64_t> lds_done{0};
    const void* fn = reinterpret_cast<const void*>(&k_w4a16_batch<MR, MT, GS, RING>);
    if (bytes > 64 * 1024 && snx::lds_optin(fn, bytes, lds_done) != hipSuccess) {
        snx_set_error("w4a16 batch: cannot reserve %d bytes of LDS", bytes);
        return -1;
    }
    const int cols = a.glu ? BN / 2 : BN;
    const dim3 grid((a.N + cols - 1) / cols, a.splits, (a.M + MT * MR - 1) / (MT * MR));
    const int steps = a.K / BK;
    k_w4a16_batch<MR, MT, GS, RING><<<grid, 256 * KW, bytes, a.s>>>(
        Args{a.x, a.qw, a.scales, a.qz, a.y, a.bias, a.y_f32, a.M, a.N, a.K, a.gshift, a.glu, steps / a.splits,
             steps % a.splits, a.part, a.cnt});
    return snx_launch_check("k_w4a16_batch");
}

// rows of a block
int rows_of(int M) {
    if (M <= 16) return 16;
    const int blocks = (M + 95) / 96;
    return ((M + blocks - 1) / blocks + 31) / 32 * 32;
}

template <int GS>
int launch_rows(const Batch& a) {
    switch (rows_of(a.M)) {
        case 16: return launch<16, 1, GS, 5>(a);
        case 32: return launch<32, 1, GS, 4>(a);
        case 64: return launch<32, 2, GS, 2>(a);
        default: return launch<32, 3, GS, 2>(a);
    }
}

}  // namespace

extern "C" {

int snx_w4a16_batch_ok(size_t M, size_t N, size_t K, int group, const void* scales, const void* qz) {
    if (M < 1 || K % BK != 0 || group < 32 || (group & (group - 1)) != 0 || K % (size_t)group != 0) return 0;
    const size_t G = K / (size_t)group;
    // scales are read as aligned words of two; 31-bit buffer offsets
    return N * G >= 2 && ((uintptr_t)scales & 3u) == 0 && ((uintptr_t)qz & 3u) == 0 &&
           M * K * 2 < (1ull << 31) && N * K / 2 < (1ull << 31) && N * G * 2 < (1ull << 31) &&
           (M + 96) * N * 4 < (1ull << 31) && M <= 96 * 65535ull;
}

// Spans of K: as many as the CUs take at once (one workgroup's LDS is most of
// a CU's), and no more than pay: a span takes its share off the steps and adds
// its results to the meeting; the best counts measured lie near sqrt(4/3
// steps), and K = 512 stays whole (N = 1792, M = 8: 4.5 us, 2 spans 5.8).  64
// rows and more meet four spans at a time.
// N = 6144, K = 4096, M = 16: 1 span 17.9 us, 2 13.3, 4 10.5, 5 9.7, 6 (288
// workgroups, more than the CUs) 13.1; N = 961, M = 8: K = 2048 1 span 10.3, 2
// 9.0, 4 7.4, 6 7.0, 8 7.7; K = 8192 4 spans 14.4, 8 11.6, 12 11.7, 16 12.5.
int snx_w4a16_batch_splits(size_t M, size_t N, size_t K) {
    const size_t rows = (size_t)rows_of((int)M), ncu = (size_t)snx::cu_count(), steps = K / BK;
    const size_t units = ((N + BN - 1) / BN) * ((M + rows - 1) / rows), most = steps < 8 ? 1 : steps / KW;
    size_t s = ncu / units;
    if (s > most) s = most;
    while (s > 1 && 3 * s * (s - 1) >= 4 * steps) s--;
    if (rows >= 64 && s > 4) s -= s % 4;
    return s < 1 ? 1 : (int)s;
}

// Estimated time in units of 0.1 us, to set against the prefill GEMM's: a
// fixed part, the meeting of the spans, and for each round of the CUs its
// start and the steps of a wave group (0.9 us with 16 rows, 1.0, 1.6 and 2.2
// with 32, 64 and 96).  N = 7168, K = 3584 at M = 320, 394, 1049 (1, 2, 3
// rounds): 35.4, 65.0, 100 us measured, 35.3, 68.6, 102 estimated.
size_t snx_w4a16_batch_cost(size_t M, size_t N, size_t K) {
    const int rows = rows_of((int)M), splits = snx_w4a16_batch_splits(M, N, K);
    const size_t ncu = (size_t)snx::cu_count();
    const size_t units = ((N + BN - 1) / BN) * ((M + rows - 1) / rows) * splits;
    const size_t steps = (K / BK + (size_t)splits * KW - 1) / ((size_t)splits * KW);
    const size_t step = rows == 16 ? 9 : rows == 32 ? 10 : rows == 64 ? 16 : 22;
    const size_t meet = splits == 1 ? 0 : rows < 96 ? 25 : 20 + 10 * (size_t)splits;
    return 20 + meet + (units + ncu - 1) / ncu * (25 + steps * step);
}

// Whether whole-K workgroups are more than a round of the CUs and leave more than
// a sixth of their rounds idle.
int snx_w4a16_batch_uneven(size_t M, size_t N) {
    const size_t rows = (size_t)rows_of((int)M), ncu = (size_t)snx::cu_count();
    const size_t units = ((N + BN - 1) / BN) * ((M + rows - 1) / rows);
    return units > ncu && 6 * units < 5 * ncu * ((units + ncu - 1) / ncu);
}

size_t snx_w4a16_batch_part_bytes(size_t M, size_t N, int splits) {
    const size_t rows = (size_t)rows_of((int)M), tiles = ((N + BN - 1) / BN) * ((M + rows - 1) / rows);
    return tiles * (size_t)splits * rows * BN * sizeof(float);
}
size_t snx_w4a16_batch_cnt_bytes(size_t M, size_t N) {
    const size_t rows = (size_t)rows_of((int)M), tiles = ((N + BN - 1) / BN) * ((M + rows - 1) / rows);
    return tiles * 4 * KW * sizeof(uint32_t);
}

// glu: qw holds the stacked [2N][K] gate/up rows, y bf16 [M][N]; splits, part
// and cnt are those of M x 2N x K
int snx_k_w4a16_batch(const uint16_t* x, const uint32_t* qw, const uint16_t* scales, const uint32_t* qzeros,
                      void* y, const float* bias, int y_f32, size_t M, size_t N, size_t K, int group, int glu,
                      int splits, void* part, uint32_t* cnt, void* st) {
    if (!snx_w4a16_batch_ok(M, glu ? 2 * N : N, K, group, scales, qzeros) || (splits > 1 && (!part || !cnt)) ||
        (glu && y_f32)) {
        snx_set_error("w4a16 batch: M=%zu N=%zu K=%zu group %d is not a shape of this kernel", M, N, K, group);
        return -1;
    }
    const Batch a{x, qw, scales, qzeros, y, bias, y_f32, (int)M, (int)N, (int)K, __builtin_ctz((unsigned)group),
                  glu, splits, (float*)part, cnt, S(st)};
    if (group == 32) return launch_rows<32>(a);
    if (group == 64) return launch_rows<64>(a);
    return launch_rows<128>(a);
}

}  // extern "C"
