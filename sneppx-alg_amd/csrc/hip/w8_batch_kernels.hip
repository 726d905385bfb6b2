// w8_batch_kernels.hip - W8 weight-only linears with more than one row of
// fp32 activations, on the bf16 matrix cores of gfx950.
//
// y[m][n] = s[n] * sum_k x[m][k] * q[n][k] (+ bias[n]), q int8.
//
// An fp32 value is exactly p0 + 2^-8 p1 + 2^-16 p2 with bf16 p0, p1, p2 (its 24
// significant bits cut into 8 + 8 + 8, the later pieces scaled up so that they
// are bf16 values also where x is tiny or subnormal) and an int8 is exactly
// one, so three bf16 products with fp32 accumulation compute what fp32
// arithmetic does.  1. k_w8_split_x writes the pieces once; 2. k_w8_batch
// multiplies.  The leading pieces' products meet in accumulators that are added
// to the result every 128 columns, the second and third ones' (with their
// scales a 256th and a 65536th of the size) in their own: the sum's error stays
// that of short fp32 chains, 7e-8 at K = 2048 for activations of any size down to
// 1e-40 (the fp32 kernel's is 1.3e-7).  Pieces that are not scaled share one
// accumulator (53.5 against 53.8 us at 384 rows), but lose the low bits of x
// below 2^-110 and all of it below 2^-133.  Measured at N = K = 4096 (before: k_w8_gemv, one row after the
// other on the vector units): M = 16 94 -> 15.6 us, 64 371 -> 19.3, 384
// 2490 -> 58.
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

constexpr int BK = 64;          // columns of a step
constexpr int XSTEP = 3 * BK * 2;   // bytes of a row's three pieces of a step

// s_waitcnt of vmcnt `vm` and lgkmcnt 0 (expcnt not waited for)
constexpr int wait_imm(int vm) { return (vm & 15) | 0x70 | ((vm >> 4) << 14); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, voff, soff, 0, 0);
}

// ------------------------------------------------------- activation pieces
// xp [M][steps][3][64] bf16: piece p of the 64 columns of a step, zero past K.
// One thread per 4 columns; each piece is the top 16 bits of what is left, times
// 2^8 after each (cut, not rounded: no piece overflows, and the third is exact).
// An infinity or NaN is its first piece alone.
__global__ void __launch_bounds__(256) k_w8_split_x(const float* __restrict__ x, uint16_t* __restrict__ xp, int K,
                                                    uint32_t items, uint32_t per_row) {
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    if (it >= items) return;
    const uint32_t m = it / per_row, k = (it - m * per_row) * 4;
    const float* xr = x + (size_t)m * (size_t)K;
    uint32_t p[3][2] = {};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float v = k + e < (uint32_t)K ? xr[k + e] : 0.0f;
        uint32_t b = f2u(v);
        if ((b & 0x7F800000u) == 0x7F800000u) {
            p[0][e >> 1] |= ((b >> 16) | ((b & 0x7FFFFFu) ? 0x40u : 0u)) << (16 * (e & 1));
            continue;
        }
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const uint32_t hi = f2u(v) & 0xFFFF0000u;
            p[i][e >> 1] |= (e & 1) ? hi : hi >> 16;
            v = (v - u2f(hi)) * 256.0f;     // exact: the bits that were cut off
        }
    }
    uint16_t* o = xp + ((size_t)m * (per_row / 16) + k / BK) * (3 * BK) + k % BK;
#pragma unroll
    for (int i = 0; i < 3; i++) *reinterpret_cast<uint2*>(o + i * BK) = make_uint2(p[i][0], p[i][1]);
}

// ----------------------------------------------------------------- the GEMM
// LDS of one stage of one wave group: three planes of 32 MT activation rows of
// 128 bytes (16-byte chunk c of row r at c ^ ((r >> 1) & 7)), 128 weight rows
// of 64 bytes (chunk c of row r at c ^ bsw(r)).
__device__ __forceinline__ int bsw(int r) { return ((r >> 1) ^ (r >> 2)) & 3; }
constexpr int BN = 128;         // output columns of a workgroup: 4 waves of 32
template <int MT>
struct layout {
    static constexpr int PLANE = 32 * MT * 128, A = 3 * PLANE, W = BN * 64, STAGE = A + W;
};

// (one argument: see k_q8_batch)
struct Args {
    const uint16_t* xp;
    const int8_t* qw;
    const float *scales, *bias;
    float* y;
    int M, N, K, per, extra;
    float* part;
    uint32_t* cnt;
};

// four int8 of a word as two registers of bf16 pairs (exact)
__device__ __forceinline__ void bytes_to_bf16(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const float f0 = (float)(int8_t)w, f1 = (float)(int8_t)(w >> 8);
    const float f2 = (float)(int8_t)(w >> 16), f3 = (float)(int8_t)(w >> 24);
    lo = __builtin_amdgcn_perm(f2u(f1), f2u(f0), 0x07060302u);
    hi = __builtin_amdgcn_perm(f2u(f3), f2u(f2), 0x07060302u);
}

// One workgroup: 4 KW waves; wave (nw, kw) computes 32 MT rows x 32 columns over
// wave group kw's share of the workgroup's K.  What bounds it: at 384 rows the
// LDS reads of the activation pieces (one fragment per product, as much as
// LDS delivers), at few rows the fixed parts.  64 x 64 per wave (a fragment
// for two products) leaves one wave per SIMD its registers and measured
// slower: 62 against 58 us at 384 rows, 35 against 21 at 64 (N = K = 4096).
// K is split over wave groups and workgroups as in k_w4a16_batch, whose
// comments cover what is not said here.
template <int MT, int KW, int RING>
__global__ void __launch_bounds__(256 * KW) __attribute__((amdgpu_waves_per_eu(KW, KW))) k_w8_batch(
    const Args p) {
    const uint16_t* __restrict__ const xp = p.xp;
    const int8_t* __restrict__ const qw = p.qw;
    const float *__restrict__ const scales = p.scales, *__restrict__ const bias = p.bias;
    float *__restrict__ const y = p.y, *__restrict__ const part = p.part;
    uint32_t* __restrict__ const cnt = p.cnt;
    const int M = p.M, N = p.N, K = p.K, per = p.per, extra = p.extra;
    typedef layout<MT> L;
    constexpr int AL = 3 * MT, WL = 2, PER = AL + WL;
    constexpr int NP = 4 * MT, OWN = NP / KW;     // 16-byte result pieces per lane, and those a wave finishes
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = wave & 3, kw = wave >> 2;
    const int r = lane & 31, h = lane >> 5;
    const int tile = blockIdx.x, span = blockIdx.y, splits = gridDim.y;
    const int m0 = blockIdx.z * (32 * MT), n0 = tile * BN + 32 * nw;

    const int wg0 = span * per + (span < extra ? span : extra), wgn = per + (span < extra ? 1 : 0);
    const int g0 = wg0 + wgn * kw / KW, ns = wg0 + wgn * (kw + 1) / KW - g0;
    const int nmax = (wgn + KW - 1) / KW;
    const uint32_t xrow = (uint32_t)((K + BK - 1) / BK) * XSTEP;

    uint8_t* ring = lds + kw * (RING * L::STAGE);
    const __amdgpu_buffer_rsrc_t rx = rsrc(xp, (uint32_t)M * xrow), rq = rsrc(qw, (uint32_t)N * (uint32_t)K);
    // activations: load i of a plane fills rows 8 (4 i + nw) .. + 7
    uint32_t ga[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = 8 * (4 * i + nw) + (lane >> 3), gr = m0 + row < M ? m0 + row : M - 1;
        ga[i] = (uint32_t)gr * xrow + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
    // weights: load i fills rows 16 i .. + 15 of the wave's columns.  Columns
    // past K read the next row's (or nothing): they meet zero activations.
    uint32_t gb[WL];
#pragma unroll
    for (int i = 0; i < WL; i++) {
        const int row = 16 * i + (lane >> 2), n = n0 + row;
        gb[i] = (uint32_t)(n < N ? n : N - 1) * (uint32_t)K + (uint32_t)((lane & 3) ^ bsw(row)) * 16u;
    }
    auto issue = [&](int slot, int t) {
        uint8_t* st = ring + slot * L::STAGE;
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < MT; i++)
                lds_load16(rx, st + p * L::PLANE + (4 * i + nw) * 1024, ga[i], (g0 + t) * XSTEP + p * 128);
#pragma unroll
        for (int i = 0; i < WL; i++)
            lds_load16(rq, st + L::A + nw * 2048 + i * 1024, gb[i], (g0 + t) * BK);
    };

    // the result, the leading pieces' sums of 128 columns, the second and third ones'
    f32x16 yv[MT], ah[MT], am[MT], al[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) yv[i] = ah[i] = am[i] = al[i] = f32x16{};

    // what a step reads from its stage ahead of its products
    u32x4 wd[2];
    bf16x8 f0[3][MT];
    const uint8_t* st = ring;
    auto frag = [&](int p, int i, int j) {     // columns 32 h + 8 j .. + 7
        return *reinterpret_cast<const bf16x8*>(st + p * L::PLANE + (32 * i + r) * 128 + (((4 * h + j) ^ ((r >> 1) & 7)) << 4));
    };
    auto begin = [&](int slot) {
        st = ring + slot * L::STAGE;
#pragma unroll
        for (int c = 0; c < 2; c++)
            wd[c] = *reinterpret_cast<const u32x4*>(st + L::A + nw * 2048 + r * 64 + (((2 * h + c) ^ bsw(r)) << 4));
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < MT; i++) f0[p][i] = frag(p, i, 0);
    };
    auto landed = [&](int newer) {
        if (RING > 3 && newer >= 3) __builtin_amdgcn_s_waitcnt(wait_imm(3 * PER));
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
        const bool live = t < ns;
        bf16x8 fl[3][MT];
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < MT; i++) fl[p][i] = f0[p][i];
        auto mul = [&](const u32x4& w, int half, const bf16x8 (&fa)[3][MT]) {
            uint32_t b0, b1, b2, b3;
            bytes_to_bf16(w[2 * half], b0, b1);
            bytes_to_bf16(w[2 * half + 1], b2, b3);
            const u32x4 b = {b0, b1, b2, b3};
            const bf16x8 fb = __builtin_bit_cast(bf16x8, b);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                ah[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0][i], fb, ah[i], 0, 0, 0);
                am[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1][i], fb, am[i], 0, 0, 0);
                al[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[2][i], fb, al[i], 0, 0, 0);
            }
        };
        const u32x4 wl = wd[1];     // the step's last words
        if (live) {
            const u32x4 w0 = wd[0];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                bf16x8 fn[3][MT];
#pragma unroll
                for (int p = 0; p < 3; p++)
#pragma unroll
                    for (int i = 0; i < MT; i++) fn[p][i] = frag(p, i, j + 1);
                mul(j < 2 ? w0 : wl, j & 1, fl);
#pragma unroll
                for (int p = 0; p < 3; p++)
#pragma unroll
                    for (int i = 0; i < MT; i++) fl[p][i] = fn[p][i];
            }
        }
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
            mul(wl, 1, fl);
            if ((t & 1) || t + 1 == ns) {
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    yv[i] += ah[i];
                    ah[i] = f32x16{};
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            yv[i][e] = __builtin_fmaf(__builtin_fmaf(al[i][e], 0x1p-8f, am[i][e]), 0x1p-8f, yv[i][e]);

    // piece p = MT v + i: rows 8 v + 4 h .. + 3 of tile i.  The wave groups'
    // sums meet in LDS and wave (nw, kw) finishes pieces kw, kw + KW, ...
    static_assert(KW * 4 * NP * 1024 <= KW * RING * L::STAGE, "the sums fit where the rings were");
    f32x4 res[OWN];
    __builtin_amdgcn_s_waitcnt(wait_imm(0));
    __builtin_amdgcn_s_barrier();
    f32x4* red = reinterpret_cast<f32x4*>(lds) + nw * NP * 64 + lane;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = yv[p % MT][4 * (p / MT) + e];
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

    if (splits > 1) {
        constexpr int kSysCoherent = 1 | 16;
        constexpr uint32_t SLOTB = 4 * KW * OWN * 1024;
        const uint32_t tl = blockIdx.z * gridDim.x + tile;
        const __amdgpu_buffer_rsrc_t rp = rsrc(part, 0xffffffffu);
        const uint32_t first = tl * (uint32_t)splits * SLOTB + (uint32_t)(wave * OWN) * 1024u;
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const float e0 = res[o][0], e1 = res[o][1], e2 = res[o][2], e3 = res[o][3];
            const u32x4 v = {f2u(e0), f2u(e1), f2u(e2), f2u(e3)};
            __builtin_amdgcn_raw_buffer_store_b128(v, rp, lane * 16, first + (uint32_t)span * SLOTB + o * 1024, kSysCoherent);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0f70);             // vmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        uint32_t* mine = cnt + (size_t)tl * (4 * KW) + wave;
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(mine, 1u);
        if ((int)__builtin_amdgcn_readfirstlane(c) != splits - 1) return;
        __builtin_amdgcn_sched_barrier(0);
        if (lane == 0) atomicExch(mine, 0u);
#pragma unroll
        for (int o = 0; o < OWN; o++) res[o] = f32x4{0.f, 0.f, 0.f, 0.f};
        constexpr int CH = OWN >= 4 ? 4 : 8;
#pragma unroll 1
        for (int s0 = 0; s0 < splits; s0 += CH) {
            u32x4 v[CH][OWN];
#pragma unroll
            for (int c2 = 0; c2 < CH; c2++)
#pragma unroll
                for (int o = 0; o < OWN; o++)
                    v[c2][o] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                        rp, lane * 16, first + (uint32_t)(s0 + c2 < splits ? s0 + c2 : splits - 1) * SLOTB + o * 1024, kSysCoherent));
#pragma unroll
            for (int c2 = 0; c2 < CH; c2++)
                if (s0 + c2 < splits)
#pragma unroll
                    for (int o = 0; o < OWN; o++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const uint32_t d = v[c2][o][e];
                            res[o][e] += u2f(d);
                        }
        }
    }

    const __amdgpu_buffer_rsrc_t ry = rsrc(y, (uint32_t)M * (uint32_t)N * 4u);
#pragma unroll
    for (int o = 0; o < OWN; o++) {
        const int p = kw + o * KW;
        const int n = n0 + r, m = m0 + 32 * (p % MT) + 8 * (p / MT) + 4 * h, nc = n < N ? n : N - 1;
        uint32_t off = n < N ? ((uint32_t)m * (uint32_t)N + (uint32_t)n) * 4u : 0x80000000u;
        const float sc = scales[nc], bv = bias ? bias[nc] : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float f = sc * res[o][e];
            if (bias) f += bv;
            __builtin_amdgcn_raw_buffer_store_b32(f2u(f), ry, off, 0, 0);
            off += (uint32_t)N * 4u;
        }
    }
}

struct Batch {
    const uint16_t* xp;
    const int8_t* qw;
    const float* scales;
    const float* bias;
    float* y;
    int M, N, K, splits;
    float* part;
    uint32_t* cnt;
    hipStream_t s;
};

template <int MT, int KW, int RING>
int launch(const Batch& a) {
    constexpr int bytes = KW * RING * layout<MT>::STAGE;
    static_assert(bytes <= 160 * 1024, "LDS of a workgroup");
    static std::atomic<uint64_t> lds_done{0};
    const void* fn = reinterpret_cast<const void*>(&k_w8_batch<MT, KW, RING>);
    if (snx::lds_optin(fn, bytes, lds_done) != hipSuccess) {
        snx_set_error("w8 batch: cannot reserve %d bytes of LDS", bytes);
        return -1;
    }
    const dim3 grid((a.N + BN - 1) / BN, a.splits, (a.M + 32 * MT - 1) / (32 * MT));
    const int steps = (a.K + BK - 1) / BK;
    k_w8_batch<MT, KW, RING><<<grid, 256 * KW, bytes, a.s>>>(
        Args{a.xp, a.qw, a.scales, a.bias, a.y, a.M, a.N, a.K, steps / a.splits, steps % a.splits, a.part, a.cnt});
    return snx_launch_check("k_w8_batch");
}

constexpr int KWG = 2;          // wave groups of a workgroup

size_t tiles_of(size_t M, size_t N, size_t rows) { return ((N + BN - 1) / BN) * ((M + rows - 1) / rows); }

// Rows of a workgroup: 32 while those tiles are at most a quarter of the CUs
// (M = 64, N = K = 4096: 19.3 us, with 64 rows 20.8), else 64 (M = 96: 23.8,
// with 32 rows 25.2 us).
size_t rows_of(size_t M, size_t N) { return tiles_of(M, N, 32) * 4 <= (size_t)snx::cu_count() ? 32 : 64; }

// Where the three-piece form is the faster one (us of the GEMV / of it).
// K % 16 == 0: M = 5: K = 256, N = 256 11.2 / 6.8, K = 1024, N = 4096 10.8 / 10.9;
// M = 4: K = 1024, N = 4096 9.1 / 11, K = 2048, N = 4096 13.8 / 12.0, 12288 17.6 / 19.2,
// 24576 33 / 26; M = 3: K = 2048, N = 4096 11.1 / 12, K = 3072, N = 4096 14.3 / 13.2, 12288
// 23.2 / 24.6, 36864 (just past a round of the CUs) 61 / 73; M = 2: K = 4096, N = 2048
// 12.3 / 12.9, 4096 14.4 / 13.9, 12288 22 / 29, K = 6144, N = 512 13.3 / 13.2, K = 8192, N =
// 4096 24.5 / 17.0, 12288 44 / 50.
// Other K, where the GEMV loads single values: M = 5, N = 4096: K = 260 6.1 / 7.6, 772
// 10.4 / 10.7, 1000 12.8 / 11.0, N = 16384, K = 20 8.1 / 7.0; N = 256, K = 20: M = 12 5.8 / 6.8,
// 16 7.2 / 6.6; M = 2, K = 4100, N = 300 15.9 / 11.5.
bool rows_pay(size_t M, size_t N, size_t K) {
    if (K % 16 != 0) return M >= 5 ? N > 8192 || M * (K + 600) >= 7500 : M >= 2 && M * K >= 8192;
    if (M == 2) return N <= 8192 && K >= (N >= 4096 ? 4096u : 6144u);
    if (M == 3) return K >= (N > 8192 ? 4096u : 2816u) && (N <= 32768 || N > 40960);
    if (M == 4) return K >= (N > 8192 && N < 16384 ? 3072u : 2048u);
    return M >= 5;
}

}  // namespace

extern "C" {

// K a multiple of 4 (rows of weights on their 4-byte alignment), 31-bit buffer
// offsets, and rows_pay().
int snx_w8_batch_ok(size_t M, size_t N, size_t K, const void* q) {
    const size_t steps = (K + BK - 1) / BK;
    return rows_pay(M, N, K) && K % 4 == 0 && ((uintptr_t)q & 3u) == 0 && N * K < (1ull << 31) &&
           M * steps * XSTEP < (1ull << 31) && (M + 64) * N * 4 < (1ull << 31) && M <= 32 * 65535ull;
}

size_t snx_w8_batch_xp_bytes(size_t M, size_t K) { return M * ((K + BK - 1) / BK) * XSTEP; }

// spans of K: as many as fill the CUs, at least four steps of each wave group
int snx_w8_batch_splits(size_t M, size_t N, size_t K) {
    const size_t most = (K + BK - 1) / BK / (4 * KWG);
    size_t s = (size_t)snx::cu_count() / tiles_of(M, N, rows_of(M, N));
    if (s > most) s = most;
    return s < 1 ? 1 : (int)s;
}
size_t snx_w8_batch_part_bytes(size_t M, size_t N, int splits) {
    const size_t rows = rows_of(M, N);
    return tiles_of(M, N, rows) * (size_t)splits * rows * BN * sizeof(float);
}
size_t snx_w8_batch_cnt_bytes(size_t M, size_t N) {
    return tiles_of(M, N, rows_of(M, N)) * 4 * KWG * sizeof(uint32_t);
}

int snx_k_w8_batch(const float* x, const int8_t* q, const float* s, float* y, const float* bias, size_t M, size_t N,
                   size_t K, int splits, void* xp, void* part, uint32_t* cnt, void* st) {
    if (!snx_w8_batch_ok(M, N, K, q) || !xp || (splits > 1 && (!part || !cnt))) {
        snx_set_error("w8 batch: M=%zu N=%zu K=%zu is not a shape of this kernel", M, N, K);
        return -1;
    }
    const uint32_t per_row = (uint32_t)((K + BK - 1) / BK) * (BK / 4);
    const uint32_t items = (uint32_t)M * per_row;
    k_w8_split_x<<<(items + 255) / 256, 256, 0, S(st)>>>(x, (uint16_t*)xp, (int)K, items, per_row);
    if (snx_launch_check("k_w8_split_x")) return -1;
    const Batch a{(const uint16_t*)xp, q, s, bias, y, (int)M, (int)N, (int)K, splits, (float*)part, cnt, S(st)};
    return rows_of(M, N) == 32 ? launch<1, KWG, 4>(a) : launch<2, KWG, 2>(a);
}

}  // extern "C"
