// q8_batch_kernels.hip - linears of two low-precision operands (int8, fp8 and
// the MX formats) with too few rows to fill the 256 x 224 tiles of
// gemm_kernels.hip.
//
// out[m][n] = sum_k A[m][k] W[n][k], scaled; A and W K-contiguous.
//
// What bounds it: a decode batch is bound by reading W once and, before that,
// by how much of the chip has work: a large tile leaves 38 workgroups at
// 512 x 4096, and 64 x 64 tiles that load their operands straight from memory
// leave every load's latency open.  Here a workgroup takes 32 to 128 rows and
// 128 columns, K is split over its two wave groups (their sums meet in LDS)
// and over workgroups (their sums meet in memory), both operands are staged in
// LDS by direct loads, and a step is little more than its LDS reads and its
// products.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "codec.h"
#include "launch.h"
#include "../snx_internal.h"

using namespace snx;

namespace {

typedef int i32x3 __attribute__((ext_vector_type(3)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

constexpr int BN = 128;         // output columns of a workgroup: 4 waves of 32
constexpr int KW = 2;           // wave groups of a workgroup, each with a share of its K
constexpr int ROWB = 128;       // LDS bytes of a row of a step: 8 pieces of 16

// operand kinds: int8, fp8 with per-tensor scales, MX by MFMA element format
// (2 e4m3, 3 e5m2, 4 e2m3, 5 e3m2, 6 e2m1)
constexpr int INT8 = 0, FP8 = 1, MX = 2;
constexpr int kind_bits(int k) { return k == 6 ? 4 : k >= 4 ? 6 : 8; }
constexpr int kind_step(int k) { return k == 6 ? 256 : 128; }              // elements of a step
constexpr int kind_piece(int k) { return kind_bits(k) == 6 ? 12 : 16; }    // bytes of a piece

constexpr int wait_imm(int vm) { return (vm & 15) | 0x70 | ((vm >> 4) << 14); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void lds_load(__amdgpu_buffer_rsrc_t r, void* dst, int bytes, uint32_t voff, uint32_t soff) {
    if (bytes == 16)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, voff, soff, 0, 0);
    else if (bytes == 12)   // into the first 12 bytes of each lane's 16-byte slot
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 12, voff, soff, 0, 0);
    else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 4, voff, soff, 0, 0);
}
constexpr uint32_t kNoRecord = 0x7ffffff0u;     // an offset past any operand: the load writes zeros

// piece c of row r of a stage sits at slot c ^ swz(r): 16-lane reads of one
// piece of 16 rows then touch every bank once
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// four int8 exponents as E8M0 bytes: s + 127, -128 as -127
__device__ __forceinline__ uint32_t e8m0x4(uint32_t s) {
    const uint32_t u = s ^ 0x80808080u;         // s + 128
    const uint32_t nz = (((u & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | u) >> 7 & 0x01010101u;
    return u - nz;
}

// The kernel's arguments, as one: the runtime takes about 20 ns for each of a launch
// (3.8 us for this kernel's fourteen, 3.4 so).
struct Args {
    const uint8_t *A, *W;
    const void *sA, *sW;
    void* out;
    const float* bias;
    int y_f32, M, N, K, per, extra;
    uint32_t *part, *cnt;
};

template <int KIND, int MT>
struct layout {
    static constexpr int A = 32 * MT * ROWB, W = BN * ROWB;
    static constexpr int SC = KIND >= MX ? (4 + MT) * 256 : 0;      // exponent words, 64 per 32 rows
    static constexpr int STAGE = A + W + SC;
};

// One workgroup: 2 x 4 waves; wave (nw, kw) computes 32 MT rows x 32 columns
// over wave group kw's share of the workgroup's steps.  Operand lane l of the
// 32-row MFMAs: row l % 32; int8 (32 k): piece 2 j + l / 32; 8-bit floats (64 k):
// pieces 4 j + l / 32 and 4 j + 2 + l / 32; 6 and 4 bits: block 2 j + l / 32 whole.
// The scale byte of lane l is that of block 2 j + l / 32 in every format.
// K % 128 != 0 (int8, fp8): pieces past K are loaded as zeros.
template <int KIND, int MT, int RING>
__global__ void __launch_bounds__(256 * KW) __attribute__((amdgpu_waves_per_eu(KW, KW))) k_q8_batch(
    const Args p) {
    const uint8_t* __restrict__ const A = p.A;
    const uint8_t* __restrict__ const W = p.W;
    const void *__restrict__ const sA = p.sA, *__restrict__ const sW = p.sW;
    void* __restrict__ const out = p.out;
    const float* __restrict__ const bias = p.bias;
    const int y_f32 = p.y_f32, M = p.M, N = p.N, K = p.K, per = p.per, extra = p.extra;
    uint32_t *__restrict__ const part = p.part, *__restrict__ const cnt = p.cnt;
    typedef layout<KIND, MT> L;
    typedef std::conditional_t<KIND == INT8, i32x16, f32x16> acc_t;
    constexpr int STEP = kind_step(KIND), PB = kind_piece(KIND);
    constexpr int JN = KIND == INT8 || KIND == 6 ? 4 : 2;      // products of a step per tile
    constexpr int PER = MT + 4 + (KIND >= MX ? 2 : 0);         // loads per wave and stage
    constexpr int NP = 4 * MT, OWN = NP / KW;                  // 16-byte result pieces per lane, and those a wave finishes
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = wave & 3, kw = wave >> 2;
    const int r = lane & 31, h = lane >> 5;
    const int tile = blockIdx.x, span = blockIdx.y, splits = gridDim.y;
    const int m0 = blockIdx.z * (32 * MT), n0 = tile * BN + 32 * nw;

    const int wg0 = span * per + (span < extra ? span : extra), wgn = per + (span < extra ? 1 : 0);
    const int g0 = wg0 + wgn * kw / KW, ns = wg0 + wgn * (kw + 1) / KW - g0;
    const int nmax = (wgn + KW - 1) / KW;
    const uint32_t KB = (uint32_t)K * kind_bits(KIND) / 8, KS = (uint32_t)K / 32;   // code and exponent bytes per row

    uint8_t* ring = lds + kw * (RING * L::STAGE);
    const __amdgpu_buffer_rsrc_t ra = rsrc(A, (uint32_t)M * KB), rw = rsrc(W, (uint32_t)N * KB);
    const __amdgpu_buffer_rsrc_t rsa = rsrc(sA, (uint32_t)M * KS), rsw = rsrc(sW, (uint32_t)N * KS);
    // load i of wave nw: rows 8 (4 i + nw) .. + 7 of A, rows 8 i .. + 7 of the wave's columns
    const int lrow = lane >> 3;
    uint32_t ga[MT], gw[4];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = 8 * (4 * i + nw) + lrow, gr = m0 + row < M ? m0 + row : M - 1;
        ga[i] = (uint32_t)gr * KB + (uint32_t)((lane & 7) ^ swz(row)) * PB;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = 8 * i + lrow, n = n0 + row;
        gw[i] = (uint32_t)(n < N ? n : N - 1) * KB + (uint32_t)((lane & 7) ^ swz(row)) * PB;
    }
    // exponent words: lanes 0..31 the step's first of 32 rows, lanes 32..63 its
    // second (4-bit formats; past the row it meets zeros) or the first again
    uint32_t gsa = 0, gsw = 0;
    if (KIND >= MX) {
        const int ma = m0 + 32 * (nw % MT) + r, n = n0 + r;
        gsa = (uint32_t)(ma < M ? ma : M - 1) * KS + (KIND == 6 ? 4u * h : 0u);
        gsw = (uint32_t)(n < N ? n : N - 1) * KS + (KIND == 6 ? 4u * h : 0u);
    }
    auto issue = [&](int slot, int t) {
        uint8_t* st = ring + slot * L::STAGE;
        const uint32_t k0 = (uint32_t)(g0 + t) * (STEP * kind_bits(KIND) / 8);
        const bool tail = k0 + ROWB > KB && PB == 16;         // pieces past K
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const uint32_t c = (uint32_t)((lane & 7) ^ swz(8 * (4 * i + nw) + lrow)) * 16u;
            lds_load(ra, st + (4 * i + nw) * 1024, PB, tail && k0 + c >= KB ? kNoRecord : ga[i], k0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t c = (uint32_t)((lane & 7) ^ swz(8 * i + lrow)) * 16u;
            lds_load(rw, st + L::A + (4 * nw + i) * 1024, PB, tail && k0 + c >= KB ? kNoRecord : gw[i], k0);
        }
        if (KIND >= MX) {
            const uint32_t ks = (uint32_t)(g0 + t) * (STEP / 32);
            lds_load(rsa, st + L::A + L::W + (nw % MT) * 256, 4, gsa, ks);
            lds_load(rsw, st + L::A + L::W + (MT + nw) * 256, 4, gsw, ks);
        }
    };

    acc_t acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = acc_t{};

    auto landed = [&](int newer) {
        if (RING > 3 && newer >= 3) __builtin_amdgcn_s_waitcnt(wait_imm(3 * PER));
        else if (RING > 2 && newer >= 2) __builtin_amdgcn_s_waitcnt(wait_imm(2 * PER));
        else if (newer >= 1) __builtin_amdgcn_s_waitcnt(wait_imm(PER));
        else __builtin_amdgcn_s_waitcnt(wait_imm(0));
    };
    // operand of product j from a row of a stage
    auto frag = [&](const uint8_t* row, int j) -> i32x8 {
        auto at = [&](int c) { return row + ((c ^ swz(r)) << 4); };
        if constexpr (KIND == INT8 || KIND == 6) {
            const i32x4 v = *reinterpret_cast<const i32x4*>(at(2 * j + h));
            return i32x8{v[0], v[1], v[2], v[3], 0, 0, 0, 0};
        } else if constexpr (PB == 16) {
            const i32x4 lo = *reinterpret_cast<const i32x4*>(at(4 * j + h));
            const i32x4 hi = *reinterpret_cast<const i32x4*>(at(4 * j + 2 + h));
            return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            const i32x3 lo = *reinterpret_cast<const i32x3*>(at(2 * (2 * j + h)));
            const i32x3 hi = *reinterpret_cast<const i32x3*>(at(2 * (2 * j + h) + 1));
            return i32x8{lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], 0, 0};
        }
    };

#pragma unroll 1
    for (int p = 0; p < RING && p < ns; p++) issue(p, p);
    int slot = 0;
#pragma unroll 1
    for (int t = 0; t < nmax; t++) {
        // stage t landed (newer ones may fly)
        const int newest = t + RING - 1 < ns - 1 ? t + RING - 1 : ns - 1;
        landed(newest - t);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t < ns) {
            const uint8_t* st = ring + slot * L::STAGE;
            const uint8_t* wrow = st + L::A + (32 * nw + r) * ROWB;
            // every fragment of the step ahead of its products
            i32x8 fw[JN], fa[MT][JN];
#pragma unroll
            for (int j = 0; j < JN; j++) fw[j] = frag(wrow, j);
            uint32_t ea[MT][2] = {}, ew[2] = {};
            if (KIND >= MX) {
                const uint32_t* sc = reinterpret_cast<const uint32_t*>(st + L::A + L::W);
#pragma unroll
                for (int w = 0; w < (KIND == 6 ? 2 : 1); w++) {
                    ew[w] = e8m0x4(sc[(MT + nw) * 64 + 32 * w + r]) >> (8 * h);
#pragma unroll
                    for (int i = 0; i < MT; i++) ea[i][w] = e8m0x4(sc[i * 64 + 32 * w + r]) >> (8 * h);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < JN; j++) fa[i][j] = frag(st + (32 * i + r) * ROWB, j);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < JN; j++) {
                    if constexpr (KIND == INT8) {
                        const i32x4 a = __builtin_shufflevector(fa[i][j], fa[i][j], 0, 1, 2, 3);
                        const i32x4 b = __builtin_shufflevector(fw[j], fw[j], 0, 1, 2, 3);
                        acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc[i], 0, 0, 0);
                    } else if constexpr (KIND == FP8) {
                        acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i][j], fw[j], acc[i], 0, 0, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
                    } else {
                        constexpr int F = KIND - MX;
                        if (j % 2 == 0)
                            acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i][j], fw[j], acc[i], F, F, 0, (int)ea[i][j / 2], 0, (int)ew[j / 2]);
                        else
                            acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i][j], fw[j], acc[i], F, F, 2, (int)ea[i][j / 2], 2, (int)ew[j / 2]);
                    }
                }
        }
        // this wave is done reading stage t; its place takes stage t + RING
        // behind a barrier of its own (a step is short: the second barrier
        // costs less than a ring slot kept free)
        if (t + RING < nmax) {
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (t + RING < ns) issue(slot, t + RING);
        }
        slot = slot + 1 == RING ? 0 : slot + 1;
    }

    // piece p = MT v + i: rows 8 v + 4 h .. + 3 of tile i, as bits.  The wave
    // groups' sums meet in LDS; wave (nw, kw) finishes pieces kw, kw + KW, ...
    auto add = [](u32x4 a, u32x4 b) -> u32x4 {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t x = a[e], y = b[e];
            o[e] = KIND == INT8 ? x + y : f2u(u2f(x) + u2f(y));
        }
        return o;
    };
    static_assert(KW * 4 * NP * 1024 <= KW * RING * L::STAGE, "the sums fit where the rings were");
    u32x4 res[OWN];
    __builtin_amdgcn_s_waitcnt(wait_imm(0));
    __builtin_amdgcn_s_barrier();
    u32x4* red = reinterpret_cast<u32x4*>(lds) + nw * NP * 64 + lane;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const auto v = acc[p % MT][4 * (p / MT) + e];
            o[e] = __builtin_bit_cast(uint32_t, v);
        }
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
        for (int k = 1; k < KW; k++) res[o] = add(res[o], red[(k * 4 * NP + p) * 64]);
    }

    if (splits > 1) {
        // as in k_w4a16_batch: stored past the L2s, counted per wave, summed in
        // span order by the last wave to arrive
        constexpr int kSysCoherent = 1 | 16;
        constexpr uint32_t SLOTB = 4 * KW * OWN * 1024;
        const uint32_t tl = blockIdx.z * gridDim.x + tile;
        const __amdgpu_buffer_rsrc_t rp = rsrc(part, 0xffffffffu);
        const uint32_t first = tl * (uint32_t)splits * SLOTB + (uint32_t)(wave * OWN) * 1024u;
#pragma unroll
        for (int o = 0; o < OWN; o++)
            __builtin_amdgcn_raw_buffer_store_b128(res[o], rp, lane * 16, first + (uint32_t)span * SLOTB + o * 1024, kSysCoherent);
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
        for (int o = 0; o < OWN; o++) res[o] = u32x4{0u, 0u, 0u, 0u};
        constexpr int CH = OWN >= 8 ? 2 : OWN >= 4 ? 4 : 8;
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
                    for (int o = 0; o < OWN; o++) res[o] = add(res[o], v[c2][o]);
        }
    }

    // rows past M lie past the buffer's records; lanes of columns past N take
    // an offset that does
    const uint32_t eb = y_f32 ? 4 : 2;
    const __amdgpu_buffer_rsrc_t ry = rsrc(out, (uint32_t)M * (uint32_t)N * eb);
    const int n = n0 + r, nc = n < N ? n : N - 1;
    const float bv = bias ? bias[nc] : 0.0f;
    const float swn = KIND == INT8 ? static_cast<const float*>(sW)[nc] : KIND == FP8 ? static_cast<const float*>(sW)[0] : 1.0f;
    const float sa0 = KIND == FP8 ? static_cast<const float*>(sA)[0] : 1.0f;
#pragma unroll
    for (int o = 0; o < OWN; o++) {
        const int p = kw + o * KW;
        const int m = m0 + 32 * (p % MT) + 8 * (p / MT) + 4 * h;
        uint32_t off = n < N ? ((uint32_t)m * (uint32_t)N + (uint32_t)n) * eb : 0x80000000u;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t w = res[o][e];
            float f = KIND == INT8 ? (float)(int)w : u2f(w);
            if (KIND == INT8) f = (f * static_cast<const float*>(sA)[m + e < M ? m + e : M - 1]) * swn;
            if (KIND == FP8) f = (f * sa0) * swn;
            if (bias) f += bv;
            if (y_f32) __builtin_amdgcn_raw_buffer_store_b32(f2u(f), ry, off, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16(bf16_out(f), ry, off, 0, 0);
            off += (uint32_t)N * eb;
        }
    }
}

// Rows of a workgroup: the fewest whose tiles are one round of the CUs (more
// tiles, not fewer K spans, are what fills the chip cheapest), 128 when none
// are.  The MX formats of 8 and 6 bits, with exponents to load and convert for
// every row of a tile, take 3/5 of a round.  us at N = 14336, K = 4096 with 32 /
// 64 / 128 rows: int8 M = 48 17.5 / 19.2 / -, 128 29.3 / 21.7 / 27.1, 256 51 /
// 36.6 / 31.3; mxfp8 M = 48 25.9 / 22.1 / -, 128 43 / 30.4 / 26.4.
size_t tiles_of(size_t M, size_t N, size_t rows) { return ((N + BN - 1) / BN) * ((M + rows - 1) / rows); }
size_t rows_of(int kind, size_t M, size_t N) {
    const size_t round = (size_t)snx::cu_count(), most = kind >= MX && kind != 6 ? round * 3 / 5 : round;
    for (size_t rows = 32; rows < 128; rows *= 2)
        if (M <= rows || tiles_of(M, N, rows) <= most) return rows;
    return 128;
}

// spans of K: as many as fill the CUs, at least two steps of each wave group
int splits_of(size_t tiles, size_t steps) {
    const size_t most = steps / (2 * KW);
    size_t s = (size_t)snx::cu_count() / tiles;
    if (s > most) s = most;
    return s < 1 ? 1 : (int)s;
}

struct Batch {
    const uint8_t* A;
    const void* sA;
    const uint8_t* W;
    const void* sW;
    void* out;
    const float* bias;
    int y_f32, M, N, K;
    hipStream_t s;
};

template <int KIND, int MT, int RING>
int launch(const Batch& a) {
    constexpr int bytes = KW * RING * layout<KIND, MT>::STAGE;
    static_assert(bytes <= 160 * 1024, "LDS of a workgroup");
    static std::atomic<uint64_t> lds_done{0};
    const void* fn = reinterpret_cast<const void*>(&k_q8_batch<KIND, MT, RING>);
    if (snx::lds_optin(fn, bytes, lds_done) != hipSuccess) {
        snx_set_error("q8 batch: cannot reserve %d bytes of LDS", bytes);
        return -1;
    }
    const int steps = (a.K + kind_step(KIND) - 1) / kind_step(KIND);
    const size_t tiles = tiles_of(a.M, a.N, 32 * MT);
    const int splits = splits_of(tiles, steps);
    void* part = nullptr;
    uint32_t* cnt = nullptr;
    if (splits > 1 && snx_span_workspaces(tiles * splits * (32 * MT) * BN * 4, tiles * 4 * KW * sizeof(uint32_t), a.s,
                                          &part, &cnt))
        return -1;
    const dim3 grid((a.N + BN - 1) / BN, splits, (a.M + 32 * MT - 1) / (32 * MT));
    k_q8_batch<KIND, MT, RING><<<grid, 256 * KW, bytes, a.s>>>(Args{a.A, a.W, a.sA, a.sW, a.out, a.bias, a.y_f32, a.M, a.N, a.K,
        steps / splits, steps % splits, static_cast<uint32_t*>(part), cnt});
    return snx_launch_check("k_q8_batch");
}

template <int KIND>
int launch_rows(const Batch& a) {
    switch (rows_of(KIND, a.M, a.N)) {
        case 32: return launch<KIND, 1, 3>(a);
        case 64: return launch<KIND, 2, 3>(a);
        default: return launch<KIND, 4, 2>(a);
    }
}

}  // namespace

extern "C" {

// kind: 0 int8 (fp32 sA [M], sW [N]), 1 fp8 (fp32 sA[0], sW[0]), 2 + MFMA element
// format: MX (int8 exponents); 31-bit buffer offsets
int snx_q8_batch_ok(int kind, size_t M, size_t N, size_t K) {
    const size_t kb = K * (size_t)kind_bits(kind) / 8;
    return (kind < MX ? K % 16 == 0 : K % 128 == 0) && M * kb < kNoRecord && N * kb < kNoRecord &&
           (M + 128) * N * 4 < (1ull << 31) && M <= 128 * 65535ull;
}

// Where the 256 x 224 tiles of gemm_kernels.hip apply too (M, N >= 128), the
// batch kernel is the faster one while its own largest tiles are one round of
// the CUs: int8 at N = 14336, K = 4096 31 against 43 us at M = 256, equal at
// 512 (mxfp8 36 / 62 and 64 / 63); at N = K = 4096 30 / 42 at M = 1024.  The MX
// formats of 8 and 6 bits have those tiles for fewer rows too, and take them where
// they are half the rounds of the CUs (mxfp8, K = 4096, M = 100: N = 36864 67 / 59 us,
// 49152 69 / 63, 57344 71 / 66, 65536, where both are two rounds, 76 / 118; M = 32:
// 36864 54 / 53).
int snx_q8_batch_better(int kind, size_t M, size_t N, size_t K) {
    const size_t ncu = (size_t)snx::cu_count();
    if (!snx_q8_batch_ok(kind, M, N, K)) return 0;
    if (M >= 128 && N >= 128) return tiles_of(M, N, 128) <= ncu;
    if (kind < MX || kind == 6 || M <= 32) return 1;
    const size_t rounds = (tiles_of(M, N, rows_of(kind, M, N)) + ncu - 1) / ncu;
    const size_t large = ((M + 255) / 256 * ((N + 223) / 224) + ncu - 1) / ncu;
    return rounds < 2 * large;
}

int snx_k_q8_batch(int kind, const void* A, const void* sA, const void* W, const void* sW, void* out,
                   const float* bias, int y_f32, size_t M, size_t N, size_t K, void* st) {
    if (!snx_q8_batch_ok(kind, M, N, K)) {
        snx_set_error("q8 batch: M=%zu N=%zu K=%zu is not a shape of this kernel", M, N, K);
        return -1;
    }
    const Batch a{(const uint8_t*)A, sA, (const uint8_t*)W, sW, out, bias, y_f32, (int)M, (int)N, (int)K, S(st)};
    switch (kind) {
        case INT8: return launch_rows<INT8>(a);
        case FP8: return launch_rows<FP8>(a);
        case 2: return launch_rows<2>(a);
        case 3: return launch_rows<3>(a);
        case 4: return launch_rows<4>(a);
        case 5: return launch_rows<5>(a);
        default: return launch_rows<6>(a);
    }
}

}  // extern "C"
