// gemm_kernels.hpp — gfx950 products C = A . B^T of more than 64 rows (prompts and
// prompt pieces); the few-row form is gemm_skinny_kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ops_kernels.hpp"

#pragma clang fp contract(off)

namespace awo {

constexpr int kStageK = 64; // k per LDS stage: a staged row is 128 bytes, eight 16-byte chunks

// gfx9 buffer resource word 3 (32-bit data format) of the operand loads.
constexpr uint32_t kRsrcWord3 = 0x00020000u;
// An offset past every tile, whose rows the host keeps below 1 GiB: the load returns zeros.
constexpr uint32_t kOutOfRange = 0x80000000u;
constexpr uint64_t kTileBytesMax = 1ull << 30;

// s_waitcnt immediate (gfx9): vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8, no
// wait on expcnt (6:4).
constexpr short wait_imm(uint32_t vm, uint32_t lgkm) {
    return (short)((vm & 15u) | ((vm >> 4) << 14) | (7u << 4) | (lgkm << 8));
}

template <int V>
struct Int {
    static constexpr int value = V;
};

// WM x WN waves, each FM x FN MFMA tiles of 16 x 16: a work-group owns TM = 16 WM FM
// activation rows x TN = 16 WN FN weight rows.
// Its LDS holds NA stages of activations and NB (NA or NA + 1) of weights.
template <int WM_, int WN_, int FM_, int FN_, int NA_, int NB_ = NA_>
struct GemmTile {
    static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_, NA = NA_, NB = NB_;
    static constexpr int TM = 16 * WM * FM, TN = 16 * WN * FN, kWaves = WM * WN, kThreads = 64 * kWaves;
    static constexpr size_t kLdsBytes = (size_t)(NA * TM + NB * TN) * kStageK * 2;
    static_assert(NA >= 2 && (NB == NA || NB == NA + 1) && kLdsBytes <= 160 * 1024);
};

// 16 bytes at an element's alignment: one access on gfx950, whatever row of an odd
// length it lies in.
typedef uint32_t uint4_a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef float float4_a4_t __attribute__((ext_vector_type(4), aligned(4)));

// Eight results C[m][n .. n+7] of one lane, masked to M x N; all but the last of a row
// whose N % 8 != 0 are read and written 16 bytes at a time.  4096 x N x 64, the stores
// its bound, us with single values and this: N 8196 f16 80 -> 24, f32 106 -> 37,
// residual 121 -> 51; N 8197 81 -> 41, 104 -> 48, 129 -> 72 (N 8192, 16 bytes at a
// time both ways: 22, 28, 34).
template <Epi EPI, bool F32>
__device__ inline void store8(void* C, uint32_t M, uint32_t N, uint32_t m, uint32_t n, float4_t lo, float4_t hi,
                              float scale) {
    if (n + 8 > N) {
        store4<EPI, F32>(C, M, N, m, n, lo, lo, scale, false);
        store4<EPI, F32>(C, M, N, m, n + 4u, hi, hi, scale, false);
        return;
    }
    if (m >= M) return;
    if constexpr (F32) {
        float* at = (float*)C + (uint64_t)m * N + n;
        *(float4_a4_t*)at = lo * scale;
        *(float4_a4_t*)(at + 4) = hi * scale;
        return;
    }
    uint4_a2_t* at = (uint4_a2_t*)((uint16_t*)C + (uint64_t)m * N + n);
    uint4_a2_t x = (uint4_a2_t)0u, r;
    if constexpr (EPI == Epi::Residual) x = *at;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t h[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = w < 2 ? lo[2 * w + e] : hi[2 * w - 4 + e];
            h[e] = f2h(v);
            if constexpr (EPI == Epi::Residual)
                h[e] = ew_one<Ew::Add>((uint16_t)(x[w] >> (16 * e)), ew_one<Ew::Scale>((uint16_t)h[e], 0, scale), 0.0f);
        }
        r[w] = h[0] | (h[1] << 16);
    }
    *at = r;
}

// One product (or up to three that share A), K % 8 == 0 and 16-byte aligned rows.
// Both operands go from memory straight into LDS (buffer loads with the LDS flag) in
// stages of 64 k; a wave load covers 8 rows x 128 bytes, and chunks are permuted within
// a row so that neither the writes nor the fragment reads (ds_read_b128, 16 rows at
// one chunk) meet a bank conflict.  All tiles sum the same 32-k MFMA steps in the same
// order: a product's bits depend neither on the tile nor on the products beside it.
// Bound: large tiles by power (2048 x 8192 x 8192: 1.19 PFLOP/s, with zeros as operands
// 1.84), small ones by their loads into LDS (58 bytes a ns and CU).  Against 256 x 128
// tiles whose loads and fragment reads ran ahead of a stage's products, or 128 x 128
// tiles through registers where 256 x 128 did not fill the CUs, us: 2048 x 14336 x 4096
// 278 -> 222, 2048 x 4096 x 14336 241 -> 217, 512 x 4096 x 14336 313 -> 95, 512 x 14336
// x 4096 108 -> 61, 117 x 3072 x 2048 42 -> 8.3.
template <typename T, bool F32, Epi EPI>
__global__ __launch_bounds__(T::kThreads) __attribute__((amdgpu_waves_per_eu(T::kWaves == 8 ? 2 : 1))) void gemm_tile_kernel(GemmArgs a) {
    static_assert(EPI != Epi::SiluGate, "one weight matrix");
    constexpr int FM = T::FM, FN = T::FN, NA = T::NA, NB = T::NB, TM = T::TM, TN = T::TN, W = T::kWaves;
    constexpr uint32_t kBufA = (uint32_t)TM * kStageK, kBufB = (uint32_t)TN * kStageK; // halves
    // Wave loads (8 rows x 128 bytes) per stage; wave w takes loads w, w + W, ..
    constexpr int GA = TM / 8, GB = TN / 8, LA = (GA + W - 1) / W, LB = (GB + W - 1) / W;
    extern __shared__ __attribute__((aligned(16))) _Float16 gemm_lds[]; // [NB][TN weight rows][64], [NA][TM rows][64]
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % T::WN, wm = wave / T::WN;
    auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }; // divisions run on the vector ALUs

    // Work-group b runs on XCD b % 8: each XCD takes a contiguous run of tiles, up to
    // 8 row tiles of one weight tile after another.
    const uint32_t tm = uniform((a.M + TM - 1u) / TM), total = gridDim.x, xcd = blockIdx.x & 7u;
    uint32_t t = xcd * (total >> 3) + min(xcd, total & 7u) + (blockIdx.x >> 3);
    const uint32_t tn = uniform(total / tm), span = uniform(t / (8u * tn));
    t -= span * 8u * tn;
    const uint32_t width = min(8u, tm - 8u * span);
    uint32_t tile = uniform(t / width);
    const uint32_t m0 = (8u * span + t - tile * width) * (uint32_t)TM;
    const bool in0 = tile < a.g[0].tiles;
    if (!in0) tile -= a.g[0].tiles;
    const bool in1 = !in0 && (a.groups < 3 || tile < a.g[1].tiles);
    if (!in0 && !in1) tile -= a.g[1].tiles;
    const GemmGroup& G = in0 ? a.g[0] : (in1 ? a.g[1] : a.g[2]);
    const uint32_t N = G.N, K = a.K, n0 = tile * (uint32_t)TN, K2 = 2u * K;

    // The tile's rows as buffers: rows past the operand's last load zeros.
    const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(G.B + (uint64_t)n0 * K), (short)0, (int)(min((uint32_t)TN, N - n0) * K2), (int)kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.A + (uint64_t)m0 * K), (short)0, (int)(min((uint32_t)TM, a.M - m0) * K2), (int)kRsrcWord3);

    // A wave load fills 64 consecutive 16-byte slots: lane -> row lane / 8, slot lane % 8,
    // which holds chunk (slot ^ swz(row)).  swz differs over the 8 rows that one LDS
    // cycle reads: activations rows r .. r + 7, weights r .. r + 3 and r + 8 .. r + 11.
    const uint32_t lr = (uint32_t)lane >> 3, slot = (uint32_t)lane & 7u;
    auto swz_b = [](uint32_t row) { return (row & 3u) | ((row >> 1) & 4u); };
    const uint32_t n_stages = (K + kStageK - 1u) / kStageK, last = n_stages - 1u;
    // Row w * 8 + lr + 8 W j of an operand for load j: the same chunk for every j.
    static_assert(W % 2 == 0, "swz_b looks at bit 3 of a row");
    const uint32_t row0 = 8u * (uint32_t)wave + lr, cha = slot ^ (row0 & 7u), chb = slot ^ swz_b(row0);
    const uint32_t offa = row0 * K2 + 16u * cha, offb = row0 * K2 + 16u * chb, step = 8u * (uint32_t)W * K2;
    const uint32_t ktail = K - (uint32_t)kStageK * last; // k of the last stage
    // Load x of stage st: the LA of the activations, then the LB of the weights.
    auto load = [&](int x, uint32_t st, uint32_t buf) {
        const bool isa = x < LA;
        const int j = isa ? x : x - LA, g = wave + W * j, G = isa ? GA : GB, L = isa ? LA : LB;
        if (G % W != 0 && j == L - 1 && g >= G) return; // wave-uniform
        const uint32_t off = (isa ? offa : offb) + st * (uint32_t)(kStageK * 2) + (uint32_t)j * step;
        const bool in = st < last || 8u * (isa ? cha : chb) < ktail;
        _Float16* d = gemm_lds + (isa ? NB * kBufB + buf * kBufA : buf * kBufB) + (uint32_t)g * 512u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(isa ? rA : rB, (__attribute__((address_space(3))) void*)d, 16,
                                                 (int)(in ? off : kOutOfRange), 0, 0, 0);
    };
    // Waits until at most `na` + `nb` of this wave's newest loads (stages of A and of B) are in flight.
    const bool full_a = GA % W == 0 || wave < GA % W, full_b = GB % W == 0 || wave < GB % W;
    auto wait = [&](auto stages_a, auto stages_b, auto lgkm) {
        constexpr int na = decltype(stages_a)::value, nb = decltype(stages_b)::value, lg = decltype(lgkm)::value;
        if (full_a && full_b) __builtin_amdgcn_s_waitcnt(wait_imm(na * LA + nb * LB, lg));
        else if (full_a) __builtin_amdgcn_s_waitcnt(wait_imm(na * LA + nb * (LB - 1), lg));
        else if (full_b) __builtin_amdgcn_s_waitcnt(wait_imm(na * (LA - 1) + nb * LB, lg));
        else __builtin_amdgcn_s_waitcnt(wait_imm(na * (LA - 1) + nb * (LB - 1), lg));
    };

    // Fragments (halves from a buffer's start).  Weight fragments come in pairs:
    // fragment 2 p + h holds weight rows 32 p + 8 (i / 4) + 4 h + i % 4 for i < 16, so a
    // lane ends with 8 consecutive columns; the last of an odd FN holds its rows in order.
    uint32_t arow = (uint32_t)(wm * 16 * FM + li) * kStageK, brow[2], blast = 0;
    uint32_t ach[2], bch[2][2], blch[2] = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t row = (uint32_t)(wn * 16 * FN + 8 * (li >> 2) + 4 * h + (li & 3));
        brow[h] = row * kStageK;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) bch[h][ks] = (((uint32_t)(4 * ks + lg)) ^ swz_b(row)) << 3;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) ach[ks] = (((uint32_t)(4 * ks + lg)) ^ ((uint32_t)li & 7u)) << 3;
    if constexpr (FN % 2) {
        const uint32_t row = (uint32_t)(wn * 16 * FN + 16 * (FN - 1) + li);
        blast = row * kStageK;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) blch[ks] = (((uint32_t)(4 * ks + lg)) ^ swz_b(row)) << 3;
    }
    struct Frags {
        half8_t a[FM], b[FN];
    };
    // Fragment x of a half stage: the FN of the weights, then the FM of the activations.
    auto read = [&](Frags& f, int x, uint32_t bufa, uint32_t bufb, int ks) {
        const _Float16 *sb = gemm_lds + bufb * kBufB, *sa = gemm_lds + NB * kBufB + bufa * kBufA;
        if (x >= FN) f.a[x - FN] = *(const half8_t*)(sa + arow + ach[ks] + (x - FN) * 16 * kStageK);
        else if (FN % 2 && x == FN - 1) f.b[x] = *(const half8_t*)(sb + blast + blch[ks]);
        else f.b[x] = *(const half8_t*)(sb + brow[x & 1] + bch[x & 1][ks] + (x >> 1) * 32 * kStageK);
    };
    float4_t acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = (float4_t)0.0f;
    // Half a stage's products; between them, in this order and spread over them, the
    // other half's fragments are read and the loads of a later stage issued (issued
    // in one run, the loads hold every wave at the barrier until they are taken).
    constexpr int RPG = (4 * (FN + FM) + 3 * FN - 1) / (3 * FN), LPG = (LA + LB + FN - 1) / FN;
    auto multiply = [&](const Frags& f, auto read_x, auto load_x) {
#pragma unroll
        for (int i = 0; i < FN; ++i) {
#pragma unroll
            for (int x = i * RPG; x < (i + 1) * RPG && x < FN + FM; ++x) read_x(x);
#pragma unroll
            for (int x = i * LPG; x < (i + 1) * LPG && x < LA + LB; ++x) load_x(x);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = mfma(f.b[i], f.a[j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // Stage s sits in buffers s % NA and s % NB.  Half a stage's products run from
    // fragments read during the other half's; in the middle of stage s every wave has
    // read all of it and waited for its own loads of stage s + 1, so after one barrier
    // its buffers take stages s + NA and s + NB and the next stage's fragments are read.
    if (n_stages > 0) {
#pragma unroll
        for (uint32_t s = 0; s < (uint32_t)NB; ++s)
#pragma unroll
            for (int x = 0; x < LA + LB; ++x)
                if (s < n_stages && (x >= LA || s < (uint32_t)NA)) load(x, s, s);
        if (n_stages >= (uint32_t)NB) wait(Int<NA - 1>{}, Int<NB - 1>{}, Int<15>{});
        else wait(Int<0>{}, Int<0>{}, Int<15>{});
        barrier();
        Frags f0, f1;
#pragma unroll
        for (int x = 0; x < FN + FM; ++x) read(f0, x, 0, 0, 0);
        uint32_t s = 0, ba = 0, bb = 0;
        auto stage = [&](auto steady) {
            constexpr bool kSteady = decltype(steady)::value != 0; // stages s + NA and s + NB exist
            multiply(f0, [&](int x) { read(f1, x, ba, bb, 1); }, [](int) {});
            if (kSteady || s + (uint32_t)NB <= n_stages) wait(Int<NA - 2>{}, Int<NB - 2>{}, Int<0>{});
            else wait(Int<0>{}, Int<0>{}, Int<0>{});
            barrier();
            const uint32_t oa = ba, ob = bb;
            ba = ba + 1u == (uint32_t)NA ? 0u : ba + 1u;
            bb = bb + 1u == (uint32_t)NB ? 0u : bb + 1u;
            multiply(
                f1,
                [&](int x) {
                    if (kSteady || s < last) read(f0, x, ba, bb, 0);
                },
                [&](int x) {
                    const uint32_t st = s + (uint32_t)(x < LA ? NA : NB);
                    if (kSteady || st < n_stages) load(x, st, x < LA ? oa : ob);
                });
            ++s;
        };
        while (s + (uint32_t)NB < n_stages) stage(Int<1>{});
        while (s < n_stages) stage(Int<0>{});
    }
    const uint32_t mrow = m0 + (uint32_t)(wm * 16 * FM + li);
    const uint32_t ncol = n0 + (uint32_t)(wn * 16 * FN);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
#pragma unroll
        for (int p = 0; p < FN / 2; ++p)
            store8<EPI, F32>(G.C, a.M, N, mrow + 16u * j, ncol + 32u * p + 8u * (uint32_t)lg, acc[2 * p][j],
                             acc[2 * p + 1][j], a.scale);
        if constexpr (FN % 2)
            store4<EPI, F32>(G.C, a.M, N, mrow + 16u * j, ncol + 16u * (FN - 1) + 4u * (uint32_t)lg, acc[FN - 1][j],
                             acc[FN - 1][j], a.scale, G.vec_out);
    }
}

} // namespace awo
