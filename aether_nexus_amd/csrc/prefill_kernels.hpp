// prefill_kernels.hpp — gfx950 causal attention over contiguous caches for many
// new tokens (prompts and prompt pieces); the few-query form is hot_kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "weaver_kernels.hpp"

namespace aw {

typedef float float16_t __attribute__((ext_vector_type(16)));

struct PrefillArgs {
    const uint16_t* q;       // [n][q_heads][HD]
    const uint16_t* k;       // [kv_len][kv_heads][HD], 16-byte aligned
    const uint16_t* v;
    uint16_t* out;           // [n][q_heads][HD] (one split)
    float* part_m;           // [kv_heads][splits][rows] (several splits)
    float* part_l;
    float* part_o;           // [kv_heads][splits][rows][HD]
    uint32_t n, kv_len, q_heads, kv_heads, gqa;
    uint32_t rows, tiles;    // n * gqa query rows per kv head, in tiles of kPrefillRows
    uint32_t splits;
    float scale_log2;
};

// Work-group = 128 query rows of one kv head (row r: query r / G, head r % G, so
// the G heads of a group share the staged keys and values) x one part of the
// positions those rows see; 4 waves of 32 rows, 64 positions a step.  K and V of a
// step go from memory straight into LDS, the next step's while this one is
// multiplied; two work-groups per CU (64 KiB each at 128 dims) cover each
// other's softmax.  Rows past kv_len load zeros (the resource's range).
//   S^T = K Q^T on v_mfma_f32_32x32x16_f16 (lane l: row l % 32, hf = l / 32):
//     A = K (position l % 32, dims 16 j + 8 hf ..), B = Q^T from registers; a lane
//     ends with 16 of 32 positions, 8 (i / 4) + 4 hf + i % 4, of its row: the
//     softmax is per lane but for one exchange with lane l ^ 32, and
//   O^T += V^T P^T takes P from the same registers: k-index 8 hf + j is position
//     4 hf + j (j < 4) or 8 + 4 hf + j - 4; A = V^T by transposing LDS reads.
// Staged rows are HD / 8 16-byte chunks, chunk c of K row r at c ^ (r % chunks),
// of V row r at c ^ 4 (r % 4) ^ (r / 4) % 4 (128 dims) so that the 4 rows of a
// transposing read lie in different quarters: no bank conflict at 128 dims.
// A row's sums are rescaled whenever its maximum grows: its largest weight so far is
// exactly 1, as in the decode kernel, whose 32-position groups the second half of a
// step equals.  The first 32 positions' weights, whose maximum the second half may
// still raise, are multiplied as two f16 terms.  Error against 64 bits, against groups
// of decodes: random scores 2.1e-4 (2.4e-4) at 600 positions, 2.4e-4 (2.6e-4) at 2000;
// rows where a later position takes most of the weight equal to within 0.2%.  (Rescaled
// only after a growth of 2^8: 62.8 us instead of 66.4 at 2048 queries, and such rows
// up to 27% above; without the second term 59.4 us and up to 7% above; with it for
// all positions 69.2.)
// Bound: a wave's own chain of products, softmax, products (MFMA busy 28% of the cycles).
// 2048 queries of 32 heads x 128 dims: 2930 -> 66 us (0.52 PFLOP/s of the pairs
// that are seen), against 128 decodes of 16 queries each; 509 of 14 x 64 behind
// 1022 positions 585 -> 19 us.
constexpr int kPrefillRows = 128;   // query rows of one kv head per work-group: 4 waves x 32
constexpr int kPrefillTokens = 64;  // cache tokens per staged tile
constexpr int kPrefillThreads = 256;
constexpr size_t prefill_lds_bytes(int HD) { return (size_t)2 * 2 * kPrefillTokens * HD * 2; }

// x with its infinities and NaNs replaced by zeros.
__device__ __forceinline__ half8_t finite_part(half8_t x) {
    uint4_t w = __builtin_bit_cast(uint4_t, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t v = w[e];
        w[e] = ((v & 0x7C00u) == 0x7C00u ? 0u : v & 0xFFFFu) | ((v & 0x7C000000u) == 0x7C000000u ? 0u : v & 0xFFFF0000u);
    }
    return as_h8(w);
}

template <int HD>
__global__ __launch_bounds__(kPrefillThreads) __attribute__((amdgpu_waves_per_eu(2))) void prefill_kernel(PrefillArgs a) {
    constexpr int CH = HD / 8, KS = HD / 16, NB = HD / 32;         // 16-byte chunks per row, k-steps, dim blocks
    constexpr int LPT = kPrefillTokens * CH / kPrefillThreads;     // loads per thread, operand and tile
    constexpr uint32_t OP = kPrefillTokens * HD;                   // halves per staged operand
    extern __shared__ __attribute__((aligned(16))) _Float16 pre_lds[]; // [2][K, V][kPrefillTokens][HD]
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t t = blockIdx.x;
    auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }; // divisions run on the vector ALUs
    const uint32_t g = uniform(t % a.kv_heads);
    t /= a.kv_heads;
    const uint32_t s = t % a.splits, rank = uniform(t / a.splits);
    const uint32_t tile = a.tiles - 1u - rank; // the longest first

    // Rows of this lane and the positions they see: [0, lim).
    const uint32_t row0 = tile * (uint32_t)kPrefillRows, wrow0 = row0 + 32u * (uint32_t)wave;
    const int base = (int)a.kv_len - (int)a.n + 1;
    auto lim_of = [&](uint32_t r) -> int { return base + (int)(min(r, a.rows - 1u) / a.gqa); };
    const uint32_t r = wrow0 + (uint32_t)li;
    const uint32_t rc = min(r, a.rows - 1u), qi = rc / a.gqa, head = g * a.gqa + rc % a.gqa;
    const int lim = lim_of(r);
    const int wmax = wrow0 < a.rows ? (int)uniform((uint32_t)lim_of(wrow0 + 31u)) : 0, wmin = (int)uniform((uint32_t)lim_of(wrow0));
    const uint32_t nt = (uint32_t)(max(lim_of(row0 + (uint32_t)kPrefillRows - 1u), 0) + kPrefillTokens - 1) / kPrefillTokens;
    const uint32_t t0 = uniform(nt * s / a.splits), t1 = uniform(nt * (s + 1u) / a.splits); // nt * splits < 2^32

    half8_t qop[KS];
    {
        const uint16_t* p = a.q + ((uint64_t)qi * a.q_heads + head) * HD;
#pragma unroll
        for (int j = 0; j < KS; ++j) qop[j] = as_h8(*(const uint4_t*)(p + 16 * j + 8 * hf));
    }

    // Staging: load j fills slots tid + 256 * j of the operand; slot -> row, chunk.
    auto ksw = [](uint32_t row) { return row & (uint32_t)(CH - 1); };
    auto vsw = [](uint32_t row) {
        return CH == 16 ? ((row & 3u) << 2) | ((row >> 2) & 3u) : ((row >> 1) & 1u) << 2;
    };
    const uint32_t rstride = a.kv_heads * (uint32_t)HD; // halves
    uint32_t koff[LPT], voff[LPT];
#pragma unroll
    for (int j = 0; j < LPT; ++j) {
        const uint32_t q = (uint32_t)tid + (uint32_t)(kPrefillThreads * j), row = q / CH, c = q % CH;
        koff[j] = (row * rstride + 8u * (c ^ ksw(row))) * 2u;
        voff[j] = (row * rstride + 8u * (c ^ vsw(row))) * 2u;
    }
    auto issue = [&](uint32_t tt, uint32_t buf) {
        const uint32_t tok0 = tt * (uint32_t)kPrefillTokens;
        const uint64_t at = (uint64_t)tok0 * rstride + (uint64_t)g * HD;
        const uint32_t rows = min((uint32_t)kPrefillTokens, a.kv_len - tok0);
        const int bytes = (int)(((rows - 1u) * rstride + (uint32_t)HD) * 2u); // rows past kv_len load zeros
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(a.k + at), (short)0, bytes, (int)kBufferWord3);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(a.v + at), (short)0, bytes, (int)kBufferWord3);
        _Float16* dst = pre_lds + buf * 2u * OP;
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            _Float16* d = dst + ((uint32_t)wave * 64u + (uint32_t)(kPrefillThreads * j)) * 8u; // wave-uniform
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)d, 16, (int)koff[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            _Float16* d = dst + OP + ((uint32_t)wave * 64u + (uint32_t)(kPrefillThreads * j)) * 8u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)d, 16, (int)voff[j], 0, 0, 0);
        }
    };
    auto barrier = [] {
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
    };

    float m_run, l_run;
    float16_t oacc[NB];

    // LDS offsets (halves) of this lane's operands in a staged tile.
    uint32_t kat[KS], va[NB], vb[NB];
#pragma unroll
    for (int j = 0; j < KS; ++j) kat[j] = (uint32_t)li * HD + 8u * (((uint32_t)(2 * j + hf)) ^ ksw((uint32_t)li));
    {
        const uint32_t i16 = (uint32_t)lane & 15u, ra = 4u * (uint32_t)hf + (i16 >> 2), rb = ra + 8u;
        const uint32_t c = (((uint32_t)lane >> 4) & 1u) * 2u + ((i16 & 3u) >> 1), lo = 4u * (i16 & 1u);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            va[nb] = OP + ra * HD + 8u * ((4u * nb + c) ^ vsw(ra)) + lo;
            vb[nb] = OP + rb * HD + 8u * ((4u * nb + c) ^ vsw(rb)) + lo;
        }
    }

    // SPLIT: the products take the values' finite part, and positions with an inf or NaN
    // are then added to the rows that see them one by one, weights in f32.
    auto process = [&](auto split, uint32_t tt, uint32_t buf) {
        constexpr bool SPLIT = decltype(split)::value;
        const int c0 = (int)(tt * (uint32_t)kPrefillTokens);
        if (c0 >= wmax) return; // wave-uniform: every row of the wave ends before this tile
        const _Float16* sb = pre_lds + buf * 2u * OP;
        float16_t sacc[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            sacc[tb] = (float16_t)0.0f;
#pragma unroll
            for (int j = 0; j < KS; ++j)
                sacc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8_t*)(sb + kat[j] + tb * 32 * HD), qop[j],
                                                                  sacc[tb], 0, 0, 0);
        }
        const bool masked = c0 + kPrefillTokens > wmin; // wave-uniform
        if (masked) {
            int see = lim - c0 - 4 * hf;
            __asm__ volatile("" : "+v"(see)); // compared with constants here, not as 32 values kept over the loop
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (32 * tb + 8 * (i / 4) + i % 4 >= see) sacc[tb][i] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sacc[tb][i]);
        const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mx), __builtin_bit_cast(uint32_t, mx), false, false);
        const uint32_t sw0 = sw[0], sw1 = sw[1]; // the row's two halves
        mx = fmaxf(__builtin_bit_cast(float, sw0), __builtin_bit_cast(float, sw1)) * a.scale_log2;
        if (__any(mx > m_run)) {
            const float mnew = fmaxf(m_run, mx);
            const float alpha = mnew == -INFINITY ? 1.0f : fast_exp2(m_run - mnew);
            m_run = mnew;
            l_run *= alpha;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) oacc[nb] *= alpha;
        }
        const float mref = m_run == -INFINITY ? 0.0f : m_run; // nothing seen yet: every score is -inf, p = 0
        half8_t pop[2][2], plo[2]; // plo: what f16 left of the first 32 positions' weights
        float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                const float p0 = fast_exp2(fmaf(sacc[tb][i], a.scale_log2, -mref));
                const float p1 = fast_exp2(fmaf(sacc[tb][i + 1], a.scale_log2, -mref));
                ps0 += p0;
                ps1 += p1;
                pop[tb][i / 8][i % 8] = (_Float16)p0;
                pop[tb][i / 8][i % 8 + 1] = (_Float16)p1;
                if (tb == 0) {
                    plo[i / 8][i % 8] = (_Float16)(p0 - (float)pop[0][i / 8][i % 8]);
                    plo[i / 8][i % 8 + 1] = (_Float16)(p1 - (float)pop[0][i / 8][i % 8 + 1]);
                }
            }
        l_run += ps0 + ps1;
        // The transposed V operand of dims 32 * nb .. + 31, the 16 tokens of pop[tb][kk].
        auto vfrag = [&](int tb, int kk, int nb) -> half8_t {
            const int ro = (32 * tb + 16 * kk) * HD;
            return __builtin_bit_cast(half8_t, __builtin_shufflevector(lds_read_tr16(sb + va[nb] + ro),
                                                                       lds_read_tr16(sb + vb[nb] + ro), 0, 1, 2, 3, 4, 5, 6, 7));
        };
#pragma unroll
        for (int x = 0; x < 4 * NB; ++x) {
            const int tb = x / (2 * NB), kk = (x / NB) % 2, nb = x % NB;
            half8_t v = vfrag(tb, kk, nb);
            if constexpr (SPLIT) v = finite_part(v);
            oacc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, pop[tb][kk], oacc[nb], 0, 0, 0);
            if (tb == 0) oacc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, plo[kk], oacc[nb], 0, 0, 0);
            if constexpr (SPLIT) __builtin_amdgcn_sched_barrier(0); // fewer fragments at once: no spills
        }
        if constexpr (SPLIT) {
            // Whether slot c of the tile's row holds an inf or NaN.
            auto nonfinite = [&](uint32_t row, uint32_t c) -> bool {
                const uint4_t w = *(const uint4_t*)(sb + OP + row * HD + 8u * c);
                bool any = false;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t v = w[e];
                    any |= (v & 0x7C00u) == 0x7C00u || (v & 0x7C000000u) == 0x7C000000u;
                }
                return any;
            };
            bool any = false; // row `lane`, from another slot on in each lane (banks)
#pragma unroll 4
            for (uint32_t c = 0; c < (uint32_t)CH; ++c) any |= nonfinite((uint32_t)lane, (c + (uint32_t)lane) % (uint32_t)CH);
#pragma unroll 1
            for (uint64_t todo = __ballot(any); todo; todo &= todo - 1u) {
                const uint32_t at = (uint32_t)__builtin_ctzll(todo);
                const uint32_t slots = (uint32_t)__ballot(lane < CH && nonfinite(at, (uint32_t)lane % (uint32_t)CH));
                float x = 0.0f;
#pragma unroll
                for (int j = 0; j < KS; ++j) {
                    const half8_t kv = *(const half8_t*)(sb + at * HD + 8u * (((uint32_t)(2 * j + hf)) ^ ksw(at)));
#pragma unroll
                    for (int e = 0; e < 8; ++e) x = fmaf((float)qop[j][e], (float)kv[e], x);
                }
                x += __shfl_xor(x, 32);
                const float p = fast_exp2(fmaf(x, a.scale_log2, -mref));
                const bool sees = c0 + (int)at < lim;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        const uint32_t slot = (uint32_t)(4 * nb + i / 4) ^ vsw(at);
                        if (!((slots >> slot) & 1u)) continue; // uniform
                        const half4_t v = *(const half4_t*)(sb + OP + at * HD + 8u * slot + 4 * hf);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float f = (float)v[e];
                            if (sees && !(fabsf(f) < INFINITY)) oacc[nb][i + e] = fmaf(p, f, oacc[nb][i + e]);
                        }
                    }
            }
        }
    };

    constexpr short kWaitAll = (short)0x0070; // vmcnt(0), lgkmcnt(0): this wave's loads are in LDS, its LDS reads done
    auto pass = [&](auto split) {
        m_run = -INFINITY;
        l_run = 0.0f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) oacc[nb] = (float16_t)0.0f;
        if (t0 >= t1) return;
        issue(t0, 0);
        __builtin_amdgcn_s_waitcnt(kWaitAll);
        barrier();
        uint32_t buf = 0;
        for (uint32_t tt = t0; tt < t1; ++tt) {
            if (tt + 1u < t1) issue(tt + 1u, buf ^ 1u); // its readers (tile tt - 1) passed the previous barrier
            process(split, tt, buf);
            __builtin_amdgcn_s_waitcnt(kWaitAll);
            barrier();
            buf ^= 1u;
        }
    };
    pass(std::false_type{});
    // An inf or NaN among the sums, under finite weights: it comes from the values, and
    // may have reached rows that do not see it (0 * inf) or have a weight there that f16
    // rounds to 0.  The work-group then takes its positions once more, split.  2048
    // queries of 32/8 heads x 128 dims, us: finite values 66, one inf in each head 220
    // (its rows one at a time without matrix instructions 10500), an inf at every
    // position 1790; as groups of decodes 2920.
    float l = l_run + __shfl_xor(l_run, 32), chk = 0.0f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) chk = fmaf(oacc[nb][i], 0.0f, chk);
    uint32_t* flags = (uint32_t*)pre_lds; // every tile has been read
    const bool redo = __any(chk != 0.0f && l * 0.0f == 0.0f && r < a.rows);
    if (lane == 0) flags[wave] = redo ? 1u : 0u;
    __syncthreads();
    const uint32_t again = flags[0] | flags[1] | flags[2] | flags[3];
    if (again) { // the same in every wave
        __syncthreads();
        pass(std::true_type{});
        l = l_run + __shfl_xor(l_run, 32);
    }
    uint32_t ro = wrow0 + (uint32_t)li;
    __asm__ volatile("" : "+v"(ro)); // its addresses are made here, not kept over the loops
    if (ro >= a.rows) return;
    if (a.splits == 1u) {
        const float inv = l == 0.0f ? 0.0f : 1.0f / l;
        uint16_t* po = a.out + ((uint64_t)(ro / a.gqa) * a.q_heads + g * a.gqa + ro % a.gqa) * HD;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = (_Float16)(oacc[nb][i + e] * inv);
                *(half4_t*)(po + 32 * nb + 2 * i + 4 * hf) = h;
            }
    } else {
        const uint64_t at = ((uint64_t)g * a.splits + s) * a.rows + ro;
        if (hf == 0) {
            a.part_m[at] = m_run;
            a.part_l[at] = l;
        }
        float* po = a.part_o + at * HD;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; i += 4)
                *(float4_t*)(po + 32 * nb + 2 * i + 4 * hf) =
                    (float4_t){oacc[nb][i], oacc[nb][i + 1], oacc[nb][i + 2], oacc[nb][i + 3]};
    }
}

} // namespace aw
