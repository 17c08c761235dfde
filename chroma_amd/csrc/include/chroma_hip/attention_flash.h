// Grouped-query attention with sinks for few query rows (bfloat16) and for float prefills: the chain of attention.h on
// the matrix cores, one pass over the keys, each wave on key blocks of its own.
//
// The group-shared kernel (``attention_heads_mfma_bf16``) gives a workgroup 16 queries and every key; with few queries
// the chip idles (100 queries x 8 heads: 56 workgroups), and below 16 queries most of a tile is padding. Here a tile is
// 16 (query, head of the group) rows, so one query of 8 heads fills half of one and 36 queries 18, and the keys are
// split over the 4 waves of a workgroup and over ``splits`` workgroups. A wave copies its 64-key block of K and of V
// global -> LDS into buffers of its own (no barrier in the loop), reads V^T fragments with the transposing LDS read,
// and keeps (max, sum, p . v) of its keys; the waves of a workgroup meet in LDS, workgroups through ``partial`` (added
// by ``attention_flash_combine``). What bounds it is latency: a block's copies, one round trip, behind the block before.
// Measured back to back on 8 KV heads of 8 heads of 64 over 128-key windows, with the combining launch, against the kernels
// that took them before: 3 queries over 137 keys 25.5 -> 4.8 us, 36 over 4072 291 -> 7.5, 100 over 1100 22.2 (with its live
// tiles) -> 7.2.
//
// Float products run on v_mfma_f32_16x16x4f32 (256 queries of one KV head of 8 heads of 16 over 512 keys: 8.7 us with a wave
// per query head, 6.0 here).
//
// Rounding: the scores, scaled scores and masked scores are rounded as attention.h says; a probability is rounded to
// bfloat16 as exp(s - m), m a running maximum of the row, before it meets V, and the row is divided by the float sum at
// the end (the same relative rounding of each probability as when it is divided first). Where every wave has at most one
// block (up to 256 keys, one workgroup a row group) the waves exchange their (max, sum) before the second product and
// the probabilities are divided first, as attention.h's are: a row of few live keys then has the very probabilities of
// the unfused chain, at the price of one barrier.
#pragma once

#include "attention.h"
#include "kwave.h"

namespace chroma {

constexpr uint32_t kFlashWaves = 4, kFlashKeys = 64;
// A wave's maximum is only raised (its sums rescaled) once a score exceeds it by more than this: probabilities then
// stay below e^8, far inside float and bfloat16 range.
constexpr float kFlashHeadroom = 8.0f;

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

// Floats of one (KV head, row group, split): per row the maximum and the sum, then the D sums of p . v.
template <int D, int RT> constexpr uint32_t flash_partial_floats() { return 16u * RT * (D + 2u); }

// The result of a row from its (max, sum, p . v) parts: weights exp(max_i - M) with M the largest of them and the sink.
// A row whose scores and sink are all -inf divides 0 by 0, as the reference does.
struct FlashMerge {
    float top, total;
    __device__ __forceinline__ float weight(float peak) const { return peak == -__builtin_inff() ? 0.0f : fast_exp(peak - top); }
};

// MASK4: the mask's rows, first element and key count are multiples of 4 elements, so its entries are read 4 at a time.
template <class T, int D, int G, int RT, bool POW2, bool MASK4>
__device__ __forceinline__ void attention_flash(const AttentionOperandsOf<T>& a, uint32_t splits, float* __restrict__ partial) {
    constexpr bool BF16 = sizeof(T) == 2;
    constexpr uint32_t CHUNK = 16u / sizeof(T), PER_ROW = D / CHUNK;  // elements of a 16-byte chunk, chunks of a key's row
    static_assert(PER_ROW % 4u == 0 && 64u % PER_ROW == 0 && G >= 1, "head dimension and group");
    constexpr uint32_t WAVE = 2u * kFlashKeys * D;  // LDS elements per wave: a K block and a V block
    constexpr uint32_t ROWS = 16u * RT, OPAD = D + 4u;
    static_assert(ROWS * (OPAD + 2u) * 4u <= WAVE * sizeof(T), "a wave's sums fit its buffers");
    constexpr int COPIES = kFlashKeys * D * sizeof(T) / 1024;  // 1 KB copies per block and operand
    constexpr int PARTS = PER_ROW / 4u;                        // matrix-core operands of a row: 64 bytes of it each
    constexpr uint32_t SWZ = PER_ROW % 8u == 0 ? 7u : 3u;  // chunk c of row r lies at c ^ ((r / 2) & SWZ)
    __shared__ __attribute__((aligned(1024))) T lds[kFlashWaves * WAVE];
    const uint32_t lane = threadIdx.x % 64u, quad = lane / 16u, col = lane % 16u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
    const uint32_t kv = blockIdx.x, row0 = blockIdx.y * ROWS, split = blockIdx.z;
    const uint32_t total_rows = a.tokens * G;
    const float neg_inf = -__builtin_inff();
    T* ks = lds + wave * WAVE;
    T* vs = ks + kFlashKeys * D;
    __shared__ float stats[BF16 ? kFlashWaves : 1][BF16 ? ROWS : 1][2];
    const bool divided = BF16 && splits == 1u && a.keys <= kFlashWaves * kFlashKeys;

    uint32_t query[RT];
    uint4 qf[RT][PARTS];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint32_t row = row0 + rt * 16u + col < total_rows ? row0 + rt * 16u + col : total_rows - 1u;
        query[rt] = row / G;
#pragma unroll
        for (int c = 0; c < PARTS; ++c) {
            qf[rt][c] = *reinterpret_cast<const uint4*>(a.q + size_t(query[rt]) * a.qt + kv * a.qh + (row % G) * a.qg + (c * 4u + quad) * CHUNK);
        }
    }

    auto minus_infinity = [](T v) {
        if constexpr (BF16) {
            return v == 0xff80u;
        } else {
            return v == -__builtin_inff();
        }
    };
    // This wave's key blocks: split * 4 + wave, then every 4 * splits. With more than one, those that a mask entry of
    // this group's queries leaves alive are found first (a bit each; past 64 they all count as alive).
    const uint32_t blocks = (a.keys + kFlashKeys - 1u) / kFlashKeys, stride = kFlashWaves * splits, first = split * kFlashWaves + wave;
    const uint32_t mine = first < blocks ? (blocks - first + stride - 1u) / stride : 0u;
    unsigned long long alive = ~0ull;
    if (mine > 1u) {
        constexpr int TQ = (ROWS + G - 1) / G + 1;  // queries a group's rows can touch
        const uint32_t q_first = row0 / G, q_last = (row0 + ROWS < total_rows ? row0 + ROWS - 1u : total_rows - 1u) / G;
        alive = 0ull;
        for (uint32_t n0 = 0; n0 < (mine < 64u ? mine : 64u); n0 += 4u) {
            T bits[4][TQ];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t j = (first + (n0 + i) * stride) * kFlashKeys + lane;
#pragma unroll
                for (int t = 0; t < TQ; ++t) {
                    const uint32_t q = q_first + t < q_last ? q_first + t : q_last;
                    bits[i][t] = a.mask[size_t(q) * a.mt + (j < a.keys ? j : a.keys - 1u)];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bool any = false;
#pragma unroll
                for (int t = 0; t < TQ; ++t) {
                    any |= !minus_infinity(bits[i][t]);
                }
                any = any && n0 + i < mine && (first + (n0 + i) * stride) * kFlashKeys + lane < a.keys;
                if (__ballot(any) != 0ull) {
                    alive |= 1ull << (n0 + i);
                }
            }
        }
    }
    auto next_of = [&](uint32_t n) {
        while (n < mine && n < 64u && !((alive >> n) & 1ull)) {
            ++n;
        }
        return n;
    };

    // Copies: lane l moves position l % PER_ROW of row l / PER_ROW of each 1 KB piece. Keys past the end repeat the last.
    auto copy = [&](T* to, const T* past, uint32_t pj, uint32_t ph, const T* fresh, uint32_t nj, uint32_t nh, uint32_t block) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) {
            const uint32_t r = i * (64u / PER_ROW) + lane / PER_ROW, chunk = (lane % PER_ROW) ^ ((r / 2u) & SWZ);
            const uint32_t j = block * kFlashKeys + r < a.keys ? block * kFlashKeys + r : a.keys - 1u;
            const bool old = j < a.past;
            const T* row = old ? past + (size_t(j) * pj + kv * ph) : fresh + (size_t(j - a.past) * nj + kv * nh);
            __builtin_amdgcn_global_load_lds((global_void*)(row + chunk * CHUNK), (lds_void*)(to + i * (1024u / sizeof(T))), 16, 0, 0);
        }
    };
    auto copy_k = [&](uint32_t block) { copy(ks, a.k_past, a.kpj, a.kph, a.k_new, a.knj, a.knh, block); };
    auto copy_v = [&](uint32_t block) { copy(vs, a.v_past, a.vpj, a.vph, a.v_new, a.vnj, a.vnh, block); };

    float peak[RT], total[RT];
    f32x4_t o[RT][D / 16];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        peak[rt] = neg_inf;
        total[rt] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            o[rt][dt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    uint32_t n = next_of(0);
    if (n < mine) {
        copy_k(first + n * stride);
        copy_v(first + n * stride);
    }
    if constexpr (BF16) {
        if (divided && mine == 0u) {  // (a wave without a block; the others meet it at the barrier in the loop, run once)
            for (uint32_t r = lane; r < ROWS; r += 64u) {
                stats[wave][r][0] = neg_inf;
                stats[wave][r][1] = 0.0f;
            }
            __syncthreads();
        }
    }
    while (n < mine) {
        const uint32_t block = first + n * stride, next = next_of(n + 1u);
        // mask entries of this lane: keys 16 t + 4 quad .. + 3 of the block, its query
        // (every load unconditional, clamped: a guarded load would end its branch with a wait)
        struct alignas(4 * sizeof(T)) Four {
            T v[4];
        } m[RT][4];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t j = block * kFlashKeys + t * 16u + quad * 4u;
                const T* row = a.mask + size_t(query[rt]) * a.mt;
                if constexpr (MASK4) {
                    m[rt][t] = *reinterpret_cast<const Four*>(row + (j < a.keys ? j : a.keys - 4u));
                } else {
#pragma unroll
                    for (uint32_t r = 0; r < 4u; ++r) {
                        m[rt][t].v[r] = row[j + r < a.keys ? j + r : a.keys - 1u];
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(vmcnt_wait(0));  // K, V and the mask of this block
        __builtin_amdgcn_sched_barrier(0);
        if (block * kFlashKeys + kFlashKeys > a.keys) {
            // the copies of the last key stand for none: their probability is 0, and 0 times an infinite value would be NaN
            const uint32_t from = (a.keys - block * kFlashKeys) * PER_ROW;
            for (uint32_t c = from + lane; c < kFlashKeys * PER_ROW; c += 64u) {
                *reinterpret_cast<uint4*>(vs + c * CHUNK) = uint4{0u, 0u, 0u, 0u};
            }
        }
        // scores of keys 16 t + 4 quad + r for this lane's row, in u units: s = u * cs (attention_heads_mfma_bf16)
        float u[RT][4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4_t s[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                s[rt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int c = 0; c < PARTS; ++c) {
                const uint32_t r = t * 16u + col;
                const uint4 kf = *reinterpret_cast<const uint4*>(ks + r * D + ((c * 4u + quad) ^ ((r / 2u) & SWZ)) * CHUNK);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    if constexpr (BF16) {
                        kwave_mfma<T>(kf, qf[rt][c], s[rt]);
                    } else {
                        s[rt] += kwave_unit(kf, qf[rt][c]);
                    }
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    const bool in_x = block * kFlashKeys + t * 16u + quad * 4u + r < a.keys, in_y = block * kFlashKeys + t * 16u + quad * 4u + r + 1u < a.keys;
                    const float mx = in_x ? widen_of<T>(m[rt][t].v[r]) : neg_inf, my = in_y ? widen_of<T>(m[rt][t].v[r + 1]) : neg_inf;
                    float x = s[rt][r], y = s[rt][r + 1];
                    if constexpr (BF16) {
                        round_bf16_pair(x, y);
                    }
                    x *= a.scale;
                    y *= a.scale;
                    if constexpr (BF16 && !POW2) {
                        round_bf16_pair(x, y);
                    }
                    x += mx;
                    y += my;
                    if constexpr (BF16) {
                        round_bf16_pair(x, y);
                    }
                    u[rt][t][r] = x;
                    u[rt][t][r + 1] = y;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        bf16x8_t pf[RT][2];  // bfloat16: probabilities of the products' operands; float ones replace u
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float top = neg_inf;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                top = __builtin_fmaxf(top, __builtin_fmaxf(__builtin_fmaxf(u[rt][t][0], u[rt][t][1]), __builtin_fmaxf(u[rt][t][2], u[rt][t][3])));
            }
            if (__ballot(top > peak[rt] + kFlashHeadroom || (peak[rt] == neg_inf && top != neg_inf)) != 0ull) {
                top = __builtin_fmaxf(top, __shfl_xor(top, 16, kWave));
                top = __builtin_fmaxf(top, __shfl_xor(top, 32, kWave));
                top = __builtin_fmaxf(top, peak[rt]);
                const float shrink = peak[rt] == neg_inf ? 0.0f : fast_exp(peak[rt] - top);
                total[rt] *= shrink;
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt) {
                    o[rt][dt] *= shrink;
                }
                peak[rt] = top;
            }
            // subtracted before it is scaled: the rounding of peak * log2(e) alone would grow with the scores (2.6e-6 of a
            // float result at scores around 100, and an infinite power for a row that has met only a finite masking value)
            const float base = peak[rt] == neg_inf ? 0.0f : peak[rt];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    u[rt][t][r] = fast_exp(u[rt][t][r] - base);
                    total[rt] += u[rt][t][r];
                }
            }
        }
        if constexpr (BF16) {
            float factor[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                factor[rt] = 1.0f;
            }
            if (divided) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    float sum = total[rt] + __shfl_xor(total[rt], 16, kWave);
                    sum += __shfl_xor(sum, 32, kWave);
                    if (quad == 0) {
                        stats[wave][rt * 16 + col][0] = peak[rt];
                        stats[wave][rt * 16 + col][1] = sum;
                    }
                }
                __syncthreads();
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const uint32_t row = row0 + rt * 16u + col < total_rows ? row0 + rt * 16u + col : total_rows - 1u;
                    const float sink = widen_of<T>(a.sinks[kv * a.sh + (row % G) * a.sg]);
                    FlashMerge merge{sink, 0.0f};
#pragma unroll
                    for (uint32_t w = 0; w < kFlashWaves; ++w) {
                        merge.top = __builtin_fmaxf(merge.top, stats[w][rt * 16 + col][0]);
                    }
#pragma unroll
                    for (uint32_t w = 0; w < kFlashWaves; ++w) {
                        merge.total += merge.weight(stats[w][rt * 16 + col][0]) * stats[w][rt * 16 + col][1];
                    }
                    merge.total += merge.weight(sink);
                    factor[rt] = merge.weight(peak[rt]) / merge.total;
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; r += 2) {
                        const bf16x2_t pair = __builtin_convertvector(f32x2_t{u[rt][t][r] * factor[rt], u[rt][t][r + 1] * factor[rt]}, bf16x2_t);
                        pf[rt][t / 2][t % 2 * 4 + r] = pair[0];
                        pf[rt][t / 2][t % 2 * 4 + r + 1] = pair[1];
                    }
                }
            }
        }
        // slots 0-3 and 4-7 of lane (d, quad) hold keys 32 h + 4 quad + r and 32 h + 16 + 4 quad + r: one transposing
        // read each (lane 4 r + c of a quad gives the address of key r's columns 4 c .. + 3 and receives column
        // 4 r + c of the four keys)
        if constexpr (BF16) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) {
                s16x4_t half[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const uint32_t r = h * 32u + x * 16u + quad * 4u + col / 4u;
                    const uint32_t chunk = (dt * 2u + (col % 4u) / 2u) ^ ((r / 2u) & SWZ);
                    half[x] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vs + r * D + chunk * 8u + (col % 2u) * 4u));
                }
                const uint2 lo = __builtin_bit_cast(uint2, half[0]), hi = __builtin_bit_cast(uint2, half[1]);
                const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, uint4{lo.x, lo.y, hi.x, hi.y});
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[rt][h], o[rt][dt], 0, 0, 0);
                }
            }
        }
        } else {
            // product (t, r) takes keys 16 t + 4 quad + r: this lane's own probability, V's element (key, d = 16 dt + col).
            // 16 keys are summed before they join the row's: over 512 keys of 16 the result's error is 1.8e-7 of it
            // (2.9e-7 with one chain over a wave's keys and over each score's products, 2.1e-7 on the vector units)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f32x4_t sum[RT][D / 16];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t key = t * 16u + quad * 4u + r;
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) {
                        const float v = vs[key * D + ((dt * 4u + col / 4u) ^ ((key / 2u) & SWZ)) * 4u + col % 4u];
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) {
                            const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                            sum[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, u[rt][t][r], r == 0 ? zero : sum[rt][dt], 0, 0, 0);
                        }
                    }
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) {
                        o[rt][dt] += sum[rt][dt];
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // Both buffers have been read. (Copies issued earlier would be waited for by the reads above: the compiler
        // cannot tell the buffers apart. The other waves of the compute unit cover the round trip.)
        if (next < mine) {
            copy_k(first + next * stride);
            copy_v(first + next * stride);
        }
        n = next;
    }

    // The waves' parts: rows of (D + 4) floats in each wave's own buffers, then [row][max, sum].
    float* mine_o = reinterpret_cast<float*>(lds + wave * WAVE);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        total[rt] += __shfl_xor(total[rt], 16, kWave);
        total[rt] += __shfl_xor(total[rt], 32, kWave);
        const uint32_t r = rt * 16u + col;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            *reinterpret_cast<f32x4_t*>(mine_o + r * OPAD + dt * 16u + quad * 4u) = o[rt][dt];
        }
        if (quad == 0) {
            mine_o[ROWS * OPAD + 2u * r] = peak[rt];
            mine_o[ROWS * OPAD + 2u * r + 1u] = total[rt];
        }
    }
    __syncthreads();
    const float* parts = reinterpret_cast<const float*>(lds);
    constexpr uint32_t PART = WAVE * sizeof(T) / 4u;  // floats of a wave's buffers
    for (uint32_t i = threadIdx.x; i < ROWS * (D / 4u); i += 64u * kFlashWaves) {
        const uint32_t r = i / (D / 4u), d = i % (D / 4u) * 4u, row = row0 + r;
        if (row >= total_rows) {
            continue;
        }
        FlashMerge merge{splits == 1u ? widen_of<T>(a.sinks[kv * a.sh + (row % G) * a.sg]) : neg_inf, 0.0f};
        const float sink = merge.top;
#pragma unroll
        for (uint32_t w = 0; w < kFlashWaves; ++w) {
            merge.top = __builtin_fmaxf(merge.top, parts[w * PART + ROWS * OPAD + 2u * r]);
        }
        f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t w = 0; w < kFlashWaves; ++w) {
            const float scale = divided ? 1.0f : merge.weight(parts[w * PART + ROWS * OPAD + 2u * r]);
            merge.total += scale * parts[w * PART + ROWS * OPAD + 2u * r + 1u];
            sum += scale * *reinterpret_cast<const f32x4_t*>(parts + w * PART + r * OPAD + d);
        }
        if (splits == 1u) {
            merge.total += merge.weight(sink);
            sum *= divided ? 1.0f : 1.0f / merge.total;
            const float y[4] = {sum[0], sum[1], sum[2], sum[3]};
            kwave_store<T>(a.out + ((size_t(row / G) * a.kv_heads + kv) * G + row % G) * D + d, y, d, D);
        } else {
            float* to = partial + size_t((kv * gridDim.y + blockIdx.y) * splits + split) * flash_partial_floats<D, RT>();
            *reinterpret_cast<f32x4_t*>(to + 2u * ROWS + r * D + d) = sum;
            if (d == 0) {
                to[2u * r] = merge.top;
                to[2u * r + 1u] = merge.total;
            }
        }
    }
}

// The splits of every row, in order, and the sink (grid: KV heads x row groups, 256 threads).
template <class T, int D, int G, int RT>
__device__ __forceinline__ void attention_flash_combine(const float* __restrict__ partial, const T* __restrict__ sinks, uint32_t sh,
                                                        uint32_t sg, T* __restrict__ out, uint32_t tokens, uint32_t splits) {
    constexpr uint32_t ROWS = 16u * RT, PART = flash_partial_floats<D, RT>();
    const uint32_t kv = blockIdx.x, row0 = blockIdx.y * ROWS;
    const float* parts = partial + size_t(kv * gridDim.y + blockIdx.y) * splits * PART;
    for (uint32_t i = threadIdx.x; i < ROWS * (D / 4u); i += 256u) {
        const uint32_t r = i / (D / 4u), d = i % (D / 4u) * 4u, row = row0 + r;
        if (row >= tokens * G) {
            continue;
        }
        const float sink = widen_of<T>(sinks[kv * sh + (row % G) * sg]);
        FlashMerge merge{sink, 0.0f};
        for (uint32_t s = 0; s < splits; ++s) {
            merge.top = __builtin_fmaxf(merge.top, parts[s * PART + 2u * r]);
        }
        f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t s = 0; s < splits; ++s) {
            const float scale = merge.weight(parts[s * PART + 2u * r]);
            merge.total += scale * parts[s * PART + 2u * r + 1u];
            sum += scale * *reinterpret_cast<const f32x4_t*>(parts + s * PART + 2u * ROWS + r * D + d);
        }
        merge.total += merge.weight(sink);
        sum *= 1.0f / merge.total;
        const float y[4] = {sum[0], sum[1], sum[2], sum[3]};
        kwave_store<T>(out + ((size_t(row / G) * gridDim.x + kv) * G + row % G) * D + d, y, d, D);
    }
}

}  // namespace chroma
