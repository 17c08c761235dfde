// Matrix-core products of few output tiles: Y[M, N] = X[M, K] . W[N, K]^T with K split over a workgroup's waves.
//
// The tiled bodies in linear.h walk K in slices that all of a workgroup's waves share, a barrier and a round trip per
// slice; with few output tiles most of the chip idles while a handful of workgroups walk K serially (a 100 x 5120
// product over K = 2880: 40 workgroups, 45 slices). Here each of NW waves computes the whole 16 TM x 16 TN output
// tile over its own contiguous share of K: it copies its operands global -> LDS into a ring of its own (no barrier
// in the loop: a wave waits only for its own copies), and the waves' float partial sums meet once, in LDS, added
// in wave order. What bounds it is the compute unit's load path, (16 TM + 16 TN) K elements per workgroup at 41-55 GB/s per
// compute unit with 4 lanes to every 64-byte row piece, its first round trip included (operand fragments read straight into
// registers, a lane to a row, move about half of that: the path is bound by the addresses of neighbouring lanes, not by
// bytes), and for weights too large for the caches HBM at 4.3 TB/s.
#pragma once

#include "linear.h"

namespace chroma {

// A unit is 64 bytes of every operand row (32 bfloat16 or 16 float values of K): lane l holds the 16-byte chunk
// l / 16 of row l % 16 of a 16-row block. One v_mfma_f32_16x16x32_bf16 takes a bfloat16 unit as it lies; for float,
// element e of every lane's 4 forms the operand of one v_mfma_f32_16x16x4f32 (both operands pair the same k, whose
// order inside a unit is then 0 4 8 12, 1 5 9 13, ...).
template <class T>
__device__ __forceinline__ void kwave_mfma(const uint4& b, const uint4& a, f32x4_t& acc) {
    if constexpr (sizeof(T) == 2) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), acc, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.x), __uint_as_float(a.x), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.y), __uint_as_float(a.y), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.z), __uint_as_float(a.z), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.w), __uint_as_float(a.w), acc, 0, 0, 0);
    }
}

// A float unit's 16 products of one element, summed 8 + 8.
__device__ __forceinline__ f32x4_t kwave_unit(const uint4& b, const uint4& a) {
    const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t lo = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.x), __uint_as_float(a.x), zero, 0, 0, 0);
    f32x4_t hi = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.z), __uint_as_float(a.z), zero, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.y), __uint_as_float(a.y), lo, 0, 0, 0);
    hi = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.w), __uint_as_float(a.w), hi, 0, 0, 0);
    return lo + hi;
}

// Elements of the LDS array: S units of TM + TN 16-row blocks (1 KiB each) per wave; a wave's partial sums (TM TN
// KiB) take the place of its own ring.
template <int TM, int TN, int NW, int S>
constexpr int kwave_elements() {
    return NW * 512 * (S * (TM + TN) > TM * TN ? S * (TM + TN) : TM * TN);
}

// The row of a 16-row block that this lane copies from.
__device__ __forceinline__ uint32_t kwave_row() { return threadIdx.x % 64u / 4u; }

// One output tile. ``a`` and ``b`` are the operands' first bytes; ``oa`` and
// ``ob`` hold the byte offset of row ``kwave_row`` of each 16-row block (rows past the edge repeat a valid row):
// 32-bit, so the caller guarantees operands below 2 GiB. ``row_bytes`` (a multiple of 16) is K's extent. The ring's
// 16-byte chunks are swizzled as the ring body's (``wide_swizzle``). ``store(i, j, v)`` is called once per 16 x 16
// block (i, j) on the wave that sums it: lane l has row 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3.
template <class T, int TM, int TN, int NW, int S, bool FINE, class Store>
__device__ __forceinline__ void kwave_tile(const char* __restrict__ a, const uint32_t (&oa)[TM], const char* __restrict__ b,
                                           const uint32_t (&ob)[TN], uint32_t row_bytes, uint16_t* lds, Store store) {
    static_assert(S >= 2, "a unit being read and at least one in flight");
    constexpr int PER = TM + TN;
    constexpr uint32_t WAVE = kwave_elements<TM, TN, 1, S>();
    const uint32_t lane = threadIdx.x % 64u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
    const uint32_t units = (row_bytes + 63u) / 64u, begin = units * wave / NW, end = units * (wave + 1u) / NW;
    uint16_t* ring = lds + wave * WAVE;
    const uint32_t chunk = 16u * ((lane % 4u) ^ wide_swizzle(lane / 4u));                               // copied byte of the row's unit
    const uint32_t at = (lane % 16u) * 32u + (((lane / 16u) ^ wide_swizzle(lane % 16u)) * 8u);  // fragment element in a block
    const uint32_t tail = row_bytes % 64u;  // bytes of a ragged last unit
    // Float sums are kept in levels, so that their rounding errors grow with the root of a level's length and not of the whole
    // (3 x 2880 x 11520: 6.2e-7 relative in one chain, 1.9e-7 with levels of FLUSH = 4 units, a wave's share, the waves).
    // FINE adds a unit's two halves of 8 products and takes 8 units a level, as exact as the weight stream it stands in for:
    // 8 x 4096 x 1024 9.6e-8 (1.55e-7 without), 3 x 2880 x 11520 1.3e-7. Its additions cost nothing beside the copies of few
    // rows, but a product of many rows is bound by the matrix cores: 1000 rows, 1024 -> 4096, +16%.
    constexpr bool LEVELS = sizeof(T) == 4;
    constexpr uint32_t FLUSH = FINE ? 8u : 4u;
    f32x4_t acc[TM][TN];
    unroll<TM>([&](auto i) { unroll<TN>([&](auto j) { acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}; }); });
    // past the row's end (a ragged last unit) a lane copies the unit's first 16 bytes instead; the reader drops them
    auto copy = [&](uint32_t u) {
        const uint32_t from = u * 64u + chunk < row_bytes ? chunk : 0u;
        uint16_t* slot = ring + (u - begin) % S * (PER * 512u);
        unroll<PER>([&](auto ic) {
            constexpr int i = ic;
            const char* source;
            if constexpr (i < TM) {
                source = a + u * 64u + (oa[i] + from);
            } else {
                source = b + u * 64u + (ob[i - TM] + from);
            }
            __builtin_amdgcn_global_load_lds((global_void*)source, (lds_void*)(slot + i * 512u), 16, 0, 0);
        });
    };
    auto multiply = [&](uint32_t u) {
        const uint16_t* slot = ring + (u - begin) % S * (PER * 512u) + at;
        uint4 fa[TM], fb[TN];
        unroll<TM>([&](auto i) { fa[i] = *reinterpret_cast<const uint4*>(slot + i * 512u); });
        unroll<TN>([&](auto j) { fb[j] = *reinterpret_cast<const uint4*>(slot + (TM + j) * 512u); });
        if (tail && u * 64u + 64u > row_bytes && 16u * (lane / 16u) >= tail) {
            unroll<TM>([&](auto i) { fa[i] = uint4{0u, 0u, 0u, 0u}; });
            unroll<TN>([&](auto j) { fb[j] = uint4{0u, 0u, 0u, 0u}; });
        }
        unroll<TM>([&](auto i) {
            unroll<TN>([&](auto j) {
                if constexpr (LEVELS && FINE) {
                    acc[i][j] += kwave_unit(fb[j], fa[i]);
                } else {
                    kwave_mfma<T>(fb[j], fa[i], acc[i][j]);
                }
            });
        });
    };
    unroll<S - 1>([&](auto n) {
        if (begin + uint32_t(n) < end) {
            copy(begin + uint32_t(n));
        }
    });
    f32x4_t sums[LEVELS ? TM : 1][LEVELS ? TN : 1];
    if constexpr (LEVELS) {
        unroll<TM>([&](auto i) { unroll<TN>([&](auto j) { sums[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}; }); });
    }
    auto level = [&](uint32_t u) {
        if constexpr (LEVELS) {
            if ((u - begin) % FLUSH == FLUSH - 1u || u + 1u == end) {
                unroll<TM>([&](auto i) {
                    unroll<TN>([&](auto j) {
                        sums[i][j] += acc[i][j];
                        acc[i][j] = u + 1u == end ? sums[i][j] : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    });
                });
            }
        }
    };
    uint32_t u = begin;
    for (; u + (S - 1) < end; ++u) {
        __builtin_amdgcn_s_waitcnt(vmcnt_wait((S - 2) * PER));  // unit u landed; the S - 2 after it may be in flight
        __builtin_amdgcn_sched_barrier(0);
        copy(u + (S - 1));  // into the slot unit u - 1 was read from
        multiply(u);
        level(u);
        __builtin_amdgcn_sched_barrier(0);
    }
    unroll<S - 1>([&](auto n) {
        constexpr int left = S - 2 - int(n);  // units in flight behind this one
        if (end - u > uint32_t(left)) {
            __builtin_amdgcn_s_waitcnt(vmcnt_wait(left * PER));
            __builtin_amdgcn_sched_barrier(0);
            multiply(u);
            level(u);
            __builtin_amdgcn_sched_barrier(0);
            ++u;
        }
    });
    if constexpr (NW == 1) {
        unroll<TM>([&](auto i) { unroll<TN>([&](auto j) { store(i, j, acc[i][j]); }); });
    } else {
        // (each wave's last fragment reads are done: they fed its products)
        f32x4_t* partial = reinterpret_cast<f32x4_t*>(lds) + lane;
        constexpr uint32_t STRIDE = WAVE / 8u;
        unroll<TM>([&](auto i) { unroll<TN>([&](auto j) { partial[wave * STRIDE + (i * TN + j) * 64u] = acc[i][j]; }); });
        __syncthreads();
        unroll<(TM * TN + NW - 1) / NW>([&](auto n) {
            const uint32_t t = n * NW + wave;
            if (t < uint32_t(TM * TN)) {
                f32x4_t sum = partial[t * 64u];
                unroll<NW - 1>([&](auto w) { sum += partial[(w + 1) * STRIDE + t * 64u]; });
                store(t / TN, t % TN, sum);
            }
        });
    }
}

// Four consecutive columns n .. n + 3 of a row of ``columns``, rounded once; whole chunks when rows are.
template <class T>
__device__ __forceinline__ void kwave_store(T* to, const float (&y)[4], uint32_t n, uint32_t columns) {
    if (columns % 4u == 0) {
        if constexpr (sizeof(T) == 2) {
            *reinterpret_cast<uint2*>(to) = uint2{uint32_t(f32_to_bf16(y[0])) | uint32_t(f32_to_bf16(y[1])) << 16,
                                                  uint32_t(f32_to_bf16(y[2])) | uint32_t(f32_to_bf16(y[3])) << 16};
        } else {
            *reinterpret_cast<float4*>(to) = float4{y[0], y[1], y[2], y[3]};
        }
        return;
    }
#pragma unroll
    for (uint32_t r = 0; r < 4u; ++r) {
        if (n + r < columns) {
            store1<T>(to + r, y[r]);
        }
    }
}

// A linear layer on ``kwave_tile``: 8 * ceil(tiles / 8) workgroups of 64 NW threads, the row tiles of one column tile
// adjacent (one XCD's L2 reads each weight row once). Requires 16-byte aligned operands and rows (K a multiple of 8
// bfloat16 or 4 float values), and X and a column tile of W below 2 GiB. Measured on cold weights, back to back, NW = 4, against
// the bodies that took them before (M x N x K): bfloat16 100 x 5120 x 2880 41.4 -> 16.4 us, 100 x 2880 x 4096 52.5 -> 14.7, 300 x
// 1024 x 4096 50.9 -> 14.6, 600 x 2880 x 4096 54.1 -> 30.4; float 256 x 160 x 128 12.2 -> 1.9, 100 x 4000 x 1000 87 -> 15.5.
template <class T, int TM, int TN, int NW, int S, bool FINE>
__device__ __forceinline__ void kwave_linear(const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ bias, T* __restrict__ out,
                                             uint32_t m_total, uint32_t n_total, uint32_t k_total) {
    __shared__ __attribute__((aligned(1024))) uint16_t lds[kwave_elements<TM, TN, NW, S>()];
    const uint32_t gy = (m_total + 16u * TM - 1u) / (16u * TM), gx = (n_total + 16u * TN - 1u) / (16u * TN);
    uint32_t logical;
    if (!xcd_logical_tile(gx * gy, logical)) {
        return;
    }
    const uint32_t m0 = logical % gy * (16u * TM), n0 = logical / gy * (16u * TN);
    const uint32_t lane = threadIdx.x % 64u, row_bytes = k_total * sizeof(T);
    uint32_t oa[TM], ob[TN];
    unroll<TM>([&](auto i) {
        const uint32_t m = m0 + i * 16u + kwave_row();
        oa[i] = (m < m_total ? m : m_total - 1u) * row_bytes;
    });
    unroll<TN>([&](auto j) {
        const uint32_t n = n0 + j * 16u + kwave_row();
        ob[j] = ((n < n_total ? n : n_total - 1u) - n0) * row_bytes;
    });
    kwave_tile<T, TM, TN, NW, S, FINE>(reinterpret_cast<const char*>(x), oa, reinterpret_cast<const char*>(w) + size_t(n0) * row_bytes, ob, row_bytes, lds,
                                 [&](uint32_t i, uint32_t j, f32x4_t v) {
        const uint32_t m = m0 + i * 16u + lane % 16u, n = n0 + j * 16u + 4u * (lane / 16u);
        if (m >= m_total || n >= n_total) {
            return;
        }
        T* row = out + size_t(m) * n_total + n;
        float y[4];
#pragma unroll
        for (uint32_t r = 0; r < 4u; ++r) {
            y[r] = v[r] + (bias ? load1<T>(bias + (n + r < n_total ? n + r : n_total - 1u)) : 0.0f);
        }
        kwave_store<T>(row, y, n, n_total);
    });
}

// The piece of ``logical`` among the experts' pieces of ``size`` slots, expert by expert, column by column, an expert's
// pieces of one column adjacent (the order of ``expert_tile_of``, from the counts alone: no piece is ever empty). Every
// wave scans the counts; ``total`` receives the number of pieces. False when ``logical`` >= gx * total.
struct ExpertPiece {
    uint32_t expert, first, column;  // first: the piece's first slot inside its expert
};
__device__ __forceinline__ uint32_t expert_pieces(const int32_t* __restrict__ counts, uint32_t experts, uint32_t size) {
    uint32_t total = 0;
    for (uint32_t e0 = 0; e0 < experts; e0 += kWave) {
        const uint32_t e = e0 + threadIdx.x % kWave;
        uint32_t n = e < experts ? (uint32_t(counts[e]) + size - 1u) / size : 0u;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            n += __shfl_xor(n, d, kWave);
        }
        total += n;
    }
    return total;
}
__device__ __forceinline__ ExpertPiece expert_piece_of(const int32_t* __restrict__ counts, uint32_t experts, uint32_t size, uint32_t gx,
                                                       uint32_t logical) {
    const uint32_t lane = threadIdx.x % kWave;
    uint32_t carry = 0;
    for (uint32_t e0 = 0; e0 < experts; e0 += kWave) {
        const uint32_t e = e0 + lane;
        const uint32_t n = e < experts ? (uint32_t(counts[e]) + size - 1u) / size : 0u;
        uint32_t inclusive = n;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t up = __shfl_up(inclusive, d, kWave);
            inclusive += lane >= uint32_t(d) ? up : 0u;
        }
        const uint32_t first = carry + inclusive - n;
        const unsigned long long hit = __ballot(n > 0 && gx * first <= logical && logical < gx * (first + n));
        if (hit) {
            const int source = __ffsll(hit) - 1;
            const uint32_t r = logical - gx * uint32_t(__shfl(first, source, kWave)), pieces = __shfl(n, source, kWave);
            return ExpertPiece{e0 + uint32_t(source), r % pieces * size, r / pieces};
        }
        carry += __shfl(inclusive, kWave - 1, kWave);
    }
    return ExpertPiece{0u, 0u, 0u};  // not reached: ``logical`` < gx * (pieces)
}

// Expert-grouped products on ``kwave_tile``: the slots of an expert (grouped by ``route_slots``) in pieces of 16 TM, each
// times TN 16-channel blocks; a piece with fewer live 16-row blocks runs a body of 1, 2, 4 or TM of them (float, 1024
// slots over 12 experts: 256 x 128 products 19 -> 5.7 us with their gated activation, 128 x 128 ones 18 -> 4.2, against the
// 128 x 128 tiles' serial slices). What bounds it is the chain of routing loads before a piece's first copy. Operands, order on the XCDs and ``epilogue`` as
// ``grouped_expert_linear``; launched as 8 * ceil(ceil(C / 16 TN) * (slots / 16 TM + experts) / 8) workgroups of 64 NW threads.
template <class T, bool PER_SLOT, int TM, int TN, int NW, int S, class Epilogue = std::nullptr_t>
__device__ __forceinline__ void grouped_expert_kwave(const T* __restrict__ w, const T* __restrict__ x, T* __restrict__ out,
                                                     const int32_t* __restrict__ scratch, uint32_t selected, uint32_t experts,
                                                     uint32_t channels, uint32_t inner, Epilogue epilogue = nullptr) {
    __shared__ __attribute__((aligned(1024))) uint16_t lds[kwave_elements<TM, TN, NW, S>()];
    const int32_t* offsets = scratch + experts;
    const int32_t* permutation = scratch + 2 * experts + 2;
    const uint32_t gx = (channels + 16u * TN - 1u) / (16u * TN);
    uint32_t logical;
    if (!xcd_logical_tile(gx * expert_pieces(scratch, experts, 16u * TM), logical)) {
        return;
    }
    const ExpertPiece piece = expert_piece_of(scratch, experts, 16u * TM, gx, logical);
    const uint32_t expert = __builtin_amdgcn_readfirstlane(piece.expert), first = __builtin_amdgcn_readfirstlane(piece.first);
    const uint32_t n0 = __builtin_amdgcn_readfirstlane(piece.column) * (16u * TN);
    const uint32_t left = uint32_t(scratch[expert]) - first, rows = left < 16u * TM ? left : 16u * TM;
    const int32_t* slot_of = permutation + offsets[expert] + first;
    const uint32_t lane = threadIdx.x % 64u, row_bytes = inner * sizeof(T);
    uint32_t ob[TN];
    unroll<TN>([&](auto j) {
        const uint32_t n = n0 + j * 16u + kwave_row();
        ob[j] = ((n < channels ? n : channels - 1u) - n0) * row_bytes;
    });
    auto body = [&](auto live) {
        constexpr int L = live;
        uint32_t oa[L];
        unroll<L>([&](auto i) {
            const uint32_t r = i * 16u + kwave_row();
            const uint32_t slot = uint32_t(slot_of[r < rows ? r : rows - 1u]);
            oa[i] = (PER_SLOT ? slot : slot / selected) * row_bytes;
        });
        kwave_tile<T, L, TN, NW, S, false>(reinterpret_cast<const char*>(x), oa,
                                    reinterpret_cast<const char*>(w) + (size_t(expert) * channels + n0) * row_bytes, ob, row_bytes, lds,
                                    [&](uint32_t i, uint32_t j, f32x4_t v) {
            const uint32_t r = i * 16u + lane % 16u, n = n0 + j * 16u + 4u * (lane / 16u);
            if (r >= rows || n >= channels) {
                return;
            }
            const uint32_t slot = uint32_t(slot_of[r]);
            float y[4] = {v[0], v[1], v[2], v[3]};
            if constexpr (!std::is_same_v<Epilogue, std::nullptr_t>) {
                epilogue(slot, n, y, expert);  // channels are a multiple of 4 (the code generator's condition)
            } else {
                kwave_store<T>(out + size_t(slot) * channels + n, y, n, channels);
            }
        });
    };
    if constexpr (TM > 1) {
        if (rows <= 16u) {
            body(std::integral_constant<int, 1>{});
            return;
        }
    }
    if constexpr (TM > 2) {
        if (rows <= 32u) {
            body(std::integral_constant<int, 2>{});
            return;
        }
    }
    if constexpr (TM > 4) {
        if (rows <= 64u) {
            body(std::integral_constant<int, 4>{});
            return;
        }
    }
    body(std::integral_constant<int, TM>{});
}

}  // namespace chroma
