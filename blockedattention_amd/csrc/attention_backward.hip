// Backward of the one-pass varlen attention (attention.hip): dQ, dK and dV per segment and head from dO, with the
// probabilities recomputed from the row sums the forward pass kept (base-2 logarithms, one float per query) and never
// written to memory.  It is what a caller of the reference gets from the backward passes of blockGEMM, blockSoftmax
// and blockGEMM (csrc/sparseBlockedAttention.cpp:52-72, 95-114): that chain writes and reads six M x N arrays.
//
//   P  = 2^(c Q K^T - lse)      dP = dO V^T      dS = P o (dP - delta),  delta = sum over columns of dO o O
//   dV = P^T dO                 dK = scale dS^T Q                        dQ = scale dS K
//
// Two kernels, each owning its results (no atomics, the same sums every time): attention_dq_kernel walks the keys for a
// block of queries and leaves delta for attention_dkdv_kernel, which walks the queries for a block of keys.  The scores
// and dP are computed in both, seven products instead of five; adding dQ to memory from the second kernel instead
// would move N / 128 times the size of dQ in fp32 atomics.
//
// Measured on 16 segments x 16 heads of 1024 .. 4096 rows, K = 128, bf16: dQ 1.21 ms (1.22 PFLOP/s over its three
// products), dK and dV 1.75 ms (1.13 over four), 2.96 ms together against 9.3 ms of the chain.  By counters the clock is 2.0
// GHz under dQ and 2.2 under dK and dV, and of the cycles the matrix unit is busy 59 and 50 %, the vector issue port 43 and
// 36 %, LDS 39 and 39 %, no bank conflicts: the phases of a block still follow each other in part.
//
// Operands lie in LDS as rows (one copy of each): a matrix operand whose reduction runs over the head dimension is read
// 16 bytes per lane, one whose reduction runs over the rows by the transposing read (ds_read_b64_tr_b16).  The lane that
// holds scores of (row 16 t + 4 rg + e, column 16 u + j) packs them, over two row tiles, into the second operand of the
// product that reduces over those rows, so that P and dS stay where they are.
#include <algorithm>

#include "att_common.hpp"
#include "ba_host.hpp"

namespace ba {

typedef __attribute__((address_space(3))) unsigned char *LdsPtr;
__device__ __forceinline__ LdsPtr lds_ptr(void *p) { return (LdsPtr)p; }
__device__ __forceinline__ u32x4 lds_row16(LdsPtr p, int off) {
    return *reinterpret_cast<__attribute__((address_space(3))) const u32x4 *>(p + off);
}
// Eight rows of one column (see lds_tr8 in gemm_any16.hip): four rows from p + off, four from `next` bytes on.
__device__ __forceinline__ u32x4 lds_col8(LdsPtr p, int off, int next) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *Ptr;
    const u32x2 l = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Ptr)(p + off)));
    const u32x2 h = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((Ptr)(p + off + next)));
    return u32x4{l[0], l[1], h[0], h[1]};
}
template <int DT> __device__ __forceinline__ float lo16(uint32_t w) { return Elem<DT>::to_float((uint16_t)w); }
template <int DT> __device__ __forceinline__ float hi16(uint32_t w) { return Elem<DT>::to_float((uint16_t)(w >> 16)); }

// Four consecutive results (columns c0 .. c0 + 3 of a row of K) to memory.
template <int DT> __device__ __forceinline__ void store4(uint16_t *row, int c0, int K, f32x4 v, float f) {
    if (c0 + 4 <= K) {
        *reinterpret_cast<u32x2_unaligned *>(row + c0) =
            u32x2{Elem<DT>::pack2(v[0] * f, v[1] * f), Elem<DT>::pack2(v[2] * f, v[3] * f)};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e < K) row[c0 + e] = Elem<DT>::from_float(v[e] * f);
    }
}

// LDS pitch of staged rows: 16 * (2 * odd) bytes, the 16-byte operand reads and the transposing reads meet no conflict
constexpr int att_pitch(int nk) { return 64 * nk + 32; }

struct AttBwdArgs {
    const void *V, *O, *dO;
    const float *lse;
    float *delta;
    void *dQ, *dK, *dV;
    int min_K;                                         // of the summary that lse and delta were sized from
};

// The ROWS rows of an array staged per block: thread -> (row, piece), kSteps pieces an array.
template <int NK, int THREADS, int ROWS = kAttKeys> struct AttStage {
    static constexpr int kPieces = 4 * NK;
    static constexpr int kLpr = NK == 3 ? 16 : kPieces;      // lanes per row (a power of two)
    static constexpr int kRowsStep = THREADS / kLpr;
    static constexpr int kSteps = ROWS / kRowsStep > 0 ? ROWS / kRowsStep : 1;
};

// ---------------------------------------------------------------------------------------------------------- dQ
// Workgroup = 4 wavefronts; a wavefront owns QT strips of 16 queries (64 apart), their Q and dO fragments in registers,
// and walks the keys in blocks of 64 staged in LDS (K and V rows), 32 at a time: scores and dP transposed (lane = query
// j, keys 4 rg + e), dS packed over two key tiles, dQ^T += K^T dS^T.
template <int DT, int NK, int QT, bool VEC>
__device__ __forceinline__ void att_dq_body(const RunArgs &a, const AttBwdArgs &w, const SegRec &rec, int64_t h, int64_t row0,
                                            int block, unsigned char *sK, unsigned char *sV) {
    using St = AttStage<NK, 256>;
    constexpr int kPitch = att_pitch(NK);
    constexpr int kOutTiles = 2 * NK;
    const int M = rec.M, N = rec.N, K = rec.K;
    const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = lane_id(), j = lane & 15, rg = lane >> 4;
    const int64_t o1 = h * a.Dm1 + rec.off1, o2 = h * a.Dm2 + rec.off2;
    const RowPieces<VEC> pq((const uint16_t *)a.A + o1, M, K), pg((const uint16_t *)w.dO + o1, M, K), po((const uint16_t *)w.O + o1, M, K);
    const RowPieces<VEC> pk((const uint16_t *)a.B + o2, N, K), pv((const uint16_t *)w.V + o2, N, K);
    const float c = a.scale * kLog2e;

    const int s_row = tid / St::kLpr, s_piece = tid % St::kLpr;
    u32x4 kw[St::kSteps], vw[St::kSteps];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int s = 0; s < St::kSteps; ++s) {
            const uint32_t off = pk.offset(kb + s * St::kRowsStep + s_row, s_piece);
            kw[s] = pk.load(off);
            vw[s] = pv.load(off);
        }
    };
    if (N > 0) fetch(0);

    const int r0 = block * kAttBlockRows * QT + wave * 16;
    u32x4 qf[QT][NK], gf[QT][NK];
    float lse[QT], delta[QT];
    f32x4 acc[QT][kOutTiles];
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int row = r0 + kAttBlockRows * q + j;
        float d = 0.f;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            qf[q][s] = pq.get(row, 4 * s + rg);
            gf[q][s] = pg.get(row, 4 * s + rg);
            const u32x4 of = po.get(row, 4 * s + rg);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d = fmaf(lo16<DT>(gf[q][s][i]), lo16<DT>(of[i]), d);
                d = fmaf(hi16<DT>(gf[q][s][i]), hi16<DT>(of[i]), d);
            }
        }
        delta[q] = quad_column_sum(d);
        lse[q] = row < M && N > 0 ? w.lse[row0 + row] : INFINITY;        // 2^-inf: rows that do not exist have no probabilities
        if (row < M && N > 0 && rg == 0) w.delta[row0 + row] = delta[q];
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const LdsPtr k_row = lds_ptr(sK) + j * kPitch + rg * 16, v_row = lds_ptr(sV) + j * kPitch + rg * 16;
    const LdsPtr k_col = lds_ptr(sK) + (4 * rg + (j >> 2)) * kPitch + (j & 3) * 8;

    auto put = [&](int kb) {
        if (St::kLpr == St::kPieces || s_piece < St::kPieces) {
#pragma unroll
            for (int s = 0; s < St::kSteps; ++s) {
                const int row = s * St::kRowsStep + s_row;
                const uint32_t off = pk.offset(kb + row, s_piece);
                *reinterpret_cast<u32x4 *>(sK + row * kPitch + s_piece * 16) = pk.finish(kw[s], off, s_piece);
                *reinterpret_cast<u32x4 *>(sV + row * kPitch + s_piece * 16) = pv.finish(vw[s], off, s_piece);
            }
        }
    };
    // The operands and delta's rows arrive under the first block's way into LDS: waited for in front of it, 64 x 8 segments of
    // 8 .. 32 rows, K = 128, took 13.6 us backward instead of 13.0, 338 x 14 of 5 .. 28 74 instead of 72.  Not at 32 < K <= 64,
    // where that costs 16 registers and the fifth wavefront per SIMD (512 x 8 of 100 .. 120 rows and 30 .. 60 keys 111 -> 115 us),
    // nor for rows that are cleared on that way (51 segments of 13 .. 43, K = 31: 11.1 -> 11.5).
    constexpr bool kPeeled = VEC && NK != 2;
    if constexpr (kPeeled) {
        if (N > 0) put(0);
        att_lds_barrier();
    }
    arrived(qf);
    arrived(gf);

    for (int kb = 0; kb < N; kb += kAttKeys) {
        if (!kPeeled || kb > 0) {
            att_lds_barrier();                         // the previous block is consumed
            put(kb);
            att_lds_barrier();
        }
        if (kb + kAttKeys < N) fetch(kb + kAttKeys);
        if (r0 >= M) continue;                         // the wavefront only stages
        const int left = N - kb;
        auto half = [&](auto h_tag) {                  // (a strip whose rows do not exist runs along: one code path)
            constexpr int NQ = QT, H0 = decltype(h_tag)::value;       // key tiles 2 H0, 2 H0 + 1
            f32x4 s[NQ][2], dp[NQ][2];
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t) s[q][t] = dp[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < NK; ++st)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u32x4 kf = lds_row16(k_row, 16 * (2 * H0 + t) * kPitch + 64 * st);
#pragma unroll
                    for (int q = 0; q < NQ; ++q) s[q][t] = Elem<DT>::mfma(kf, qf[q][st], s[q][t]);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < NK; ++st)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u32x4 vf = lds_row16(v_row, 16 * (2 * H0 + t) * kPitch + 64 * st);
#pragma unroll
                    for (int q = 0; q < NQ; ++q) dp[q][t] = Elem<DT>::mfma(vf, gf[q][st], dp[q][t]);
                }
            __builtin_amdgcn_sched_barrier(0);
            u32x4 ds[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[q][t][e] = __builtin_amdgcn_exp2f(fmaf(s[q][t][e], c, -lse[q]));
                if (left < kAttKeys) {                 // keys past the last one (their scores are zeros, lse may be anything)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[q][t][e] = 16 * (2 * H0 + t) + 4 * rg + e < left ? s[q][t][e] : 0.f;
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[q][t][e] *= dp[q][t][e] - delta[q];
                    ds[q][2 * t] = Elem<DT>::pack2(s[q][t][0], s[q][t][1]);
                    ds[q][2 * t + 1] = Elem<DT>::pack2(s[q][t][2], s[q][t][3]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < kOutTiles; ++t) {
                const u32x4 kc = lds_col8(k_col, 32 * H0 * kPitch + 32 * t, 16 * kPitch);
#pragma unroll
                for (int q = 0; q < NQ; ++q) acc[q][t] = Elem<DT>::mfma(kc, ds[q], acc[q][t]);
            }
        };
        half(std::integral_constant<int, 0>{});
        if (left > 32) half(std::integral_constant<int, 1>{});
    }
    uint16_t *dq = (uint16_t *)w.dQ + o1;
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int row = r0 + kAttBlockRows * q + j;
        if (row >= M) continue;
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) store4<DT>(dq + (int64_t)row * K, 16 * t + 4 * rg, K, acc[q][t], a.scale);
    }
}

// The same for two strips a wavefront: two LDS stages and one barrier a block.  Each half of a block is one
// stream of operand reads, kRing of them in flight across its three products (and into the next half); the exponentials
// stand between the matrix instructions of dP, and the pieces of the next block are written, and those of the block after
// it requested, between all of them: its values during the first half, its keys during the second, in one set of registers.
// Before, staging stood between two barriers a block and every product began with an LDS round trip.  16 x 16 pairs of
// 1024 .. 4096 rows, K = 128, bf16: 1378 -> 1241 us a launch; forward and backward 4104 -> 4025..4081 (the other kernels
// clock lower then), of 24 x 4 pairs of 1000 .. 2000 634 -> 610, of 48 x 4 of 200 .. 400 104 -> 101, K = 64 79 -> 78.
template <int DT, int NK, bool VEC>
__device__ __forceinline__ void att_dq_pipe_body(const RunArgs &a, const AttBwdArgs &w, const SegRec &rec, int64_t h, int64_t row0,
                                                 int block, unsigned char *lds) {
    using St = AttStage<NK, 256>;
    constexpr int QT = 2;
    constexpr int kPitch = att_pitch(NK);
    constexpr int kArray = kAttKeys * kPitch, kStage = 2 * kArray;       // keys, then values
    constexpr int kOutTiles = 2 * NK;
    constexpr int kRing = 4, kTail = 3;
    const int M = rec.M, N = rec.N, K = rec.K;
    const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = lane_id(), j = lane & 15, rg = lane >> 4;
    const int64_t o1 = h * a.Dm1 + rec.off1, o2 = h * a.Dm2 + rec.off2;
    const RowPieces<VEC> pq((const uint16_t *)a.A + o1, M, K), pg((const uint16_t *)w.dO + o1, M, K), po((const uint16_t *)w.O + o1, M, K);
    const RowPieces<VEC> pk((const uint16_t *)a.B + o2, N, K), pv((const uint16_t *)w.V + o2, N, K);
    const float c = a.scale * kLog2e;

    const int s_row = tid / St::kLpr, s_piece = tid % St::kLpr;
    const bool stages = St::kLpr == St::kPieces || s_piece < St::kPieces;
    u32x4 piece[St::kSteps];
    auto offset = [&](int s, int kb) { return pk.offset(kb + s * St::kRowsStep + s_row, s_piece); };
    auto put = [&](int s, int kb, int at, u32x4 x) {
        x = pk.finish(x, offset(s, kb), s_piece);
        if (stages) *reinterpret_cast<u32x4 *>(lds + at + (s * St::kRowsStep + s_row) * kPitch + s_piece * 16) = x;
    };
    {
        u32x4 values[St::kSteps];
#pragma unroll
        for (int s = 0; s < St::kSteps; ++s) {
            piece[s] = pk.load(offset(s, 0));
            values[s] = pv.load(offset(s, 0));
        }
#pragma unroll
        for (int s = 0; s < St::kSteps; ++s) {
            put(s, 0, 0, piece[s]);
            put(s, 0, kArray, values[s]);
            piece[s] = pv.load(offset(s, kAttKeys));
        }
    }
    const int r0 = block * kAttBlockRows * QT + wave * 16;
    u32x4 qf[QT][NK], gf[QT][NK];
    float lse[QT], delta[QT];
    f32x4 acc[QT][kOutTiles];
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int row = r0 + kAttBlockRows * q + j;
        float d = 0.f;
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            qf[q][s] = pq.get(row, 4 * s + rg);
            gf[q][s] = pg.get(row, 4 * s + rg);
            const u32x4 of = po.get(row, 4 * s + rg);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d = fmaf(lo16<DT>(gf[q][s][i]), lo16<DT>(of[i]), d);
                d = fmaf(hi16<DT>(gf[q][s][i]), hi16<DT>(of[i]), d);
            }
        }
        delta[q] = quad_column_sum(d);
        lse[q] = row < M && N > 0 ? w.lse[row0 + row] : INFINITY;        // 2^-inf: rows that do not exist have no probabilities
        if (row < M && N > 0 && rg == 0) w.delta[row0 + row] = delta[q];
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    arrived(qf);
    arrived(gf);
    att_lds_barrier();

    int kb = 0, stage = 0;
    // (past the last block: a stage that nobody reads, and loads of rows that do not exist)
    auto exchange = [&](auto sc, auto half_tag) {
        constexpr int s = decltype(sc)::value, H0 = decltype(half_tag)::value;
        put(s, kb + kAttKeys, (kStage - stage) + (H0 ? 0 : kArray), piece[s]);
        piece[s] = H0 ? pv.load(offset(s, kb + 2 * kAttKeys)) : pk.load(offset(s, kb + kAttKeys));
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, 0> first;
    constexpr std::integral_constant<int, 1> second;
    auto turn = [&]() {
        stage = kStage - stage;
        att_lds_barrier();
    };
    if (r0 >= M) {                                     // the wavefront only stages
        for (; kb < N; kb += kAttKeys, turn()) {
            static_for<St::kSteps>([&](auto sc) { exchange(sc, first); });
            static_for<St::kSteps>([&](auto sc) { exchange(sc, second); });
        }
        return;
    }
    const uint32_t row_base = lds_offset(lds) + (uint32_t)(j * kPitch + rg * 16);
    const uint32_t col_base = lds_offset(lds) + (uint32_t)((4 * rg + (j >> 2)) * kPitch + (j & 3) * 8);
    constexpr int kRows = 4 * NK, kCols = kOutTiles, kSteps = kRows + kCols;
    constexpr int kAheadC = kRing < kCols ? kRing : kCols;
    static_assert(kTail + 2 * kAheadC <= 15 && 2 * kTail + kRing <= 15);  // (the counter of outstanding reads has four bits)
    u32x4 ring[kRing];
    u32x2 lo[kRing], hi[kRing];
    // read I of half H0: scores (key row tiles 2 H0 and the next, step by step), then dP (value rows)
    auto read_row = [&](auto ic, auto half_tag) {
        constexpr int I = decltype(ic)::value, H0 = decltype(half_tag)::value;
        lds_read128<(I >= 2 * NK ? kArray : 0) + 16 * (2 * H0 + I % 2) * kPitch + 64 * (I % (2 * NK) / 2)>(ring[I % kRing], row_base + stage);
    };
    auto read_col = [&](auto ic, auto half_tag) {
        constexpr int I = decltype(ic)::value, H0 = decltype(half_tag)::value;
        lds_read_tr<32 * H0 * kPitch + 32 * I, 16 * kPitch>(lo[I % kRing], hi[I % kRing], col_base + stage);
    };
    auto half = [&](auto half_tag, int left) {         // (a strip whose rows do not exist runs along: one code path)
        constexpr int H0 = decltype(half_tag)::value;
        f32x4 s[QT][2], dp[QT][2];
        auto spread = [&](auto ic) {                   // the half's exchanges, evenly behind its steps
            constexpr int I = decltype(ic)::value, now = I * St::kSteps / kSteps, then = (I + 1) * St::kSteps / kSteps;
            if constexpr (then > now) exchange(std::integral_constant<int, now>{}, half_tag);
        };
        static_for<kRows>([&](auto ic) {
            constexpr int I = decltype(ic)::value, R = I % kRing, J = I + kRing, t = I % 2, st = I % (2 * NK) / 2;
            constexpr int kBehind = (J < kRows ? J : kRows) - (I + 1) + (I >= kRows - kTail ? 2 * kAheadC : 0);
            if constexpr (I == kRows - kTail) static_for<kAheadC>([&](auto xc) { read_col(xc, half_tag); });
            lds_wait<kBehind>(ring[R]);
#pragma unroll
            for (int q = 0; q < QT; ++q) {
                if constexpr (I < 2 * NK) s[q][t] = Elem<DT>::mfma(ring[R], qf[q][st], st ? s[q][t] : f32x4{0.f, 0.f, 0.f, 0.f});
                else dp[q][t] = Elem<DT>::mfma(ring[R], gf[q][st], st ? dp[q][t] : f32x4{-delta[q], -delta[q], -delta[q], -delta[q]});
            }
            // (from the second step of dP on: the scores have left the matrix unit)
            if constexpr (I > 2 * NK) {
                constexpr int kParts = 2 * NK - 1, from = (I - 2 * NK - 1) * 16 / kParts, to = (I - 2 * NK) * 16 / kParts;
                static_for<to - from>([&](auto xc) {
                    constexpr int x = from + decltype(xc)::value, tt = x / 8, q = x / 4 % 2, e = x % 4;
                    s[q][tt][e] = __builtin_amdgcn_exp2f(fmaf(s[q][tt][e], c, -lse[q]));
                });
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (J < kRows) read_row(std::integral_constant<int, (J < kRows ? J : 0)>{}, half_tag);
            spread(ic);
        });
        if (left < kAttKeys) {                         // keys past the last one (their scores are zeros, lse may be anything)
            const int mine = left - 4 * rg;
#pragma unroll
            for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[q][t][e] = 16 * (2 * H0 + t) + e < mine ? s[q][t][e] : 0.f;
        }
        u32x4 ds[QT];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < QT; ++q) {
                ds[q][2 * t] = Elem<DT>::pack2(s[q][t][0] * dp[q][t][0], s[q][t][1] * dp[q][t][1]);
                ds[q][2 * t + 1] = Elem<DT>::pack2(s[q][t][2] * dp[q][t][2], s[q][t][3] * dp[q][t][3]);
            }
        static_for<kCols>([&](auto ic) {
            constexpr int I = decltype(ic)::value, R = I % kRing, J = I + kRing;
            constexpr int kBehind = 2 * ((J < kCols ? J : kCols) - (I + 1)) + (H0 == 0 && I >= kCols - kTail ? kRing : 0);
            if constexpr (H0 == 0 && I == kCols - kTail) static_for<kRing>([&](auto xc) { read_row(xc, second); });
            lds_wait_tr<kBehind>(lo[R], hi[R]);
            const u32x4 kc = u32x4{lo[R][0], lo[R][1], hi[R][0], hi[R][1]};
#pragma unroll
            for (int q = 0; q < QT; ++q) acc[q][I] = Elem<DT>::mfma(kc, ds[q], acc[q][I]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (J < kCols) read_col(std::integral_constant<int, (J < kCols ? J : 0)>{}, half_tag);
            spread(std::integral_constant<int, kRows + I>{});
        });
    };
    for (; kb < N; kb += kAttKeys, turn()) {
        const int left = N - kb;
        static_for<kRing>([&](auto xc) { read_row(xc, first); });
        half(first, left);
        if (left > 32) half(second, left);
        else lds_drain(ring);                          // (what was read for it)
    }
    uint16_t *dq = (uint16_t *)w.dQ + o1;
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int row = r0 + kAttBlockRows * q + j;
        if (row >= M) continue;
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) store4<DT>(dq + (int64_t)row * K, 16 * t + 4 * rg, K, acc[q][t], a.scale);
    }
}

// Work item of a workgroup: item u of the (head, segment, block) items, head-major, cut into eight contiguous shares, one
// per die (as in attention_kernel: the blocks of a pair read the same rows and run side by side on one die).
// prefix: blocks of the segments before each segment; per_head: all of them.
__device__ __forceinline__ bool att_item(const RunArgs &a, int which, int64_t per_head, int64_t &h, int &g, int &block) {
    const unsigned id = flat_block(), die = id & 7u, kk = id >> 3;
    const int32_t *pfx = plan_rowblocks(a.plan, a.nseg, which);
    const int64_t items = per_head * a.H, share = (items + 7) >> 3;
    const int64_t u = (int64_t)die * share + kk;
    // a grid too small for the plan's items: the summary the launch was sized from is not this plan's
    if (id == 0 && threadIdx.x == 0 && share * 8 > flat_blocks())
        atomicAdd(&reinterpret_cast<PlanHeader *>(a.plan)->run_errors, 1);
    if (kk >= share || u >= items) return false;
    h = u / per_head;
    const int item = (int)(u % per_head);
    g = prefix_search(pfx, a.nseg, item);
    block = item - ((ConstI32)(uintptr_t)pfx)[g];
    return true;
}
// The head dimension fits the build and every byte offset inside the segment fits 32 bits.
__device__ __forceinline__ bool att_fits(const RunArgs &a, const SegRec &rec, int kp, int64_t h, int block) {
    if (rec.K <= kp && att_offsets_fit(max(rec.M, rec.N), rec.K)) return true;
    if (h == 0 && block == 0 && threadIdx.x == 0) atomicAdd(&reinterpret_cast<PlanHeader *>(a.plan)->run_errors, 1);
    return false;
}

template <int DT, int NK, int QT, bool PIPE>
__global__ __launch_bounds__(256, 2) void attention_dq_kernel(RunArgs a, AttBwdArgs w) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[(PIPE ? 4 : 2) * kAttKeys * att_pitch(NK)];
    const ConstHdr hdr = (ConstHdr)(uintptr_t)a.plan;
    const int64_t per_head = QT == 2 ? hdr->att_blocks128 : hdr->att_blocks64;
    const bool rows_ok = hdr->min_K == w.min_K;
    if (!header_ok(a) || !rows_ok) { report_mismatch(a); return; }
    int64_t h;
    int g, block;
    if (!att_item(a, QT - 1, per_head, h, g, block)) return;
    const SegRec rec = load_rec(plan_ro(a.plan, a.nseg).recs, g);
    if (rec.M < 1 || rec.K < 1 || !att_fits(a, rec, 32 * NK, h, block)) return;
    const int64_t row0 = att_row_base(w.min_K, a.Dm1, h, rec.off1);
    if constexpr (PIPE) {
        if ((rec.K & 7) == 0) att_dq_pipe_body<DT, NK, true>(a, w, rec, h, row0, block, lds);
        else att_dq_pipe_body<DT, NK, false>(a, w, rec, h, row0, block, lds);
    } else {
        unsigned char *values = lds + kAttKeys * att_pitch(NK);
        if ((rec.K & 7) == 0) att_dq_body<DT, NK, QT, true>(a, w, rec, h, row0, block, lds, values);
        else att_dq_body<DT, NK, QT, false>(a, w, rec, h, row0, block, lds, values);
    }
}

// ------------------------------------------------------------------------------------------------------- dK and dV
// Workgroup = PAIRS pairs of wavefronts; a pair owns 32 keys and walks the queries in blocks of QB staged in LDS (Q and
// dO rows, two stages).  One wavefront of a pair (side 0) holds K's fragments and dV's sums, the other (side 1) V's
// fragments and dK's sums, which keeps either within the registers of two wavefronts per SIMD at a head dimension of 128
// (both sums and both operands in one wavefront would take 192 registers before the first score):
//   step 1   side 0: P = 2^(c Q K^T - lse), packed, handed over through LDS;   side 1: dP = dO V^T
//   step 2   side 0: dV^T += dO^T P;                                           side 1: dS = P o (dP - delta), dK^T += Q^T dS
// Both sides run the same code on the two arrays in exchanged roles, two products each.
template <int DT, int NK, int PAIRS, int QB, bool VEC>
__device__ __forceinline__ void att_dkdv_body(const RunArgs &a, const AttBwdArgs &w, const SegRec &rec, int64_t h, int64_t row0,
                                              int block, unsigned char *lds) {
    constexpr int kThreads = 128 * PAIRS;
    using St = AttStage<NK, kThreads, QB>;
    constexpr int kTiles = QB / 16;
    constexpr int kPitch = att_pitch(NK);
    constexpr int kArray = QB * kPitch;          // bytes of one staged array
    constexpr int kStage = 2 * kArray + 8 * QB;        // Q, dO, lse, delta
    constexpr int kOutTiles = 2 * NK;
    const int M = rec.M, N = rec.N, K = rec.K;
    const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = lane_id(), j = lane & 15, rg = lane >> 4;
    const int side = wave / PAIRS, pair = wave % PAIRS;
    const int64_t o1 = h * a.Dm1 + rec.off1, o2 = h * a.Dm2 + rec.off2;
    const RowPieces<VEC> pq((const uint16_t *)a.A + o1, M, K), pg((const uint16_t *)w.dO + o1, M, K);
    const RowPieces<VEC> pf((const uint16_t *)(side ? w.V : a.B) + o2, N, K);
    const float c = a.scale * kLog2e;

    const int s_row = tid / St::kLpr, s_piece = tid % St::kLpr;
    u32x4 qw[St::kSteps], gw[St::kSteps];
    float aux = 0.f;                                   // threads 0 .. QB - 1: lse, QB .. 2 QB - 1: delta of a row of the block
    auto fetch = [&](int qb) {
#pragma unroll
        for (int s = 0; s < St::kSteps; ++s) {
            const uint32_t off = pq.offset(qb + s * St::kRowsStep + s_row, s_piece);
            qw[s] = pq.load(off);
            gw[s] = pg.load(off);
        }
        if (tid < 2 * QB) {
            const int row = qb + (tid & (QB - 1));
            // 2^-inf: rows that do not exist have no probabilities
            aux = row < M ? (tid < QB ? w.lse : w.delta)[row0 + row] : tid < QB ? INFINITY : 0.f;
        }
    };
    auto put = [&](int qb, unsigned char *stage) {
        if ((St::kLpr == St::kPieces || s_piece < St::kPieces) && (St::kRowsStep <= QB || s_row < QB)) {
#pragma unroll
            for (int s = 0; s < St::kSteps; ++s) {
                const int row = s * St::kRowsStep + s_row;
                const uint32_t off = pq.offset(qb + row, s_piece);
                *reinterpret_cast<u32x4 *>(stage + row * kPitch + s_piece * 16) = pq.finish(qw[s], off, s_piece);
                *reinterpret_cast<u32x4 *>(stage + kArray + row * kPitch + s_piece * 16) = pg.finish(gw[s], off, s_piece);
            }
        }
        if (tid < 2 * QB) *reinterpret_cast<float *>(stage + 2 * kArray + 4 * tid) = aux;
    };
    if (M > 0) fetch(0);

    const int key0 = block * 32 * PAIRS + 32 * pair;
    const bool alive = key0 < N;
    u32x4 kf[2][NK];
    f32x4 acc[kOutTiles][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int s = 0; s < NK; ++s) kf[u][s] = pf.get(key0 + 16 * u + j, 4 * s + rg);
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // this side's arrays: rows for the scores (Q / dO), columns for the sums (dO / Q)
    const LdsPtr row_base = lds_ptr(lds) + side * kArray + j * kPitch + rg * 16;
    const LdsPtr col_base = lds_ptr(lds) + (1 - side) * kArray + (4 * rg + (j >> 2)) * kPitch + (j & 3) * 8;
    const LdsPtr aux_base = lds_ptr(lds) + 2 * kArray + side * 4 * QB + rg * 16;
    unsigned char *hand = lds + 2 * kStage + pair * (64 * QB) + lane * 16;        // kTiles 16-byte slots of 64 lanes a pair
    // (the operands arrive under the first block's way into LDS: backward of 338 x 14 segments of 5 .. 28 rows, K = 128, 73 -> 72
    // us; before it at 32 < K <= 64, 16 x 8 of 600 .. 760 85 us against 86, and for rows that are cleared on that way)
    if constexpr (!VEC || NK == 2) arrived(kf);
    if (M > 0) put(0, lds);
    att_lds_barrier();
    if constexpr (VEC && NK != 2) arrived(kf);

    for (int qb = 0, stage = 0; qb < M; qb += QB, stage ^= 1) {
        const bool more = qb + QB < M;
        if (more) fetch(qb + QB);
        f32x4 s[kTiles][2];
        u32x4 pk[kTiles / 2][2];                                // [row tile pair][key tile]
        if (alive) {
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int u = 0; u < 2; ++u) s[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < NK; ++st)
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    const u32x4 rf = lds_row16(row_base, stage * kStage + 16 * t * kPitch + 64 * st);
#pragma unroll
                    for (int u = 0; u < 2; ++u) s[t][u] = Elem<DT>::mfma(rf, kf[u][st], s[t][u]);
                }
            if (side == 0) {
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    const f32x4 l = __builtin_bit_cast(f32x4, lds_row16(aux_base, stage * kStage + 64 * t));
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[t][u][e] = __builtin_amdgcn_exp2f(fmaf(s[t][u][e], c, -l[e]));
                        pk[t >> 1][u][2 * (t & 1)] = Elem<DT>::pack2(s[t][u][0], s[t][u][1]);
                        pk[t >> 1][u][2 * (t & 1) + 1] = Elem<DT>::pack2(s[t][u][2], s[t][u][3]);
                    }
                }
#pragma unroll
                for (int tt = 0; tt < kTiles / 2; ++tt)
#pragma unroll
                    for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4 *>(hand + (2 * tt + u) * 1024) = pk[tt][u];
            }
        }
        att_lds_barrier();
        if (alive) {
            if (side == 1) {
#pragma unroll
                for (int tt = 0; tt < kTiles / 2; ++tt)
#pragma unroll
                    for (int u = 0; u < 2; ++u) pk[tt][u] = *reinterpret_cast<const u32x4 *>(hand + (2 * tt + u) * 1024);
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    const f32x4 d = __builtin_bit_cast(f32x4, lds_row16(aux_base, stage * kStage + 64 * t));
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            const uint32_t p = pk[t >> 1][u][2 * (t & 1) + i];
                            pk[t >> 1][u][2 * (t & 1) + i] =
                                Elem<DT>::pack2(lo16<DT>(p) * (s[t][u][2 * i] - d[2 * i]),
                                                hi16<DT>(p) * (s[t][u][2 * i + 1] - d[2 * i + 1]));
                        }
                }
            }
#pragma unroll
            for (int tt = 0; tt < kTiles / 2; ++tt)
#pragma unroll
                for (int t = 0; t < kOutTiles; ++t) {
                    const u32x4 cf = lds_col8(col_base, stage * kStage + 32 * tt * kPitch + 32 * t, 16 * kPitch);
#pragma unroll
                    for (int u = 0; u < 2; ++u) acc[t][u] = Elem<DT>::mfma(cf, pk[tt][u], acc[t][u]);
                }
        }
        if (more) put(qb + QB, lds + (stage ^ 1) * kStage);
        att_lds_barrier();
    }
    uint16_t *out = (uint16_t *)(side ? w.dK : w.dV) + o2;
    const float f = side ? a.scale : 1.0f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int key = key0 + 16 * u + j;
        if (key >= N) continue;
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) store4<DT>(out + (int64_t)key * K, 16 * t + 4 * rg, K, acc[t][u], f);
    }
}

// The same for tall segments, eight wavefronts and one barrier a block: side 1 runs half a block behind side 0, so that on
// every SIMD one wavefront's exponentials stand beside the other's matrix instructions, and neither waits inside a block
// for what the other makes in it.  In iteration i
//   side 0   P = 2^(c Q K^T - lse) of block i, packed, handed over; dV^T += dO^T P
//   side 1   dS = P o (dP - delta) of block i - 1, dK^T += Q^T dS; then dP - delta = dO V^T - delta of block i, kept in registers
// Three stages (blocks i - 1 and i are read while i + 1 is written), two buffers of the handed probabilities.
// 16 x 16 pairs of 1024 .. 4096 rows, K = 128, bf16: two barriers a block, both sides in the same block 2.10 ms; one barrier
// 2.07; LDS reads in flight across the phases 2.01; staging spread over the matrix instructions, delta as their starting
// value 1.86; a loop for each side without branches in it 1.82.  An iteration takes 4100 cycles, of them 2048 of the matrix unit
// (counters; the ends of a workgroup, which has its compute unit alone, included).
template <int DT, int NK, int PAIRS, int QB, bool VEC>
__device__ __forceinline__ void att_dkdv_pipe_body(const RunArgs &a, const AttBwdArgs &w, const SegRec &rec, int64_t h,
                                                   int64_t row0, int block, unsigned char *lds) {
    constexpr int kThreads = 128 * PAIRS;
    using St = AttStage<NK, kThreads, QB>;
    constexpr int kTiles = QB / 16;
    constexpr int kPitch = att_pitch(NK);
    constexpr int kArray = QB * kPitch;          // bytes of one staged array
    constexpr int kStage = 2 * kArray + 8 * QB;        // Q, dO, lse, delta
    constexpr int kHand = 64 * QB;                     // bytes of a pair's probabilities
    constexpr int kRing = 5;                           // operand reads in flight (the counter of outstanding reads has four bits)
    constexpr int kOutTiles = 2 * NK;
    static_assert(QB == 64 && PAIRS % 2 == 0);
    const int M = rec.M, N = rec.N, K = rec.K;
    const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = lane_id(), j = lane & 15, rg = lane >> 4;
    const int side = wave / PAIRS, pair = wave % PAIRS;
    const int64_t o1 = h * a.Dm1 + rec.off1, o2 = h * a.Dm2 + rec.off2;
    const RowPieces<VEC> pq((const uint16_t *)a.A + o1, M, K), pg((const uint16_t *)w.dO + o1, M, K);
    const RowPieces<VEC> pf((const uint16_t *)(side ? w.V : a.B) + o2, N, K);
    const float c = a.scale * kLog2e;

    // Staging: kPuts pieces a thread and block (Q and dO of kSteps rows); a piece's registers are written to LDS and loaded
    // again for the block after the next in one place, and these places are spread over the matrix instructions: eight
    // wavefronts that issue all their loads at once stand in front of the texture unit for 400 cycles an iteration.
    const int s_row = tid / St::kLpr, s_piece = tid % St::kLpr;
    const bool stages = (St::kLpr == St::kPieces || s_piece < St::kPieces) && (St::kRowsStep <= QB || s_row < QB);
    constexpr int kPuts = 2 * St::kSteps;
    u32x4 piece[kPuts];
    float aux = 0.f;
    auto fetch = [&](int x, int qb) {
        const uint32_t off = pq.offset(qb + (x >> 1) * St::kRowsStep + s_row, s_piece);
        piece[x] = x & 1 ? pg.load(off) : pq.load(off);
    };
    auto put = [&](int x, int qb, int stage) {
        const int row = (x >> 1) * St::kRowsStep + s_row;
        const uint32_t off = pq.offset(qb + row, s_piece);
        const u32x4 done = x & 1 ? pg.finish(piece[x], off, s_piece) : pq.finish(piece[x], off, s_piece);
        if (stages) *reinterpret_cast<u32x4 *>(lds + stage + (x & 1) * kArray + row * kPitch + s_piece * 16) = done;
    };
    // (per-query values: the wavefronts of side 0, those of odd number delta, the two halves of a side the same ones)
    const int aux_row = tid & (QB - 1);
    const bool aux_delta = wave & 1;
    const __amdgpu_buffer_rsrc_t aux_res =
        __builtin_amdgcn_make_buffer_rsrc((void *)((aux_delta ? w.delta : w.lse) + row0), 0, 4u * (uint32_t)M, kRsrcFlags);
    auto fetch_aux = [&](int qb) { aux = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(aux_res, 4u * (uint32_t)(qb + aux_row), 0, 0)); };
    auto put_aux = [&](int qb, int stage) {
        // 2^-inf: rows that do not exist have no probabilities (past 2^30 rows the offset wraps: delta is not taken as read either)
        const float x = qb + aux_row < M ? (aux_delta ? -aux : aux) : (aux_delta ? 0.f : INFINITY);
        *reinterpret_cast<float *>(lds + stage + 2 * kArray + (aux_delta ? 4 * QB : 0) + 4 * aux_row) = x;
    };
    static_for<kPuts>([&](auto xc) { fetch(decltype(xc)::value, 0); });
    fetch_aux(0);

    const int key0 = block * 32 * PAIRS + 32 * pair;
    const bool alive = key0 < N;
    u32x4 kf[2][NK];
    f32x4 acc[kOutTiles][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int s = 0; s < NK; ++s) kf[u][s] = pf.get(key0 + 16 * u + j, 4 * s + rg);
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    arrived(kf);
    // this side's arrays: rows for the scores (Q / dO), columns for the sums (dO / Q)
    const uint32_t row_base = lds_offset(lds) + (uint32_t)(side * kArray + j * kPitch + rg * 16);
    const uint32_t col_base = lds_offset(lds) + (uint32_t)((1 - side) * kArray + (4 * rg + (j >> 2)) * kPitch + (j & 3) * 8);
    const uint32_t aux_base = lds_offset(lds) + (uint32_t)(2 * kArray + side * 4 * QB + rg * 16);
    const uint32_t hand_base = lds_offset(lds) + (uint32_t)(3 * kStage + pair * kHand + lane * 16);   // kTiles 16-byte slots of 64 lanes a pair
    f32x4 s[kTiles][2];
    u32x4 pk[kTiles / 2][2];                           // [row tile pair][key tile]
    u32x4 aux4[kTiles];                                // lse (side 0) or -delta (side 1) of the rows 16 t + 4 rg ..
    // Two products a block, each a stream of LDS operand reads, kRing of them in flight; towards the end of a stream
    // (kTail steps before it) the first reads of the next one are issued (`ahead`, kOps of them), so that it starts at once.
    constexpr int kRows = NK * kTiles, kCols = (kTiles / 2) * kOutTiles, kTail = 3;
    constexpr int kAheadR = kRing < kRows ? kRing : kRows, kAheadC = kRing < kCols ? kRing : kCols;
    static_assert(2 * kTail + kTiles + kAheadR <= 15 && kTail + 2 * kAheadC <= 15);      // (the counter has four bits)
    u32x4 ring[kRing];
    u32x2 lo[kRing], hi[kRing];
    auto read_aux = [&](int stage) {
        static_for<kTiles>([&](auto tc) { lds_read128<64 * decltype(tc)::value>(aux4[decltype(tc)::value], aux_base + stage); });
    };
    auto rows_ahead = [&](int stage) {
        static_for<kAheadR>([&](auto ic) {
            constexpr int I = decltype(ic)::value;
            lds_read128<16 * (I % kTiles) * kPitch + 64 * (I / kTiles)>(ring[I], row_base + stage);
        });
    };
    auto cols_ahead = [&](int stage) {
        static_for<kAheadC>([&](auto ic) {
            constexpr int I = decltype(ic)::value;
            lds_read_tr<32 * (I / kOutTiles) * kPitch + 32 * (I % kOutTiles), 16 * kPitch>(lo[I], hi[I], col_base + stage);
        });
    };
    // scores of a stage's rows with the operand held in registers, from zero (side 0) or -delta (side 1) on
    auto scores = [&](int stage, auto side_tag, auto &&between, auto ops, auto &&ahead) {
        constexpr bool kDelta = decltype(side_tag)::value == 1;
        const uint32_t at = row_base + stage;
        static_for<kRows>([&](auto ic) {
            constexpr int I = decltype(ic)::value, R = I % kRing, J = I + kRing, t = I % kTiles;
            constexpr int kBehind = (J < kRows ? J : kRows) - (I + 1) + (I >= kRows - kTail ? decltype(ops)::value : 0);
            if constexpr (I == kRows - kTail) ahead();
            if constexpr (kDelta && I < kTiles) lds_wait<kBehind>(aux4[t]);
            lds_wait<kBehind>(ring[R]);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const f32x4 from = I >= kTiles ? s[t][u] : kDelta ? __builtin_bit_cast(f32x4, aux4[t]) : f32x4{0.f, 0.f, 0.f, 0.f};
                s[t][u] = Elem<DT>::mfma(ring[R], kf[u][I / kTiles], from);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (J < kRows) lds_read128<16 * (J % kTiles) * kPitch + 64 * (J / kTiles)>(ring[R], at);
            between(ic, std::integral_constant<int, kRows>{});
        });
    };
    // sums over a stage's rows
    auto sums = [&](int stage, auto &&between, auto ops, auto &&ahead) {
        const uint32_t at = col_base + stage;
        static_for<kCols>([&](auto ic) {
            constexpr int I = decltype(ic)::value, R = I % kRing, J = I + kRing;
            constexpr int kBehind = 2 * ((J < kCols ? J : kCols) - (I + 1)) + (I >= kCols - kTail ? decltype(ops)::value : 0);
            if constexpr (I == kCols - kTail) ahead();
            lds_wait_tr<kBehind>(lo[R], hi[R]);
            const u32x4 cf = u32x4{lo[R][0], lo[R][1], hi[R][0], hi[R][1]};
#pragma unroll
            for (int u = 0; u < 2; ++u) acc[I % kOutTiles][u] = Elem<DT>::mfma(cf, pk[I / kOutTiles][u], acc[I % kOutTiles][u]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (J < kCols)
                lds_read_tr<32 * (J / kOutTiles) * kPitch + 32 * (J % kOutTiles), 16 * kPitch>(lo[R], hi[R], at);
            between(ic, std::integral_constant<int, kCols>{});
        });
    };
    static_for<kPuts>([&](auto xc) { put(decltype(xc)::value, 0, 0); fetch(decltype(xc)::value, QB); });
    if (side == 0) { put_aux(0, 0); fetch_aux(QB); }
    att_lds_barrier();

    // The three kinds of wavefronts have a loop each, one barrier a block.
    const int blocks = (M + QB - 1) / QB;
    int now = 0, before = 2 * kStage, next = kStage;   // stages of blocks i, i - 1 and i + 1
    int i = 0;
    // (past the last block: a stage that nobody reads, and loads of rows that do not exist)
    auto exchange = [&](auto xc) {
        put(decltype(xc)::value, (i + 1) * QB, next);
        fetch(decltype(xc)::value, (i + 2) * QB);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto spread = [&](auto ic, auto reads) {           // exchange x behind step (x + 1) reads / kPuts - 1
        constexpr int I = decltype(ic)::value, kEvery = decltype(reads)::value / kPuts;
        static_assert(kEvery * kPuts == decltype(reads)::value);
        if constexpr (I % kEvery == kEvery - 1) exchange(std::integral_constant<int, I / kEvery>{});
    };
    auto nothing = [](auto...) {};
    constexpr std::integral_constant<int, 0> zero;
    constexpr std::integral_constant<int, 1> one;
    auto turn = [&]() {
        att_lds_barrier();
        const int was = before;
        before = now; now = next; next = was;
    };
    auto aux_turn = [&]() { put_aux((i + 1) * QB, next); fetch_aux((i + 2) * QB); };
    if (!alive) {
        for (; i < blocks; ++i, turn()) {
            static_for<kPuts>(exchange);
            if (side == 0) aux_turn();
        }
    } else if (side == 0) {
        for (; i < blocks; ++i, turn()) {
            read_aux(now);
            rows_ahead(now);
            scores(now, zero, spread, std::integral_constant<int, 2 * kAheadC>{}, [&]() { cols_ahead(now); });
            static_for<kTiles>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                lds_wait<15>(aux4[t]);                 // (read before the first operand)
                const f32x4 l = __builtin_bit_cast(f32x4, aux4[t]);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[t][u][e] = __builtin_amdgcn_exp2f(fmaf(s[t][u][e], c, -l[e]));
                    pk[t >> 1][u][2 * (t & 1)] = Elem<DT>::pack2(s[t][u][0], s[t][u][1]);
                    pk[t >> 1][u][2 * (t & 1) + 1] = Elem<DT>::pack2(s[t][u][2], s[t][u][3]);
                }
            });
            unsigned char *hand = lds + 3 * kStage + pair * kHand + lane * 16 + (i & 1) * (PAIRS * kHand);
#pragma unroll
            for (int tt = 0; tt < kTiles / 2; ++tt)
#pragma unroll
                for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4 *>(hand + (2 * tt + u) * 1024) = pk[tt][u];
            sums(now, nothing, zero, nothing);
            aux_turn();
        }
    } else {
        auto handed = [&]() {                          // dS of block i - 1
            const uint32_t hand = hand_base + (1 - (i & 1)) * (PAIRS * kHand);
            static_for<kTiles>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                lds_read128<1024 * t>(pk[t >> 1][t & 1], hand);
            });
            cols_ahead(before);
            static_for<kTiles>([&](auto tc) {          // slot t: row tiles 2 (t / 2) and the next, key tile t % 2
                constexpr int t = decltype(tc)::value, tt = t >> 1, u = t & 1;
                lds_wait<kTiles - 1 - t + 2 * kAheadC>(pk[tt][u]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x4 &d = s[2 * tt + (e >> 1)][u];
                    pk[tt][u][e] = Elem<DT>::pack2(lo16<DT>(pk[tt][u][e]) * d[2 * (e & 1)], hi16<DT>(pk[tt][u][e]) * d[2 * (e & 1) + 1]);
                }
            });
        };
        auto dp_ahead = [&]() { read_aux(now); rows_ahead(now); };
        if (blocks > 0) {
            dp_ahead();
            scores(now, one, spread, zero, nothing);
            ++i;
            turn();
            for (; i < blocks; ++i, turn()) {
                handed();
                sums(before, spread, std::integral_constant<int, kTiles + kAheadR>{}, dp_ahead);
                scores(now, one, nothing, zero, nothing);
            }
            handed();
            sums(before, nothing, zero, nothing);
        }
    }
    uint16_t *out = (uint16_t *)(side ? w.dK : w.dV) + o2;
    const float f = side ? a.scale : 1.0f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int key = key0 + 16 * u + j;
        if (key >= N) continue;
#pragma unroll
        for (int t = 0; t < kOutTiles; ++t) store4<DT>(out + (int64_t)key * K, 16 * t + 4 * rg, K, acc[t][u], f);
    }
}

constexpr int att_dkdv_lds(int nk, int pairs, int qb, bool pipe) {
    return (pipe ? 3 : 2) * (2 * qb * att_pitch(nk) + 8 * qb) + (pipe ? 2 : 1) * pairs * 64 * qb;
}
static_assert(att_dkdv_lds(4, 4, 64, true) <= 160 * 1024);

// The build for short segments is bound by the life of a workgroup: three wavefronts per SIMD, not the two that its 197
// registers at a head dimension of 128 would leave (30 of them spilled), 1024 x 4 pairs of 2 .. 512 rows: 133 -> 110 us.
template <int DT, int NK, int PAIRS, int QB, bool PIPE>
__global__ __launch_bounds__(128 * PAIRS, QB == 32 ? 3 : 2) void attention_dkdv_kernel(RunArgs a, AttBwdArgs w) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    static_assert(PAIRS == 2 || PAIRS == 4, "the plan's column-block prefixes count blocks of 64 and of 128");
    const ConstHdr hdr = (ConstHdr)(uintptr_t)a.plan;
    const int64_t per_head = PAIRS == 4 ? hdr->att_cols128 : hdr->att_cols64;
    const bool rows_ok = hdr->min_K == w.min_K;
    if (!header_ok(a) || !rows_ok) return;            // reported by the dQ kernel
    int64_t h;
    int g, block;
    if (!att_item(a, PAIRS == 4 ? 3 : 2, per_head, h, g, block)) return;
    const SegRec rec = load_rec(plan_ro(a.plan, a.nseg).recs, g);
    if (rec.N < 1 || rec.K < 1 || !att_fits(a, rec, 32 * NK, h, block)) return;
    const int64_t row0 = att_row_base(w.min_K, a.Dm1, h, rec.off1);
    if constexpr (PIPE) {
        if ((rec.K & 7) == 0) att_dkdv_pipe_body<DT, NK, PAIRS, QB, true>(a, w, rec, h, row0, block, lds);
        else att_dkdv_pipe_body<DT, NK, PAIRS, QB, false>(a, w, rec, h, row0, block, lds);
    } else {
        if ((rec.K & 7) == 0) att_dkdv_body<DT, NK, PAIRS, QB, true>(a, w, rec, h, row0, block, lds);
        else att_dkdv_body<DT, NK, PAIRS, QB, false>(a, w, rec, h, row0, block, lds);
    }
}

// Blocks of 128 columns a head: at most half of the blocks of 64 and a half more for every segment.
static int64_t att_cols128_most(const ba_plan_info *info) { return ((int64_t)info->att_cols64 + info->nseg) / 2; }

template <int DT, int NK, int QT, int PAIRS, int QB, bool PIPE>
static int launch_bwd(const RunArgs &args, const AttBwdArgs &w, const ba_plan_info *info, hipStream_t stream) {
    constexpr int kLds = att_dkdv_lds(NK, PAIRS, QB, PIPE);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&attention_dkdv_kernel<DT, NK, PAIRS, QB, PIPE>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return BA_ERR_LAUNCH;
    const int64_t rows = ((QT == 2 ? info->att_blocks128 : info->att_blocks64) * args.H + 7) / 8 * 8;
    const int64_t blocks = PAIRS == 4 ? att_cols128_most(info) : info->att_cols64;
    const int64_t cols = (blocks * args.H + 7) / 8 * 8;
    if (rows > 0x7fffffff || cols > 0x7fffffff) return BA_ERR_UNSUPPORTED;
    if (rows > 0) {
        auto dq = [&](auto pipe) {
            hipLaunchKernelGGL((attention_dq_kernel<DT, NK, QT, decltype(pipe)::value>), flat_grid(rows), dim3(256), 0, stream, args, w);
        };
        // K <= 32: too few matrix instructions to spread the staging over.  Rows at any alignment and fewer than 256 keys a query
        // (the mean over the queries): the first blocks, which nothing overlaps, weigh more than the others gain (backward of
        // 48 x 8 pairs of 900 .. 1400 rows, K = 61 / 77 / 101, us, two stages and one: 64 keys 132 / 194 / 238, 128 / 182 / 225; 192 keys
        // 186 / 277 / 333, 184 / 270 / 324; 16 x 4 of 1000 .. 2000 242 / 334 / 378, 249 / 354 / 404).  Aligned rows are within 2 %
        // either way below 256 keys (K = 64, 128 keys 107, 106; K = 128, 64 keys 178, 177).
        const bool unaligned = (info->min_K | info->max_K) & 7;
        if constexpr (QT == 2 && NK > 1) {
            if (unaligned && info->Dout < 256 * info->total_rows) dq(std::false_type{});
            else dq(std::true_type{});
        } else {
            dq(std::false_type{});
        }
    }
    if (cols > 0)
        hipLaunchKernelGGL((attention_dkdv_kernel<DT, NK, PAIRS, QB, PIPE>), flat_grid(cols), dim3(128 * PAIRS), kLds, stream, args, w);
    return hipGetLastError() == hipSuccess ? BA_OK : BA_ERR_LAUNCH;
}

template <int DT, int QT, int PAIRS, int QB, bool PIPE>
static int launch_bwd_nk(int nk, const RunArgs &args, const AttBwdArgs &w, const ba_plan_info *info, hipStream_t stream) {
    switch (nk) {
        case 1: return launch_bwd<DT, 1, QT, PAIRS, QB, PIPE>(args, w, info, stream);
        case 2: return launch_bwd<DT, 2, QT, PAIRS, QB, PIPE>(args, w, info, stream);
        case 3: return launch_bwd<DT, 3, QT, PAIRS, QB, PIPE>(args, w, info, stream);
        default: return launch_bwd<DT, 4, QT, PAIRS, QB, PIPE>(args, w, info, stream);
    }
}

int launch_attention_backward(int dtype, const RunArgs &args, const void *V, const void *O, const void *dO, const float *lse,
                              float *delta, void *dQ, void *dK, void *dV, const ba_plan_info *info, hipStream_t stream) {
    if (info->max_K > 128 || info->nseg <= 0) return info->nseg <= 0 ? BA_OK : BA_ERR_UNSUPPORTED;
    const AttBwdArgs w{V, O, dO, lse, delta, dQ, dK, dV, info->min_K};
    const int nk = std::max(1, (info->max_K + 31) / 32);
    // Rows per segment on average: from 256 on wavefronts of two query strips (dQ), and for dK and dV a choice of workgroup
    // that is timed in backward passes, us, bf16.  128 keys that stage 64 queries, three stages of them: every query block is
    // staged once per workgroup, which has its compute unit alone.  64 keys and 32 queries: two to three times as many
    // resident workgroups.
    // - All workgroups of 128 keys find a compute unit of their own: these, they do twice the work at a time (10 x 4 of 400 ..
    //   600 rows, K = 32 / 64 / 128: 64 keys 31 / 36 / 54, 128 keys 25 / 30 / 47; 8 x 4 of 256 .. 300 18.3 / 21.8, 16.7 / 20.8).
    // - Otherwise where segments are tall enough for the stages to pay.  32 < K <= 64: 768 rows (24 x 8 of 750 .. 900 158, 168;
    //   16 x 8 of 1000 .. 1300 199, 194; 10 x 4 of 1500 .. 2500 213, 202).  Above, 576, K = 96 / 128: 50 x 8 of 450 .. 600 216 / 285,
    //   217 / 291; 64 x 8 of 600 .. 900 499 / 626, 484 / 613; 32 x 8 of 500 .. 750 rows and 100 .. 300 keys 91 / 114, 82 / 104.
    //   K <= 32 (two stages, below): 400 (K = 16 / 32: 64 x 8 of 256 .. 400 63 / 67, 65 / 70; of 400 .. 500 95 / 98, 92 / 96; 16 x 8
    //   of 600 .. 760 62.5 / 65, 57 / 59).
    // - Rows at any alignment, for which the small build has too few registers: always (64 x 8 of 200 .. 400, K = 101: 314, 230).
    const int64_t mean = info->total_rows / std::max<int64_t>(info->nseg, 1);
    const bool few = att_cols128_most(info) * args.H <= device_cu_count();
    const bool unaligned = (info->min_K | info->max_K) & 7;
    const bool strips2 = mean >= 256, keys128 = mean >= (unaligned || few ? 256 : nk == 1 ? 400 : nk == 2 ? 768 : 576);
    // K <= 32: the pipeline's LDS leaves room for one workgroup a compute unit where its two-stage form has two, and there are
    // too few matrix instructions to hide the exchanges behind: the pipeline only where a compute unit gets no second one.
    // Backward of 16 x 16 pairs of 1024 .. 4096 rows, K = 16 1273 us, two stages 1185; K = 32 1308, 1227; of 32 x 8 of 768 ..
    // 1100 190, 175; of 2 x 2 of 1000 .. 2000 49, 56; 32 x 8 of 768 .. 1100 rows with 64 keys 33, 37.
    auto launch = [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (keys128 && nk == 1 && !few) return launch_bwd<DT, 1, 2, 4, 64, false>(args, w, info, stream);
        if (keys128) return launch_bwd_nk<DT, 2, 4, 64, true>(nk, args, w, info, stream);
        if (strips2) return launch_bwd_nk<DT, 2, 2, 32, false>(nk, args, w, info, stream);
        return launch_bwd_nk<DT, 1, 2, 32, false>(nk, args, w, info, stream);
    };
    if (dtype == BA_F16) return launch(std::integral_constant<int, 0>{});
    if (dtype == BA_BF16) return launch(std::integral_constant<int, 1>{});
    return BA_ERR_UNSUPPORTED;
}

}  // namespace ba
