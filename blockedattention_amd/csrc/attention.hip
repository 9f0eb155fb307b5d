// Varlen attention in one pass: O_g = softmax(scale * Q_g K_g^T) V_g per segment and head, with the
// probabilities never written to memory.  It is what a caller of the reference gets from
// blockGEMM -> blockSoftmax -> blockGEMM (README.md:3; csrc/sparseBlockedAttention.cpp:118-131) when
// the probabilities themselves are not wanted: the M x N array, which bounds every other kernel of
// this library, stays in registers.
//
// Layout: Q_g is the M x K operand of the plan (offset off1), K_g and V_g are N x K (offset off2,
// both with the per-head stride Dm2), O_g is M x K at off1 of a [H, Dm1] buffer.  K <= 128.
//
// Workgroup = 4 wavefronts = 64 queries of one segment and head; the keys go by in blocks of 64.
// Per block the workgroup stages K_g's and V_g's rows as they lie, zero padded to a multiple of 32
// columns, in LDS; the second product reads V through the transposing LDS read.  A wavefront owns
// 16 queries:
//   S^T block  = K_blk Q^T   (matrix instructions, A operand = key rows from LDS, B operand = the
//                wavefront's query rows, held in registers for the whole pass); the lane
//                (j = lane%16, rg = lane/16) then holds query j's scores for keys 16t + 4rg + e;
//   online softmax: reference value m (a lazily raised row maximum) and row sum l per query (per lane;
//                the four lanes of a query exchange the block maximum), accumulators rescaled by
//                2^((m_old - m_new) c) when m is raised;
//   O^T       += V_blk^T P^T (A operand = columns of the value rows, gathered from LDS four keys at a
//                time by ds_read_b64_tr_b16, B operand = the lane's own
//                probabilities rounded to the 16-bit type: the k index of the instruction runs over
//                keys in the order the score registers hold them, so P never moves between lanes).
// The query index is lane%16 in scores and outputs alike, so m, l and the rescaling are per lane.
// Value rows were transposed on the way into LDS before (32 v_perm and eight 8-byte writes a thread and block, two-way
// conflicts): 512 pairs of 16 .. 256 rows and columns, K 32 .. 128, 23.2 -> 22.2 us; 16 x 16 pairs of 1024 .. 4096,
// K = 128, 1084 -> 1069 us; 1024 x 4 power-law pairs with the backward 293 -> 284 us.
#include <stdlib.h>

#include <algorithm>

#include "att_common.hpp"

namespace ba {

constexpr int kAttThreads = 256;
constexpr int kAttWaves = kAttThreads / 64;
constexpr int kAttRows = 16 * kAttWaves;              // queries per workgroup round
static_assert(kAttRows == kAttBlockRows, "the plan's row-block prefixes count blocks of kAttRows and 2 kAttRows");
// LDS row pitch, keys and values alike: 64 NK + 32 bytes.  A 16-byte operand read of a wavefront is served 32 lanes at
// a time, 512 bytes wide (measured: lane * 16 and 288-byte rows run at 4.75 cycles per wavefront read, 272- and
// 144-byte rows at 8): the lanes (j, rg) and (j, rg + 1) of sixteen rows j must land in 32 different 16-byte slots
// modulo 512 bytes, which a pitch of 16 * (2 * odd) bytes does; the transposing reads meet no conflict there either.
// LDS operand reads in flight per wavefront: six; four with two stages, whose registers hold no more; three in the builds
// for short segments, which are bound by the life of a workgroup: head dimensions up to 64 then fit 128 registers and
// four wavefronts per SIMD (256 segments of 32..128 rows, 31.3 -> 29.0 us), those up to 128 spill less at three
// wavefronts (512 pairs of 16 .. 256 rows and columns, 22.2 -> 21.9 us)
constexpr int att_ring(int qt, int stages) { return qt == 1 ? 3 : stages == 1 ? 6 : 4; }

// Four accumulators times f, in place: as an assignment under a branch the compiler keeps a second copy of all of them.
__device__ __forceinline__ void scale_in_place(f32x4 &x, float f) {
    float a = x[0], b = x[1], c = x[2], d = x[3];
    asm volatile("v_mul_f32 %0, %0, %4\n\tv_mul_f32 %1, %1, %4\n\tv_mul_f32 %2, %2, %4\n\tv_mul_f32 %3, %3, %4"
                 : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : "v"(f));
    x = f32x4{a, b, c, d};
}

// NK = 32-wide k steps (head dimension padded to 32 * NK).  ST = LDS stages (the rule: launch_attention).  VEC: the
// segment's K is a multiple of 8, its rows come as 16-byte loads that need no clearing; otherwise through RowPieces
// (element by element before: 256 x 8 pairs of 32 .. 128 rows, K = 61: 103 -> 48 us; 16 x 8 pairs of 512 .. 2048, K = 101:
// 764 -> 279 us).  The two are separate instances of the whole body so that the clearing does not sit inside the fast
// path's loops.
template <int DT, int NK, int QT, int ST, bool VEC, bool LSE>
__device__ __forceinline__ void attention_body(const RunArgs &a, const void *Vbuf, float *lse_rows, const SegRec &rec, int64_t h,
                                               int zblock, unsigned char *lds) {
    constexpr int KP = 32 * NK;                       // padded head dimension
    constexpr int kPitchK = KP * 2 + 32;              // bytes per LDS row of keys
    constexpr int kPieces = KP / 8;                   // 16-byte pieces per row
    constexpr int kOutTiles = KP / 16;
    constexpr int kAttRing = att_ring(QT, ST);
    const int M = rec.M, N = rec.N, K = rec.K;
    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6);
    const int lane = lane_id();
    const int j = lane & 15, rg = lane >> 4;
    const uint16_t *qs = reinterpret_cast<const uint16_t *>(a.A) + h * a.Dm1 + rec.off1;
    const uint16_t *ks = reinterpret_cast<const uint16_t *>(a.B) + h * a.Dm2 + rec.off2;
    const uint16_t *vs = reinterpret_cast<const uint16_t *>(Vbuf) + h * a.Dm2 + rec.off2;
    uint16_t *os = reinterpret_cast<uint16_t *>(a.out) + h * a.Dm1 + rec.off1;

    // A negative scale is applied as |scale| to negated scores (sign bits of the query operand flipped),
    // so that the running maximum is always the value to subtract.
    // A scale of zero (uniform probabilities) is applied as scores of zero under a scale of one: the keys past
    // the end of a segment are masked as -inf scores, which a zero factor would turn into NaN.
    const float c_signed = a.scale * kLog2e;
    const float c = c_signed == 0.f ? 1.0f : __builtin_fabsf(c_signed);
    const uint32_t flip = c_signed < 0.f ? 0x80008000u : 0u;
    const uint32_t keep = c_signed == 0.f ? 0u : 0xffffffffu;
    const u32x4 zero4 = u32x4{0u, 0u, 0u, 0u};

    // Staging: ST LDS stages.  With two, a block's pieces are written and loaded again one by one between the matrix
    // instructions of the block before (see below).
    constexpr int kStageBytes = kAttKeys * kPitchK, kValues = ST * kStageBytes;      // keys' stages, then values' stages
    // Per thread: kSteps 16-byte pieces of the key rows and of the value rows (kLpr neighbouring lanes share
    // a row; step s takes rows s * kRowsStep ..).  Element offsets inside a segment fit 32 bits (checked by the kernel).
    constexpr int kLpr = NK == 3 ? 16 : kPieces;      // lanes per row (a power of two; 12 pieces: 4 lanes idle)
    constexpr int kSteps = kLpr / 4, kRowsStep = kAttThreads / kLpr;
    const int k_row = tid / kLpr, k_piece = tid % kLpr;
    // VEC: the loads go through buffer descriptors that span exactly the segment's keys and values, so a row
    // past the last key reads as zeros with no code; a piece past the head dimension has an offset that is
    // out of range and stays there (its advance is multiplied by zero).
    const __amdgpu_buffer_rsrc_t resK = __builtin_amdgcn_make_buffer_rsrc((void *)ks, 0, VEC ? N * K * 2 : 0, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t resV = __builtin_amdgcn_make_buffer_rsrc((void *)vs, 0, VEC ? N * K * 2 : 0, kRsrcFlags);
    // Other rows: 16-byte pieces at any alignment, cleared past the row's end on the way into LDS.
    const RowPieces<false> pq(qs, M, K), pk(ks, N, K), pv(vs, N, K);
    const uint32_t row_bytes = 2u * (uint32_t)K;      // all advances below are under 2^24 (K <= 128)
    const uint32_t k_live = 8 * k_piece < K ? 1u : 0u;
    const uint32_t k_byte0 = k_live ? (uint32_t)k_row * row_bytes + 16u * (uint32_t)k_piece : kNowhere;

    // operand reads: lane (j, rg) reads 16 bytes of key row 16 t + j at k = 32 s + 8 rg; of the values it addresses four
    // columns of key 4 rg + j / 4 and receives column j of the lane group's four keys
    const uint32_t k_addr = lds_offset(lds) + (uint32_t)(j * kPitchK + rg * 16);
    const uint32_t v_addr = lds_offset(lds) + (uint32_t)(kValues + (4 * rg + (j >> 2)) * kPitchK + (j & 3) * 8);

    constexpr int kRoundRows = kAttRows * QT;           // queries per workgroup round
    for (int round = zblock; (int64_t)round * kRoundRows < M; round += a.ride_slots ? (1 << 24) : a.tile_zdim) {
        // strip q of the wavefront: rows round * kRoundRows + 64 q + 16 wave ..; the live ones come first
        const int r0 = round * kRoundRows + wave * 16;
        const int nq = uniform(r0 >= M ? 0 : min(QT, (M - r0 + kAttRows - 1) / kAttRows));   // 0: the wavefront only stages
        // the wavefront's queries as B operand: lane (query j, rg) holds k = 32 s + 8 rg .. + 7
        u32x4 qf[QT][NK];
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const uint16_t *qrow = qs + (int64_t)min(r0 + kAttRows * q + j, M - 1) * K;
            if constexpr (VEC) {
#pragma unroll
                for (int s = 0; s < NK; ++s)
                    qf[q][s] = *reinterpret_cast<const u32x4_unaligned *>(qrow + min(32 * s + 8 * rg, K - 8));
            } else {
#pragma unroll
                for (int s = 0; s < NK; ++s) qf[q][s] = pq.get(min(r0 + kAttRows * q + j, M - 1), 4 * s + rg);
            }
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                qf[q][s] = 32 * s + 8 * rg < K ? qf[q][s] : zero4;
                qf[q][s] = u32x4{(qf[q][s][0] ^ flip) & keep, (qf[q][s][1] ^ flip) & keep, (qf[q][s][2] ^ flip) & keep,
                                 (qf[q][s][3] ^ flip) & keep};
            }
        }
        // The loads run ahead of the arithmetic and land in registers while it runs.  One stage: the loads of block kb + 64
        // (kw, vw: this thread's pieces of the key and value rows) are issued before the matrix work on block kb; they sit
        // in one branch-free sequence (index clamped, value selected afterwards): loads behind a branch wait one by one.
        // Two stages: one barrier a block, and the pieces take turns in one set of registers (kw).  Between the score
        // products of block kb the value pieces of block kb + 64 go to the other stage and its key pieces are requested;
        // between the value products these go there and the value pieces of block kb + 128 are requested.
        u32x4 kw[kSteps], vw[ST == 1 ? kSteps : 1];
        uint32_t k_byte = k_byte0;                     // of the block that is loaded next
        auto offset = [&](auto step_tag, int kb) {
            constexpr int step = decltype(step_tag)::value;
            if constexpr (VEC) return mad24(k_live, (uint32_t)(step * kRowsStep) * row_bytes, k_byte);
            else return pk.offset(kb + step * kRowsStep + k_row, k_piece);
        };
        auto load_k = [&](uint32_t off) { return VEC ? __builtin_amdgcn_raw_buffer_load_b128(resK, off, 0, 0) : pk.load(off); };
        auto load_v = [&](uint32_t off) { return VEC ? __builtin_amdgcn_raw_buffer_load_b128(resV, off, 0, 0) : pv.load(off); };
        auto advance = [&]() { k_byte = mad24(k_live, (uint32_t)kAttKeys * row_bytes, k_byte); };
        // what the loads of block kb brought -> pieces with zeros past the head dimension and past the last key
        // (values: their probabilities are zeros too, but 0 * stale bits could be NaN)
        auto finish = [&](auto step_tag, int kb, u32x4 x) {
            if constexpr (VEC) return x;
            else return pk.finish(x, pk.offset(kb + decltype(step_tag)::value * kRowsStep + k_row, k_piece), k_piece);
        };
        const bool puts = kLpr == kPieces || k_piece < kPieces;
        unsigned char *const put_at = lds + k_row * kPitchK + k_piece * 16;
        auto put = [&](auto step_tag, int array, u32x4 x) {
            if (puts) *reinterpret_cast<u32x4 *>(put_at + array + decltype(step_tag)::value * (kRowsStep * kPitchK)) = x;
        };
        int stage = 0;
        if constexpr (ST == 2) {
            if (round != zblock) att_lds_barrier();    // the previous round is consumed
            if (N > 0) {
                u32x4 first[kSteps];
                static_for<kSteps>([&](auto sc) {
                    const uint32_t off = offset(sc, 0);
                    kw[decltype(sc)::value] = load_k(off);
                    first[decltype(sc)::value] = load_v(off);
                });
                advance();
                static_for<kSteps>([&](auto sc) {
                    constexpr int step = decltype(sc)::value;
                    put(sc, 0, finish(sc, 0, kw[step]));
                    put(sc, kValues, finish(sc, 0, first[step]));
                    kw[step] = load_v(offset(sc, kAttKeys));
                });
            }
            att_lds_barrier();
        } else if (N > 0) {
            static_for<kSteps>([&](auto sc) {
                const uint32_t off = offset(sc, 0);
                kw[decltype(sc)::value] = load_k(off);
                vw[decltype(sc)::value] = load_v(off);
            });
            advance();
        }

        int kb = 0;
        // (past the last block: a stage that nobody reads, rows that do not exist)
        auto exchange_v = [&](auto sc) {
            constexpr int step = decltype(sc)::value;
            put(sc, kStageBytes - stage + kValues, finish(sc, kb + kAttKeys, kw[step]));
            kw[step] = load_k(offset(sc, kb + kAttKeys));
            __builtin_amdgcn_sched_barrier(0);
        };
        auto exchange_k = [&](auto sc) {
            constexpr int step = decltype(sc)::value;
            put(sc, kStageBytes - stage, finish(sc, kb + kAttKeys, kw[step]));
            kw[step] = load_v(offset(sc, kb + 2 * kAttKeys));
            __builtin_amdgcn_sched_barrier(0);
        };
        // All blocks and the results of a wavefront with S strips.  Two stages: a wavefront of one strip has a walk of its own
        // from its accumulators to its results (as a choice inside the loop the accumulators would be copied where the two
        // meet); computing the missing strip along instead cost 5 % on 100 x 8 segments of 320 rows and 500 keys.
        auto walk = [&](auto s_tag) {
            constexpr int S = decltype(s_tag)::value;
            float m[S], lsum[S];
            f32x4 oacc[S][kOutTiles];
#pragma unroll
            for (int q = 0; q < S; ++q) {
                m[q] = -INFINITY; lsum[q] = 0.f;
#pragma unroll
                for (int t = 0; t < kOutTiles; ++t) oacc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            for (; kb < N; kb += kAttKeys) {
                if constexpr (ST == 1) {
                    static_for<kSteps>([&](auto sc) {
                        constexpr int step = decltype(sc)::value;
                        kw[step] = finish(sc, kb, kw[step]);
                        vw[step] = finish(sc, kb, vw[step]);
                    });
                    __syncthreads();                       // the previous block (or round) is consumed
                    // ---- one 16-byte piece per thread, array and step, pieces of a row on neighbouring lanes
                    static_for<kSteps>([&](auto sc) {
                        put(sc, 0, kw[decltype(sc)::value]);
                        put(sc, kValues, vw[decltype(sc)::value]);
                    });
                    __syncthreads();
                    if (kb + kAttKeys < N) {
                        static_for<kSteps>([&](auto sc) {
                            const uint32_t off = offset(sc, kb + kAttKeys);
                            kw[decltype(sc)::value] = load_k(off);
                            vw[decltype(sc)::value] = load_v(off);
                        });
                        advance();
                    }
                    if (nq == 0) continue;
                }
                // The arithmetic on one block for NQ live strips, as straight-line code: a branch around every
                // matrix instruction of a strip that may be missing would keep the scheduler from interleaving them.
                auto block_math = [&](auto nq_tag) {
                    constexpr int NQ = decltype(nq_tag)::value;
                    // ---- scores of 64 keys x 16 queries per strip; a key operand read serves every strip
                    f32x4 sacc[NQ][4];
        #pragma unroll
                    for (int q = 0; q < NQ; ++q)
        #pragma unroll
                        for (int t = 0; t < 4; ++t) sacc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                    u32x4 ring[kAttRing];
                    const uint32_t k_at = k_addr + (ST == 2 ? stage : 0), v_at = v_addr + (ST == 2 ? stage : 0);
                    {
                        constexpr int kReads = 4 * NK;         // read i: k step i / 4, key tile i % 4
                        static_for<kAttRing>([&](auto ic) {
                            constexpr int I = decltype(ic)::value;
                            if constexpr (I < kReads) lds_read128<16 * (I % 4) * kPitchK + 64 * (I / 4)>(ring[I], k_at);
                        });
                        static_for<kReads>([&](auto ic) {
                            constexpr int I = decltype(ic)::value, R = I % kAttRing;
                            constexpr int kBehind = (I + kAttRing < kReads ? I + kAttRing : kReads) - (I + 1);
                            lds_wait<kBehind>(ring[R]);
        #pragma unroll
                            for (int q = 0; q < NQ; ++q) sacc[q][I % 4] = Elem<DT>::mfma(ring[R], qf[q][I / 4], sacc[q][I % 4]);
                            if constexpr (ST == 2) __builtin_amdgcn_sched_barrier(0);
                            if constexpr (I + kAttRing < kReads)
                                lds_read128<16 * ((I + kAttRing) % 4) * kPitchK + 64 * ((I + kAttRing) / 4)>(ring[R], k_at);
                            constexpr int kEvery = kReads / kSteps;
                            static_assert(kEvery * kSteps == kReads);
                            if constexpr (ST == 2 && I % kEvery == kEvery - 1) exchange_v(std::integral_constant<int, I / kEvery>{});
                        });
                    }
                    constexpr int kValueReads = 2 * kOutTiles; // read i: key half i / kOutTiles, output tile i % kOutTiles
                    u32x2 lo[kAttRing], hi[kAttRing];          // keys 4 rg .. + 3 of the half's two key tiles
                    auto values_ahead = [&]() {
                        static_for<kAttRing>([&](auto ic) {
                            constexpr int I = decltype(ic)::value;
                            if constexpr (I < kValueReads)
                                lds_read_tr<32 * (I / kOutTiles) * kPitchK + 32 * (I % kOutTiles), 16 * kPitchK>(lo[I], hi[I], v_at);
                        });
                    };
                    if constexpr (ST == 2) {
                        advance();
                        values_ahead();                        // in flight under the softmax
                    }
                    // ---- online softmax; lane holds keys kb + 16 t + 4 rg + e of query j of each strip
                    const int left = N - kb;                   // keys of this block that exist
                    u32x4 pf[NQ][2];
        #pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        f32x4(&sc)[4] = sacc[q];
                        // keys past the segment's last: -inf, so that they neither raise the maximum nor count
                        // (their exponentials are zeros)
                        if (left < kAttKeys) {
                            const int mine = left - 4 * rg;    // (compared with constants: no registers for 16 key numbers)
        #pragma unroll
                            for (int t = 0; t < 4; ++t)
        #pragma unroll
                                for (int e = 0; e < 4; ++e) sc[t][e] = 16 * t + e < mine ? sc[t][e] : -INFINITY;
                        }
                        settle_mfma(sc);                       // max3 reads the scores from inline assembly
                        float bm;                              // one statement: no padding between its instructions
                        asm volatile("v_max3_f32 %0, %1, %2, %3\n\tv_max3_f32 %0, %0, %4, %5\n\tv_max3_f32 %0, %0, %6, %7\n\t"
                                     "v_max3_f32 %0, %0, %8, %9\n\tv_max3_f32 %0, %0, %10, %11\n\tv_max3_f32 %0, %0, %12, %13\n\t"
                                     "v_max3_f32 %0, %0, %14, %15\n\tv_max_f32 %0, %0, %16"
                                     : "=&v"(bm)
                                     : "v"(sc[0][0]), "v"(sc[0][1]), "v"(sc[0][2]), "v"(sc[0][3]), "v"(sc[1][0]), "v"(sc[1][1]),
                                       "v"(sc[1][2]), "v"(sc[1][3]), "v"(sc[2][0]), "v"(sc[2][1]), "v"(sc[2][2]), "v"(sc[2][3]),
                                       "v"(sc[3][0]), "v"(sc[3][1]), "v"(sc[3][2]), "v"(sc[3][3]));
                        bm = quad_column_max_swap(bm);
                        // m is the reference the exponentials are taken against, not necessarily the maximum: it is
                        // raised (and the sums so far rescaled) only when a block's maximum passes it by more than
                        // 2^8 in the exponent, so probabilities stay below 256 (fine for both 16-bit types and the
                        // fp32 sums) and most blocks skip the rescale.  The comparison is false, i.e. raises, for the
                        // first block (m = -inf).
                        const bool raise = !((bm - m[q]) * c <= 8.0f);
                        const float m_new = raise ? bm : m[q];
                        const float m_use = m_new == -INFINITY ? 0.f : m_new;
                        const float alpha = !raise ? 1.0f : m[q] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m[q] - m_use) * c);
                        m[q] = m_new;
                        const float bias = -m_use * c;
                        float psum = 0.f;
        #pragma unroll
                        for (int t = 0; t < 4; ++t)
        #pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float p = __builtin_amdgcn_exp2f(fmaf(sc[t][e], c, bias));
                                sc[t][e] = p;
                                psum += p;
                            }
                        lsum[q] = fmaf(lsum[q], alpha, psum);
                        if (__any(raise)) {
                            // (the matrix instructions that wrote the accumulators are a whole score product away)
        #pragma unroll
                            for (int t = 0; t < kOutTiles; ++t) {
                                if constexpr (ST == 2) scale_in_place(oacc[q][t], alpha);
                                else oacc[q][t] *= alpha;
                            }
                        }
                        // probabilities as B operand, 32 keys per step: k = 8 rg + kk is key 32 cc + 4 rg + kk (kk < 4)
                        // or 32 cc + 16 + 4 rg + kk - 4: what the lane holds in sc[2 cc] and sc[2 cc + 1]
        #pragma unroll
                        for (int cc = 0; cc < 2; ++cc)
                            pf[q][cc] = u32x4{Elem<DT>::pack2(sc[2 * cc][0], sc[2 * cc][1]), Elem<DT>::pack2(sc[2 * cc][2], sc[2 * cc][3]),
                                              Elem<DT>::pack2(sc[2 * cc + 1][0], sc[2 * cc + 1][1]),
                                              Elem<DT>::pack2(sc[2 * cc + 1][2], sc[2 * cc + 1][3])};
                    }
                    // ---- O^T += V^T P^T; a value operand read serves every strip
                    {
                        if constexpr (ST == 1) values_ahead();
                        static_for<kValueReads>([&](auto ic) {
                            constexpr int I = decltype(ic)::value, R = I % kAttRing, J = I + kAttRing;
                            lds_wait_tr<2 * ((J < kValueReads ? J : kValueReads) - (I + 1))>(lo[R], hi[R]);
                            const u32x4 v = u32x4{lo[R][0], lo[R][1], hi[R][0], hi[R][1]};
        #pragma unroll
                            for (int q = 0; q < NQ; ++q)
                                oacc[q][I % kOutTiles] = Elem<DT>::mfma(v, pf[q][I / kOutTiles], oacc[q][I % kOutTiles]);
                            if constexpr (ST == 2) __builtin_amdgcn_sched_barrier(0);
                            if constexpr (J < kValueReads)
                                lds_read_tr<32 * (J / kOutTiles) * kPitchK + 32 * (J % kOutTiles), 16 * kPitchK>(lo[R], hi[R], v_at);
                            constexpr int kEvery = kValueReads / kSteps;
                            static_assert(kEvery * kSteps == kValueReads);
                            if constexpr (ST == 2 && I % kEvery == kEvery - 1) exchange_k(std::integral_constant<int, I / kEvery>{});
                        });
                    }
                };
                if (ST == 1 && QT == 2 && nq == 1) block_math(std::integral_constant<int, 1>{});
                else block_math(std::integral_constant<int, S>{});
                if constexpr (ST == 2) {
                    stage = kStageBytes - stage;
                    att_lds_barrier();
                }
            }
            // ---- normalise and store: lane (query j, rg) holds columns 16 t + 4 rg + e.  No key at all: zeros.
            // (column numbers made here: taken out of the loop over the rounds they would hold registers through the blocks)
            int own = 4 * rg;
            if constexpr (ST == 2) asm volatile("" : "+v"(own));
#pragma unroll
            for (int q = 0; q < S; ++q) {
                if (q >= nq) continue;
                const int qr = r0 + kAttRows * q + j;
                const float l = quad_column_sum(lsum[q]);
                const float inv = N > 0 ? 1.0f / l : 0.f;
                // base-2 logarithm of the row's sum of exponentials, for the backward pass
                if (LSE && rg == 0 && qr < M && N > 0) lse_rows[qr] = fmaf(m[q], c, __builtin_amdgcn_logf(l));
                if (qr < M) {
                    uint16_t *orow = os + (int64_t)qr * K;
#pragma unroll
                    for (int t = 0; t < kOutTiles; ++t) {
                        const int c0 = 16 * t + own;
                        if (c0 + 4 <= K) {
                            *reinterpret_cast<u32x2_unaligned *>(orow + c0) =
                                u32x2{Elem<DT>::pack2(oacc[q][t][0] * inv, oacc[q][t][1] * inv),
                                      Elem<DT>::pack2(oacc[q][t][2] * inv, oacc[q][t][3] * inv)};
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (c0 + e < K) orow[c0 + e] = Elem<DT>::from_float(oacc[q][t][e] * inv);
                        }
                    }
                }
            }
        };
        if (ST == 1 || nq == QT) walk(std::integral_constant<int, QT>{});
        else if (nq == 1) walk(std::integral_constant<int, 1>{});
        else {                                         // the wavefront only stages
            for (; kb < N; kb += kAttKeys) {
                static_for<kSteps>(exchange_v);
                advance();
                static_for<kSteps>(exchange_k);
                stage = kStageBytes - stage;
                att_lds_barrier();
            }
        }
    }
}

// LSE: the build for training, which also writes the rows' sums (as a run-time choice it cost the plain one 2 % on 512
// segments of 16 .. 256 rows and columns: 23.1 -> 23.6 us).
template <int DT, int NK, int QT, int ST, bool LSE>
__global__ __launch_bounds__(kAttThreads, QT == 2 ? 2 : NK <= 2 ? 4 : 3) void attention_kernel(RunArgs a, const void *Vbuf, float *lse, int min_K) {
    constexpr int KP = 32 * NK;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * ST * kAttKeys * (KP * 2 + 32)];
    // (the row blocks per head come with the header: one memory round trip less than the prefix's last entry)
    const int64_t per_head = QT == 2 ? ((ConstHdr)(uintptr_t)a.plan)->att_blocks128 : ((ConstHdr)(uintptr_t)a.plan)->att_blocks64;
    // (lse is sized by the min_K of the host's summary)
    if (!header_ok(a) || (LSE && ((ConstHdr)(uintptr_t)a.plan)->min_K != min_K)) { report_mismatch(a); return; }
    // Workgroup -> (segment, head, row block).  Consecutive workgroup ids go to the eight dies of the chip in
    // turn, and each die has its own L2: id = die + 8 k.  All row blocks of one (segment, head) pair read the
    // same keys and values, so they should run on ONE die at about the same time.
    // With the row-block prefix (ride_slots = 1, launches that know the batch's totals): the existing
    // (head, segment, row block) items, head-major, are cut into eight contiguous shares, one per die, so the
    // row blocks of a pair sit side by side on one die and no workgroup is launched for a row block that does
    // not exist, except past the end of a share (the grid is sized from an upper bound of the item count).
    // Without it: pair = die + 8 (k mod pairs per die), row block k / pairs per die; a workgroup takes every
    // tile_zdim-th row block of its pair, and the workgroups that find no rows come last.
    const unsigned id = flat_block(), die = id & 7u, kk = id >> 3;
    int g, zblock;
    int64_t h;
    if (a.ride_slots) {
        const int32_t *pfx = plan_rowblocks(a.plan, a.nseg, QT - 1);
        const int64_t items = per_head * a.H, share = (items + 7) >> 3;
        const int64_t u = (int64_t)die * share + kk;
        // a grid too small for the plan's items: the host summary the launch was sized from is not this plan's
        if (id == 0 && threadIdx.x == 0 && share * 8 > flat_blocks())
            atomicAdd(&reinterpret_cast<PlanHeader *>(a.plan)->run_errors, 1);
        if (kk >= share || u >= items) return;
        h = u / per_head;
        const int item = (int)(u % per_head);
        g = prefix_search(pfx, a.nseg, item);
        zblock = item - ((ConstI32)(uintptr_t)pfx)[g];
    } else {
        const unsigned pairs8 = (unsigned)a.tile_groups;
        const int64_t pair = (int64_t)die + 8 * (int64_t)(kk % pairs8);
        zblock = (int)(kk / pairs8);
        if (zblock >= a.tile_zdim) return;             // (the last row of a flat grid)
        if (pair >= (int64_t)a.nseg * a.H) return;
        g = (int)(pair / a.H);
        h = pair % a.H;
    }
    const PlanRO pv = plan_ro(a.plan, a.nseg);
    const SegRec rec = load_rec(pv.recs, g);
    const int M = rec.M, K = rec.K;
    if (M < 1 || K < 1) return;
    // the launch was sized for a smaller head dimension, or byte offsets inside the segment (of a last block of
    // keys that reaches past the segment's end, too) pass 32 bits
    if (K > KP || !att_offsets_fit(max(M, rec.N), K)) {
        if (h == 0 && zblock == 0 && threadIdx.x == 0)
            atomicAdd(&reinterpret_cast<PlanHeader *>(a.plan)->run_errors, 1);
        return;
    }
    float *lse_rows = LSE ? lse + att_row_base(min_K, a.Dm1, h, rec.off1) : nullptr;
    if ((K & 7) == 0) attention_body<DT, NK, QT, ST, true, LSE>(a, Vbuf, lse_rows, rec, h, zblock, lds);
    else attention_body<DT, NK, QT, ST, false, LSE>(a, Vbuf, lse_rows, rec, h, zblock, lds);
}

template <int DT, int QT, int ST, bool LSE>
static void launch_nk(int nk, dim3 grid, hipStream_t stream, const RunArgs &args, const void *V, float *lse, int min_K) {
    // args.ride_slots = 1: work items from the plan's row-block prefix; else args.tile_zdim = row blocks per
    // (segment, head) pair, tile_groups = pairs per die
    switch (nk) {                                      // (two stages: never with nk = 1)
        case 1: hipLaunchKernelGGL((attention_kernel<DT, 1, QT, 1, LSE>), grid, dim3(kAttThreads), 0, stream, args, V, lse, min_K); break;
        case 2: hipLaunchKernelGGL((attention_kernel<DT, 2, QT, ST, LSE>), grid, dim3(kAttThreads), 0, stream, args, V, lse, min_K); break;
        case 3: hipLaunchKernelGGL((attention_kernel<DT, 3, QT, ST, LSE>), grid, dim3(kAttThreads), 0, stream, args, V, lse, min_K); break;
        default: hipLaunchKernelGGL((attention_kernel<DT, 4, QT, ST, LSE>), grid, dim3(kAttThreads), 0, stream, args, V, lse, min_K); break;
    }
}
template <int DT, int QT, int ST>
static void launch_build(int nk, dim3 grid, hipStream_t stream, const RunArgs &args, const void *V, float *lse, int min_K) {
    if (lse) launch_nk<DT, QT, ST, true>(nk, grid, stream, args, V, lse, min_K);
    else launch_nk<DT, QT, ST, false>(nk, grid, stream, args, V, lse, min_K);
}

// Strips per wavefront: two where segments are tall (each operand read from LDS then feeds two matrix
// instructions and a block of keys is staged half as often), one otherwise (more, lighter workgroups).

int launch_attention(int dtype, const RunArgs &args, const void *V, float *lse, int64_t nseg, const ba_plan_info *info,
                     hipStream_t stream) {
    if (dtype != BA_F16 && dtype != BA_BF16) return BA_ERR_UNSUPPORTED;
    static const int forced = [] { const char *e = getenv("BLOCKEDATTN_ATT_STRIPS"); return e ? atoi(e) : 0; }();
    int nk = 4, qt = 1;
    int64_t max_m = 512;
    if (info) {
        if (info->max_K > 128) return BA_ERR_UNSUPPORTED;
        nseg = info->nseg;
        nk = std::max(1, (info->max_K + 31) / 32);
        max_m = std::max<int64_t>(info->max_M, 1);
        if (info->total_rows >= 256 * std::max<int64_t>(nseg, 1)) qt = 2;   // mean segment height >= 256 (136: one strip is 6 % faster)
    }
    if (forced == 1 || forced == 2) qt = forced;
    // LDS stages for two strips.  Two keep the matrix unit busier in the steady state, but the first block waits for its
    // successor's values.  Keys per query (the mean over the queries) from which they are faster, us, one stage and two:
    // - 400 (48 x 8 segments of 600 .. 900 rows, K = 64 / 128: 128 keys 35.4 / 53.1, 36.3 / 55.9; 300 keys 56.1 / 83.7, 56.1 /
    //   81.5; 400 keys 69.0 / 103.6, 68.2 / 99.2; 800 keys 109 / 171, 106 / 165);
    // - 800 for rows at any alignment up to K = 96, where one stage leaves registers for six reads in flight and clears its
    //   pieces in one place (K = 61 / 70 / 95: 64 x 8 of 300 .. 500 71 / 93 / 102, 73 / 97 / 107; 16 x 4 of 1000 .. 2000 111 / 148 /
    //   159, 110 / 152 / 157; above, K = 101: 110 and 175, 109 and 159);
    // - K <= 32: never, too few matrix instructions to hide an exchange behind (1000 .. 2000 rows: 117, 121).
    const int64_t deep_keys = info && nk < 4 && ((info->min_K | info->max_K) & 7) ? 800 : 400;
    const bool deep = qt == 2 && nk > 1 && info && info->Dout / deep_keys >= info->total_rows;
    // Row blocks per pair: enough for the tallest segment, but no more than four times what the mean segment
    // needs (a workgroup takes every Z-th block of its pair; blocks that do not exist cost a launch each).
    const int64_t round_rows = kAttRows * qt;
    int64_t z = std::min<int64_t>((max_m + round_rows - 1) / round_rows, 64);
    if (info) z = std::min<int64_t>(z, (4 * info->total_rows / std::max<int64_t>(nseg, 1) + round_rows - 1) / round_rows);
    z = std::max<int64_t>(z, 1);
    if (nseg <= 0) return BA_OK;
    const int min_K = info ? info->min_K : 0;
    RunArgs run = args;
    dim3 grid;
    if (info && info->total_rows >= 0) {
        // the batch's totals are known: one workgroup per existing row block, found through the plan's
        // row-block prefix (segments without keys count: their output rows are zeroed)
        const int64_t items = (int64_t)(qt == 2 ? info->att_blocks128 : info->att_blocks64) * args.H;
        if (items <= 0) return BA_OK;
        const int64_t share = (items + 7) / 8;
        if (share * 8 > 0x7fffffff) return BA_ERR_UNSUPPORTED;
        run.ride_slots = 1;
        grid = flat_grid(share * 8);
    } else {
        const int64_t pairs8 = (nseg * args.H + 7) / 8;    // pairs per die, rounded up
        if (pairs8 * z * 8 > 0x7fffffff || pairs8 > 0x7fffffff) return BA_ERR_UNSUPPORTED;
        run.tile_zdim = (int)z;
        run.tile_groups = (int)pairs8;
        grid = flat_grid(pairs8 * z * 8);
    }
    auto build = [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (qt == 1) launch_build<DT, 1, 1>(nk, grid, stream, run, V, lse, min_K);
        else if (deep) launch_build<DT, 2, 2>(nk, grid, stream, run, V, lse, min_K);
        else launch_build<DT, 2, 1>(nk, grid, stream, run, V, lse, min_K);
    };
    if (dtype == BA_F16) build(std::integral_constant<int, 0>{});
    else build(std::integral_constant<int, 1>{});
    return hipGetLastError() == hipSuccess ? BA_OK : BA_ERR_LAUNCH;
}

}  // namespace ba
