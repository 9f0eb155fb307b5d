// Fused GEMM + softmax rows for segments whose operand rows are not 16-byte aligned (K not a multiple of 8, odd segment
// starts, unaligned base pointers): any M, N and K on the matrix instructions.  Runs inside segment_kernel and
// onecall_kernel, which had an element-wise loop (one multiply-add per element, every row swept twice) for them.
//
// A workgroup takes 64 rows, a wavefront 16 of them against a panel of up to 16 * MAXNT columns in registers; k goes by
// in chunks of 64: the panel's rows of B through LDS (read as 16-byte pieces at any alignment, zeros past K), the
// wavefront's A rows straight to registers, the next chunk's loads in flight under the matrix instructions.  Up to
// 16 * MAXNT columns a row is done in one sweep; wider ones sum in a first sweep over the panels and write in a second,
// which recomputes the scores.
//
// 256 x 8 pairs of 32 .. 128 rows and columns, K = 61: 4136 -> 36 us (K = 64 on the aligned path: 14.6); 128 x 4 pairs of
// 64 .. 256, K = 101: 8667 -> 52 us; one launch (measured inlined there), 128 x 4 pairs of 32 .. 128, K = 61: 1416 -> 20 us.  The loop was bound by
// 2-byte loads, one per multiply-add.  Now it is the life of a workgroup: load, barrier, matrix instructions, softmax,
// stores one after the other, three or two workgroups to a compute unit by registers.  (128 and 168 registers, one
// workgroup more, spill: 49 and 63 us.)
#pragma once
#include "row_pieces.hpp"

namespace ba {

constexpr int kAnyK = 64;                              // k per chunk
constexpr int kAnyPitch = 2 * kAnyK + 32;              // 16 * (2 * odd): the operand reads of 16 rows meet no conflict
constexpr int any_rows_lds(int tiles) { return 16 * tiles * kAnyPitch; }

template <int DT, bool F32OUT, int MAXNT>
__device__ __forceinline__ void any_rows(const Seg &s, const RunArgs &a, unsigned char *lds, int r0) {
    constexpr int kRowsStep = kSegThreads / 8;         // eight pieces a row
    constexpr int kSteps = 16 * MAXNT / kRowsStep;
    const int M = s.M, N = s.N, K = s.K;
    const int tid = threadIdx.x, lane = lane_id(), j = lane & 15, rg = lane >> 4;
    const int s_row = tid >> 3, s_piece = tid & 7;
    const RowPieces<false> pa((const uint16_t *)a.A + s.a, M, K), pb((const uint16_t *)a.B + s.b, N, K);
    const bool active = r0 < M;
    f32x4 acc[kMaxTiles];

    // scores of the wavefront's rows against columns c0 .. c0 + 16 nt - 1
    auto panel = [&](int c0, int nt) {
        u32x4 bw[kSteps], aw[2];
        auto b_off = [&](int i, int k0) {
            const int row = c0 + i * kRowsStep + s_row;
            return row < N ? pb.offset(row, (k0 >> 3) + s_piece) : kNowhere;
        };
        auto a_off = [&](int i, int k0) { return r0 + j < M ? pa.offset(r0 + j, (k0 >> 3) + 4 * i + rg) : kNowhere; };
        auto fetch = [&](int k0) {
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
                if (i * kRowsStep < 16 * nt) bw[i] = pb.load(b_off(i, k0));
#pragma unroll
            for (int i = 0; i < 2; ++i) aw[i] = pa.load(a_off(i, k0));
        };
#pragma unroll
        for (int t = 0; t < MAXNT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (K > 0) fetch(0);
        for (int k0 = 0; k0 < K; k0 += kAnyK) {
            __syncthreads();                           // the previous chunk (or panel) is consumed
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
                if (i * kRowsStep < 16 * nt)
                    *reinterpret_cast<u32x4 *>(lds + (i * kRowsStep + s_row) * kAnyPitch + 16 * s_piece) =
                        pb.finish(bw[i], b_off(i, k0), (k0 >> 3) + s_piece);
            u32x4 af[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) af[i] = pa.finish(aw[i], a_off(i, k0), (k0 >> 3) + 4 * i + rg);
            __syncthreads();
            if (k0 + kAnyK < K) fetch(k0 + kAnyK);
            if (!active) continue;
#pragma unroll
            for (int t = 0; t < MAXNT; ++t) {
                if (t < nt) {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        acc[t] = Elem<DT>::mfma(*reinterpret_cast<const u32x4 *>(lds + (16 * t + j) * kAnyPitch + 64 * i + 16 * rg),
                                                af[i], acc[t]);
                }
            }
        }
    };
    constexpr int kPanel = 16 * MAXNT;
    const bool once = N <= kPanel;
    float row_m = -INFINITY, row_l = 0.f;
    for (int sweep = once ? 1 : 0; sweep < 2; ++sweep) {
        for (int c0 = 0; c0 < N; c0 += kPanel) {
            const int nt = min(MAXNT, (N - c0 + 15) >> 4);
            panel(c0, nt);
            if (!active) continue;
            float c = a.scale * kLog2e;
            prepare_scores<MAXNT>(acc, nt, N, c0, c);
            if (once || sweep == 0) {
                float m, l;
                local_softmax<MAXNT>(acc, nt, c, m, l);
                const float top = fmaxf(row_m, m);
                row_l = once ? l : top == -INFINITY ? 0.f
                      : row_l * __builtin_amdgcn_exp2f((row_m - top) * c) + l * __builtin_amdgcn_exp2f((m - top) * c);
                row_m = top;
            } else {
                const float bias = -(row_m == -INFINITY ? 0.f : row_m) * c;
#pragma unroll
                for (int t = 0; t < MAXNT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[t][e] = __builtin_amdgcn_exp2f(fmaf(acc[t][e], c, bias));
            }
            if (sweep == 1) store_rows<DT, MAXNT, F32OUT>(acc, nt, s, a.out, r0, c0, 1.f / row_l);
        }
    }
}

}  // namespace ba
