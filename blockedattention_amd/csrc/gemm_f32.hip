// fp32 varlen GEMM in any layout on v_mfma_f32_16x16x4_f32 (products and sums in fp32; reference: the float instance of
// its generic kernel, csrc/cuda/spBlkGEMM.cu:120-271).
//
// Workgroup = 64 rows of one segment and head (four wavefronts of 16) against its columns, up to 128 at a time, k in
// chunks of 64.  The matrix instruction takes one k per lane group (q = lane / 16); since the order of a sum is free,
// group q takes k = 16 b + 4 q + s in step s of block b, so that four steps of one operand are ONE 16-byte read.  A rows
// that are stored along k go straight from memory to registers (64 contiguous bytes of a row per instruction); B goes
// through LDS as [column][k].  An operand stored k-major is read four k lines x four columns per thread and leaves as
// four 16-byte LDS writes: the transposition is a renaming of registers.
// Lane j owns G consecutive columns of a block (tile t = column G j + t, G = the 16-column tiles the block needs, one
// build each), so that four neighbouring rows leave whole, side by side: with blocks of 64 columns the same stores wrote
// 1.7 times the result (rows of 33 .. 128 words at any phase, a line in two pieces at two times), now 1.05 times.
//
// What bounds it, on 256 segments x 8 heads of 32 .. 128 rows and columns, K = 64 (145 MB, 2 GFLOP): memory, 28 us with
// the matrix instructions left out, and the matrix unit (padded to tiles: 17 us), which hardly overlap, because four
// workgroups a compute unit live through the same phases: 42 us, against 67 us of the kernel for all types before
// (one k at a time through LDS, 64 x 64 steps).  Rounds of 128 rows 46 us, five workgroups a compute unit (spills) 47 us.
#include <algorithm>
#include <type_traits>

#include "ba_gemm_common.hpp"

namespace ba {

constexpr int kF32Threads = 256;
constexpr int kF32Rows = 16 * (kF32Threads / 64);    // rows of a round
constexpr int kF32Tile = 64;                         // k of a chunk
constexpr int kF32Cols = 128;                        // columns of a step
constexpr int kF32Pitch = kF32Tile * 4 + 32;         // bytes of an LDS row: 16 * (2 * odd), reads of 16 rows meet no conflict
static_assert(kF32Rows == kAttBlockRows, "the plan's row-block prefix counts blocks of 64 rows");

// Four consecutive words from byte `off` of a line on, through a descriptor that spans the segment; kNowhere, for pieces
// that do not exist, reads as zeros.  EDGE: the piece may reach past the segment's end; the load is then moved back to its
// last 16 bytes and shifted by finish().  A segment of fewer than four elements is read word by word (the compiler may
// merge the four reads), the words past its end as zeros: offsets past it are held at 16, so that none of the four wraps.
template <bool EDGE> struct Words4 {
    // past every segment (areas are below 2^30 elements, multiples of four without EDGE); a 16-byte load at the one
    // without EDGE ends where 32-bit offsets do
    static constexpr uint32_t kNowhere = EDGE ? 0xfffffffcu : 0xfffffff0u;
    __amdgpu_buffer_rsrc_t res;
    uint32_t bytes;
    __device__ __forceinline__ Words4(const float *seg, int elements)
        : bytes((uint32_t)elements * 4u) {
        res = __builtin_amdgcn_make_buffer_rsrc((void *)seg, 0, bytes, kRsrcFlags);
    }
    __device__ __forceinline__ f32x4 load(uint32_t off) const {
        if (!EDGE || bytes >= 16)
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(res, EDGE ? min(off, bytes - 16) : off, 0, 0));
        f32x4 x;
        off = min(off, 16u);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            x[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, off + 4 * i, 0, 0));
        return x;
    }
    // `live` of the four words exist on their line (any value)
    __device__ __forceinline__ f32x4 finish(f32x4 x, uint32_t off, int live) const {
        if (EDGE) {
            if (bytes >= 16) {
                const uint32_t behind = off <= bytes - 16 ? 0u : (min(off, bytes) - (bytes - 16)) >> 2;     // 0 .. 4
                if (behind & 1) x = f32x4{x[1], x[2], x[3], 0.f};
                if (behind & 2) x = f32x4{x[2], x[3], 0.f, 0.f};
                if (behind & 4) x = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = i < live ? x[i] : 0.f;
        }
        return x;
    }
};

// A 16 G (rows or columns of the result) x 64 (k) chunk of an operand on its way into LDS as [row][k], in pieces of four
// words: kPieces a thread.  MAJOR: stored k-major (K lines of `rows`); EDGE as above.  `rows` x K operand, chunk at
// (r0, k0).  DEALT: row G j + t goes to LDS row 16 t + j.
template <bool MAJOR, bool EDGE, int G, bool DEALT> struct F32Chunk {
    // unit u = tid + kF32Threads i of a thread; along k: row u / 16, words 4 (u % 16); k-major: four lines 4 (u / 16 % 16)
    // x four columns 4 (u % 16) + 64 (u / 256)
    static constexpr int kUnits = MAJOR ? 256 * ((G + 3) / 4) : 256 * G;
    static constexpr int kPer = (kUnits + kF32Threads - 1) / kF32Threads;
    static constexpr int kPieces = MAJOR ? 4 * kPer : kPer;
    f32x4 v[kPieces];
    static __device__ __forceinline__ int unit(int tid, int i) { return tid + kF32Threads * (MAJOR ? i >> 2 : i); }
    static __device__ __forceinline__ int col(int tid, int i) { return 4 * (unit(tid, i) & 15) + 64 * (unit(tid, i) >> 8); }       // k-major
    static __device__ __forceinline__ int line(int tid, int i) {
        return MAJOR ? 4 * ((unit(tid, i) >> 4) & 15) + (i & 3) : unit(tid, i) >> 4;
    }
    static __device__ __forceinline__ int lds_row(int row) { return DEALT ? 16 * (row % G) + row / G : row; }
    static __device__ __forceinline__ uint32_t offset(int rows, int K, int r0, int k0, int tid, int i) {
        const int l = (MAJOR ? k0 : r0) + line(tid, i), pos = MAJOR ? r0 + col(tid, i) : k0 + 4 * (tid & 15);
        const int lines = MAJOR ? K : rows, len = MAJOR ? rows : K;
        return l < lines && pos < len ? 4u * (uint32_t)(l * len + pos) : Words4<EDGE>::kNowhere;
    }
    __device__ __forceinline__ void fetch(const Words4<EDGE> &src, int rows, int K, int r0, int k0, int tid) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) v[i] = src.load(offset(rows, K, r0, k0, tid, i));
    }
    __device__ __forceinline__ void put(const Words4<EDGE> &src, int rows, int K, int r0, int k0, int tid, unsigned char *dst) {
        if constexpr (EDGE) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i)
                v[i] = src.finish(v[i], offset(rows, K, r0, k0, tid, i), MAJOR ? rows - r0 - col(tid, i) : K - k0 - 4 * (tid & 15));
        }
        if constexpr (MAJOR) {
#pragma unroll
            for (int i = 0; i < kPieces; i += 4)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int row = col(tid, i) + c;
                    if (row < 16 * G)
                        *reinterpret_cast<f32x4 *>(dst + lds_row(row) * kF32Pitch + ((tid >> 4) & 15) * 16) =
                            f32x4{v[i][c], v[i + 1][c], v[i + 2][c], v[i + 3][c]};
                }
        } else {
#pragma unroll
            for (int i = 0; i < kPieces; ++i)
                if (kUnits % kF32Threads == 0 || line(tid, i) < 16 * G)
                    *reinterpret_cast<f32x4 *>(dst + lds_row(line(tid, i)) * kF32Pitch + (tid & 15) * 16) = v[i];
        }
    }
};

// One column block (G tiles of 16 columns from c0 on) of a round of 64 rows.
template <bool T1, bool T2, bool EDGE, int G>
__device__ __forceinline__ void f32_block(const Words4<EDGE || T1> &pa, const Words4<EDGE || T2> &pb, float *os, int M, int N,
                                          int K, int r0, int c0, unsigned char *lds) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));                      // keeps the staging addresses of all eight builds of this function from being computed up front
    const int wave = uniform(tid >> 6), lane = tid & 63, j = lane & 15, q = lane >> 4;
    unsigned char *sA = lds + kF32Cols * kF32Pitch;    // T1 only
    const int chunks = max(1, (K + kF32Tile - 1) / kF32Tile);
    // operand row i of a wavefront's strip is row 4 (i % 4) + i / 4: result register e of group q is row 4 e + q
    const int arow = 16 * wave + 4 * (j & 3) + (j >> 2);
    F32Chunk<T2, EDGE || T2, G, true> cb;
    F32Chunk<T1, EDGE || T1, kF32Rows / 16, false> ca;             // T1
    f32x4 av[4];                                       // !T1: four words of k = 16 b + 4 q of the lane's row
    auto aoff = [&](int k0, int b) {
        const int row = r0 + arow, k = k0 + 16 * b + 4 * q;
        return row < M && k < K ? 4u * (uint32_t)(row * K + k) : Words4<EDGE>::kNowhere;
    };
    auto fetch = [&](int k0) {
        cb.fetch(pb, N, K, c0, k0, tid);
        if constexpr (T1) ca.fetch(pa, M, K, r0, k0, tid);
        else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                av[b] = pa.load(aoff(k0, b));
            }
        }
    };
    f32x4 acc[G];
#pragma unroll
    for (int t = 0; t < G; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool alive = r0 + 16 * wave < M;
    for (int kc = 0; kc < chunks; ++kc) {
        const int k0 = kc * kF32Tile;
        fetch(k0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");       // the previous chunk is consumed
        cb.put(pb, N, K, c0, k0, tid, lds);
        f32x4 af[4];
        if constexpr (T1) ca.put(pa, M, K, r0, k0, tid, sA);
        else {
#pragma unroll
            for (int b = 0; b < 4; ++b) af[b] = pa.finish(av[b], aoff(k0, b), K - (k0 + 16 * b + 4 * q));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const auto brow = (__attribute__((address_space(3))) unsigned char *)lds + j * kF32Pitch + q * 16;      // column G j + t lies in row 16 t + j
        auto step = [&](auto b_tag) {
            constexpr int b = decltype(b_tag)::value;
            if constexpr (T1) af[b] = *reinterpret_cast<const f32x4 *>(sA + arow * kF32Pitch + q * 16 + 64 * b);
            f32x4 bf[G];
#pragma unroll
            for (int t = 0; t < G; ++t)
                bf[t] = *reinterpret_cast<__attribute__((address_space(3))) const f32x4 *>(brow + 16 * t * kF32Pitch + 64 * b);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < G; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[b][s], bf[t][s], acc[t], 0, 0, 0);
        };
        const int left = alive ? K - k0 : 0;           // (a wavefront without rows only stages)
        if (left > 0) step(std::integral_constant<int, 0>{});
        if (left > 16) step(std::integral_constant<int, 1>{});
        if (left > 32) step(std::integral_constant<int, 2>{});
        if (left > 48) step(std::integral_constant<int, 3>{});
    }
    if (!alive) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = r0 + 16 * wave + 4 * e + q, col = c0 + G * j;
        if (row >= M) continue;
        float *d = os + (int64_t)row * N + col;
        if (col + G <= N) {
#pragma unroll
            for (int t = 0; t + 4 <= G; t += 4)
                *reinterpret_cast<f32x4_unaligned *>(d + t) = f32x4{acc[t][e], acc[t + 1][e], acc[t + 2][e], acc[t + 3][e]};
            constexpr int kDone = G & ~3;
            if constexpr ((G & 2) != 0) *reinterpret_cast<f32x2_unaligned *>(d + kDone) = f32x2{acc[kDone][e], acc[kDone + 1][e]};
            if constexpr ((G & 1) != 0) d[G - 1] = acc[G - 1][e];
        } else {
#pragma unroll
            for (int t = 0; t < G; ++t)
                if (col + t < N) d[t] = acc[t][e];
        }
    }
}

template <bool T1, bool T2, bool EDGE>
__device__ __forceinline__ void f32_round(const RunArgs &a, const SegRec &rec, int64_t h, int r0, unsigned char *lds) {
    const int M = rec.M, N = rec.N, K = rec.K;
    const Words4<EDGE || T1> pa(reinterpret_cast<const float *>(a.A) + h * a.Dm1 + rec.off1, M * K);
    const Words4<EDGE || T2> pb(reinterpret_cast<const float *>(a.B) + h * a.Dm2 + rec.off2, N * K);
    float *os = reinterpret_cast<float *>(a.out) + h * a.Dout + rec.offO;
    for (int c0 = 0; c0 < N; c0 += kF32Cols) {
        switch (min(8, (N - c0 + 15) >> 4)) {
            case 1: f32_block<T1, T2, EDGE, 1>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 2: f32_block<T1, T2, EDGE, 2>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 3: f32_block<T1, T2, EDGE, 3>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 4: f32_block<T1, T2, EDGE, 4>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 5: f32_block<T1, T2, EDGE, 5>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 6: f32_block<T1, T2, EDGE, 6>(pa, pb, os, M, N, K, r0, c0, lds); break;
            case 7: f32_block<T1, T2, EDGE, 7>(pa, pb, os, M, N, K, r0, c0, lds); break;
            default: f32_block<T1, T2, EDGE, 8>(pa, pb, os, M, N, K, r0, c0, lds); break;
        }
    }
}

// a.ride_slots = 1 (launches that know the batch's totals): one workgroup per existing (head, segment, row block) item,
// head-major, cut into eight contiguous shares, one per die (as in attention_kernel).  Else grid (pair, z), the pairs flat too.
template <bool T1, bool T2>
__global__ __launch_bounds__(kF32Threads, 4) void gemm_f32_kernel(RunArgs a) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int64_t per_head = ((ConstHdr)(uintptr_t)a.plan)->att_blocks64;
    if (!header_ok(a)) { report_mismatch(a); return; }
    int g, round, step;
    int64_t h;
    if (a.ride_slots) {
        const unsigned id = flat_block(), die = id & 7u, kk = id >> 3;
        const int32_t *pfx = plan_rowblocks(a.plan, a.nseg, 0);
        const int64_t items = per_head * a.H, share = (items + 7) >> 3;
        const int64_t u = (int64_t)die * share + kk;
        if (id == 0 && threadIdx.x == 0 && share * 8 > flat_blocks())    // sized from another plan's summary
            atomicAdd(&reinterpret_cast<PlanHeader *>(a.plan)->run_errors, 1);
        if (kk >= share || u >= items) return;
        h = u / per_head;
        const int item = (int)(u % per_head);
        g = prefix_search(pfx, a.nseg, item);
        round = item - ((ConstI32)(uintptr_t)pfx)[g];
        step = 1 << 24;
    } else {
        g = (int)(flat_block() / (unsigned)a.H);
        h = flat_block() % (unsigned)a.H;
        if (g >= a.nseg) return;                       // (the last row of a flat grid)
        round = blockIdx.z;
        step = gridDim.z;
    }
    const SegRec rec = load_rec(plan_ro(a.plan, a.nseg).recs, g);
    if (rec.N < 1) return;
    for (; (int64_t)round * kF32Rows < rec.M; round += step) {
        if ((rec.K & 3) == 0) f32_round<T1, T2, false>(a, rec, h, round * kF32Rows, lds);
        else f32_round<T1, T2, true>(a, rec, h, round * kF32Rows, lds);
    }
}

template <bool T1, bool T2>
static int launch_f32(const RunArgs &run, dim3 grid, hipStream_t stream) {
    constexpr int kLds = (kF32Cols + (T1 ? kF32Rows : 0)) * kF32Pitch;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_f32_kernel<T1, T2>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return BA_ERR_LAUNCH;
    hipLaunchKernelGGL((gemm_f32_kernel<T1, T2>), grid, dim3(kF32Threads), kLds, stream, run);
    return hipGetLastError() == hipSuccess ? BA_OK : BA_ERR_LAUNCH;
}

int launch_gemm_f32(const RunArgs &args, int64_t nseg, const ba_plan_info *info, hipStream_t stream) {
    RunArgs run = args;
    if (info) nseg = info->nseg;
    if (nseg <= 0) return BA_OK;
    run.nseg = (int)nseg;
    dim3 grid;
    if (info) {
        const int64_t items = (int64_t)info->att_blocks64 * args.H;
        if (items <= 0) return BA_OK;
        if (items > 0x7ffffff0) return BA_ERR_UNSUPPORTED;
        run.ride_slots = 1;
        grid = flat_grid((items + 7) / 8 * 8);
    } else {
        if (nseg * args.H > 0x7fffffff) return BA_ERR_UNSUPPORTED;
        grid = flat_grid(nseg * args.H);
        grid.z = 4;
    }
    switch (run.flags & (kFlagTranspose1 | kFlagTranspose2)) {
        case 0: return launch_f32<false, false>(run, grid, stream);
        case kFlagTranspose1: return launch_f32<true, false>(run, grid, stream);
        case kFlagTranspose2: return launch_f32<false, true>(run, grid, stream);
        default: return launch_f32<true, true>(run, grid, stream);
    }
}

}  // namespace ba
