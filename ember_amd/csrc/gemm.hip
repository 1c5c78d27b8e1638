// The linear layers of a prompt on gfx950: C[M, N] = A[M, K] . W[N, K]^T for
// more rows than the decode-sized kernel takes (linear.hip, 64), and for wide
// batches of up to 64 where it is the faster one, with the same four epilogues
// and the same bits per row (linear.hpp: the order of the sums).
//
// What bounds it: the matrix cores, once W and A are re-read little enough; at
// few tokens, one work-group's chain of chunks. A work-group of 4 waves covers
// 64 tokens x 64 FW features; each wave owns 16 FW features and all the tokens.
// So W, packed in the MFMA operand's lane order, goes straight from memory to
// registers, every wave its own, and only A passes through LDS, where each wave
// reads it. A comes in chunks of two k steps, double-buffered, its loads two
// chunks ahead in registers; W's loads run two chunks ahead too. Taking a run's
// strided steps one at a time would read A in 64-byte pieces (1800 x 4096 x
// 1024 29.1 us against 26.4, weights in the last-level cache); two runs side by
// side read 128.
//
// Measured, packed W from HBM, against 64 rows per launch of the decode-sized
// kernel (us): 1800 x 4096 x 1024 29 (520 TFLOP/s), 128 before; 1800 x 1024 x 2048
// 18.8, 120; 1800 x 6144 x 1024 44, 229; 1800 x 1024 x 3072 26, 162; 256 x 4096 x 1024
// 8.7, 18.6; 256 x 1024 x 2048 11.7, 16.4; 48 x 12288 x 2048 16.3, 27.6; 64 x 151936 x
// 1024 76, 147.
#include <algorithm>
#include <type_traits>

#include "linear.hpp"

namespace ember::hip {
namespace {

constexpr int kGemmWaves = 4;                      // of one K group: side by side over the features
constexpr int kGemmThreads = kGemmWaves * kWave;  // of one K group
constexpr int CS = 2;                             // k steps per LDS chunk of A
constexpr int kSplitGroups = 4;                   // K groups of the split form
constexpr int kXcds = 8;
constexpr int kDescWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit data format, no swizzle

// One lane's four adjacent outputs (features n .. n + 3 of one token; all below N if vec_out).
template <int EP>
__device__ __forceinline__ void store_outputs(void *C, int64_t row, int n, int N, const f32x4 v, bool vec_out) {
    if constexpr (EP == EMBER_EPILOGUE_SILU_MUL) {
        const f16x2 h = {static_cast<f16>(clamp_half(silu(v[0]) * v[1])), static_cast<f16>(clamp_half(silu(v[2]) * v[3]))};
        f16 *o = static_cast<f16 *>(C) + row + n / 2;
        if (vec_out) {
            *reinterpret_cast<f16x2 *>(o) = h;
        } else {
            if (n + 1 < N) o[0] = h[0];
            if (n + 3 < N) o[1] = h[1];
        }
    } else if constexpr (EP == EMBER_EPILOGUE_STORE_F16) {
        f16x4 h;
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = static_cast<f16>(clamp_half(v[i]));
        f16 *o = static_cast<f16 *>(C) + row + n;
        if (vec_out) {
            *reinterpret_cast<f16x4 *>(o) = h;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (n + i < N) o[i] = h[i];
        }
    } else {
        constexpr bool add = EP == EMBER_EPILOGUE_ADD_F32;
        float *o = static_cast<float *>(C) + row + n;
        if (vec_out) {
            f32x4 *p = reinterpret_cast<f32x4 *>(o);
            *p = add ? *p + v : v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (n + i < N) o[i] = add ? o[i] + v[i] : v[i];
        }
    }
}

// MT tiles of 16 tokens and 4 x FW of 16 features per work-group. KG = 1: four
// waves take all of K; SLICES: K is in slices as the decode-sized kernel splits
// this shape. KG = 4: four K groups of four waves, group k summing runs 2 k and
// 2 k + 1 side by side; the runs' sums meet in LDS and are added in run order.
// RAGGED: the runs are not whole pairs of chunks.
template <int MT, int FW, int KG, int EP, bool SLICES, bool RAGGED>
__global__ void __launch_bounds__(kGemmThreads *KG, KG == 1 ? 2 : 1)
    gemm_kernel(const f16 *__restrict__ A, int lda, const f16 *__restrict__ W, int w_step, int64_t w_tile, int M, int N,
                int K, void *__restrict__ C, int ldc, int n_blocks, int slice_steps) {
    static_assert(KG == 1 || (KG == kSplitGroups && FW == 1 && !SLICES));
    constexpr int kRows = 16 * MT;
    constexpr int kPieces = CS * 4;  // 16-byte pieces of a row per chunk of CS k steps
    constexpr int kSwizzle = kPieces < 16 ? kPieces - 1 : 15;
    constexpr int kLoads = kRows * kPieces / kGemmThreads;  // 16-byte pieces of A per thread and chunk
    static_assert(kRows * kPieces % kGemmThreads == 0 && (CS & (CS - 1)) == 0);
    constexpr int kBufBytes = kRows * kPieces * 16;
    constexpr int kSumBytes = KG == 1 ? 0 : kLinearRuns * kGemmWaves * MT * kWave * 16;  // the runs' sums
    __shared__ __align__(16) unsigned char lds_all[kSumBytes > 2 * KG * kBufBytes ? kSumBytes : 2 * KG * kBufBytes];
    const int tid = static_cast<int>(threadIdx.x) % kGemmThreads, lane = tid % kWave;  // in the K group
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kGemmThreads);
    auto lds = [&](int buf) { return lds_all + (kg * 2 + buf) * kBufBytes; };
    const int c = lane % 16, g = lane / 16;
    // Block id -> (token block, feature block). Ids that differ by a multiple
    // of 8 run on one XCD: with feature blocks in multiples of 8, an XCD takes
    // an eighth of them for every token block, so its L2 keeps that part of W.
    int mb, nb;
    const int id = static_cast<int>(blockIdx.x);
    if (n_blocks % kXcds == 0) {
        const int per = n_blocks / kXcds, i = id / kXcds;
        nb = (id % kXcds) * per + i % per;
        mb = i / per;
    } else {
        nb = id % n_blocks;
        mb = id / n_blocks;
    }
    const int m0 = mb * kRows, rows = min(M - m0, kRows);
    const int steps = K / 32;
    const int tiles = (N + 15) / 16, t0 = (nb * kGemmWaves + wave) * FW;

    // A through a descriptor of this block's rows: rows past M (and the last
    // chunk's columns past the last row's end) read as zeros.
    const f16 *a0 = A + static_cast<int64_t>(m0) * lda;
    const uint32_t records = static_cast<uint32_t>((static_cast<int64_t>(rows - 1) * lda + K) * 2);
    const __amdgpu_buffer_rsrc_t ad = __builtin_amdgcn_make_buffer_rsrc(const_cast<f16 *>(a0), 0, records, kDescWord3);
    uint32_t aoff[kLoads];  // byte offset of this thread's pieces at k step 0
    int aslot[kLoads];      // and their place in LDS: piece q of row r at slot kPieces r + (q ^ (r & kSwizzle))
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int p = tid + j * kGemmThreads, r = p / kPieces, q = p % kPieces;
        aoff[j] = r < rows ? static_cast<uint32_t>(r * lda + 8 * q) * 2u : records;
        aslot[j] = 16 * (r * kPieces + (q ^ (r & kSwizzle)));
    }
    // W: packed, a tile's k steps are 1 KiB blocks in lane order; row-major, this lane's row (rows past N repeat the last).
    const f16 *w[FW];
#pragma unroll
    for (int f = 0; f < FW; f++)
        w[f] = w_tile ? W + min(t0 + f, tiles - 1) * w_tile + 8 * lane
                      : W + static_cast<int64_t>(min(16 * (t0 + f) + c, N - 1)) * K + 8 * g;

    // A chunk is two adjacent k steps (128 bytes of a row of A). Unsplit, they
    // belong to runs 2 p and 2 p + 1, which are summed side by side: chunks 2 p,
    // 2 p + 8, ..., then the next pair of runs. In a slice they follow each
    // other in one run. A K group takes one pair of runs. next_chunk(b): the chunk after the one at step b (S: none).
    auto next_chunk = [&](int b) {
        if (SLICES) return b + 2;
        if (KG > 1) return min(b + kLinearRuns, steps);
        return b + kLinearRuns < steps ? b + kLinearRuns
               : b < steps && b % kLinearRuns + 2 < min(kLinearRuns, steps) ? b % kLinearRuns + 2
                                                                            : steps;
    };
    int a_chunk = min(2 * kg, steps);  // the chunk that load_a takes next
    auto load_a = [&](uint4 (&v)[kLoads]) {
        const uint32_t k = 64u * static_cast<uint32_t>(a_chunk);
        a_chunk = next_chunk(a_chunk);
#pragma unroll
        for (int j = 0; j < kLoads; j++)  // an offset at or past the records reads zeros
            v[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ad, min(aoff[j] + k, records), 0, 0));
    };
    auto store_a = [&](int buf, const uint4 (&v)[kLoads]) {
#pragma unroll
        for (int j = 0; j < kLoads; j++) *reinterpret_cast<uint4 *>(lds(buf) + aslot[j]) = v[j];
    };
    int w_chunk = min(2 * kg, steps);  // the chunk whose W goes out next
    auto load_w = [&](int v, f16x8 (&wv)[FW]) {
        const int64_t at = static_cast<int64_t>(min(w_chunk + v, steps - 1)) * w_step;
        if (v == CS - 1) w_chunk = next_chunk(w_chunk);
#pragma unroll
        for (int f = 0; f < FW; f++) wv[f] = *reinterpret_cast<const f16x8 *>(w[f] + at);
    };

    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int kAccs = SLICES ? 1 : 2;  // runs summed side by side
    f32x4 acc[kAccs][FW][MT], sum[KG == 1 ? FW : 1][KG == 1 ? MT : 1], total[SLICES ? FW : 1][SLICES ? MT : 1];
#pragma unroll
    for (int f = 0; f < FW; f++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int r = 0; r < kAccs; r++) acc[r][f][mt] = zero;
            if constexpr (KG == 1) sum[f][mt] = zero;
            if constexpr (SLICES) total[f][mt] = zero;
        }
    // The MFMAs of a chunk's k step v: every tile of the wave, from zero at the start of a run.
    auto mfmas = [&](auto first, int v, const f16x8 (&x)[MT], const f16x8 (&wv)[FW]) {
        f32x4(&ac)[FW][MT] = acc[SLICES ? 0 : v];
#pragma unroll
        for (int f = 0; f < FW; f++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                ac[f][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[f], x[mt], decltype(first)::value ? zero : ac[f][mt],
                                                                   0, 0, 0);
    };
    auto end_runs = [&]() {  // the runs' sums join the slice's
        if constexpr (KG == 1) {
#pragma unroll
        for (int r = 0; r < kAccs; r++)
#pragma unroll
            for (int f = 0; f < FW; f++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) sum[f][mt] = sum[f][mt] + acc[r][f][mt];
        }
    };
    auto end_slice = [&]() {  // the slice's sum joins the total
        if constexpr (SLICES) {
#pragma unroll
            for (int f = 0; f < FW; f++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    total[f][mt] = total[f][mt] + sum[f][mt];
                    sum[f][mt] = zero;
                }
        }
    };
    auto read_x = [&](int buf, int u, f16x8 (&x)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int r = 16 * mt + c, q = 4 * u + g;
            x[mt] = *reinterpret_cast<const f16x8 *>(lds(buf) + 16 * (r * kPieces + (q ^ (r & kSwizzle))));
        }
    };

    uint4 a0v[kLoads], a1v[kLoads];
    f16x8 wv[2][CS][FW];
    load_a(a0v);
#pragma unroll
    for (int v = 0; v < CS; v++) load_w(v, wv[0][v]);
    load_a(a1v);
#pragma unroll
    for (int v = 0; v < CS; v++) load_w(v, wv[1][v]);
    store_a(0, a0v);
    __syncthreads();
    // Two chunks: each computes from its buffer, with the A of the chunk after
    // next going out first, and ends by storing the next chunk's A into the
    // other buffer, whose readers finished before the last barrier. A step's W
    // registers take the W of two chunks on as soon as its MFMAs have read
    // them. The scheduling barriers keep the loads there: left alone, the
    // compiler moves them down to just ahead of their use.
    // step(i, v, x, w): k step v of chunk i of the pair.
    auto pair = [&](auto step) {
        auto chunk = [&](int i, uint4 (&a_free)[kLoads], uint4 (&a_next)[kLoads]) {
            f16x8 x[CS][MT];
#pragma unroll
            for (int v = 0; v < CS; v++) read_x(i, v, x[v]);
            load_a(a_free);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < CS; v++) {
                step(i, v, x[v], wv[i][v]);
                load_w(v, wv[i][v]);
                __builtin_amdgcn_sched_barrier(0);
            }
            store_a(i ^ 1, a_next);
            __syncthreads();
        };
        chunk(0, a0v, a1v);
        chunk(1, a1v, a0v);
    };
    using First = std::true_type;
    using Later = std::false_type;
    if constexpr (KG > 1) {  // one pair of runs, from zero; the groups take the same number of pairs
        for (int b = 2 * kg, at = 0; at < steps; at += 2 * kLinearRuns)
            pair([&](int, int v, const f16x8 (&x)[MT], const f16x8 (&w)[FW]) {
                if (!RAGGED || b + v < steps) mfmas(Later{}, v, x, w);
                if (RAGGED && v == CS - 1) b += kLinearRuns;
            });
    } else if constexpr (!RAGGED) {  // whole pairs of chunks per run (or pair of runs): no branch inside a pair
        const int run_chunks = SLICES ? slice_steps / kLinearRuns / CS : steps / kLinearRuns;
        for (int at = 0, run = 0; at < steps / CS;) {
            pair([&](int i, int v, const f16x8 (&x)[MT], const f16x8 (&w)[FW]) {
                if (i == 0 && (v == 0 || !SLICES)) mfmas(First{}, v, x, w);
                else mfmas(Later{}, v, x, w);
            });
            for (at += 2; at % run_chunks != 0; at += 2)
                pair([&](int, int v, const f16x8 (&x)[MT], const f16x8 (&w)[FW]) { mfmas(Later{}, v, x, w); });
            end_runs();
            if (SLICES && ++run == kLinearRuns) {
                end_slice();
                run = 0;
            }
        }
    } else if constexpr (!SLICES) {
        int b = 0;  // the chunk's first step
        while (b < steps)
            pair([&](int, int v, const f16x8 (&x)[MT], const f16x8 (&w)[FW]) {
                if (b >= steps) return;  // the second chunk of the last pair
                if (b + v < steps) {
                    if (b < kLinearRuns) mfmas(First{}, v, x, w);
                    else mfmas(Later{}, v, x, w);
                } else if (b < kLinearRuns) {  // run b + 1 is empty
#pragma unroll
                    for (int f = 0; f < FW; f++)
#pragma unroll
                        for (int mt = 0; mt < MT; mt++) acc[kAccs - 1][f][mt] = zero;
                }
                if (v == 0) return;
                if (b + kLinearRuns >= steps) end_runs();
                b = next_chunk(b);
            });
    } else {
        // Steps taken, the run in progress, its slice's first step, and the step it ends before (runs may be empty).
        int s = 0, run = 0, slice0 = 0, run_end = 0;
        while (run_end == 0) run_end = ++run * slice_steps / kLinearRuns;
        bool fresh = true;  // this step starts a run
        while (s < steps)
            pair([&](int, int v, const f16x8 (&x)[MT], const f16x8 (&w)[FW]) {
                if (s >= steps) return;
                if (fresh) mfmas(First{}, v, x, w);
                else mfmas(Later{}, v, x, w);
                fresh = ++s == run_end;
                if (!fresh) return;
                end_runs();
                if (s == slice0 + slice_steps) {
                    end_slice();
                    slice0 = s;
                    run = 0;
                }
                while (run < kLinearRuns && run_end == s) run_end = slice0 + ++run * slice_steps / kLinearRuns;
            });
    }

    // sum[f][mt][i] = C[token 16 mt + c][feature 16 (t0 + f) + 4 g + i]
    const auto whole = [&](int n0) { return ((reinterpret_cast<uintptr_t>(C) & 15) | (ldc & 3)) == 0 && n0 + 16 <= N; };
    if constexpr (KG > 1) {
        // Every group is past the last chunk's barrier: the buffers take the runs' sums, and group k adds and stores
        // token tile k.
        f32x4 *sums = reinterpret_cast<f32x4 *>(lds_all) + wave * MT * kWave + lane;  // [run][wave][mt][lane]
        constexpr int kRunSums = kGemmWaves * MT * kWave;
#pragma unroll
        for (int r = 0; r < kAccs; r++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) sums[(2 * kg + r) * kRunSums + mt * kWave] = acc[r][0][mt];
        __syncthreads();
        const int tok = 16 * kg + c;
        if (kg >= MT || tok >= rows) return;
        f32x4 v = zero;
#pragma unroll
        for (int r = 0; r < kLinearRuns; r++) v = v + sums[r * kRunSums + kg * kWave];
        store_outputs<EP>(C, static_cast<int64_t>(m0 + tok) * ldc, 16 * t0 + 4 * g, N, v, whole(16 * t0));
    } else {
#pragma unroll
        for (int f = 0; f < FW; f++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int tok = 16 * mt + c;
                if (tok >= rows) continue;
                store_outputs<EP>(C, static_cast<int64_t>(m0 + tok) * ldc, 16 * (t0 + f) + 4 * g, N,
                                  SLICES ? total[SLICES ? f : 0][SLICES ? mt : 0] : sum[f][mt], whole(16 * (t0 + f)));
            }
    }
}

// K slices: only with a workspace that launch_gemv would split with, at its most rows.
int slices(const EmberGemvArgs &a) {
    const bool room = a.workspace && a.workspace_bytes >= gemv_workspace_bytes(64, a.N, a.K);
    return room ? gemv_split(a.N, a.K) : 1;
}

// form: 0 the split form, 1 or 2 feature tiles per wave of the other; ks: K slices (1 with the split form).
template <int EP>
hipError_t launch_gemm_ep(const EmberGemvArgs &a, int form, int ks, hipStream_t stream) {
    const int steps = a.K / 32, slice_steps = steps / ks;
    const bool ragged = slice_steps % (2 * kLinearRuns * (ks > 1 ? CS : 1)) != 0;  // a run is pairs of chunks
    const int mt = form > 0 || a.M > 32 ? 4 : 2;
    const int fw = std::max(form, 1);
    const int n_blocks = (a.N + 64 * fw - 1) / (64 * fw), m_blocks = (a.M + 16 * mt - 1) / (16 * mt);
    const f16 *A = static_cast<const f16 *>(a.A), *W = static_cast<const f16 *>(a.W);
    auto go = [&](auto kernel, int groups) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n_blocks * m_blocks)), dim3(kGemmThreads * groups), 0, stream,
                           A, a.lda, W, a.w_packed ? kPackBlock : 32,
                           a.w_packed ? static_cast<int64_t>(steps) * kPackBlock : int64_t{0}, a.M, a.N, a.K, a.C, a.ldc,
                           n_blocks, slice_steps);
        return hipGetLastError();
    };
    if (form == 0) {
        switch (mt + (ragged ? 1 : 0)) {
            case 2: return go(gemm_kernel<2, 1, kSplitGroups, EP, false, false>, kSplitGroups);
            case 3: return go(gemm_kernel<2, 1, kSplitGroups, EP, false, true>, kSplitGroups);
            case 4: return go(gemm_kernel<4, 1, kSplitGroups, EP, false, false>, kSplitGroups);
            default: return go(gemm_kernel<4, 1, kSplitGroups, EP, false, true>, kSplitGroups);
        }
    }
    switch ((fw == 2 ? 4 : 0) + (ks > 1 ? 2 : 0) + (ragged ? 1 : 0)) {
        case 0: return go(gemm_kernel<4, 1, 1, EP, false, false>, 1);
        case 1: return go(gemm_kernel<4, 1, 1, EP, false, true>, 1);
        case 2: return go(gemm_kernel<4, 1, 1, EP, true, false>, 1);
        case 3: return go(gemm_kernel<4, 1, 1, EP, true, true>, 1);
        case 4: return go(gemm_kernel<4, 2, 1, EP, false, false>, 1);
        case 5: return go(gemm_kernel<4, 2, 1, EP, false, true>, 1);
        case 6: return go(gemm_kernel<4, 2, 1, EP, true, false>, 1);
        default: return go(gemm_kernel<4, 2, 1, EP, true, true>, 1);
    }
}

}  // namespace

// 65 to 128 rows of few features: two launches of the decode-sized kernel, whose
// work-groups are more (per 16 features and 16 tokens, or K slice) and each walk
// less of K. Time by the tiles over theirs, packed, W from HBM: up to 1024
// features, K 256 to 4096, 1.2 to 1.7; up to 2048 features, K 256 to 1024, 1.03
// to 1.26, in K slices (K above 4096) 1.26 to 3; K 2048, up to 1536 features, 1.01 to
// 1.18, 2048 features 1.03 to 1.06 up to 96 rows, 0.94 beyond; K 3072 and 4096 0.75
// to 1.0 (1280 features 0.84 to 1.14); 2560 and 3072 features, K 256 and 512, 1.02 to 1.19
// up to 96 rows, K 1024 0.79 to 0.98; 4080 features 0.4 to 0.9. From 129 rows on the tiles win
// unsplit (129 x 1024 x 2048 11.9 / 10.5), three launches against one.
bool gemm_by_gemv(const EmberGemvArgs &a) {
    if (a.M <= 64 || a.M > 128) return false;
    const bool split = slices(a) > 1;
    if (a.N <= 1024) return split || a.K <= 4096;
    if (a.N <= 1536) return split || a.K <= 2048;
    if (a.N <= 2048) return split || a.K <= 1024 || (a.K <= 2048 && a.M <= 96);
    return a.N <= 3072 && a.K <= 512 && a.M <= 96;
}

// The form by the number of work-groups (us; packed W from HBM):
//  - the split form while its 64 x 64 blocks fit one round at one per CU: its
//    waves each walk a quarter of K (256 x 1024 x 2048, 64 work-groups, 11.7
//    against 13.1 with one feature tile per wave and 16.3 with two; 256 x 4096 x
//    1024, 256, 8.7 / 9.0 / 10.7; 256 x 6144 x 1024, 384, 14.5 / 11.3 / 11.8).
//    Its LDS reads, 64 rows per feature tile, bound it beyond;
//  - two feature tiles per wave, which read A half as often, from 200
//    work-groups on (1800 x 12288 x 2048, one against two, 169 / 142; 1800 x 1024 x
//    2048, 232 work-groups, 19.2 / 18.8; 700 x 2048 x 2048, 176, 17.8 / 18.4); up to 64
//    rows, where W's one pass is what counts, one (64 x 151936 x 1024 75.9 / 78);
//  - else one. Four feature tiles spilled and were within 2% of two; 128 tokens
//    per work-group, at one wave per SIMD, lost (1800 x 4096 x 1024 34.3 / 27.1,
//    weights in the last-level cache).
// A row-major W's split form is no faster than one tile per wave (48 x 6144 x
// 2048 16.5 / 16.4).
hipError_t launch_gemm(const EmberGemvArgs &a, hipStream_t stream) {
    const int m_blocks = (a.M + 63) / 64;
    const int ks = slices(a);
    int form = 1;
    if (a.w_packed && ks == 1 && m_blocks * ((a.N + 63) / 64) <= 256) form = 0;
    else if (a.M > 64 && m_blocks * ((a.N + 127) / 128) >= 200) form = 2;
    switch (a.epilogue) {
        case EMBER_EPILOGUE_STORE_F16: return launch_gemm_ep<EMBER_EPILOGUE_STORE_F16>(a, form, ks, stream);
        case EMBER_EPILOGUE_STORE_F32: return launch_gemm_ep<EMBER_EPILOGUE_STORE_F32>(a, form, ks, stream);
        case EMBER_EPILOGUE_ADD_F32: return launch_gemm_ep<EMBER_EPILOGUE_ADD_F32>(a, form, ks, stream);
        case EMBER_EPILOGUE_SILU_MUL: return launch_gemm_ep<EMBER_EPILOGUE_SILU_MUL>(a, form, ks, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ember::hip
