// W8A8 for 2 .. 64 activation rows and blocks of up to 64: all tiles of a workgroup side by side, K in chunks.
//
//   acc[M,N] = A[M,K] . W[N,K]^T  (int32, bit exact);  Y = fp16((float)acc * s_tok[m] * s_ch[n])
//
// The structure of the K-streaming kernel (w4a16_kstream.h) on v_mfma_i32_16x16x64_i8, without anything to unpack: one workgroup of eight
// wavefronts per CU keeps the sums of up to T 16-row weight tiles and MB blocks of 16 activation rows in registers; of a chunk of
// 8 x U bytes of K wavefront w takes the U bytes w of every row, through an LDS slot of its own as whole 128-byte lines (global -> LDS without
// registers), refilled for the next chunk as it is read; no barrier until the wavefronts' sums meet in LDS at the end.
// blockIdx.z: blocks of 16 MB rows.
#include "nnf_device.h"
#include "nnf_launch.h"

#include "../nnf_workspace.h"

namespace nnf
{
    namespace
    {
        constexpr int QS_WAVES = workspace::KSTREAM_WAVES;
        typedef const void __attribute__((address_space(1))) * qs_global_ptr_t;
        typedef void __attribute__((address_space(3))) * qs_lds_ptr_t;
        template <int N>
        __device__ __forceinline__ void qs_wait_loads() // until at most the last N loads of the wavefront are outstanding
        {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
        }

        // LDS (bytes): per wavefront [MB + T][16 rows x U]; at the end, over all of it, the wavefronts' sums [8][tiles of a round][MB KiB]
        template <int T, int MB, int U, bool RAW>
        __global__ __launch_bounds__(QS_WAVES * 64) void w8a8_kstream_kernel(const int8_t* __restrict__ A, const int8_t* __restrict__ W,
                                                                             half_t* __restrict__ Y, int32_t* __restrict__ acc_out, int N, int K,
                                                                             int tiles_q, int tiles_r, int M_all, const float* __restrict__ s_tok,
                                                                             const float* __restrict__ s_ch)
        {
            static_assert(U == 128 || U == 256, "whole lines");
            constexpr int BLOCK = 16 * U, LB = BLOCK / 1024; // a block of 16 rows: bytes, wavefront-wide loads
            constexpr int PIECES = U / 16, ROWS = 64 / PIECES; // 16-byte pieces of a row; rows of a load
            constexpr int J = U / 64;                        // MFMAs of a tile and block
            constexpr int L = LB * (MB + T);                 // loads of a chunk
            constexpr int RT = workspace::kstream_round(T, MB);
            extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
            const int tid = threadIdx.x, lane = tid & 63;
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int col = lane & 15, kq = lane >> 4;
            const int first_row = (int)blockIdx.z * (MB * 16), M = min(M_all - first_row, MB * 16);
            A += (size_t)first_row * K;
            const int b = blockIdx.x;
            const int t0 = b * tiles_q + min(b, tiles_r);
            const int TW = tiles_q + (b < tiles_r ? 1 : 0); // tiles of this workgroup, at most T
            // (past its tiles: the last one again, not used; the last tile of an N that is no multiple of 16: rows N-16 .. N-1)
            auto row0_of = [&](int i) { return __builtin_amdgcn_readfirstlane(min((t0 + min(i, TW - 1)) * 16, N - 16)); };
            const int units = K / U; // wavefront w: w, w + 8, ...
            uint8_t* slot = smem + wave * ((MB + T) * BLOCK);

            // the 16-byte piece q of row r of a block lies at position q ^ swz(r): conflict-free 128-bit reads of a column of 16 rows
            auto swz = [](int r) { return U == 256 ? r & 15 : (r >> 1) & 7; };
            const int last_block = (M - 1) >> 4;
            uint32_t off[LB], a_off_last[LB];
#pragma unroll
            for (int c = 0; c < LB; ++c)
            {
                const int r = c * ROWS + lane / PIECES;
                const uint32_t piece = (uint32_t)(((lane % PIECES) ^ swz(r)) * 16);
                off[c] = (uint32_t)r * (uint32_t)K + piece;
                a_off_last[c] = (uint32_t)min(r, M - 1 - last_block * 16) * (uint32_t)K + piece;
            }
            auto fetch_a = [&](int u, int mb) {
                const int8_t* base = A + (size_t)(min(mb, last_block) * 16) * (size_t)K + (size_t)u * U;
#pragma unroll
                for (int c = 0; c < LB; ++c)
                    __builtin_amdgcn_global_load_lds((qs_global_ptr_t)(base + (mb >= last_block ? a_off_last[c] : off[c])),
                                                     (qs_lds_ptr_t)(slot + mb * BLOCK + c * 1024), 16, 0, 0);
            };
            const int8_t* w_row[T];
#pragma unroll
            for (int t = 0; t < T; ++t)
                w_row[t] = W + (size_t)row0_of(t) * (size_t)K;
            auto fetch_w = [&](int u, int t) {
#pragma unroll
                for (int c = 0; c < LB; ++c)
                    __builtin_amdgcn_global_load_lds((qs_global_ptr_t)(w_row[t] + (size_t)u * U + off[c]),
                                                     (qs_lds_ptr_t)(slot + (MB + t) * BLOCK + c * 1024), 16, 0, 0);
            };
            const int chunks = (units - wave + QS_WAVES - 1) / QS_WAVES;
            // A workgroup starts at the chunk of its place on its XCD (workgroups are dealt out to the eight XCDs in turn) and wraps around: in step,
            // all of them read the same 2 KiB of every row at a time, with rows of 4 or 8 KiB a part of the memory channels
            // (16 x 8192 x 8192 19.7 -> 15.4 us, 32 x 8192 x 4096 11.1 -> 9.9, rows of 5.5 or 14 KiB level)
            const int first_chunk = (b >> 3) % max(chunks, 1);
            auto unit_of = [&](int c) {
                const int i = c + first_chunk;
                return min(wave + max(i >= chunks ? i - chunks : i, 0) * QS_WAVES, units - 1);
            };
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                fetch_a(unit_of(0), mb);
#pragma unroll
            for (int t = 0; t < T; ++t)
                fetch_w(unit_of(0), t);

            intx4 acc[T][MB];
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    acc[t][mb] = intx4{0, 0, 0, 0};
            uint32_t rd[J]; // operand reads: piece kq * J + j of row col
#pragma unroll
            for (int j = 0; j < J; ++j)
                rd[j] = (uint32_t)(col * U + (((kq * J + j) ^ swz(col)) << 4));

            // Loads of a wavefront in order: chunk by chunk [MB blocks of activations] [T tiles of weights], those of the next chunk asked for
            // where their place has just been read; the wait counts are the loads that follow the one waited for (LAST: no next chunk).
            auto chunk = [&](int c, auto last) {
                constexpr bool LAST = decltype(last)::value;
                const int next = unit_of(c + 1);
                intx4 areg[MB][J];
                unroll_for<0, MB>([&](auto mb_c) {
                    constexpr int mb = decltype(mb_c)::value;
                    qs_wait_loads<LAST ? L - LB * (mb + 1) : L - LB>();
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        areg[mb][j] = *reinterpret_cast<const intx4*>(slot + mb * BLOCK + rd[j]);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // read before it is refilled
                    if constexpr (!LAST)
                        fetch_a(next, mb);
                });
                intx4 wnext[J];
                auto read_w = [&](auto t_c) {
                    constexpr int t = decltype(t_c)::value;
                    qs_wait_loads<LAST ? LB * (T - 1 - t) : L - LB>();
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        wnext[j] = *reinterpret_cast<const intx4*>(slot + (MB + t) * BLOCK + rd[j]);
                };
                read_w(std::integral_constant<int, 0>());
                unroll_for<0, T>([&](auto t_c) {
                    constexpr int t = decltype(t_c)::value;
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    intx4 wv[J];
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        wv[j] = wnext[j];
                    if constexpr (!LAST)
                        fetch_w(next, t);
                    if constexpr (t + 1 < T)
                        read_w(std::integral_constant<int, (t + 1 < T ? t + 1 : 0)>());
#pragma unroll
                    for (int j = 0; j < J; ++j)
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb)
                            acc[t][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(areg[mb][j], wv[j], acc[t][mb], 0, 0, 0);
                });
            };
            for (int c = 0; c < chunks - 1; ++c)
                chunk(c, std::false_type());
            if (chunks > 0)
                chunk(chunks - 1, std::true_type());
            qs_wait_loads<0>(); // (a wavefront without a unit of its own has asked for one all the same)
            __syncthreads();

            // ---- the wavefronts' sums meet: lane (n = col, kq), element e: row m = 16 mb + 4 kq + e --------------------------------
            int32_t* red = reinterpret_cast<int32_t*>(smem);
            unroll_for<0, (T + RT - 1) / RT>([&](auto round) {
                constexpr int first = decltype(round)::value * RT;
                if constexpr (first > 0)
                    __syncthreads();
#pragma unroll
                for (int tt = 0; tt < RT; ++tt)
                    if (first + tt < T)
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb)
                            *reinterpret_cast<intx4*>(red + ((wave * RT + tt) * MB + mb) * 256 + lane * 4) = acc[first + tt < T ? first + tt : 0][mb];
                __syncthreads();
                for (int o = tid; o < min(RT, TW - first) * (MB * 64); o += QS_WAVES * 64)
                {
                    const int tt = (o >> 6) / MB, mb = (o >> 6) % MB; // (o & 63 == lane)
                    const int n0 = (t0 + first + tt) * 16, nn = min(n0, N - 16) + col;
                    if (nn < n0) // (a last tile moved back: these columns belong to the tile before it)
                        continue;
                    intx4 s = {0, 0, 0, 0};
#pragma unroll
                    for (int w = 0; w < QS_WAVES; ++w)
                        s += *reinterpret_cast<const intx4*>(red + ((w * RT + tt) * MB + mb) * 256 + lane * 4);
                    const int v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                    {
                        const int m = mb * 16 + kq * 4 + e;
                        if (m >= M)
                            continue;
                        const size_t at = (size_t)(first_row + m) * N + nn;
                        if constexpr (RAW)
                            acc_out[at] = v[e];
                        else
                        {
                            const float t = (float)v[e] * s_tok[first_row + m];
                            Y[at] = f32_to_f16_two_step(t * s_ch[nn]);
                        }
                    }
                }
            });
        }

        template <int T, int MB, int U>
        hipError_t launch_q8_kstream(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* s_tok, const void* W,
                                     const void* s_ch, void* Y, void* acc, int M, int N, int K)
        {
            auto run = [&](auto kernel, LdsGrant& granted) {
                const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), granted, (int)MAX_LDS_BYTES);
                if (e != hipSuccess)
                    return e;
                hipLaunchKernelGGL(kernel, dim3(plan.grid, 1, plan.row_blocks), dim3(QS_WAVES * 64), workspace::w8a8_kstream_lds_bytes(T, MB, U),
                                   stream, (const int8_t*)A, (const int8_t*)W, (half_t*)Y, (int32_t*)acc, N, K, plan.tiles_q, plan.tiles_r, M,
                                   (const float*)s_tok, (const float*)s_ch);
                return hipGetLastError();
            };
            static LdsGrant granted_raw, granted;
            return acc ? run(&w8a8_kstream_kernel<T, MB, U, true>, granted_raw) : run(&w8a8_kstream_kernel<T, MB, U, false>, granted);
        }
    } // namespace

    hipError_t launch_w8a8_kstream(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* s_tok, const void* W,
                                   const void* s_ch, void* Y, void* acc, int M, int N, int K)
    {
        hipError_t e = hipErrorInvalidValue;
        unroll_for<1, 5>([&](auto mb) {
            unroll_for<1, workspace::KSTREAM_MAX_TILES + 1>([&](auto t) {
                if (plan.row_tiles != mb.value || plan.tiles != t.value)
                    return;
                if (workspace::w8a8_kstream_unit(t.value, mb.value, K) == 128)
                    e = launch_q8_kstream<t.value, mb.value, 128>(stream, plan, A, s_tok, W, s_ch, Y, acc, M, N, K);
                else if constexpr (workspace::w8a8_kstream_unit(t.value, mb.value, 256) == 256)
                    e = launch_q8_kstream<t.value, mb.value, 256>(stream, plan, A, s_tok, W, s_ch, Y, acc, M, N, K);
            });
        });
        return e;
    }
} // namespace nnf
