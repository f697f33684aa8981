// fp16 x int4 / int8 for blocks of 2 .. 64 activation rows: all tiles of a workgroup side by side, K in chunks.
//
//   Y[M,N] = A[M,K] . ((Wq - zp) * S)^T
//
// Replaces the cublasHgemm call of cuda::Dot (src/nnfusion/core/kernels/cuda_gpu/kernels/dot.cpp:271-363) for a
// weight-quantized Dot node with a few activation rows, where it is ahead of the row-streaming kernels (w4a16_mrows.hip), which keep
// the activations of all of K in registers, and of the tile GEMM (w4a16_gemm_sk.h): workspace::kstream_choice.
//
//   * One workgroup of eight wavefronts per CU owns up to T 16-row weight tiles and keeps the fp32 sums of all of them in
//     registers (T x MB accumulators of 16 x 16, MB blocks of 16 activation rows).  K is walked in chunks of eight groups
//     of 128, wavefront w the group w of each: a wavefront sums its own groups, nothing but its own loads feeds its MFMAs,
//     and there is no barrier between the first load and the last.  The eight wavefronts' sums meet in LDS once, at the end.
//   * With 33 .. 64 rows what bounds it is the activations: every CU fetches all M x K of them from its L2 (48 x 4096: 384 KiB against
//     96 KiB of weights with three tiles), and of the 3500 cycles of a chunk (1.9 GHz) the load issue, the way of the activations through
//     LDS and the unpacking take about 2000 each.  They are asked for as whole 128-byte lines, global -> LDS without registers, through a
//     ring of RB blocks (16 rows x 256 bytes) per wavefront that is refilled block by block as the blocks are copied into operand
//     registers.  45 x 12288 x 4096: 14.1 us (21.6 on the tile GEMM); with up to 16 rows HBM and the latency of the first chunk bound it:
//     16 x 12288 x 2560 7.4 us (10.4 on the row-streaming kernel), 8 x 4096 x 2560 3.9 (5.2).
//     Measured level or slower: the chunks in another order on each CU of an XCD (14.9 at 45 rows); the weights through registers and an
//     LDS write (14.5); the next chunk's loads one at a time between the MFMAs (14.5); two or three chunks ahead
//     (8 - 15 % slower with two and more tiles; with one tile and up to 16 rows two chunks are 4 - 10 % faster: D).
//   * The weights of a lane (32 of one row and group) are unpacked to the exact integers q - zp in fp16 (the nibble in the
//     mantissa of 1024.0 or 64.0, minus 1024 + zp or 64 + zp) once per chunk and meet MB blocks of rows; the group's sum times its scale
//     joins the accumulator in fp32.
//   * BITS 8 (groups of 32 / 64 / 128 with their scales in the weights, as QG of 4 bits): a byte b behind 0x64 is 1024 + b in fp16, less 1024 + zp
//     exact; lanes read 32 bytes of a row's 128, pieces 2 kq and 2 kq + 1 swizzled over eight places: no bank conflicts.  Against the
//     row-streaming kernel on bytes, the tile kernel and the passes of the nodes around them: 45 x 12288 x 4096 28.3 -> 18.2 us
//     (16.0 at 32 rows, where the weights alone bound it), 16 x 4096 x 4096 with RMSNorm and SiLU-gate 17.0 -> 12.9, 5 x 1000 x 1280 5.4 -> 3.9.
//   * RMS: rstd from the squares of the activations as they pass (fp32), applied to the sums; gamma[k] multiplies the
//     unpacked weights, as in the tile GEMM: gamma times an activation alone may leave the range of fp16.  (q - zp) times gamma is rounded
//     to eleven bits, as a normalised activation is in a pass of its own: at most 15 gamma, and a multiple of 2^-24 like gamma, so exact where it
//     is a subnormal number.  Gamma is used as it is, a sixteenth of it where a group has one of 4096 and more (16 on that group's sum).
//     QG: a weight is (q - zp) times its scale, rounded, and that times gamma, rounded, as a weight and a normalised activation are rounded
//     once each elsewhere.  The scales of a row's group of 128 are multiplied by a power of two, which the group's sum takes back in fp32: with
//     the exponent e of the largest of them by 2^(18 - BITS - e), a weight stays below 2^4, times gamma below 2^16 (where the group has a gamma of 4096
//     and more a sixteenth of that, where all are below 1 256 times that), and only products 2^15 below the largest possible lose bits.
//     Costs 4 % (45 x 11008 x 4096, groups of 64 with zero points 16.9 -> 17.5 us); RMSNorm as a launch ahead takes 2.8 us.
//   * Ranges of K (blockIdx.y): fp32 sums to scratch memory, added up in range order by the workgroup that arrives last,
//     as in w4a16_mrows_any_kernel.
#pragma once

#include "nnf_device.h"
#include "nnf_launch.h"

#include "../nnf_workspace.h"

namespace nnf
{
    namespace
    {
        constexpr int KS_WAVES = workspace::KSTREAM_WAVES;
        typedef const void __attribute__((address_space(1))) * ks_global_ptr_t;
        typedef void __attribute__((address_space(3))) * ks_lds_ptr_t;

        template <int N>
        __device__ __forceinline__ void wait_loads() // until at most the last N loads of the wavefront are outstanding
        {
            static_assert(N >= 0, "");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
        }
    } // namespace

    // blockIdx.z: blocks of 16 MB activation rows.
    // pack = M | zp << 13 | gate << 21 | range_groups << 22 (ten bits, all set for one range); tiles = tiles_q | tiles_r << 16: output
    // tiles of a workgroup, one more for the first tiles_r (gate: twice as many weight tiles, the gate and the up tile of each in turn).
    // LDS (bytes): per wavefront [RB][4096] activations | [T][256 BITS] weights | (RMS) 256 gamma; then the scales of the
    //              workgroup's range of K, [T][16][32] words.  At the end, over all of it: (RMS) the wavefronts' sums of squares
    //              [8][16 MB] and rstd[16 MB] | from byte 4096 on the wavefronts' sums [8][tiles of a round][MB KiB].
    template <int T, int MB, bool RMS, int QG, int BITS>
    __global__ __launch_bounds__(KS_WAVES * 64) void w4a16_kstream_kernel(const half_t* __restrict__ A, const uint8_t* __restrict__ Wq,
                                                                          const half_t* __restrict__ S, half_t* __restrict__ Y, int N,
                                                                          int K, int tiles, int pack, float* __restrict__ partial,
                                                                          uint32_t* sync, GemvFusionArgs f,
                                                                          const uint8_t* __restrict__ zps)
    {
        static_assert(T >= 1 && MB >= 1 && MB <= 4, "");
        constexpr int D = workspace::kstream_depth(T, MB); // chunks asked for ahead
        constexpr int RB = workspace::kstream_ring(MB);    // blocks of activations in a slot of a wavefront's ring
        static_assert(RB == MB || (RB < MB && D == 1), "");
        // QG: scales of a tile's row and group of 128 as words, 64 words a load; then loads of bytes with their zero points
        static_assert(BITS == 4 || (BITS == 8 && QG != 0), "");
        constexpr int SPW = QG == 5 ? 2 : 1, NSL = QG ? workspace::kstream_scale_loads(T, QG) : 0;
        constexpr int ZPB = BITS == 8 ? 1 << (7 - QG) : QG == 5 ? 2 : 1, NZL = QG ? workspace::kstream_zero_loads(T, QG, BITS) : 0;
        constexpr int NS = NSL + NZL;
        constexpr int NW = BITS / 4, WB = NW * 1024, LW = NW * T;      // of a tile's weights: loads, bytes; loads of all of them
        constexpr int NG = RMS ? 1 : 0, L = NG + 4 * MB + NS + LW; // loads of a chunk
        constexpr int SLOT = RB * ROW_BLOCK_BYTES + T * WB + NG * 256 + NS * 256;
        constexpr int W_AT = RB * ROW_BLOCK_BYTES, G_AT = W_AT + T * WB, S_AT = G_AT + NG * 256; // parts of a slot
        constexpr int WAVE_BYTES = workspace::kstream_wave_bytes(T, MB, RMS, QG, BITS);
        constexpr int RT = workspace::kstream_round(T, MB); // tiles whose sums are in LDS at a time
        extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
        uint32_t MAGIC, MAGIC_HI, MASK_LO, MASK_HI;
        asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(MAGIC));
        asm volatile("v_mov_b32 %0, 0x54005400" : "=v"(MAGIC_HI));
        asm volatile("s_mov_b32 %0, 0x000F000F" : "=s"(MASK_LO));
        asm volatile("s_mov_b32 %0, 0x00F000F0" : "=s"(MASK_HI));

        const int tid = threadIdx.x;
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int col = lane & 15; // n within the tile (B operand / D column), m for the A operand
        const int kq = lane >> 4;  // K quarter of the MFMA operands, row quad of D
        const int M_all = pack & 0x1fff, zp = (pack >> 13) & 0xff, gate = (pack >> 21) & 1, range_groups = (int)((unsigned)pack >> 22);
        const int tiles_q = tiles & 0xffff, tiles_r = (int)((unsigned)tiles >> 16);
        const int G = K >> 7, ROW_BYTES = BITS == 8 ? K : K >> 1;
        // rows first_row .. first_row + M - 1 of the activations, as a product of its own
        const int first_row = (int)blockIdx.z * (MB * 16), M = min(M_all - first_row, MB * 16);
        A += (size_t)first_row * K;
        Y += (size_t)first_row * N;
        if (f.residual)
            f.residual += (size_t)first_row * N;
        const int b = blockIdx.x;
        const int t0 = b * tiles_q + min(b, tiles_r);
        const int T_out = tiles_q + (b < tiles_r ? 1 : 0);
        const int TW = gate ? 2 * T_out : T_out; // weight tiles of this workgroup, at most T
        // weight rows of the workgroup's tile i (past its tiles: the last one again, its sums not used; the last tile of
        // an N that is not a multiple of 16 is moved back to rows N-16 .. N-1)
        auto row0_of = [&](int i) {
            const int it = min(i, TW - 1);
            if (gate)
                return __builtin_amdgcn_readfirstlane(((it & 1) ? N : 0) + min((t0 + (it >> 1)) * 16, N - 16));
            return __builtin_amdgcn_readfirstlane(min((t0 + it) * 16, N - 16));
        };
        const int g_lo = (int)blockIdx.y * range_groups, g_hi = min(G, g_lo + range_groups); // this workgroup's part of K
        const int Gr = g_hi - g_lo;

        uint8_t* ring = smem + wave * WAVE_BYTES;
        uint8_t* sc = smem + KS_WAVES * WAVE_BYTES;

        // ---- (groups of 128) the scales of the range: asked for first, into LDS as rows of 32 words ---------------------------------------
        // Wavefront w fetches rows 2 w and 2 w + 1 of every tile, a half of the lanes each, from the 4-byte word at or below the
        // row's first group of the range (odd numbers of groups: every other row starts in the middle of one; N is even then).
        // Word i of row r lies at position i ^ 2 r: the sixteen rows of a tile are read without bank conflicts.
        if constexpr (QG == 0)
        {
            const int r = 2 * wave + (lane >> 5);
            const uint32_t word = min((uint32_t)((lane & 31) ^ (2 * r)), (uint32_t)(Gr >> 1));
            const uint32_t last_word = (((uint32_t)(gate ? 2 * N : N) * (uint32_t)G) >> 1) - 1u; // of the matrix
#pragma unroll
            for (int t = 0; t < T; ++t)
            {
                const uint32_t at = min((((uint32_t)(row0_of(t) + r) * (uint32_t)G + (uint32_t)g_lo) >> 1) + word, last_word);
                __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(reinterpret_cast<const uint8_t*>(S) + (size_t)at * 4),
                                                 (ks_lds_ptr_t)(sc + t * 2048 + wave * 256), 4, 0, 0);
            }
        }

        // ---- what each lane fetches -------------------------------------------------------------------------------------
        // weights: lane l the 16-byte piece (l & 3) ^ (r >> 2) of row r = l >> 2 of a tile's group
        // (8 bits: piece (l & 7) ^ (r >> 1) & 7 of row r = 8 c + l / 8 in load c)
        uint32_t w_off[NW];
        if constexpr (BITS == 8)
        {
#pragma unroll
            for (int c = 0; c < NW; ++c)
                w_off[c] = (uint32_t)(c * 8 + (lane >> 3)) * (uint32_t)ROW_BYTES + (uint32_t)(((lane & 7) ^ (((c * 8 + (lane >> 3)) >> 1) & 7)) << 4);
        }
        else
            w_off[0] = (uint32_t)(lane >> 2) * (uint32_t)ROW_BYTES + (uint32_t)(((lane & 3) ^ (lane >> 4)) << 4);
        const uint8_t* w_row[T];
#pragma unroll
        for (int t = 0; t < T; ++t)
            w_row[t] = Wq + (size_t)row0_of(t) * (size_t)ROW_BYTES;
        auto fetch_w = [&](int g, int t, uint8_t* to) {
#pragma unroll
            for (int c = 0; c < NW; ++c)
                __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(w_row[t] + (uint32_t)g * (uint32_t)(16 * BITS) + w_off[c]),
                                                 (ks_lds_ptr_t)(to + W_AT + t * WB + c * 1024), 16, 0, 0);
        };
        // activations: as row_block_fetch (nnf_device.h); rows past M: the last row again, blocks past its block: that block again
        const int last_block = (M - 1) >> 4;
        uint32_t a_off[4], a_off_last[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const int r = c * 4 + (lane >> 4);
            const uint32_t piece = (uint32_t)(((lane & 15) ^ r) * 16);
            a_off[c] = (uint32_t)r * (uint32_t)(K * 2) + piece;
            a_off_last[c] = (uint32_t)min(r, M - 1 - last_block * 16) * (uint32_t)(K * 2) + piece;
        }
        auto fetch_a = [&](int g, int mb, uint8_t* to) {
            const uint8_t* base = reinterpret_cast<const uint8_t*>(A) + (size_t)(min(mb, last_block) * 16) * (size_t)(K * 2) + (size_t)g * 256;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(base + (mb >= last_block ? a_off_last[c] : a_off[c])),
                                                 (ks_lds_ptr_t)(to + c * 1024), 16, 0, 0);
        };
        auto fetch_gamma = [&](int g, uint8_t* to) {
            if constexpr (RMS)
                __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(reinterpret_cast<const uint8_t*>(f.gamma) + (size_t)g * 256 + lane * 4),
                                                 (ks_lds_ptr_t)(to + G_AT), 4, 0, 0);
        };

        // QG: lane l of load i fetches word (64 i + l) % SPW of a group of 128's scales in row (64 i + l) / SPW of the tiles; of the zero points
        // likewise one of ZPB bytes (a byte load lands in the lane's four bytes; without a tensor the scales again, unused)
        // (128: an odd number of groups starts every other row in the middle of a word; N is even then, and the tiles' first rows start in none)
        const int GQ = QG ? K >> QG : 0; // scales of a row
        uint32_t s_at[NSL ? NSL : 1], z_at[NZL ? NZL : 1];
        if constexpr (QG != 0)
        {
            auto weight_row = [&](int at) { // row at % 16 of tile at / 16
                const int it = min(at >> 4, TW - 1);
                return (gate ? ((it & 1) ? N : 0) + min((t0 + (it >> 1)) * 16, N - 16) : min((t0 + it) * 16, N - 16)) + (at & 15);
            };
#pragma unroll
            for (int i = 0; i < NSL; ++i)
                s_at[i] = (uint32_t)weight_row((i * 64 + lane) / SPW) * (uint32_t)GQ + (uint32_t)((i * 64 + lane) % SPW) * 2u;
#pragma unroll
            for (int i = 0; i < NZL; ++i)
                z_at[i] = (uint32_t)weight_row((i * 64 + lane) / ZPB) * (uint32_t)(BITS == 8 ? GQ : (GQ + 1) >> 1) + (uint32_t)((i * 64 + lane) % ZPB);
        }
        auto fetch_s = [&](int g, uint8_t* to) {
            if constexpr (QG != 0)
            {
                const uint32_t s0 = (uint32_t)(g << (7 - QG)), z0 = (uint32_t)(BITS == 8 ? g << (7 - QG) : (g << (7 - QG)) >> 1);
#pragma unroll
                for (int i = 0; i < NSL; ++i)
                    __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(reinterpret_cast<const uint8_t*>(S) + (size_t)((s_at[i] + s0) & ~1u) * 2),
                                                     (ks_lds_ptr_t)(to + S_AT + i * 256), 4, 0, 0);
#pragma unroll
                for (int i = 0; i < NZL; ++i)
                    __builtin_amdgcn_global_load_lds((ks_global_ptr_t)(zps ? zps + (z_at[i] + z0) : reinterpret_cast<const uint8_t*>(S)),
                                                     (ks_lds_ptr_t)(to + S_AT + (NSL + i) * 256), 1, 0, 0);
            }
        };
        // groups of this wavefront: g_lo + wave + 8 c
        const int chunks = (Gr - wave + KS_WAVES - 1) / KS_WAVES;
        auto group_of = [&](int c) { return min(g_lo + wave + c * KS_WAVES, g_hi - 1); };
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            fetch_gamma(group_of(d), ring + d * SLOT);
#pragma unroll
            for (int p = 0; p < RB; ++p)
                fetch_a(group_of(d), p, ring + d * SLOT + p * ROW_BLOCK_BYTES);
            fetch_s(group_of(d), ring + d * SLOT);
#pragma unroll
            for (int t = 0; t < T; ++t)
                fetch_w(group_of(d), t, ring + d * SLOT);
        }
        if constexpr (QG == 0)
            wait_loads<D*(NG + 4 * RB + LW)>(); // the scales
        lds_barrier();

        const half_t clo = (half_t)(-(1024.0f + (float)zp)), chi = (half_t)(-(64.0f + (float)zp)); // exact
        const half2_t c_lo = {clo, clo}, c_hi = {chi, chi};
        floatx4 acc[T][MB];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[t][mb] = floatx4{0.f, 0.f, 0.f, 0.f};
        float ss[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
            ss[mb] = 0.f;

        // operand reads: piece kq * 4 + j of row col of a block, piece kq of row col of a tile's group
        uint32_t a_rd[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            a_rd[j] = (uint32_t)(col * 256 + (((kq * 4 + j) ^ col) << 4));
        uint32_t w_rd[NW];
        if constexpr (BITS == 8)
        {
#pragma unroll
            for (int c = 0; c < NW; ++c)
                w_rd[c] = (uint32_t)(col * 128 + (((2 * kq + c) ^ ((col >> 1) & 7)) << 4));
        }
        else
            w_rd[0] = (uint32_t)(col * 64 + ((kq ^ (col >> 2)) << 4));
        const int sc_first = ((col * G + g_lo) & 1) + wave; // place of the wavefront's first scale in row col (row0_of() * G is even)

        // activations and gamma in the order in which the weights are unpacked: the pairs of the nibble trick, 8 bits memory order
        auto operand_order = [](uintx4 v) { return BITS == 8 ? v : permute_a8(v); };
        // Loads of a wavefront in order: chunk by chunk [gamma] [MB blocks of activations] [QG: scales, zero points] [T tiles of weights];
        // those of chunk c + D (RB < MB: of the activations, the first RB blocks) are asked for during chunk c, each where its slot has just been
        // read.  Loads come back in order: the wait counts below are the loads that follow the one waited for.  AHEAD: the chunks still to come,
        // as far as they matter: below D nothing more is asked for.  Weights asked for ahead of the chunk's last activations
        // (RB < MB) need no wait of their own.
        int block = 0;                 // RB < MB: block p of the activations sits in place p % RB
        uint8_t* at_slot = ring;       // chunk c: slot c % D
        auto chunk = [&](int c, auto ahead) {
            constexpr int AHEAD = decltype(ahead)::value;
            constexpr bool FULL = AHEAD == D;
            constexpr int LATER = FULL ? (D - 1) * L : AHEAD * L; // of later chunks, asked for before this one began
            count_down_priority<AHEAD == 0>(chunks - 1 - c);
            const int g = group_of(c), gn = group_of(c + D);
            const uint8_t* slot = at_slot;
            uintx4 gm[4];
            uint32_t gamma_own = 0; // two of the group's 128, without their signs
            if constexpr (RMS)
            {
                wait_loads<LATER + 4 * RB + NS + LW>();
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    gm[j] = operand_order(*reinterpret_cast<const uintx4*>(slot + G_AT + kq * 64 + j * 16));
                gamma_own = *reinterpret_cast<const uint32_t*>(slot + G_AT + lane * 4) & 0x7fff7fffu;
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if constexpr (FULL)
                    fetch_gamma(gn, at_slot);
            }
            const int sc_place = sc_first + c * KS_WAVES;
            const uint8_t* sc_rd = sc + (uint32_t)(col * 128 + ((((sc_place >> 1) ^ (2 * col)) & 31) << 2) + (sc_place & 1) * 2);
            // block p of the chunk's activations from its place in the ring, in operand order; the place is refilled
            auto read_a = [&](auto p_c, uintx4(&a)[4]) {
                constexpr int p = decltype(p_c)::value;
                if constexpr (FULL)
                    wait_loads<LATER + 4 * (RB - 1) + (p < RB ? NS + LW + NG : 0)>();
                else
                {
                    constexpr int fetched = p < MB - RB ? p : MB - RB; // RB < MB: blocks asked for in this chunk so far
                    wait_loads<(p < RB ? LATER + 4 * (RB - 1 - p) + NS + LW + 4 * fetched : 4 * (p - 1 + RB < MB ? RB - 1 : MB - 1 - p))>();
                }
                uint8_t* at = at_slot + (RB == MB ? p : block) * ROW_BLOCK_BYTES;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    a[j] = *reinterpret_cast<const uintx4*>(at + a_rd[j]);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the slot has been read before it is refilled
                if constexpr (p + RB < MB)
                    fetch_a(g, p + RB, at);
                else if constexpr (FULL)
                    fetch_a(gn, p + RB - MB, at);
                block = block + 1 == RB ? 0 : block + 1;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    a[j] = operand_order(a[j]);
                    if constexpr (RMS)
                    {
                        ss[p] = dot2(as_half2(a[j].x), as_half2(a[j].x), ss[p]);
                        ss[p] = dot2(as_half2(a[j].y), as_half2(a[j].y), ss[p]);
                        ss[p] = dot2(as_half2(a[j].z), as_half2(a[j].z), ss[p]);
                        ss[p] = dot2(as_half2(a[j].w), as_half2(a[j].w), ss[p]);
                    }
                }
            };
            auto wait_w = [&](auto t_c) {
                constexpr int t = decltype(t_c)::value;
                if constexpr (RB == MB)
                    wait_loads<FULL ? D * L - NW : LATER + NW * (T - 1 - t)>();
            };
            // weights 8 j .. 8 j + 7 of a lane's 32: exact integers q - zp (QG: times their scale, rounded once), times gamma
            // lo, hi: -(1024 + zp) and -(64 + zp) in both halves
            // (8 bits: w4, w5 the eight bytes; a byte behind 0x64 is 1024 + b)
            auto unpack = [&](uint32_t w4, uint32_t w5, int j, half2_t lo, half2_t hi, half2_t scale2) {
                if constexpr (BITS == 8)
                {
                    half2_t b[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                    {
                        b[i] = as_half2(__builtin_amdgcn_perm(MAGIC, i < 2 ? w4 : w5, i & 1 ? 0x07030702u : 0x07010700u)) + lo;
                        b[i] *= scale2;
                    }
                    if constexpr (RMS)
                    {
                        b[0] *= as_half2(gm[j].x);
                        b[1] *= as_half2(gm[j].y);
                        b[2] *= as_half2(gm[j].z);
                        b[3] *= as_half2(gm[j].w);
                    }
                    return uintx4{as_u32(b[0]), as_u32(b[1]), as_u32(b[2]), as_u32(b[3])};
                }
                const uint32_t w8 = w4 >> 8;
                half2_t q0 = as_half2((w4 & MASK_LO) | MAGIC) + lo;    // (q0, q4) - zp
                half2_t q1 = as_half2((w4 & MASK_HI) | MAGIC_HI) + hi; // (q1, q5) - zp
                half2_t q2 = as_half2((w8 & MASK_LO) | MAGIC) + lo;    // (q2, q6) - zp
                half2_t q3 = as_half2((w8 & MASK_HI) | MAGIC_HI) + hi; // (q3, q7) - zp
                if constexpr (QG != 0)
                {
                    q0 *= scale2;
                    q1 *= scale2;
                    q2 *= scale2;
                    q3 *= scale2;
                }
                if constexpr (RMS)
                {
                    q0 *= as_half2(gm[j].x);
                    q1 *= as_half2(gm[j].y);
                    q2 *= as_half2(gm[j].z);
                    q3 *= as_half2(gm[j].w);
                }
                return uintx4{as_u32(q0), as_u32(q1), as_u32(q2), as_u32(q3)};
            };
            auto add_scaled = [](floatx4& to, const floatx4& sum, float scale) {
                to.x = __builtin_fmaf(sum.x, scale, to.x);
                to.y = __builtin_fmaf(sum.y, scale, to.y);
                to.z = __builtin_fmaf(sum.z, scale, to.z);
                to.w = __builtin_fmaf(sum.w, scale, to.w);
            };
            uintx4 areg[MB][4];
            unroll_for<0, MB>([&](auto p_c) { read_a(p_c, areg[decltype(p_c)::value]); });
            bool large = false;
            int x_first = 0; // (QG) 2^(x_first - e) goes onto scales below 2^(e - 14)
            if constexpr (RMS)
            {
                const uint32_t own_largest = max(gamma_own & 0xffffu, gamma_own >> 16);
                large = __builtin_amdgcn_ballot_w64(own_largest >= 0x6c00u) != 0; // 4096.0 and more: 15 times it may leave fp16
                const bool below_one = __builtin_amdgcn_ballot_w64(own_largest >= 0x3c00u) == 0;
                x_first = (large ? 14 : below_one ? 26 : 18) - BITS;
            }
            // QG: scale (low half) and zero point (eight bits) of the lane's 32 weights of every tile: group (128 g + 32 kq) >> QG of row col;
            // RMS: and e in the upper eight bits
            uint32_t scale_zero[QG ? T : 1];
            if constexpr (QG != 0)
            {
                if constexpr (RB == MB)
                    wait_loads<FULL ? (D - 1) * L + LW + NG + 4 * MB : LATER + LW>();
                const int sub = QG == 5 ? kq : QG == 6 ? kq >> 1 : g & 1;     // of the group of 128 (128: of the byte)
                const int half = QG == 7 ? (col * GQ + g) & 1 : sub & 1; // of the word
#pragma unroll
                for (int t = 0; t < T; ++t)
                {
                    const uint8_t* at = slot + S_AT + (((t * 16 + col) * SPW + (SPW == 2 ? sub >> 1 : 0)) << 2);
                    const int byte = BITS == 8 ? (QG == 7 ? 0 : sub) : QG == 5 ? sub >> 1 : 0;
                    const uint32_t zb = slot[S_AT + NSL * 256 + (((t * 16 + col) * ZPB + byte) << 2)];
                    const uint32_t z = !zps ? (uint32_t)zp : BITS == 8 ? zb : (zb >> ((sub & 1) * 4)) & 0xfu;
                    if constexpr (RMS)
                    {
                        // the row's scales of this group of 128: 2, or 4 in two words, or one half of a word
                        const uint32_t own = *reinterpret_cast<const uint32_t*>(at);
                        uint32_t all = own;
                        if constexpr (QG == 5)
                        {
                            const uint32_t other = *reinterpret_cast<const uint32_t*>(slot + S_AT + (((t * 16 + col) * SPW + 1 - (sub >> 1)) << 2));
                            all = max((own >> 16) & 0x7fffu, (other >> 16) & 0x7fffu) << 16 | max(own & 0x7fffu, other & 0x7fffu);
                        }
                        const uint32_t scale = half ? own >> 16 : own & 0xffffu;
                        const uint32_t largest = QG == 7 ? scale & 0x7fffu : max((all >> 16) & 0x7fffu, all & 0x7fffu);
                        scale_zero[t] = scale | (z << 16) | ((largest >> 10) << 24);
                    }
                    else
                        scale_zero[t] = *reinterpret_cast<const uint16_t*>(at + half * 2) | (z << 16);
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if constexpr (FULL)
                    fetch_s(gn, at_slot);
            }
            uintx4 wnext[NW];
            half_t snext = (half_t)0.f;
            auto read_w = [&](auto t_c) {
                constexpr int t = decltype(t_c)::value;
                wait_w(t_c);
#pragma unroll
                for (int c = 0; c < NW; ++c)
                    wnext[c] = *reinterpret_cast<const uintx4*>(slot + W_AT + t * WB + w_rd[c]);
                if constexpr (QG == 0)
                    snext = *reinterpret_cast<const half_t*>(sc_rd + t * 2048);
            };
            read_w(std::integral_constant<int, 0>());
            float sum_factor = 1.0f; // (RMS, scales on the sums) the reciprocal of what gamma is multiplied by
            if constexpr (RMS && QG == 0)
                if (large)
                {
                    sum_factor = 16.0f;
                    const half2_t sixteenth = {(half_t)0.0625f, (half_t)0.0625f};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        gm[j] = uintx4{as_u32(as_half2(gm[j].x) * sixteenth), as_u32(as_half2(gm[j].y) * sixteenth),
                                       as_u32(as_half2(gm[j].z) * sixteenth), as_u32(as_half2(gm[j].w) * sixteenth)};
                }
            unroll_for<0, T>([&](auto t_c) {
                constexpr int t = decltype(t_c)::value;
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                uint32_t ww[4 * NW];
#pragma unroll
                for (int c = 0; c < NW; ++c)
                {
                    ww[4 * c] = wnext[c].x;
                    ww[4 * c + 1] = wnext[c].y;
                    ww[4 * c + 2] = wnext[c].z;
                    ww[4 * c + 3] = wnext[c].w;
                }
                float scale = RMS ? (float)snext * sum_factor : (float)snext;
                if constexpr (FULL)
                    fetch_w(gn, t, at_slot);
                if constexpr (t + 1 < T)
                    read_w(std::integral_constant<int, (t + 1 < T ? t + 1 : 0)>());
                // (QG: scales differ within an MFMA's K: they are in the weights, and the accumulators take the sums as they are)
                half2_t lo = c_lo, hi = c_hi, scale2 = {};
                if constexpr (QG != 0)
                {
                    const uint32_t z2 = ((scale_zero[t] >> 16) & 0xffu) * 0x10001u, e = scale_zero[t] >> 24;
                    uint32_t s1 = scale_zero[t] & 0xffffu;
                    if constexpr (RMS)
                    {
                        s1 = __builtin_bit_cast(uint16_t, __builtin_amdgcn_ldexph(__builtin_bit_cast(half_t, (uint16_t)s1), x_first - (int)e));
                        scale = __builtin_bit_cast(float, ((uint32_t)(127 - x_first) + e) << 23); // 2^(e - x_first)
                    }
                    lo = as_half2(0xE400E400u | z2);
                    hi = as_half2(0xD400D400u | (z2 << 4));
                    scale2 = as_half2(s1 | (s1 << 16));
                }
                constexpr bool OWN_SUM = QG == 0 || RMS; // the group's sum, which meets a factor, or the accumulators themselves
                floatx4 sum[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    sum[mb] = OWN_SUM ? floatx4{0.f, 0.f, 0.f, 0.f} : acc[t][mb];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    const uintx4 bq = unpack(ww[NW * j], ww[NW * j + NW - 1], j, lo, hi, scale2);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                        sum[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, areg[mb][j]),
                                                                         __builtin_bit_cast(half8_t, bq), sum[mb], 0, 0, 0);
                }
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    if constexpr (OWN_SUM)
                        add_scaled(acc[t][mb], sum[mb], scale);
                    else
                        acc[t][mb] = sum[mb];
            });
            if constexpr (D > 1)
                at_slot = at_slot == ring + (D - 1) * SLOT ? ring : at_slot + SLOT;
        };
        __builtin_amdgcn_s_setprio(3);
        int c = 0;
        for (; c < chunks - D; ++c)
            chunk(c, std::integral_constant<int, D>());
        unroll_for<0, D>([&](auto i) { // the last D chunks, of which the last one has none ahead (fewer in all: nothing is waited for too little)
            constexpr int AHEAD = D - 1 - decltype(i)::value;
            if (c + AHEAD < chunks)
                chunk(c++, std::integral_constant<int, AHEAD>());
        });
        wait_loads<0>(); // (a wavefront without a group of its own has asked for one all the same)
        __syncthreads();

        // ---- the wavefronts' sums meet ------------------------------------------------------------------------------------
        // D layout: lane (n = col, kq), element e: row m = 16 mb + 4 kq + e
        float* sum_sq = reinterpret_cast<float*>(smem); // [8][16 MB]
        float* rstd = sum_sq + KS_WAVES * MB * 16;      // [16 MB]
        float* red = reinterpret_cast<float*>(smem + 4096);
        if constexpr (RMS)
        {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
            {
                ss[mb] += __shfl_xor(ss[mb], 16, 64);
                ss[mb] += __shfl_xor(ss[mb], 32, 64);
                if (kq == 0)
                    sum_sq[wave * (MB * 16) + mb * 16 + col] = ss[mb];
            }
            __syncthreads();
            if (tid < MB * 16)
            {
                float total = 0.f;
#pragma unroll
                for (int w = 0; w < KS_WAVES; ++w)
                    total += sum_sq[w * (MB * 16) + tid];
                rstd[tid] = 1.0f / __builtin_sqrtf(total / (float)K + f.rms_eps);
            }
        }
        const int n_tiles = (N + 15) / 16;
        // the sums of output tile `it`, block mb, lane `l` (rows 16 mb + 4 (l / 16) .. + 3, below M rounded up to a multiple of four) of a
        // range: where the ranges of K meet in scratch memory
        const int quads = gridDim.z == 1 ? (M + 3) >> 2 : MB * 4;
        auto partial_at = [&](int range, int it, int mb, int l) {
            return reinterpret_cast<unsigned long long*>(partial) +
                   (((((size_t)blockIdx.z * gridDim.y + range) * n_tiles + t0 + it) * quads + mb * 4 + (l >> 4)) * 16 + (l & 15)) * 2;
        };
        auto write_out = [&](int it, int mb, int l, const floatx4& s) {
            const int nn = min((t0 + it) * 16, N - 16) + (l & 15);
            // (a last tile moved back: these columns belong to the tile before it; a residual in place is added once)
            if (nn < (t0 + it) * 16)
                return;
            const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const int m = mb * 16 + (l >> 4) * 4 + e;
                if (m < M)
                    Y[(size_t)m * N + nn] =
                        finish_bias_residual(RMS ? f32_product(v[e], rstd[m]) : v[e], f.bias, nn, f.residual, (size_t)m * N + nn);
            }
        };
        unroll_for<0, (T + RT - 1) / RT>([&](auto round) {
            constexpr int first = decltype(round)::value * RT;
            if constexpr (first > 0)
                __syncthreads();
#pragma unroll
            for (int tt = 0; tt < RT; ++tt)
                if (first + tt < T)
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                        *reinterpret_cast<floatx4*>(red + ((wave * RT + tt) * MB + mb) * 256 + lane * 4) = acc[first + tt < T ? first + tt : 0][mb];
            __syncthreads();
            auto total = [&](int tt, int mb, int l) {
                floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < KS_WAVES; ++w)
                    s += *reinterpret_cast<const floatx4*>(red + ((w * RT + tt) * MB + mb) * 256 + l * 4);
                return s;
            };
            const int here = min(RT, TW - first);
            for (int o = tid; o < (gate ? here >> 1 : here) * (MB * 64); o += KS_WAVES * 64)
            {
                const int tt = (o >> 6) / MB, mb = (o >> 6) % MB; // (o & 63 == lane)
                if (gate)
                {
                    const floatx4 sg = total(2 * tt, mb, lane), su = total(2 * tt + 1, mb, lane);
                    const int it = (first >> 1) + tt;
                    const int nn = min((t0 + it) * 16, N - 16) + col;
                    const float vg[4] = {sg.x, sg.y, sg.z, sg.w}, vu[4] = {su.x, su.y, su.z, su.w};
                    if (nn >= (t0 + it) * 16)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                        {
                            const int m = mb * 16 + kq * 4 + e;
                            const float rs = RMS ? rstd[m] : 1.0f;
                            if (m < M)
                                Y[(size_t)m * N + nn] = finish_silu_gate(vg[e] * rs, vu[e] * rs);
                        }
                }
                else
                {
                    const floatx4 s = total(tt, mb, lane);
                    if (!partial)
                        write_out(first + tt, mb, lane, s);
                    else if (mb * 4 + kq < quads)
                    {
                        unsigned long long* to = partial_at((int)blockIdx.y, first + tt, mb, lane);
                        const unsigned long long* from = reinterpret_cast<const unsigned long long*>(&s);
                        __hip_atomic_store(to, from[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(to + 1, from[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            }
        });
        if constexpr (!RMS)
        {
            if (!partial)
                return;
            // ---- ranges of K: the last of the workgroups that share these tiles adds them up in order (as in
            // w4a16_mrows_any_kernel: stores at device scope, completed, then counted; nobody waits; the word is left zero) ----
            __builtin_amdgcn_s_waitcnt(vmcnt_only(0)); // (counts stores too)
            volatile uint32_t* arrived_before = reinterpret_cast<volatile uint32_t*>(smem);
            __syncthreads();
            if (tid == 0)
                *arrived_before = atomicAdd(sync + blockIdx.z * gridDim.x + blockIdx.x, 1u);
            __syncthreads();
            if (*arrived_before != gridDim.y - 1)
                return;
            const int ranges = (int)gridDim.y;
            for (int o = tid; o < TW * (MB * 64); o += KS_WAVES * 64)
            {
                const int it = (o >> 6) / MB, mb = (o >> 6) % MB;
                if (mb * 4 + kq >= quads)
                    continue;
                floatx4 s = {0.f, 0.f, 0.f, 0.f};
                for (int r0 = 0; r0 < ranges; r0 += 4) // (four ranges in flight, added in order)
                {
                    unsigned long long part[4][2];
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                    {
                        const unsigned long long* at = partial_at(min(r0 + d, ranges - 1), it, mb, lane);
                        part[d][0] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        part[d][1] = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        if (r0 + d < ranges)
                            s += *reinterpret_cast<const floatx4*>(&part[d][0]);
                }
                write_out(it, mb, lane, s);
            }
            if (tid == 0)
                atomicExch(sync + blockIdx.z * gridDim.x + blockIdx.x, 0u);
        }
    }

    namespace
    {
        template <int T, int MB, bool RMS, int QG, int BITS>
        hipError_t launch_kstream(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* Wq, const void* S,
                                  void* Y, int M, int N, int K, int zp, const GemvFusion& fusion, float* partial, uint32_t* sync, const void* zps)
        {
            auto kernel = &w4a16_kstream_kernel<T, MB, RMS, QG, BITS>;
            constexpr size_t lds = workspace::kstream_lds_bytes(T, MB, RMS, QG, BITS);
            static_assert(lds <= MAX_LDS_BYTES, "");
            static LdsGrant granted;
            const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), granted, (int)MAX_LDS_BYTES);
            if (e != hipSuccess)
                return e;
            const GemvFusionArgs args{(const half_t*)fusion.gamma, nullptr, (const half_t*)fusion.bias, (const half_t*)fusion.residual,
                                      fusion.rms_eps};
            const unsigned pack = (unsigned)(M | (zp << 13) | (fusion.gate ? 1 << 21 : 0)) |
                                  ((unsigned)(plan.ranges > 1 ? plan.range_groups : 1023) << 22);
            hipLaunchKernelGGL(kernel, dim3(plan.grid, plan.ranges, plan.row_blocks), dim3(KS_WAVES * 64), lds, stream,
                               (const half_t*)A, (const uint8_t*)Wq, (const half_t*)S, (half_t*)Y, N, K, plan.tiles_q | (plan.tiles_r << 16),
                               (int)pack, plan.ranges > 1 ? partial : nullptr, plan.ranges > 1 ? sync : nullptr, args,
                               (const uint8_t*)zps);
            return hipGetLastError();
        }
        template <int MB, int QG, int BITS>
        hipError_t launch_kstream_t(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* Wq, const void* S,
                                    void* Y, int M, int N, int K, int zp, const GemvFusion& fusion, float* partial, uint32_t* sync, const void* zps)
        {
            hipError_t e = hipErrorInvalidValue;
            unroll_for<1, workspace::KSTREAM_MAX_TILES + 1>([&](auto t) {
                if (plan.tiles != t.value)
                    return;
                if constexpr (workspace::kstream_built(t.value, MB, true, QG, BITS))
                    if (fusion.gamma)
                        e = launch_kstream<t.value, MB, true, QG, BITS>(stream, plan, A, Wq, S, Y, M, N, K, zp, fusion, partial, sync, zps);
                if constexpr (workspace::kstream_built(t.value, MB, false, QG, BITS))
                    if (!fusion.gamma)
                        e = launch_kstream<t.value, MB, false, QG, BITS>(stream, plan, A, Wq, S, Y, M, N, K, zp, fusion, partial, sync, zps);
            });
            return e;
        }
    } // namespace

    // QG: 0 groups of 128 and a scalar zero point, else the group's log2, with zero points from `zps` (or null: zp)
    template <int QG, int BITS = 4>
    hipError_t launch_w4a16_kstream_g(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* Wq, const void* S,
                                      void* Y, int M, int N, int K, int zp, const GemvFusion& fusion, float* partial, uint32_t* sync,
                                      const void* zps)
    {
        if (plan.tiles < 1 || (plan.ranges > 1 && (!partial || !sync || fusion.gate || fusion.gamma)) || fusion.rstd ||
            (fusion.gate && (fusion.bias || fusion.residual)))
            return hipErrorInvalidValue;
        hipError_t e = hipErrorInvalidValue;
        unroll_for<1, 5>([&](auto mb) {
            if (plan.row_tiles == mb.value)
                e = launch_kstream_t<mb.value, QG, BITS>(stream, plan, A, Wq, S, Y, M, N, K, zp, fusion, partial, sync, zps);
        });
        return e;
    }
} // namespace nnf
