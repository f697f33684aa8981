// Host side of one tile height of the fp16 x int4 tile GEMM (w4a16_gemm_sk.h): picks the instantiation for the
// epilogue asked for and launches it.  Included by one translation unit per tile height, so that they compile in
// parallel.
#pragma once

#include "w4a16_gemm_sk.h"

namespace nnf
{
    namespace gemm_sk
    {
        template <class T, bool GATE, bool BIAS, bool RESID, bool RMS, int QG, bool ODD>
        hipError_t launch_product(hipStream_t stream, const SkGemmParams& p, int grid)
        {
            auto kernel = &w4a16_gemm_sk_kernel<T::TM, T::TN, T::NW, T::KH, GATE, BIAS, RESID, RMS, QG, ODD>;
            if (T::LDS_BYTES > 48 * 1024)
            {
                static LdsGrant granted;
                const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), granted, T::LDS_BYTES);
                if (e != hipSuccess)
                    return e;
            }
            launch_sk_kernel<T>(kernel, grid, stream, p);
            return hipGetLastError();
        }

        template <class T, bool GATE, bool BIAS, bool RESID, bool RMS, int QG = 0>
        hipError_t launch_instance(hipStream_t stream, const SkGemmParams& p, int grid)
        {
            if constexpr (!T::SHARED) // (even multiples of 128 only, too)
                return launch_product<T, GATE, BIAS, RESID, RMS, QG, false>(stream, p, grid);
            else
            {
                const hipError_t e = (p.K & 128) ? launch_product<T, GATE, BIAS, RESID, RMS, QG, true>(stream, p, grid)
                                                 : launch_product<T, GATE, BIAS, RESID, RMS, QG, false>(stream, p, grid);
                if (e != hipSuccess || !p.partial || p.sync)
                    return e;
                // tiles shared by several workgroups: their parts are added and finished by a second launch (unless the
                // workgroups did it themselves: p.sync); it does not depend on the block parameters
                using Parts = Tile<T::TM, T::TN, T::NW, T::KH>;
                constexpr int ROUNDS = T::TM; // blocks of 32 rows
                hipLaunchKernelGGL((w4a16_gemm_sk_fixup_kernel<Parts, GATE, BIAS, RESID, RMS>), dim3(p.tiles_m * p.tiles_n * ROUNDS * T::NW),
                                   dim3(64), 0, stream, p, grid);
                return hipGetLastError();
            }
        }

        template <class T>
        hipError_t launch_tile_height(hipStream_t stream, const SkGemmParams& p, int grid, bool gate)
        {
            const bool hb = p.bias != nullptr, hr = p.residual != nullptr, rms = p.gamma != nullptr;
            if (gate)
                return rms ? launch_instance<T, true, false, false, true>(stream, p, grid)
                           : launch_instance<T, true, false, false, false>(stream, p, grid);
            if (hb && hr)
                return rms ? launch_instance<T, false, true, true, true>(stream, p, grid)
                           : launch_instance<T, false, true, true, false>(stream, p, grid);
            if (hb)
                return rms ? launch_instance<T, false, true, false, true>(stream, p, grid)
                           : launch_instance<T, false, true, false, false>(stream, p, grid);
            if (hr)
                return rms ? launch_instance<T, false, false, true, true>(stream, p, grid)
                           : launch_instance<T, false, false, true, false>(stream, p, grid);
            return rms ? launch_instance<T, false, false, false, true>(stream, p, grid)
                       : launch_instance<T, false, false, false, false>(stream, p, grid);
        }
        // the forms without SiLU-gate (128-wide tiles have none)
        template <class T>
        hipError_t launch_tile_height_plain(hipStream_t stream, const SkGemmParams& p, int grid)
        {
            const bool hb = p.bias != nullptr, hr = p.residual != nullptr, rms = p.gamma != nullptr;
            if (hb && hr)
                return rms ? launch_instance<T, false, true, true, true>(stream, p, grid)
                           : launch_instance<T, false, true, true, false>(stream, p, grid);
            if (hb)
                return rms ? launch_instance<T, false, true, false, true>(stream, p, grid)
                           : launch_instance<T, false, true, false, false>(stream, p, grid);
            if (hr)
                return rms ? launch_instance<T, false, false, true, true>(stream, p, grid)
                           : launch_instance<T, false, false, true, false>(stream, p, grid);
            return rms ? launch_instance<T, false, false, false, true>(stream, p, grid)
                       : launch_instance<T, false, false, false, false>(stream, p, grid);
        }
        // other block parameters (QG = log2 of the group size; zero points per (row, group) when p.zps is set): the
        // plain product; tile_rows x tile_cols as sk_tile_shape chooses them for it
        template <int QG, bool EIGHT>
        hipError_t launch_low_tiles_q(hipStream_t stream, const SkGemmParams& p, int grid, int tile_rows, int tile_cols)
        {
            if (tile_cols == 128)
                return tile_rows == 128 ? launch_instance<TileOf<128, 128, EIGHT>, false, false, false, false, QG>(stream, p, grid)
                                        : launch_instance<TileOf<64, 128, EIGHT>, false, false, false, false, QG>(stream, p, grid);
            return tile_rows == 128 ? launch_instance<TileOf<128, 256, EIGHT>, false, false, false, false, QG>(stream, p, grid)
                                    : hipErrorInvalidValue; // (64 x 256: SiLU-gate only)
        }
        template <int QG>
        hipError_t launch_tiles_q(hipStream_t stream, const SkGemmParams& p, int grid, int tile_rows, int tile_cols, bool eight)
        {
            if (tile_rows == 64 || tile_rows == 128)
                return eight ? launch_low_tiles_q<QG, true>(stream, p, grid, tile_rows, tile_cols)
                             : launch_low_tiles_q<QG, false>(stream, p, grid, tile_rows, tile_cols);
            if (tile_rows == 256)
                return tile_cols == 128 ? launch_instance<TileOf<256, 128>, false, false, false, false, QG>(stream, p, grid)
                                        : launch_instance<TileOf<256, 256>, false, false, false, false, QG>(stream, p, grid);
            return tile_rows == 32 && tile_cols == 256 ? launch_instance<TileOf<32, 256>, false, false, false, false, QG>(stream, p, grid)
                                                       : hipErrorInvalidValue;
        }
    } // namespace gemm_sk

    // groups of 32 / 64 / 128 with p.zps or p.zp (w4a16_gemm_sk_q5.hip ... _q7.hip)
    hipError_t launch_gemm_sk_q5(hipStream_t stream, const SkGemmParams& p, int grid, int tile_rows, int tile_cols, bool eight);
    hipError_t launch_gemm_sk_q6(hipStream_t stream, const SkGemmParams& p, int grid, int tile_rows, int tile_cols, bool eight);
    hipError_t launch_gemm_sk_q7(hipStream_t stream, const SkGemmParams& p, int grid, int tile_rows, int tile_cols, bool eight);
    // one per tile height (w4a16_gemm_sk_32.hip ... _256.hip); narrow: tiles 128 wide, plain product, bias, residual, RMSNorm;
    // eight: on eight wavefronts
    hipError_t launch_gemm_sk_64_narrow(hipStream_t stream, const SkGemmParams& p, int grid, bool eight);
    hipError_t launch_gemm_sk_128_narrow(hipStream_t stream, const SkGemmParams& p, int grid, bool eight);
    hipError_t launch_gemm_sk_256_narrow(hipStream_t stream, const SkGemmParams& p, int grid);
    hipError_t launch_gemm_sk_32(hipStream_t stream, const SkGemmParams& p, int grid, bool gate);
    hipError_t launch_gemm_sk_64(hipStream_t stream, const SkGemmParams& p, int grid, bool gate, bool eight);
    hipError_t launch_gemm_sk_128(hipStream_t stream, const SkGemmParams& p, int grid, bool gate, bool eight);
    hipError_t launch_gemm_sk_256(hipStream_t stream, const SkGemmParams& p, int grid, bool gate);
    // tiles of 128 x 192, whole ones (w4a16_gemm_sk_192.hip)
    hipError_t launch_gemm_sk_192(hipStream_t stream, const SkGemmParams& p, int grid, bool gate);
} // namespace nnf
