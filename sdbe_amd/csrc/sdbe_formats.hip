// Input-format variants of the stage: the 2015-format B-engine reorder.
//
// sdbe_reorder_2015 restates reorderTz_smem
// (software/prototyping/cuda/kernel_template.py:107-164) as one launch over all
// output frames.  Workgroup = (128-channel tile, 32-snapshot quarter, output
// frame); 256 threads move 128 x 32 complex values through an LDS tile:
//   read:  lanes run along the input snapshots of two channels (the input is
//          channel-major, snapshots contiguous), all 16 loads of a thread in
//          flight together;
//   write: lanes run along the channels of one output snapshot (output rows are
//          channel-contiguous), 512 B per wave-store.
// Pure data movement: HBM-bound, 2 x 8 B per element.  Output rows are 16385
// values, so a row's runs start anywhere in a 128-byte line and the reads of the
// shifted channels and of frame f + 1 do too.  Neighbouring tiles of a frame
// therefore run one after another on one XCD (an eighth of the channels each),
// whose L2 puts the parts of a line together, and the runs a tile writes are 1 KB
// long.  39 frames, 1.29 GB: 261 us = 4.95 TB/s, a plain copy of as many bytes
// 252.  64 x 64 tiles, their neighbours on other XCDs and 4 loads in flight: 326;
// on one XCD, 16 in flight: 293; 64 x 32: 266; 128 x 64: 261; 32 x 128: 275;
// 128 x 128: 262.  Non-temporal loads or stores cost 2 to 8%: they keep the parts
// of a line apart.
#include <hip/hip_runtime.h>

#include "../../include/sdbe_formats.h"

namespace {

constexpr int NCH = SDBE_REORDER2015_CHANNELS;
constexpr int NSN = SDBE_REORDER2015_SNAPSHOTS;
constexpr int SPLIT = SDBE_REORDER2015_SPLIT;
constexpr int CT = 128, ST = 32;                    // channels and snapshots of a tile
constexpr int HT = NSN / ST;                        // tiles along the snapshots
constexpr int TILES = (NCH / CT) * HT;              // tiles of one output frame
constexpr int WG = 256, RR = WG / ST, WR = WG / CT; // rows read / written at a time
static_assert(TILES % 8 == 0, "an eighth of the channels per XCD");

__global__ void __launch_bounds__(WG)
k_reorder_2015(const float2 *__restrict__ in, int n_frames, float2 *__restrict__ out) {
    __shared__ float2 tile[CT][ST + 1];
    const int t = threadIdx.x;
    const int L = (blockIdx.x & 7) * (TILES / 8) + (blockIdx.x >> 3);
    const int c0 = L / HT * CT;                // channel tile
    const int s0 = L % HT * ST;                // first output snapshot
    const int f = blockIdx.z;                  // output frame, < n_frames - 1
    // read: j = output snapshot in the tile, channel rows i + RR k
    {
        const int j = t % ST, i = t / ST, s = s0 + j;
        const int fi = f + (s >= SPLIT ? 1 : 0);
        float2 v[CT / RR];
#pragma unroll
        for (int k = 0; k < CT / RR; ++k) {
            const int c = c0 + i + RR * k;
            const int si = ((c >> 2) & 1) == 0 ? ((s + 2) & (NSN - 1)) : s;
            v[k] = in[((size_t)c * n_frames + fi) * NSN + si];
        }
#pragma unroll
        for (int k = 0; k < CT / RR; ++k) tile[i + RR * k][j] = v[k];
    }
    __syncthreads();
    // write: i = channel in the tile, snapshots j + WR k
    {
        const int i = t % CT, j = t / CT;
#pragma unroll
        for (int k = 0; k < ST / WR; ++k) {
            float2 *row = out + ((size_t)f * NSN + s0 + j + WR * k) * (NCH + 1);
            row[c0 + i] = tile[i][j + WR * k];
            if (c0 + CT == NCH && i == 0) row[NCH] = make_float2(0.f, 0.f);
        }
    }
}

}  // namespace

extern "C" int sdbe_reorder_2015(const void *d_in, int32_t n_frames, void *d_out, void *stream) {
    if (!d_in || !d_out || n_frames < 2) return SDBE_ERR_ARG;
    // in and out must not overlap
    const char *ib = (const char *)d_in, *ob = (const char *)d_out;
    const size_t in_bytes = (size_t)NCH * n_frames * NSN * sizeof(float2);
    const size_t out_bytes = (size_t)(n_frames - 1) * NSN * (NCH + 1) * sizeof(float2);
    if (ib < ob + out_bytes && ob < ib + in_bytes) return SDBE_ERR_ARG;
    if (n_frames - 1 > 65535) return SDBE_ERR_ARG;   // grid z limit
    hipLaunchKernelGGL(k_reorder_2015, dim3(TILES, 1, n_frames - 1), dim3(WG), 0,
                       (hipStream_t)stream, (const float2 *)d_in, (int)n_frames, (float2 *)d_out);
    return hipGetLastError() == hipSuccess ? SDBE_OK : SDBE_ERR_HIP;
}
