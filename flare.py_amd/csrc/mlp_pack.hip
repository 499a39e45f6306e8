// Operands of the token-wise MLP launches from the parameters, in one launch: the [L,C,C] tiles in the compute type, the LDS
// images of the tiles and of their transposes (what the backward loads straight into its weight slots; the position
// formula is in include/flare_hip.h) and the fp32 bias rows.  Every parameter is read where it lies (row stride, element
// type and row count per tile), so nothing is stacked or converted beforehand.
//
// A few hundred KB: what it costs is the launch.  The same from torch calls (stack, cast, stack, two index expansions and
// an indexed read) was six launches per stack; an 8-block model's training step on 4096 points packs 34 stacks
// (4.27 -> 3.68 ms replayed, about 190 launches fewer), a block's k and v stacks in one launch.
#include "common.hpp"

namespace flare {

namespace {

__device__ __forceinline__ float load_as_float(const void* p, int64_t i, int dt)
{
    if (dt == 0) return static_cast<const float*>(p)[i];
    if (dt == 1) return (float)static_cast<const __bf16*>(p)[i];
    return (float)static_cast<const _Float16*>(p)[i];
}

// thread = four consecutive 16-bit outputs of one array: blockIdx.z = 0 the tiles, 1 their images, 2 the transposes' images;
// a.tiled: 0 the tiles, 1 the transposes, both with every matrix operand's 64 lanes x 16 bytes in one piece
template <typename V>
__global__ __launch_bounds__(256) void mlp_pack_kernel(MlpPackArgs a)
{
    typedef V vec4 __attribute__((ext_vector_type(4)));
    const int l = blockIdx.y, what = blockIdx.z;
    const int C = a.C;
    if (l == a.L) {          // further rows (a block's latents): as a cast of its own every training step it cost 6 us a block
        if (what != 0) return;
        const int64_t n = a.n_rows * a.cols_out;
        for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; e < n; e += (int64_t)gridDim.x * 1024) {
            const int64_t row = e / a.cols_out;
            const int col = (int)(e % a.cols_out);
            vec4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = col + j < a.cols ? (V)load_as_float(a.rows_src, row * a.cols + col + j, a.rows_dtype) : (V)0.f;
            *reinterpret_cast<vec4*>(reinterpret_cast<V*>(a.rows_out) + e) = v;
        }
        return;
    }
    V* out = reinterpret_cast<V*>(what == 0 ? a.w : what == 1 && !a.tiled ? a.w_img : a.wt_img);
    const bool transposed = what == (a.tiled ? 1 : 2);
    const int e = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
    if (out && e < C * C) {
        int row = e / C, rem = e % C;
        int col = rem;
        if (a.tiled) {      // [C / 16 row blocks][C / 32 k-steps][4 lane groups][16 rows][8 columns]
            row = e / (16 * C) * 16 + (e >> 3) % 16;
            col = e % (16 * C) / 512 * 32 + (e >> 7) % 4 * 8 + (e & 7);
        } else if (what > 0) {
            const int key = (row & 15) >> (C == 128 ? 0 : C == 64 ? 1 : 2);
            const int c = (rem >> 3) ^ key, half = (rem >> 2) & 1;
            col = 8 * (4 * (c >> 2) + 2 * half + ((c & 3) >> 1)) + 4 * (c & 1);
        }
        vec4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = transposed ? col + j : row, k = transposed ? row : col + j;      // [out][in] element of the tile
            v[j] = r < a.rows[l] ? (V)load_as_float(a.src[l], (int64_t)r * a.ld[l] + k, a.src_dtype[l]) : (V)0.f;
        }
        *reinterpret_cast<vec4*>(out + (size_t)l * C * C + e) = v;
    }
    if (what == 0 && blockIdx.x == 0 && (int)threadIdx.x < C) {
        const int c = threadIdx.x;
        a.bias[(size_t)l * C + c] = a.bsrc[l] && c < a.rows[l] ? load_as_float(a.bsrc[l], c, a.b_dtype[l]) : 0.f;
    }
}

}  // namespace

hipError_t launch_mlp_pack(const MlpPackArgs& a, int w_dtype, hipStream_t st)
{
    const dim3 grid((unsigned)((a.C * a.C / 4 + 255) / 256), (unsigned)(a.L + (a.rows_src ? 1 : 0)), a.tiled ? (a.wt_img ? 2 : 1) : a.w_img ? 3 : 1);
    if (w_dtype == 1) hipLaunchKernelGGL(mlp_pack_kernel<__bf16>, grid, dim3(256), 0, st, a);
    else              hipLaunchKernelGGL(mlp_pack_kernel<_Float16>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace flare
