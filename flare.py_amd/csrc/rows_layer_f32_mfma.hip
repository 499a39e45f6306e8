// Backward of one fp32 token-wise layer y = [x +] act(x W^T + b) over long rows, in one pass over the rows (pdebench/models/flare.py:45-59
// run as separate torch layers): dt = dy act'(t), dx = [dy +] dt W, and per workgroup the partial sums dW = dt^T x, db = column sums of
// dt, which one small launch adds up in a fixed order.  fp32 [T,C] rows, C in {64, 128}, products on v_mfma_f32_16x16x4_f32.
//
// The arrays a layer's backward cannot do without are dy, t, x in and dx out (134 MB for 65,536 rows of 128 channels: 27 us at this
// card's copy rate) and the two products are 4.3 GFLOP (28 us at its fp32 matrix rate), so both pipes are near their limit when they
// overlap.  As separate passes (slope, bias sums and copy; product; batched product of the weight gradient; sum over its slices;
// residual's sum) the rows crossed the memory eight times more.  A GELU layer of that size inside a block's step: 102 us in six
// launches before, 58 us in two now (53 + 5; without activation 72 / 51); 131,072 rows of 64 channels alone 89 / 43 us.  What is left
// above the floors: the matrix instructions (32 us at the 2 GHz this load runs at) and the vector instructions of the slopes hardly
// overlap, measured with either part left out.
//
// A workgroup is 16 waves and owns a contiguous token range, taken in tiles through two LDS buffers.  dx^T = W^T dt^T: a wave holds
// 16 columns of W as A operands in registers for the whole range, and a lane ends up with four consecutive channels of a row.
// dW: a wave owns a block of it in its accumulators for the whole range, both operands read from the tile.  While a tile is
// multiplied, the next one is turned into dt and stored into the other buffer; half of the waves do that before their products
// and half after, so that a SIMD's vector and matrix pipes work at the same time.
#include <algorithm>

#include "rows_f32.hpp"

namespace flare {

namespace {

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// the wave's LDS writes are done, then every wave's are; loads of the next tile stay in flight across it
__device__ __forceinline__ void tile_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int C> struct Shape;
template <> struct Shape<128> { static constexpr int TM = 32, DO = 2, DI = 2; };      // tile's tokens; 16-blocks of dW per wave
template <> struct Shape<64>  { static constexpr int TM = 64, DO = 1, DI = 1; };

template <int C, int ACT>
__global__ __launch_bounds__(1024) void rows_layer_bwd_kernel(RowsLayerArgs a)
{
    using S = Shape<C>;
    constexpr int TM = S::TM, P = C + 4, Q = C / 4;                  // pitch: 16 rows' quads meet different banks
    constexpr int VPT = TM * C / 4 / 1024;                           // quads of a tile per thread and array
    constexpr int IW = C / 16, TG = 16 / IW, GPW = TM / 16 / TG;     // waves along dx's channels, along its tokens; 16-token groups each
    constexpr int WO = C / 16 / S::DO;                               // waves along dW's rows
    static_assert(WO * (C / 16 / S::DI) == 16 && 1024 % Q == 0, "one wave per block of dW");
    extern __shared__ __attribute__((aligned(16))) float lds[];      // [2][dt | x][TM][P]

    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    const int64_t first = (int64_t)blockIdx.x * a.rows_per_wg;
    const int n_rows = (int)(a.T - first < a.rows_per_wg ? a.T - first : a.rows_per_wg);
    const int tiles = (n_rows + TM - 1) / TM;
    const float* dy = a.dy + first * C;
    const float* t = ACT != 0 ? a.t + first * C : nullptr;
    const float* x = a.x + first * C;

    // A operands of dx: W[o][i0 + c16], o = 16 j + 4 g + e
    const int i0 = 16 * (w % IW), tg = w / IW;
    f32x4 wa[C / 16];
    if (a.dx)
#pragma unroll
        for (int j = 0; j < C / 16; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) wa[j][e] = a.w[(16 * j + 4 * g + e) * C + i0 + c16];

    const int wo = 16 * S::DO * (w % WO), wi = 16 * S::DI * (w / WO);
    f32x4 dw[S::DO][S::DI], db = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int o = 0; o < S::DO; ++o)
#pragma unroll
        for (int i = 0; i < S::DI; ++i) dw[o][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 rv[VPT], rt[VPT], rx[VPT];
    auto fetch = [&](int r0) {                                        // rows past the range repeat its last one
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int c = tid + 1024 * k, row = min(r0 + c / Q, n_rows - 1);
            const int at = row * C + 4 * (c % Q);
            rv[k] = *reinterpret_cast<const f32x4*>(dy + at);
            if (ACT != 0) rt[k] = *reinterpret_cast<const f32x4*>(t + at);
            rx[k] = *reinterpret_cast<const f32x4*>(x + at);
        }
    };
    auto stage = [&](int r0, float* buf) {                            // ... and take no part
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int c = tid + 1024 * k, row = c / Q;
            const bool live = r0 + row < n_rows;
            f32x4 v = rv[k];
            if (ACT != 0)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= act_slope<ACT>(rt[k][r]);
            v = live ? v : f32x4{0.f, 0.f, 0.f, 0.f};
            db += v;
            *reinterpret_cast<f32x4*>(buf + row * P + 4 * (c % Q)) = v;
            *reinterpret_cast<f32x4*>(buf + (TM + row) * P + 4 * (c % Q)) = live ? rx[k] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // The residual's part of dx, requested before the rows of a later tile, so that waiting for it does not wait for those.  Loads
    // stand under no branch: behind one the compiler could not count them and would wait for all.
    f32x4 res[GPW];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto fetch_res = [&](int r0) {
#pragma unroll
        for (int k = 0; k < GPW; ++k)
            res[k] = *reinterpret_cast<const f32x4*>(dy + min(r0 + 16 * (tg * GPW + k) + c16, n_rows - 1) * C + i0 + 4 * g);
    };
    auto products = [&](int r0, const float* buf) {
        const float* bx = buf + TM * P;
        if (a.dx) {
#pragma unroll
            for (int k = 0; k < GPW; ++k) {
                const int row = 16 * (tg * GPW + k) + c16;
                f32x4 acc[2] = {zero, zero};
#pragma unroll
                for (int j = 0; j < C / 16; ++j) {
                    const f32x4 b = *reinterpret_cast<const f32x4*>(buf + row * P + 16 * j + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e % 2] = mma4(wa[j][e], b[e], acc[e % 2]);
                }
                const f32x4 v = acc[0] + acc[1] + (a.add ? res[k] : zero);
                if (r0 + row < n_rows) *reinterpret_cast<f32x4*>(a.dx + (first + r0 + row) * C + i0 + 4 * g) = v;
            }
        }
#pragma unroll
        for (int t0 = 0; t0 < TM; t0 += 16) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int row = t0 + 4 * g + s;
                float ao[S::DO], bi[S::DI];
#pragma unroll
                for (int o = 0; o < S::DO; ++o) ao[o] = buf[row * P + wo + 16 * o + c16];
#pragma unroll
                for (int i = 0; i < S::DI; ++i) bi[i] = bx[row * P + wi + 16 * i + c16];
#pragma unroll
                for (int o = 0; o < S::DO; ++o)
#pragma unroll
                    for (int i = 0; i < S::DI; ++i) dw[o][i] = mma4(ao[o], bi[i], dw[o][i]);
            }
        }
    };

    constexpr int BUF = 2 * TM * P;
    fetch(0);
    stage(0, lds);
    if (w >= 8) fetch_res(0);
    fetch(TM);
    tile_barrier();
    if (w < 8) {
        for (int i = 0; i + 1 < tiles; ++i) {
            fetch_res(i * TM);
            stage((i + 1) * TM, lds + (~i & 1) * BUF);
            fetch((i + 2) * TM);
            products(i * TM, lds + (i & 1) * BUF);
            tile_barrier();
        }
        fetch_res((tiles - 1) * TM);
    } else {
        for (int i = 0; i + 1 < tiles; ++i) {
            products(i * TM, lds + (i & 1) * BUF);
            stage((i + 1) * TM, lds + (~i & 1) * BUF);
            fetch_res((i + 1) * TM);
            fetch((i + 2) * TM);
            tile_barrier();
        }
    }
    products((tiles - 1) * TM, lds + ((tiles - 1) & 1) * BUF);
    tile_barrier();

    float* out = a.dw_part + (size_t)blockIdx.x * C * C;
#pragma unroll
    for (int o = 0; o < S::DO; ++o)
#pragma unroll
        for (int i = 0; i < S::DI; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(wo + 16 * o + 4 * g + r) * C + wi + 16 * i + c16] = dw[o][i][r];
    if (a.db_part) {                                                  // thread tid owns the four channels of quad tid % Q in every row
        f32x4* red = reinterpret_cast<f32x4*>(lds);
        red[tid] = db;
        tile_barrier();
        if (tid < Q) {
            f32x4 s = red[tid];
            for (int k = tid + Q; k < 1024; k += Q) s += red[k];
            *reinterpret_cast<f32x4*>(a.db_part + (size_t)blockIdx.x * C + 4 * tid) = s;
        }
    }
}

template <int C> hipError_t launch_c(int act, const RowsLayerArgs& a, unsigned grid, hipStream_t st)
{
    const size_t lds = (size_t)4 * Shape<C>::TM * (C + 4) * sizeof(float);
    return with_row_act(act, [&](auto ac) {
        auto kern = rows_layer_bwd_kernel<C, decltype(ac)::value>;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(1024), lds, st, a);
    });
}

}  // namespace

bool rows_layer_bwd_supported(int C) { return C == 64 || C == 128; }

// Rows of a workgroup: an equal share of the compute units' (one workgroup each: its 16 waves hold 74 to 119 registers a lane, and two
// workgroups would need 64; of the LDS the two buffers take 70 of 160 KB), a multiple of the 16 rows a product takes, and not fewer
// than 64, below which writing the partial dW costs more than the rows.
static int64_t rows_per_wg(int64_t T)
{
    const int64_t share = (T + device_cus() - 1) / device_cus();
    return std::max<int64_t>(64, (share + 15) / 16 * 16);
}
int rows_layer_bwd_parts(int64_t T)
{
    const int64_t per = rows_per_wg(T);
    return (int)((T + per - 1) / per);
}

hipError_t launch_rows_layer_bwd(int act, const RowsLayerArgs& a0, float* dw, float* db, hipStream_t st)
{
    RowsLayerArgs a = a0;
    a.rows_per_wg = rows_per_wg(a.T);
    const unsigned grid = (unsigned)rows_layer_bwd_parts(a.T);
    const hipError_t e = a.C == 128 ? launch_c<128>(act, a, grid, st) : launch_c<64>(act, a, grid, st);
    return e != hipSuccess ? e : launch_sum_two_parts(a.dw_part, dw, (int64_t)a.C * a.C, a.db_part, db, a.C, (int)grid, st);
}

}  // namespace flare
