// The token-wise MLP chain and its backward for launches of few tokens (bf16 / f16 weights, C in {32, 64, 128}): the
// contracts of mlp_mfma.hip (chain mode, head-padded rows) and of mlp_bwd_mfma.hip, the backward for one chain or for two that
// read the same rows through the same norm (the k and v projections of a block).
//
// With few tokens nothing but latency counts.  The many-token kernels give a wave 16 tokens and all C output channels: every
// layer waits for its C x C weight tile to travel through LDS behind a barrier and then runs C / 16 products one after the
// other -- about 3.8 us per layer at C = 128, whatever the token count.  Here a workgroup owns 16 tokens and has C / 16
// waves, each of which owns 16 output channels: its share of every layer's weights (C / 32 registers quads per layer) is
// requested at the very start, straight into registers, and a layer is one LDS exchange of the 16 x C activations (each wave
// writes its 16 channels in B-operand order, one barrier, everybody reads all of them) and C / 32 products.  The price is
// that every 16 tokens read all weights again from the L2, which is what ends the range this is used in.
// Two chains that read the same rows (a block's k and v projections) are one launch each way: with the
// forward pair, one packing launch a block and the residual's gradient added here, the step of 8 blocks went from 1689 to 1608 us.
// 4096 tokens, C = 128, five layers, in a replayed graph: forward 17.3 -> 9.1 us, backward 37.6 + 8.6 + 4.6 (norm sums) -> 16.2
// us, two chains of it 102 -> 27 us; the 8-block model's training step 3.68 -> 1.81 ms (with one launch for the sums over
// partial results and 256-token ranges in mlp_wgrad_mfma.hip).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace flare {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mf;
template <> struct Mf<bf16_t> {
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi)
    {
        bf16x2 v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float lo(uint32_t p) { return __uint_as_float(p << 16); }
    static __device__ __forceinline__ float hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }
};
template <> struct Mf<f16_t> {
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi)
    {
        f16x2 v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float lo(uint32_t p) { return (float)__builtin_bit_cast(f16x2, p)[0]; }
    static __device__ __forceinline__ float hi(uint32_t p) { return (float)__builtin_bit_cast(f16x2, p)[1]; }
};

// element type of a row (0 f32, 1 bf16, 2 f16): one uniform branch, not one per load
template <typename F> __device__ __forceinline__ void with_dtype(int dt, F&& f)
{
    if (dt == 0) f(std::integral_constant<int, 0>{});
    else if (dt == 1) f(std::integral_constant<int, 1>{});
    else f(std::integral_constant<int, 2>{});
}
template <int DT> __device__ __forceinline__ f32x4 load4(const void* base, int64_t e)
{
    if constexpr (DT == 0) {
        return *reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + e);
    } else {
        const uint2 r = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + e);
        using M_ = Mf<std::conditional_t<DT == 1, bf16_t, f16_t>>;
        return f32x4{M_::lo(r.x), M_::hi(r.x), M_::lo(r.y), M_::hi(r.y)};
    }
}
template <int DT> __device__ __forceinline__ void store4(void* base, int64_t e, f32x4 v)
{
    if constexpr (DT == 0) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(base) + e) = v;
    } else {
        using M_ = Mf<std::conditional_t<DT == 1, bf16_t, f16_t>>;
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(base) + e) = make_uint2(M_::pack2(v[0], v[1]), M_::pack2(v[2], v[3]));
    }
}

// a value as it is after a store and a load of the type
template <int DT> __device__ __forceinline__ f32x4 round4(f32x4 v)
{
    if constexpr (DT == 0) {
        return v;
    } else {
        using M_ = Mf<std::conditional_t<DT == 1, bf16_t, f16_t>>;
        const uint32_t a = M_::pack2(v[0], v[1]), b = M_::pack2(v[2], v[3]);
        return f32x4{M_::lo(a), M_::hi(a), M_::lo(b), M_::hi(b)};
    }
}

__device__ __forceinline__ float tok_sum(float v)      // sum over the 4 lane groups that share a token
{
    v = sum_xor16(v);
    v = sum_xor32(v);
    return v;
}

// act(t) and its derivative as in mlp_bwd_mfma.hip, without a branch on the kind: tanh-GELU has the gate
// sigmoid(t (1.5957691 + 0.0713548 t^2)), SiLU sigmoid(t), so the kinds differ in four coefficients (in log2 units for the
// gate).  The square is kept finite: a zero coefficient times infinity would not be zero.
struct ActCoef { float g0, g1, s0, s1; };
__device__ __forceinline__ ActCoef act_coef(int kind)
{
    return kind == 0 ? ActCoef{2.3022081f, 0.10294324f, 1.5957691f, 0.2140645f} : ActCoef{kLog2e, 0.f, 1.f, 0.f};
}
__device__ __forceinline__ void act_and_slope(const ActCoef& k, float t, float& value, float& slope)
{
    const float t2 = fminf(t * t, 3.0e38f);
    const float gate = __builtin_amdgcn_rcpf(1.f + fast_exp2(-t * fmaf(k.g1, t2, k.g0)));
    value = t * gate;
    slope = gate * fmaf(t * (1.f - gate), fmaf(k.s1, t2, k.s0), 1.f);
}

// LDS writes of this wave are done, then every wave's are.  The bare barrier: __syncthreads() would wait for the weights and
// rows in flight as well.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One 16-token activation tile on its way to every wave, in B-operand order: k-step ks, lane (g, c16) = token c16, channels
// 32 ks + 8 g .. + 7 (the accumulators of wave w hold channels 16 w + 4 g .. + 3).  Two buffers alternate: a wave is at most one barrier ahead of another.
template <int C> struct Exchange {
    static constexpr int KS = C / 32;
    u32x4 q[2][KS][64];
};
template <int C>
__device__ __forceinline__ void publish(Exchange<C>& x, int buf, int w, int lane, uint32_t p0, uint32_t p1)
{
    const int g = lane >> 4, to = 16 * (2 * (w & 1) + (g >> 1)) + (lane & 15);
    *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(&x.q[buf][w >> 1][to]) + 8 * (g & 1)) = make_uint2(p0, p1);
    lds_barrier();
}

// A published tile leaves as 16-bit rows [T,C]: wave ks < C / 32 stores its k-step, a token's four lanes cover 64 contiguous bytes.
template <int C>
__device__ __forceinline__ void store_rows(const Exchange<C>& x, int buf, int w, int lane, uint16_t* base, int64_t t, bool live)
{
    if (w < C / 32 && live) *reinterpret_cast<u32x4*>(base + t * C + 32 * w + 8 * (lane >> 4)) = x.q[buf][w][lane];
}

// Matrix operand of 16 output channels: the tiled weights keep the 64 lanes x 16 bytes of one operand in one piece (row by row,
// 16 rows of 64 bytes per load, the forward took 16 us instead of 9)
template <int C>
__device__ __forceinline__ u32x4 operand(const uint16_t* wts, size_t tile, int w, int ks, int lane)
{
    return *reinterpret_cast<const u32x4*>(wts + tile * C * C + ((w * (C / 32) + ks) * 64 + lane) * 8);
}

// mean and 1/std of the lane's token, from the whole row (every wave reads it: 16 rows, mostly from the L1)
template <int C>
__device__ __forceinline__ void row_stats(const f32x4 (&x)[C / 16], int norm, float eps, float& mean, float& rstd)
{
    float s = 0.f;
#pragma unroll
    for (int ft = 0; ft < C / 16; ++ft) s += x[ft][0] + x[ft][1] + x[ft][2] + x[ft][3];
    const float rowmean = tok_sum(s) * (1.f / C);
    mean = norm == 1 ? rowmean : 0.f;
    float ss = 0.f;
#pragma unroll
    for (int ft = 0; ft < C / 16; ++ft)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float d = x[ft][r] - mean;
            ss = fmaf(d, d, ss);
        }
    rstd = rsqrtf(tok_sum(ss) * (1.f / C) + eps);
}

// The layers run in a loop: unrolled they took the same time, at a multiple of the code.  Registers cannot be indexed by the
// layer number, so the tiles turn by one place per layer instead.  pin: the loads have returned here, and nothing inside the loop waits for memory.
template <int N, int KS> __device__ __forceinline__ void turn(u32x4 (&r)[N][KS])
{
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int l = 0; l + 1 < N; ++l) r[l][ks] = r[l + 1][ks];
    }
}
template <int N, int KS> __device__ __forceinline__ void pin(u32x4 (&r)[N][KS])
{
#pragma unroll
    for (int l = 0; l < N; ++l)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(r[l][ks]));
}
template <int N> __device__ __forceinline__ void pin(f32x4 (&r)[N])
{
#pragma unroll
    for (int l = 0; l < N; ++l) asm volatile("" : "+v"(r[l]));
}

// column of channels f = 16 ft + 4 g .. of a row: f itself, or 16 (f / head) + f % head in head-padded rows
__device__ __forceinline__ int col_of(int head, int ft, int g)
{
    return head == 0 ? 16 * ft + 4 * g : head == 8 ? 32 * ft + 8 * g - 4 * (g & 1) : 64 * ft + 16 * g;
}
// the zeros of head-padded rows up to 16 columns, by the lane that holds the head's last four channels
template <int DT> __device__ __forceinline__ void store_pad(void* base, int64_t e, int head, int g)
{
    const int nz = head == 0 ? 0 : head == 8 ? ((g & 1) ? 2 : 0) : 3;
    for (int z = 1; z <= nz; ++z) store4<DT>(base, e + 4 * z, f32x4{0.f, 0.f, 0.f, 0.f});
}

// Forward.  LMAX: layers held in registers, L <= LMAX (the surplus tiles are the last one again: no branch around a load).
// PRE: a Linear and a residual in front, in the same launch (a block's output projection before its feed-forward); what the chain
// reads then goes from wave to wave through LDS in fp32, in the order row_stats takes it from memory, so the results are the
// same bits as those of two launches.  What goes away is a launch's latency (start, one trip to memory, end) each way: 8 blocks, bf16, training
// step at 4096 tokens 1342 -> 1261 us (C = 128) and 1024 -> 966 us (C = 64), inference forward at 3973 tokens, C = 64, 360 -> 340 us.
// At most 128 registers up to five layers: two workgroups of C = 128 share a CU, which a pair of chains needs from 2049 tokens and a
// single one from 4097 (with 160 registers they came one after the other: 4 blocks, 9001 tokens, inference 341 -> 282 us; training step at
// 12,000 tokens 1325 -> 1252 us, of 8 blocks at 4096 tokens 1258 -> 1238 us).
template <typename T, int C, int LMAX, bool PRE>
__global__ __launch_bounds__(4 * C, LMAX <= 5 ? 4 : 2) void few_mlp_mfma_kernel(MlpArgs a)
{
    constexpr int FT = C / 16, KS = C / 32;
    using M_ = Mf<T>;
    __shared__ Exchange<C> ex;
    __shared__ __attribute__((aligned(16))) float xs[PRE ? 16 : 1][C + 4];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = a.L;
    const bool has_bias = a.bias != nullptr;
    const int ch0 = 16 * w + 4 * g;                               // this lane's four channels of the stream
    const int chain = blockIdx.y;                                 // 1: the second chain of a pair

    const int64_t t = (int64_t)blockIdx.x * 16 + c16;
    const bool live = t < a.T;
    const int64_t tok = live ? t : a.T - 1;

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 x0[FT], own;
    uint2 pre = {};
    u32x4 pw[KS];
    f32x4 pb = zero;
    if constexpr (PRE) {
        pre = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.pre_x) + tok * a.pre_xs + col_of(a.pre_head, w, g));
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) pw[ks] = operand<C>(a.pre_w, 0, w, ks, lane);
        if (a.pre_bias) pb = *reinterpret_cast<const f32x4*>(a.pre_bias + ch0);
        with_dtype(a.res_dtype, [&](auto dc) { own = load4<decltype(dc)::value>(a.res, tok * a.rs + ch0); });
    } else {
        with_dtype(a.x_dtype, [&](auto dc) {
            constexpr int DT = decltype(dc)::value;
            own = load4<DT>(a.x, tok * a.xs + col_of(a.x_head, w, g));
            if (a.norm != 0) {
#pragma unroll
                for (int ft = 0; ft < FT; ++ft) x0[ft] = load4<DT>(a.x, tok * a.xs + col_of(a.x_head, ft, g));
            }
        });
    }
    f32x4 gm = zero, bt = zero;
    if (a.norm != 0) {
        gm = *reinterpret_cast<const f32x4*>(a.gamma + ch0);
        if (a.beta) bt = *reinterpret_cast<const f32x4*>(a.beta + ch0);
    }
    // the first layers' weights travel beside the rows, the others take the rows' registers once the norm is done with them
    constexpr int FIRST = C == 128 ? (LMAX + 1) / 2 : LMAX;
    u32x4 wr[LMAX][KS];
    f32x4 bias[LMAX];
    auto request = [&](int l) {
        const size_t tile = (size_t)chain * L + (l < L ? l : L - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) wr[l][ks] = operand<C>(a.w, tile, w, ks, lane);
        // a missing bias reads the weights instead (any mapped memory will do) and is replaced by zeros where it is used
        bias[l] = *reinterpret_cast<const f32x4*>((has_bias ? a.bias + tile * C : reinterpret_cast<const float*>(a.w)) + ch0);
    };
#pragma unroll
    for (int l = 0; l < FIRST; ++l) request(l);
    if constexpr (PRE) {
        publish<C>(ex, 1, w, lane, pre.x, pre.y);
        f32x4 x1, acc = pb;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc = M_::mma(pw[ks], ex.q[1][ks][lane], acc);
        x1 = acc + own;
        with_dtype(a.x_dtype, [&](auto dc) {
            constexpr int DT = decltype(dc)::value;
            if (live && a.pre_y) store4<DT>(a.pre_y, tok * a.xs + ch0, x1);
            x1 = round4<DT>(x1);
        });
        own = x1;
        *reinterpret_cast<f32x4*>(&xs[c16][ch0]) = x1;            // also kept there for the residual
        if (a.norm != 0) {
            lds_barrier();
#pragma unroll
            for (int ft = 0; ft < FT; ++ft) x0[ft] = *reinterpret_cast<const f32x4*>(&xs[c16][16 * ft + 4 * g]);
        }
    }
    if (a.norm != 0) {
        float mean, rstd;
        row_stats<C>(x0, a.norm, a.eps, mean, rstd);
#pragma unroll
        for (int r = 0; r < 4; ++r) own[r] = (own[r] - mean) * rstd * gm[r] + bt[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(own[r]));
#pragma unroll
    for (int l = FIRST; l < LMAX; ++l) request(l);
    pin(wr);
    pin(bias);
    const ActCoef coef = act_coef(a.act);
    f32x4 s = own;
#pragma unroll 1
    for (int l = 0; l < L; ++l) {
        publish<C>(ex, l & 1, w, lane, M_::pack2(s[0], s[1]), M_::pack2(s[2], s[3]));
        u32x4 xb[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) xb[ks] = ex.q[l & 1][ks][lane];
        f32x4 acc = has_bias ? bias[0] : zero;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc = M_::mma(wr[0][ks], xb[ks], acc);
        const bool act = (a.act_mask >> l) & 1u, add = (a.add_mask >> l) & 1u;
        turn(wr);
#pragma unroll
        for (int i = 0; i + 1 < LMAX; ++i) bias[i] = bias[i + 1];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float u, slope;
            act_and_slope(coef, acc[r], u, slope);
            u = act ? u : acc[r];
            s[r] = add ? s[r] + u : u;
        }
    }
    // the lane's place again, from its number: kept through the layers it would cost the registers that they need
    int id = tid;
    asm volatile("" : "+v"(id));
    const int g_ = (id & 63) >> 4, c_ = id & 15, f_ = 16 * w + 4 * g_;
    const int64_t t_ = (int64_t)blockIdx.x * 16 + c_, tok_ = t_ < a.T ? t_ : a.T - 1;
    if constexpr (PRE) s += *reinterpret_cast<const f32x4*>(&xs[c_][f_]);
    else if (a.res) with_dtype(a.res_dtype, [&](auto dc) { s += load4<decltype(dc)::value>(a.res, tok_ * a.rs + f_); });
    if (t_ < a.T) {
        with_dtype(a.y_dtype, [&](auto dc) {
            constexpr int DT = decltype(dc)::value;
            const int64_t e = tok_ * a.ys + col_of(a.y_head, w, g_);
            void* y = chain ? a.y2 : a.y;
            store4<DT>(y, e, s);
            store_pad<DT>(y, e, a.y_head, g_);
        });
    }
}

// Backward: the forward recomputed, the chain walked back with the transposed weights, the norm's backward, dx; the rows s_l
// and dt_l for the weight gradients leave as they are published.  Two chains: their gradients at the norm's output are added
// before the norm's backward.  dgamma and dbeta are summed here over the workgroup's tokens (gb_part, one row per workgroup).
// PRE: on through the Linear in front of the chain (see the forward), with dx as the gradient of its output.
template <typename T, int C, int LMAX, int CH, bool PRE>
__global__ __launch_bounds__(4 * C) void few_mlp_bwd_kernel(MlpBwdArgs a)
{
    constexpr int FT = C / 16, KS = C / 32, NW = C / 16;
    using M_ = Mf<T>;
    __shared__ Exchange<C> ex;
    __shared__ float red[2][NW][16];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = a.L;
    const bool has_bias = a.bias != nullptr;
    const int ch0 = 16 * w + 4 * g;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

    const int64_t t = (int64_t)blockIdx.x * 16 + c16;
    const bool live = t < a.T;
    const int64_t tok = live ? t : a.T - 1;

    f32x4 x0[FT], own, dy[CH];
    with_dtype(a.x_dtype, [&](auto dc) {
        constexpr int DT = decltype(dc)::value;
        own = load4<DT>(a.x, tok * a.xs + col_of(a.x_head, w, g));
        if (a.norm != 0) {
#pragma unroll
            for (int ft = 0; ft < FT; ++ft) x0[ft] = load4<DT>(a.x, tok * a.xs + col_of(a.x_head, ft, g));
        }
    });
    f32x4 gm = zero, bt = zero;
    if (a.norm != 0) {
        gm = *reinterpret_cast<const f32x4*>(a.gamma + ch0);
        if (a.beta) bt = *reinterpret_cast<const f32x4*>(a.beta + ch0);
    }
    with_dtype(a.dy_dtype, [&](auto dc) {
#pragma unroll
        for (int c = 0; c < CH; ++c) dy[c] = load4<decltype(dc)::value>(c == 0 ? a.dy : a.dy2, tok * a.dys + col_of(a.y_head, w, g));
    });
    u32x4 wr[LMAX][KS], wt[LMAX][KS];
    f32x4 bias[LMAX];
    auto tile_of = [&](int c, int l) { return (size_t)c * L + (l < L ? l : L - 1); };
    auto request_w = [&](int c) {
#pragma unroll
        for (int l = 0; l < LMAX; ++l) {
            const size_t tile = tile_of(c, l);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) wr[l][ks] = operand<C>(a.w, tile, w, ks, lane);
            bias[l] = *reinterpret_cast<const f32x4*>((has_bias ? a.bias + tile * C : reinterpret_cast<const float*>(a.w)) + ch0);
        }
    };
    auto request_wt = [&](int c) {
#pragma unroll
        for (int i = 0; i < LMAX; ++i)      // in the order of use: the last layer's first
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) wt[i][ks] = operand<C>(a.wt, (size_t)c * L + (i < L ? L - 1 - i : 0), w, ks, lane);
    };
    request_w(0);
    request_wt(0);
    float mean = 0.f, rstd = 1.f;
    f32x4 xhat = zero, s0 = own;
    if (a.norm != 0) {
        row_stats<C>(x0, a.norm, a.eps, mean, rstd);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            xhat[r] = (own[r] - mean) * rstd;
            s0[r] = xhat[r] * gm[r] + bt[r];
        }
    }
    const ActCoef coef = act_coef(a.act);
    int buf = 0;
    f32x4 total = zero;
    uint2 pre = {};
    u32x4 pw[KS];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        uint16_t* a_row = a.a_in + (size_t)c * L * a.T * C;
        uint16_t* g_row = a.g_out + (size_t)(c * L + L - 1) * a.T * C;
        uint2 slope[LMAX] = {};                                    // act'(t_l), packed to 16 bits, the latest layer in front
        f32x4 s = s0;
        pin(wr);
        pin(bias);
#pragma unroll 1
        for (int l = 0; l < L; ++l) {
            publish<C>(ex, buf, w, lane, M_::pack2(s[0], s[1]), M_::pack2(s[2], s[3]));
            u32x4 xb[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) xb[ks] = ex.q[buf][ks][lane];
            f32x4 acc = has_bias ? bias[0] : zero;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) acc = M_::mma(wr[0][ks], xb[ks], acc);
            store_rows<C>(ex, buf, w, lane, a_row, t, live);
            a_row += (size_t)a.T * C;
            buf ^= 1;
            const bool act = (a.act_mask >> l) & 1u, add = (a.add_mask >> l) & 1u;
            turn(wr);
#pragma unroll
            for (int i = 0; i + 1 < LMAX; ++i) bias[i] = bias[i + 1];
#pragma unroll
            for (int i = LMAX - 1; i > 0; --i) slope[i] = slope[i - 1];
            float sl[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float u;
                act_and_slope(coef, acc[r], u, sl[r]);
                u = act ? u : acc[r];
                s[r] = add ? s[r] + u : u;
            }
            slope[0] = make_uint2(M_::pack2(sl[0], sl[1]), M_::pack2(sl[2], sl[3]));
        }
        if (c + 1 < CH) request_w(c + 1);
        if constexpr (PRE) {
            pre = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.pre_x) + tok * a.pre_xs + col_of(a.pre_head, w, g));
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) pw[ks] = operand<C>(a.pre_wt, 0, w, ks, lane);
        }
        f32x4 ds = live ? dy[c] : zero;
        pin(wt);
#pragma unroll 1
        for (int l = L - 1; l >= 0; --l) {
            const bool act = (a.act_mask >> l) & 1u, add = (a.add_mask >> l) & 1u;
            f32x4 dt = ds;
            if (act) {
                dt[0] *= M_::lo(slope[0].x); dt[1] *= M_::hi(slope[0].x);
                dt[2] *= M_::lo(slope[0].y); dt[3] *= M_::hi(slope[0].y);
            }
            publish<C>(ex, buf, w, lane, M_::pack2(dt[0], dt[1]), M_::pack2(dt[2], dt[3]));
            u32x4 db[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) db[ks] = ex.q[buf][ks][lane];
            f32x4 acc = add ? ds : zero;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) acc = M_::mma(wt[0][ks], db[ks], acc);
            store_rows<C>(ex, buf, w, lane, g_row, t, live);
            g_row -= (size_t)a.T * C;
            buf ^= 1;
            turn(wt);
#pragma unroll
            for (int i = 0; i + 1 < LMAX; ++i) slope[i] = slope[i + 1];
            ds = acc;
        }
        if (c + 1 < CH) request_wt(c + 1);
        total += ds;
    }

    if (a.norm != 0) {
        f32x4 gs, bs = live ? total : zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) gs[r] = bs[r] * xhat[r];
#pragma unroll
        for (int r = 0; r < 4; ++r) {       // over the 16 tokens of the lane group
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                gs[r] += __shfl_xor(gs[r], o);
                bs[r] += __shfl_xor(bs[r], o);
            }
        }
        if (c16 == 0) {
            float* part = a.gb_part + (size_t)blockIdx.x * 2 * C + ch0;
            *reinterpret_cast<f32x4*>(part) = gs;
            *reinterpret_cast<f32x4*>(part + C) = bs;
        }
        float m1 = 0.f, m2 = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            total[r] *= gm[r];
            m1 += total[r];
            m2 = fmaf(total[r], xhat[r], m2);
        }
        m1 = tok_sum(m1);
        m2 = tok_sum(m2);
        if (g == 0) {
            red[0][w][c16] = m1;
            red[1][w][c16] = m2;
        }
        lds_barrier();
        m1 = m2 = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            m1 += red[0][i][c16];
            m2 += red[1][i][c16];
        }
        m1 = a.norm == 1 ? m1 * (1.f / C) : 0.f;
        m2 *= 1.f / C;
#pragma unroll
        for (int r = 0; r < 4; ++r) total[r] = rstd * (total[r] - m1 - xhat[r] * m2);
    }
    if (live) {
        if (a.add_dy & 1) total += dy[0];
        with_dtype(a.dx_dtype, [&](auto dc) {
            constexpr int DT = decltype(dc)::value;
            const int64_t e = tok * a.dxs + col_of(a.x_head, w, g);
            if (a.dres) total += load4<DT>(a.dres, e);            // another path's gradient of x (a residual's)
            if (a.add_dy & 2) total += load4<DT>(a.dx, e);        // dx holds another path's gradient of the same x
            store4<DT>(a.dx, e, total);
            store_pad<DT>(a.dx, e, a.x_head, g);
            if constexpr (PRE) total = round4<DT>(total);
        });
    }
    if constexpr (PRE) {
        publish<C>(ex, buf, w, lane, pre.x, pre.y);
        store_rows<C>(ex, buf, w, lane, a.pre_a, t, live);
        buf ^= 1;
        publish<C>(ex, buf, w, lane, M_::pack2(total[0], total[1]), M_::pack2(total[2], total[3]));
        f32x4 acc = zero;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc = M_::mma(pw[ks], ex.q[buf][ks][lane], acc);
        store_rows<C>(ex, buf, w, lane, a.pre_g, t, live);
        if (live) {
            constexpr int DT = std::is_same_v<T, bf16_t> ? 1 : 2;
            const int64_t e = tok * (a.pre_head ? 16 * (C / a.pre_head) : C) + col_of(a.pre_head, w, g);
            store4<DT>(a.pre_dx, e, acc);
            store_pad<DT>(a.pre_dx, e, a.pre_head, g);
        }
    }
}

template <typename T, int C, int LMAX>
hipError_t fwd_l(const MlpArgs& a, hipStream_t st)
{
    const dim3 grid((unsigned)((a.T + 15) / 16), a.y2 ? 2 : 1);
    if constexpr (LMAX > 1) {
        if (a.pre_x) {
            hipLaunchKernelGGL((few_mlp_mfma_kernel<T, C, LMAX, true>), grid, dim3(4 * C), 0, st, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((few_mlp_mfma_kernel<T, C, LMAX, false>), grid, dim3(4 * C), 0, st, a);
    return hipGetLastError();
}
template <typename T, int C, int LMAX>
hipError_t bwd_l(const MlpBwdArgs& a, hipStream_t st)
{
    const dim3 grid((unsigned)mlp_few_bwd_rows(a.T));
    if constexpr (LMAX > 1) {
        if (a.pre_x) {
            hipLaunchKernelGGL((few_mlp_bwd_kernel<T, C, LMAX, 1, true>), grid, dim3(4 * C), 0, st, a);
            return hipGetLastError();
        }
    }
    if (a.dy2) hipLaunchKernelGGL((few_mlp_bwd_kernel<T, C, LMAX, 2, false>), grid, dim3(4 * C), 0, st, a);
    else       hipLaunchKernelGGL((few_mlp_bwd_kernel<T, C, LMAX, 1, false>), grid, dim3(4 * C), 0, st, a);
    return hipGetLastError();
}

template <typename T, int C> hipError_t fwd_c(const MlpArgs& a, hipStream_t st)
{
    if (a.L <= 1 && !a.pre_x) return fwd_l<T, C, 1>(a, st);
    if (a.L <= 5) return fwd_l<T, C, 5>(a, st);
    if constexpr (C < 128) { if (a.L <= 8) return fwd_l<T, C, 8>(a, st); }
    return hipErrorInvalidValue;
}
template <typename T, int C> hipError_t bwd_c(const MlpBwdArgs& a, hipStream_t st)
{
    if (a.L <= 1 && !a.pre_x) return bwd_l<T, C, 1>(a, st);
    if (a.L <= 5) return bwd_l<T, C, 5>(a, st);
    if constexpr (C < 128) { if (a.L <= 8) return bwd_l<T, C, 8>(a, st); }
    return hipErrorInvalidValue;
}

}  // namespace

// Where the few-token kernels are the faster ones: their time grows with the tokens (every 16 read all weights again), that of
// the many-token kernels does not up to 32,768.  A training step of a 4-block model, the many-token against the few-token
// kernels (with everything around them alike): C = 128, 12,001 tokens 1949 / 1723 us, 16,384 tokens 1974 / 2010 us;
// C = 64, 12,001 tokens 1657 / 1367 us, 16,384 tokens 1635 / 1415 us.  fused.py knows the same limits.
bool mlp_few_ok(int64_t T, int C, int L) { return T >= 1 && T <= (C == 128 ? 12288 : 16384) && L >= 1 && L <= (C == 128 ? 5 : 8); }

// workgroups of the backward, and rows of gb_part it writes
int mlp_few_bwd_rows(int64_t T) { return (int)((T + 15) / 16); }

hipError_t launch_mlp_few(const MlpArgs& a, int w_dtype, hipStream_t st)
{
    if (w_dtype == 1) return a.C == 32 ? fwd_c<bf16_t, 32>(a, st) : a.C == 64 ? fwd_c<bf16_t, 64>(a, st) : fwd_c<bf16_t, 128>(a, st);
    return a.C == 32 ? fwd_c<f16_t, 32>(a, st) : a.C == 64 ? fwd_c<f16_t, 64>(a, st) : fwd_c<f16_t, 128>(a, st);
}

hipError_t launch_mlp_few_bwd(const MlpBwdArgs& a, int w_dtype, hipStream_t st)
{
    if (w_dtype == 1) return a.C == 32 ? bwd_c<bf16_t, 32>(a, st) : a.C == 64 ? bwd_c<bf16_t, 64>(a, st) : bwd_c<bf16_t, 128>(a, st);
    return a.C == 32 ? bwd_c<f16_t, 32>(a, st) : a.C == 64 ? bwd_c<f16_t, 64>(a, st) : bwd_c<f16_t, 128>(a, st);
}

}  // namespace flare
