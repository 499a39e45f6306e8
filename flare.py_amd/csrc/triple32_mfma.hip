// Triple attention with head dims of 32 (Dq = Dv = 32, bf16 / f16, rows 16-byte aligned) on v_mfma_f32_32x32x16.
//
//   state[i,j,k] = (1/N) sum_n f(k1)[n,i] v[n,j] f(k2)[n,k],   out[n,j] = sum_{i,k} f(q1)[n,i] state[i,j,k] f(q2)[n,k]
//
// as in triple_mfma.hip, but with the 32 x 32 x 32 state as one block instead of eight of 16 x 16 x 16, which re-read every
// input four times, rebuilt every product f(k1) f(k2) twice and kept the output's contraction over i at a quarter of the
// matrix instruction's depth.  Measured at B=1, H=8, N=32,768 f16: state 62 -> 27 us, output 81 -> 24 us, the backward's five
// outputs 406 -> 91 us (one launch); forward + backward 591 -> 193 us.
//
// What bounds them: vector issue and power.  An output slice of 32 tokens is 64 matrix cycles and sixteen FMAs of 4 cycles; the
// five-output launch runs at 1.75 GHz with the matrix pipe 49 % and vector issue 64 % busy, and neither a deeper pipeline nor
// plain FMAs in place of v_fma_mix moved it by more than 4 %.  The state kernel's partials (132 KB of fp32 per workgroup,
// written and merged) are a third of its 27 + 9 us.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace flare {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Tx;
template <> struct Tx<bf16_t> {
    static __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi)
    {
        bf16x2 v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
    static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};
template <> struct Tx<f16_t> {
    static __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi)
    {
        f16x2 v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float lo(uint32_t w) { return float(__builtin_bit_cast(f16x2, w)[0]); }
    static __device__ __forceinline__ float hi(uint32_t w) { return float(__builtin_bit_cast(f16x2, w)[1]); }
};

__device__ __forceinline__ uint2 tr16(const void* lds_addr)
{
    typedef s16x4 __attribute__((address_space(3))) * lds_ptr_t;
    asm volatile("" ::: "memory");
    const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(uintptr_t)lds_addr);
    asm volatile("" ::: "memory");
    return __builtin_bit_cast(uint2, r);
}

__device__ __forceinline__ float featf(float x) { return x > 0.f ? x + 1.f : __expf(x); }

// eight elements through the feature map and back to the element type
template <typename T> __device__ __forceinline__ u32x4 feat8(u32x4 raw)
{
    u32x4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = raw[i];
        f[i] = Tx<T>::pack2(featf(Tx<T>::lo(w)), featf(Tx<T>::hi(w)));
    }
    return f;
}

constexpr int kD = 32, kWaves = 8, kThreads = 64 * kWaves;
constexpr int kTok = 128;                 // tokens per staged tile of the state kernel
constexpr int kRow = kD + 8;              // LDS row stride in elements: 16-byte aligned, rows 20 banks apart
constexpr size_t kStateLds = (size_t)2 * 3 * kTok * kRow * 2;
constexpr int kTab = kD * 2 * 64;         // 16-byte entries of a state table (64 KB)

// x times the value y holds R lanes down the lane's row of 16 (see triple_mfma.hip: the caller spends the DPP wait states)
template <int R> __device__ __forceinline__ float mul_ror(float x, float y)
{
    if constexpr (R == 0) return x * y;
    float d;
    asm("v_mul_f32_dpp %0, %1, %2 row_ror:%3 row_mask:0xf bank_mask:0xf" : "=v"(d) : "v"(y), "v"(x), "i"(R));
    return d;
}
template <int R> __device__ __forceinline__ uint32_t ror(uint32_t y)
{
    if constexpr (R == 0) return y;
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)y, 0x120 + R, 0xf, 0xf, true);
}

// State.  grid (splits, H, B), one workgroup of eight waves per compute unit.  Tiles of 128 tokens (feature map applied once,
// as they are staged) are shared by the waves; a wave takes k1, k2 and v of 16 tokens at a time with the tokens in the
// k-slots (transpose reads: lane = feature, 8 tokens per lane half).  As in the 16-wide kernel the accumulators run along
// diagonals, so that a factor f(k2)[n,k] never has to be broadcast: wave w owns the four diagonals c = 4 w + R,
//   S_c[i][j] = state[i][j][k],  k = 16 ((i >> 4) ^ (w >> 2)) + ((i - 4 (w & 3) - R) mod 16),
// the half and the multiple of four chosen by the addresses of the transpose read, R = 0..3 by a DPP rotate of the row.
// The waves' diagonals are disjoint: no sum across waves, the partial leaves in accumulator order, 16 bytes per lane and
// store.  The f16 products use the packed multiply (exact product, one rounding: the
// bits of an fp32 product rounded to f16).
template <typename T, bool NORM>
__global__ __launch_bounds__(kThreads, 2) void triple_state32_kernel(TripleArgs a)
{
    using M_ = Tx<T>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint16_t* buf = reinterpret_cast<uint16_t*>(smem);          // [2][3][kTok][kRow]

    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c16 = lane & 15, ih = (lane >> 4) & 1, half = lane >> 5;
    const int split = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const uint16_t* k1 = (const uint16_t*)a.k1 + b * a.k1s[0] + h * a.k1s[1];
    const uint16_t* k2 = (const uint16_t*)a.k2 + b * a.k2s[0] + h * a.k2s[1];
    const uint16_t* v = (const uint16_t*)a.v + b * a.vs[0] + h * a.vs[1];
    const int n_begin = split * a.tokens_per_split, n_end = min(a.N, n_begin + a.tokens_per_split);
    const int tiles = (n_end - n_begin + kTok - 1) / kTok;
    const int tok = tid >> 2, ch = (tid & 3) * 8;

    f32x16 S[4], kk;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        kk[e] = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r][e] = 0.f;
    }

    u32x4 r1, r2, rv;
    auto fetch = [&](int n0) {      // rows past the end repeat the last one (no branch around a load), staged as zeros
        const int64_t n = min(n0 + tok, n_end - 1);
        r1 = *reinterpret_cast<const u32x4*>(k1 + n * a.k1s[2] + ch);
        r2 = *reinterpret_cast<const u32x4*>(k2 + n * a.k2s[2] + ch);
        rv = *reinterpret_cast<const u32x4*>(v + n * a.vs[2] + ch);
    };
    auto stage = [&](int n0, int p) {
        const u32x4 z = {0u, 0u, 0u, 0u};
        const bool live = n0 + tok < n_end;
        const u32x4 f1 = a.feature_map ? feat8<T>(r1) : r1, f2 = a.feature_map ? feat8<T>(r2) : r2;
        uint16_t* d = buf + (size_t)p * 3 * kTok * kRow + tok * kRow + ch;
        *reinterpret_cast<u32x4*>(d) = live ? f1 : z;
        *reinterpret_cast<u32x4*>(d + kTok * kRow) = live ? f2 : z;
        *reinterpret_cast<u32x4*>(d + 2 * kTok * kRow) = live ? rv : z;
    };
    // lane (half, ih, c16): eight tokens 8 half .. + 7 of column `col` of the 16-token step
    const int trow = 8 * half + (c16 >> 2);
    auto take = [&](const uint16_t* tile, int m, int col) {
        const uint2 lo = tr16(tile + (16 * m + trow) * kRow + col);
        const uint2 hi = tr16(tile + (16 * m + trow + 4) * kRow + col);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    const int col_nat = 16 * ih + 4 * (c16 & 3);                                              // columns as they are
    const int col_k2 = 16 * (ih ^ (w >> 2)) + 4 * (((c16 & 3) - (w & 3)) & 3);                // half swapped, rotated by 4 (w & 3)

    fetch(n_begin);
    stage(n_begin, 0);
    __syncthreads();
    for (int t = 0, n0 = n_begin; t < tiles; ++t, n0 += kTok) {
        fetch(n0 + kTok);
        const uint16_t* t1 = buf + (size_t)(t & 1) * 3 * kTok * kRow;
        const uint16_t* t2 = t1 + kTok * kRow;
        const uint16_t* tv = t2 + kTok * kRow;
        u32x4 y1 = take(t1, 0, col_nat), y2 = take(t2, 0, col_k2), yv = take(tv, 0, col_nat);
#pragma unroll
        for (int m = 0; m < kTok / 16; ++m) {
            const u32x4 x1 = y1, x2 = y2, xv = yv;
            if (m + 1 < kTok / 16) {        // the next step's operands travel under this step's products
                y1 = take(t1, m + 1, col_nat);
                y2 = take(t2, m + 1, col_k2);
                yv = take(tv, m + 1, col_nat);
            }
            auto product = [&](auto r_c) {
                constexpr int R = decltype(r_c)::value;
                return u32x4{ror<R>(x2[0]), ror<R>(x2[1]), ror<R>(x2[2]), ror<R>(x2[3])};
            };
            if constexpr (std::is_same<T, f16_t>::value) {
                auto step = [&](auto r_c, f32x16& acc) {
                    const f16x8 p = __builtin_bit_cast(f16x8, x1) * __builtin_bit_cast(f16x8, product(r_c));
                    acc = M_::mma(__builtin_bit_cast(u32x4, p), xv, acc);
                };
                step(std::integral_constant<int, 0>{}, S[0]);
                step(std::integral_constant<int, 1>{}, S[1]);
                step(std::integral_constant<int, 2>{}, S[2]);
                step(std::integral_constant<int, 3>{}, S[3]);
            } else {
                float f1[8], f2[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t w1 = x1[e], w2 = x2[e];
                    f1[2 * e] = M_::lo(w1); f1[2 * e + 1] = M_::hi(w1);
                    f2[2 * e] = M_::lo(w2); f2[2 * e + 1] = M_::hi(w2);
                }
                // the DPP reads below sit in assembly: this statement orders them behind the writes of f2 and spends the
                // two wait states a DPP read of a fresh register needs
                asm volatile("s_nop 1" : "+v"(f2[0]), "+v"(f2[1]), "+v"(f2[2]), "+v"(f2[3]), "+v"(f2[4]), "+v"(f2[5]), "+v"(f2[6]), "+v"(f2[7]));
                auto step = [&](auto r_c, f32x16& acc) {
                    constexpr int R = decltype(r_c)::value;
                    u32x4 p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) p[e] = M_::pack2(mul_ror<R>(f1[2 * e], f2[2 * e]), mul_ror<R>(f1[2 * e + 1], f2[2 * e + 1]));
                    acc = M_::mma(p, xv, acc);
                };
                step(std::integral_constant<int, 0>{}, S[0]);
                step(std::integral_constant<int, 1>{}, S[1]);
                step(std::integral_constant<int, 2>{}, S[2]);
                step(std::integral_constant<int, 3>{}, S[3]);
            }
            if (NORM && w == 0) kk = M_::mma(x1, x2, kk);      // wave 0 holds k2 unrotated: kk[i][k']
        }
        stage(n0 + kTok, (t + 1) & 1);      // the buffer of the tile before: its readers passed the last barrier
        __syncthreads();
    }

    float* part = a.part + (((size_t)b * a.H + h) * a.n_parts + split) * kTriple32Partial;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(part + ((size_t)((4 * w + r) * 4 + q) * 64 + lane) * 4) =
                f32x4{S[r][4 * q], S[r][4 * q + 1], S[r][4 * q + 2], S[r][4 * q + 3]};
    if (NORM && w == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(part + ((size_t)(128 + q) * 64 + lane) * 4) = f32x4{kk[4 * q], kk[4 * q + 1], kk[4 * q + 2], kk[4 * q + 3]};
    }
}

// Where element (i, j, k) sits in a state table (16-bit elements): entry (k, i >> 4) of lane (half = (i >> 3) & 1, j) holds
// i = 16 (i >> 4) + 8 half + e, e = 0..7: the A operand of the product over i for one slice k.
__device__ __forceinline__ int tab_pos(int i, int j, int k) { return ((k * 2 + (i >> 4)) * 64 + ((i >> 3) & 1) * 32 + j) * 8 + (i & 7); }

// Partials summed in split order into the state (and kk), plus dstate / N when given, and the tables the outputs read: as it
// is, with i and j exchanged, with j and k exchanged; for the backward also the two exchanged tables of the forward's state.
template <typename T>
__global__ __launch_bounds__(256) void triple_merge32_kernel(Triple32MergeArgs a)
{
    const size_t ns = (size_t)kD * kD * kD;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t bh = idx / kTriple32Partial, e = idx % kTriple32Partial;
    if (bh >= (size_t)a.BH) return;
    if (e >= ns && !a.kk) return;
    const float* p = a.part + bh * a.n_parts * kTriple32Partial + e;
    float s = 0.f;
    for (int sp = 0; sp < a.n_parts; sp += 8) {      // eight partials requested at a time
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = p[(size_t)min(sp + u, a.n_parts - 1) * kTriple32Partial];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += sp + u < a.n_parts ? t[u] : 0.f;
    }
    s *= a.inv_n;
    const int q = (int)(e >> 8) & 3, lane = (int)(e >> 2) & 63, rr = (int)e & 3;
    const int i = 8 * q + 4 * (lane >> 5) + rr, j = lane & 31;
    if (e >= ns) {
        a.kk[bh * kD * kD + i * kD + j] = s;
        return;
    }
    const int c = (int)(e >> 10), w = c >> 2, R = c & 3;
    const int k = 16 * ((i >> 4) ^ (w >> 2)) + ((i - 4 * (w & 3) - R) & 15);
    const size_t at = bh * ns + (size_t)(i * kD + j) * kD + k;
    if (a.dstate) s += a.dstate[at] * a.inv_n;
    if (a.state) a.state[at] = s;
    auto put = [&](uint16_t* tab, int x, int y, int z, float val) {
        if (tab) tab[bh * kTab * 8 + tab_pos(x, y, z)] = (uint16_t)Tx<T>::pack2(val, 0.f);
    };
    put(a.tab, i, j, k, s);
    put(a.tab_ji, j, i, k, s);
    put(a.tab_kj, i, k, j, s);
    if (a.fwd_state) {
        const float f = a.fwd_state[at];
        put(a.fwd_tab_ji, j, i, k, f);
        put(a.fwd_tab_kj, i, k, j, f);
    }
}

// Outputs, up to five contractions per launch (the backward's).  grid (ranges, H * ops, B), eight waves.  The state's table (64 KB, 16-bit
// A operands) is resident in LDS; products are taken transposed, T_k^T[j,n] = sum_i state[i,j,k] f(q1)[n,i]: two 32x32x16
// products per slice k and 32 tokens, f(q1) rows straight from global memory as B operands, the token in the lane, so that
// f(q2)[n,k] is a per-lane factor: out[n,j] += T_k f(q2)[n,k], sixteen FMAs per slice.  A wave carries two 32-token tiles per
// pass so that one table read serves two products (with one, the table reads alone take the LDS as long as the products
// take the matrix cores), slice k's products issued ahead of slice k-1's FMAs.
template <typename T>
__global__ __launch_bounds__(kThreads, 2) void triple_out32_kernel(Triple32OutArgs a)
{
    using M_ = Tx<T>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    u32x4* tab = reinterpret_cast<u32x4*>(smem);           // [k][i half][lane]
    u32x4* kkt = tab + kTab;                                // [i half][lane] (normalised outputs only)

    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int op = blockIdx.y / a.H, h = blockIdx.y % a.H, b = blockIdx.z;
    const size_t bh = (size_t)b * a.H + h;
    const Triple32OutOp o = a.op[op];
    const uint16_t* q1 = (const uint16_t*)o.q1 + b * o.q1s[0] + h * o.q1s[1];
    const uint16_t* q2 = (const uint16_t*)o.q2 + b * o.q2s[0] + h * o.q2s[1];
    uint16_t* out = (uint16_t*)o.out + b * o.os[0] + h * o.os[1];
    const int wg_n0 = blockIdx.x * a.tokens_per_wg, wg_n1 = min(a.N, wg_n0 + a.tokens_per_wg);

    u32x4 r1[2][2], r2[2][4];
    auto fetch = [&](int n0) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int64_t n = min(n0 + 32 * t + l32, wg_n1 - 1);
#pragma unroll
            for (int c = 0; c < 2; ++c) r1[t][c] = *reinterpret_cast<const u32x4*>(q1 + n * o.q1s[2] + 16 * c + 8 * half);
#pragma unroll
            for (int c = 0; c < 4; ++c) r2[t][c] = *reinterpret_cast<const u32x4*>(q2 + n * o.q2s[2] + 8 * c);
        }
    };
    fetch(wg_n0 + 64 * w);

    if (o.tab) {
        const u32x4* src = reinterpret_cast<const u32x4*>(o.tab) + bh * kTab;
#pragma unroll
        for (int i = 0; i < kTab / kThreads; ++i) tab[tid + i * kThreads] = src[tid + i * kThreads];
    } else {
        // from the fp32 state: a thread takes eight rows i of one j and four slices k; eight lanes cover a 128-byte line
        // of each row, and their 16-byte stores (consecutive j) fall into different banks
        const float* st = o.state + bh * kD * kD * kD;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int rest = w + 8 * it, k4 = (lane >> 3) & 7, j = (lane & 7) + 8 * (rest & 3), io = rest >> 2;
            f32x4 x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = *reinterpret_cast<const f32x4*>(st + (size_t)((8 * io + e) * kD + j) * kD + 4 * k4);
#pragma unroll
            for (int c = 0; c < 4; ++c)
                tab[((4 * k4 + c) * 2 + (io >> 1)) * 64 + (io & 1) * 32 + j] =
                    u32x4{M_::pack2(x[0][c], x[1][c]), M_::pack2(x[2][c], x[3][c]), M_::pack2(x[4][c], x[5][c]), M_::pack2(x[6][c], x[7][c])};
        }
    }
    if (a.normalize && tid < 128) {      // kk[i][k'] as A operands: rows k', contraction over i
        const float* kp = o.kk + bh * kD * kD + (size_t)(16 * (tid >> 6) + 8 * half) * kD + l32;
        kkt[tid] = u32x4{M_::pack2(kp[0], kp[kD]), M_::pack2(kp[2 * kD], kp[3 * kD]), M_::pack2(kp[4 * kD], kp[5 * kD]), M_::pack2(kp[6 * kD], kp[7 * kD])};
    }
    __syncthreads();

    f32x16 zero;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0.f;
    for (int n0 = wg_n0 + 64 * w; n0 < wg_n1; n0 += 64 * kWaves) {
        u32x4 f1[2][2], f2[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int c = 0; c < 2; ++c) f1[t][c] = a.feature_map ? feat8<T>(r1[t][c]) : r1[t][c];
#pragma unroll
            for (int c = 0; c < 4; ++c) f2[t][c] = a.feature_map ? feat8<T>(r2[t][c]) : r2[t][c];
        }
        fetch(n0 + 64 * kWaves);        // unconditional: past the end the last row is read again and never used
        f32x16 acc[2] = {zero, zero};   // out[n][j = 8 (e / 4) + 4 half + e % 4]
        // slice k's products of both tiles are issued ahead of slice k - 1's FMAs, the second product of a tile half a slice
        // behind the first (a product waits at issue for the one it accumulates onto).  The fences keep the compiler from
        // spreading many slices' table reads over the registers.
        auto add = [&](int k, int u, const f32x16& t) {
            const uint32_t word = f2[u][k >> 3][(k >> 1) & 3];
            float f = (k & 1) ? M_::hi(word) : M_::lo(word);
            asm("" : "+v"(f));      // a plain FMA (2.4 cycles): with the f16 factor in view this becomes v_fma_mix, at half the rate
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[u][e] = fmaf(t[e], f, acc[u][e]);
        };
        f32x16 ta[2], tb[2];
        u32x4 a0 = tab[lane], a1 = tab[64 + lane];
#pragma unroll
        for (int k = 0; k <= kD; ++k) {
            f32x16 (&tn)[2] = k & 1 ? tb : ta;
            f32x16 (&tp)[2] = k & 1 ? ta : tb;
            u32x4 b0 = a0, b1 = a1;
            if (k < kD) {
                tn[0] = M_::mma(a0, f1[0][0], zero);
                tn[1] = M_::mma(a0, f1[1][0], zero);
                if (k + 1 < kD) {
                    b0 = tab[(k + 1) * 128 + lane];
                    b1 = tab[(k + 1) * 128 + 64 + lane];
                }
            }
            if (k > 0) add(k - 1, 0, tp[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (k < kD) {
                tn[0] = M_::mma(a1, f1[0][1], tn[0]);
                tn[1] = M_::mma(a1, f1[1][1], tn[1]);
            }
            if (k > 0) add(k - 1, 1, tp[1]);
            a0 = b0;
            a1 = b1;
            __builtin_amdgcn_sched_barrier(0);
        }
        if (a.normalize) {
            // den[n] = sum_k' (sum_i kk[i,k'] f(q1)[n,i]) f(q2)[n,k']: the lane holds k' = 8 (e / 4) + 4 half + e % 4
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f32x16 wv = M_::mma(kkt[lane], f1[u][0], zero);
                wv = M_::mma(kkt[64 + lane], f1[u][1], wv);
                float den = 0.f;
#pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    const uint32_t w0 = f2[u][e >> 2][(e & 3) >> 1], w1 = f2[u][e >> 2][2 + ((e & 3) >> 1)];
                    const uint32_t word = half ? w1 : w0;
                    den = fmaf(wv[e], M_::lo(word), den);
                    den = fmaf(wv[e + 1], M_::hi(word), den);
                }
                const float inv = 1.f / sum_xor32(den);
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[u][e] *= inv;
            }
        }
        // a lane holds 4-element pieces j = 8 c + 4 half ..: lanes 32 apart swap pieces so that each stores 16 contiguous bytes
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n = n0 + 32 * u + l32;
#pragma unroll
            for (int c = 0; c < 4; c += 2) {
                u32x4 row;
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const flare_u32x2 x = __builtin_amdgcn_permlane32_swap(M_::pack2(acc[u][4 * c + 2 * d], acc[u][4 * c + 2 * d + 1]),
                                                                           M_::pack2(acc[u][4 * c + 4 + 2 * d], acc[u][4 * c + 5 + 2 * d]), false, false);
                    row[d] = x[0];
                    row[2 + d] = x[1];
                }
                if (n < wg_n1) *reinterpret_cast<u32x4*>(out + (int64_t)n * o.os[2] + 8 * (c + half)) = row;
            }
        }
    }
}

}  // namespace

bool triple32_supported(int dtype, int Dq, int Dv) { return (dtype == 1 || dtype == 2) && Dq == kD && Dv == kD; }

size_t triple32_table_bytes() { return (size_t)kTab * 16; }

hipError_t launch_triple_state32(const TripleArgs& a, int dtype, hipStream_t st)
{
    auto kern = dtype == 1 ? (a.normalize ? triple_state32_kernel<bf16_t, true> : triple_state32_kernel<bf16_t, false>)
                           : (a.normalize ? triple_state32_kernel<f16_t, true> : triple_state32_kernel<f16_t, false>);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStateLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(a.n_splits, a.H, a.B), dim3(kThreads), kStateLds, st, a);
    return hipGetLastError();
}

hipError_t launch_triple_merge32(const Triple32MergeArgs& a, int dtype, hipStream_t st)
{
    const dim3 grid((unsigned)(((size_t)a.BH * kTriple32Partial + 255) / 256));
    if (dtype == 1) hipLaunchKernelGGL(triple_merge32_kernel<bf16_t>, grid, dim3(256), 0, st, a);
    else            hipLaunchKernelGGL(triple_merge32_kernel<f16_t>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

// Tokens per workgroup of the state kernel.  A 128-token tile takes a workgroup about 1.5 us; a workgroup's partial (132 KB) is
// written and read back at the memory's pace, about 0.05 us of the whole launch each.
int triple32_tokens_per_split(int64_t N, int64_t BH)
{
    const int64_t cus = device_cus(), tiles = (N + kTok - 1) / kTok;
    int64_t best = 1;
    double best_cost = 1e30;
    for (int64_t s = 1; s <= std::min<int64_t>(tiles, 256); ++s) {
        const int64_t wgs = BH * ((tiles + s - 1) / s);
        const double cost = (double)((wgs + cus - 1) / cus) * s * 1.5 + wgs * 0.05;
        if (cost < best_cost) { best_cost = cost; best = s; }
    }
    return (int)std::max(best, (tiles + 4095) / 4096) * kTok;
}

hipError_t launch_triple_out32(Triple32OutArgs& a, int dtype, hipStream_t st)
{
    // One workgroup per compute unit at a time.  The eight waves take 512 tokens per pass (about 7 us); starting up with the
    // table costs a workgroup about one pass more: the range that ends the launch first, in whole rounds of workgroups.
    constexpr int step = 64 * kWaves;
    const int64_t rows = (int64_t)a.B * a.H * a.n_ops, steps = (a.N + step - 1) / step, cus = device_cus();
    int64_t best = 1, best_cost = INT64_MAX;
    for (int64_t s = 1; s <= std::min<int64_t>(steps, 256); ++s) {
        const int64_t cost = (rows * ((steps + s - 1) / s) + cus - 1) / cus * (s + 1);
        if (cost < best_cost) { best_cost = cost; best = s; }
    }
    a.tokens_per_wg = (int)(best * step);
    auto kern = dtype == 1 ? triple_out32_kernel<bf16_t> : triple_out32_kernel<f16_t>;
    constexpr size_t lds = (size_t)(kTab + 128) * 16;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.N + a.tokens_per_wg - 1) / a.tokens_per_wg), a.H * a.n_ops, a.B), dim3(kThreads), lds, st, a);
    return hipGetLastError();
}

}  // namespace flare
