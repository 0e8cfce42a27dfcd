// The decoder layers' small operations around the attention (the reference runs them in vLLM's
// stock Llama, starkv_serve/model.py:77-106): RoPE on q and k with the cache write of an
// uncompressed layer, the SiLU gate, and the weight products of a decode step's few tokens with
// the norm in front of them and the gate or the residual sum behind.
//
// rope_qkv_kernel: a lane takes 8 head dimensions and their rotation partners of one (token, head):
// q and k rows are rotated (fp32 products and sums rounded one by one, the result rounded once to
// the model dtype, as the elementwise form), v rows are copied; k and v go to their cache slots
// and, for prompts, also to the contiguous fp16 rows the prefill attention reads. Every value is
// read once and written once per destination; the bound is HBM for prompts, one launch for a
// decode step. 2048 tokens of 32 + 64 rows with cache and fp16 rows 26 us (134 MB), where 22
// elementwise launches, the write and two conversions took 330.
//
// silu_mul_kernel: silu(gate) * up, the gate rounded to the model dtype before the product as the
// two elementwise kernels did. 2048 tokens of 2 x 11008: 31 us (135 MB) against 56.
//
// few_linear_kernel: y[n][N] = x[n][K] W[N][K]^T for n <= 16 tokens on v_mfma_f32_16x16x32 (M = 16
// rows of W, N = the tokens, K = 32 a step). A decode step reads every weight once, so the bound is
// HBM: a workgroup of 8 waves takes 16 rows of W (GATE: 16 of the gate's and the same 16 of the
// up projection's) and splits K over its waves, each with 8 KB of loads in flight; the waves' sums
// meet in LDS. NORM (RMSNorm in front): the operand is x times the norm's weight, rounded to the
// model dtype, the squares are summed beside the products, and the sum is scaled by the token's
// 1 / rms at the end, so no pass over x comes before the weights' loads (normalising x into LDS
// first cost 3 to 5 us a product at one token). Epilogues: silu(gate) * up in fp32, or the residual
// row added; one rounding to the model dtype.
// bf16, one token, weights from HBM, us (GB/s): 4096 x 4096 with the sum 10.5 (3.2) against 17.6 for
// the library's product and torch's sum, with the norm 11.7 against 20.8; 12288 x 4096 with the norm
// 26.9 (3.7) against 33.0; the gate of 2 x 11008 x 4096 42.3 (4.3) against 63.9; 4096 x 11008 with the
// sum 21.4 (4.2) against 40.6; 32000 x 4096 with the norm 57.2 (4.6) against 67.7.
#include <type_traits>

#include "decode_pages.hpp"
#include "index_rules.hpp"

namespace starkv {

namespace {

// ---------------------------------------------------------------------------
// RoPE, cache write, fp16 rows
// ---------------------------------------------------------------------------
struct RopeParams {
    const void* q; int64_t q_s0, q_s1;  // elements; v null: q only, or q and k
    const void* k; int64_t k_s0, k_s1;
    const void* v; int64_t v_s0, v_s1;
    int dt, H, Hkv;
    const void* pos; int pos64;
    const void* cs; int64_t cs_s0; int cs_dt; int64_t cs_rows;
    void* q_out; void* k_out;           // contiguous [T][heads][128] of the model dtype, or null
    void* kc; void* vc; int64_t c_s0, c_s1, c_s2;  // paged caches, or null
    int64_t block_size, num_blocks;
    const void* slots; int slot64;
    uint16_t* k16; uint16_t* v16;       // contiguous fp16 [T][Hkv][128], or null
};

__device__ __forceinline__ void store8(void* p, int64_t i, int dt, const float* f) {
    if (dt == STARKV_F32) {
        *(float4*)((float*)p + i) = make_float4(f[0], f[1], f[2], f[3]);
        *(float4*)((float*)p + i + 4) = make_float4(f[4], f[5], f[6], f[7]);
        return;
    }
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        w[e] = dt == STARKV_F16 ? h2_bits(cvt_h2(f[2 * e], f[2 * e + 1]))
                                : (uint32_t)f32_to_bf16_rne(f[2 * e]) | ((uint32_t)f32_to_bf16_rne(f[2 * e + 1]) << 16);
    *(uint4*)((uint16_t*)p + i) = make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ float round_to(float f, int dt) {
    if (dt == STARKV_F16) return (float)(_Float16)f;
    if (dt == STARKV_BF16) return bf16_bits_to_f32(f32_to_bf16_rne(f));
    return f;
}

__device__ __forceinline__ float2 rotate(float x1, float x2, float c, float s) {
#pragma clang fp contract(off)
    return make_float2(x1 * c - x2 * s, x2 * c + x1 * s);
}

__global__ __launch_bounds__(256) void rope_qkv_kernel(const RopeParams p) {
    const int rows = p.H + (p.k ? p.Hkv : 0) + (p.v ? p.Hkv : 0);
    const int t = blockIdx.x, it = blockIdx.y * 256 + threadIdx.x;
    const int r = it >> 3, d = 8 * (it & 7);
    if (r >= rows) return;
    const bool isq = r < p.H, isv = r >= p.H + p.Hkv;
    const int h = isq ? r : isv ? r - p.H - p.Hkv : r - p.H;
    const void* src = isq ? p.q : isv ? p.v : p.k;
    const int64_t at = isq ? t * p.q_s0 + h * p.q_s1 : isv ? t * p.v_s0 + h * p.v_s1 : t * p.k_s0 + h * p.k_s1;
    float a[8], b[8];
    load8_f(src, at + d, p.dt, a);
    load8_f(src, at + 64 + d, p.dt, b);
    if (!isv) {
        int64_t pos = p.pos64 ? ((const int64_t*)p.pos)[t] : (int64_t)((const int32_t*)p.pos)[t];
        if (!wrap_index(pos, p.cs_rows)) __builtin_trap();
        float c[8], s[8];
        load8_f(p.cs, pos * p.cs_s0 + d, p.cs_dt, c);
        load8_f(p.cs, pos * p.cs_s0 + 64 + d, p.cs_dt, s);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float2 r = rotate(a[e], b[e], c[e], s[e]);
            a[e] = round_to(r.x, p.dt);
            b[e] = round_to(r.y, p.dt);
        }
    }
    const int64_t o = ((int64_t)t * (isq ? p.H : p.Hkv) + h) * 128 + d;
    if (isq) {
        store8(p.q_out, o, p.dt, a);
        store8(p.q_out, o + 64, p.dt, b);
        return;
    }
    if (!isv && p.k_out) {
        store8(p.k_out, o, p.dt, a);
        store8(p.k_out, o + 64, p.dt, b);
    }
    uint16_t* x16 = isv ? p.v16 : p.k16;
    if (x16) {
        store8(x16, o, STARKV_F16, a);
        store8(x16, o + 64, STARKV_F16, b);
    }
    if (p.kc) {
        const int64_t slot = p.slot64 ? ((const int64_t*)p.slots)[t] : (int64_t)((const int32_t*)p.slots)[t];
        if (slot < 0 || slot >= p.num_blocks * p.block_size) return;
        const int64_t c = (slot / p.block_size) * p.c_s0 + (slot % p.block_size) * p.c_s1 + h * p.c_s2 + d;
        store8(isv ? p.vc : p.kc, c, p.dt, a);
        store8(isv ? p.vc : p.kc, c + 64, p.dt, b);
    }
}

// ---------------------------------------------------------------------------
// A decode step's slots and lengths from its positions: one launch for what took ten of torch's
// on a step's critical path. A block index counts from the row's end when negative, as an index
// does; one outside the row ends the launch.
// ---------------------------------------------------------------------------
template <typename BT>
__global__ __launch_bounds__(256) void decode_slots_kernel(const BT* __restrict__ bt, int64_t s0, int64_t s1, int width,
                                                           const int64_t* __restrict__ pos, int n, int block_size,
                                                           int64_t* slots, int32_t* lens) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= n) return;
    const int64_t p = pos[b];
    int64_t blk, in;
    if (!split_position(p, block_size, width, blk, in)) __builtin_trap();
    slots[b] = (int64_t)bt[b * s0 + blk * s1] * block_size + in;
    lens[b] = (int32_t)(p + 1);
}

// ---------------------------------------------------------------------------
// The greedy step's end: tokens[b] = the first largest logit of row b (NaN largest, as argmax),
// positions[b] += 1. One workgroup a row, four 16-byte pieces a lane in flight; one
// launch for an argmax, a copy and a sum (15 + 4 + 4 us at 32,000 logits, 5 here).
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(1024) void greedy_kernel(const void* logits, int64_t s0, int width, int64_t* tokens,
                                                      int64_t* positions) {
    __shared__ unsigned long long s_k[16];
    const int b = blockIdx.x, tid = threadIdx.x;
    // A value's order as an integer (-0 as 0, every NaN above inf), then the lower index.
    const auto key = [](float v) -> uint32_t {
        const uint32_t u = __float_as_uint(v + 0.f);
        const uint32_t k = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
        return v != v ? 0xffffffffu : k;
    };
    uint32_t best = 0;
    int at = 0x7fffffff;
    const auto take = [&](float v, int i) {  // indices ascend in a lane: the first of equals stays
        const uint32_t k = key(v);
        if (k > best) {
            best = k;
            at = i;
        }
    };
    constexpr int U = 4;
    const int whole = width & ~7;
    for (int c0 = 8 * tid; c0 < whole; c0 += U * 8 * 1024) {
        float x[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) load8_f(logits, b * s0 + min(c0 + 8192 * u, whole - 8), DT, x[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + 8192 * u < whole) {
#pragma unroll
                for (int e = 0; e < 8; ++e) take(x[u][e], c0 + 8192 * u + e);
            }
    }
    if (whole + tid < width) take(load_f(logits, b * s0 + whole + tid, DT), whole + tid);
    unsigned long long m = ((unsigned long long)best << 32) | (0xffffffffu - (uint32_t)at);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_xor(m, d);
        m = o > m ? o : m;
    }
    if ((tid & 63) == 0) s_k[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w) m = s_k[w] > m ? s_k[w] : m;
        tokens[b] = (int64_t)(0xffffffffu - (uint32_t)m);
        positions[b] += 1;
    }
}

// ---------------------------------------------------------------------------
// SiLU gate
// ---------------------------------------------------------------------------
__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }

template <int DT>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ x, int64_t x_s0, uint16_t* out, int width) {
    const int64_t t = blockIdx.x;
    const int c = 8 * (blockIdx.y * 256 + (int)threadIdx.x);
    if (c >= width) return;
    float g[8], u[8];
    load8_f(x, t * x_s0 + c, DT, g);
    load8_f(x, t * x_s0 + width + c, DT, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = round_to(silu(g[e]), DT) * u[e];
    store8(out, t * width + c, DT, g);
}

// ---------------------------------------------------------------------------
// Weight products of a decode step
// ---------------------------------------------------------------------------
constexpr int FL_WAVES = 8;

struct FewParams {
    const uint16_t* x; int64_t x_s0;
    const uint16_t* w; int64_t w_s0;   // [N][K]; GATE: [2 N][K]
    const uint16_t* nw; float eps;     // NORM
    uint16_t* h;                       // NORM: the normalised rows [n][K], or null
    const uint16_t* res; int64_t r_s0;
    uint16_t* out; int64_t o_s0;
    int n, N, K;
};

enum { FEW_PLAIN = 0, FEW_ADD = 1, FEW_GATE = 2 };

template <int DT>
__device__ __forceinline__ f32x4_t few_mfma(uint4 a, uint4 b, f32x4_t c) {
    if (DT == STARKV_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                       c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0,
                                                  0, 0);
}

// Value e (of 8) of a 16-byte piece whose word e / 2 is w.
template <int DT>
__device__ __forceinline__ float few_value(uint32_t w, int e) {
    if (DT == STARKV_F16) return (float)as_h2(w)[e & 1];
    return e & 1 ? __uint_as_float(w & 0xffff0000u) : __uint_as_float(w << 16);
}

template <int DT>
__device__ __forceinline__ uint32_t few_pair(float a, float b) {
    if (DT == STARKV_F16) return h2_bits(cvt_h2(a, b));
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)b) << 16);
}

template <int DT, int MODE, bool NORM, int TILES>
__global__ __launch_bounds__(64 * FL_WAVES, 4) void few_linear_kernel(const FewParams p) {
    static_assert(MODE != FEW_GATE || TILES == 2, "the gate's rows and the up projection's");
    constexpr int U = 4 / TILES;  // steps of 32 per batch of loads, two batches in flight
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    __shared__ f32x4_t s_sum[FL_WAVES][TILES][64];
    __shared__ float s_ss[FL_WAVES][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = rfl(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    constexpr int ROWS = MODE == FEW_GATE ? 16 : 16 * TILES;  // results of the workgroup a token
    const int row0 = blockIdx.x * ROWS;
    const int steps = p.K >> 5;
    const int s0 = steps * wave / FL_WAVES, s1 = steps * (wave + 1) / FL_WAVES;
    const uint16_t* wr[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i)
        wr[i] = p.w + (MODE == FEW_GATE ? (int64_t)min(row0 + m, p.N - 1) + (int64_t)i * p.N
                                        : (int64_t)min(row0 + 16 * i + m, p.N - 1)) * p.w_s0 + 8 * g;
    const uint16_t* xr = p.x + (int64_t)min(m, p.n - 1) * p.x_s0 + 8 * g;

    u4 a[2][TILES][U], xb[2][U], nb[2][NORM ? U : 1];
    auto load = [&](auto B, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 32 * min(s + u, s1 - 1);
#pragma unroll
            for (int i = 0; i < TILES; ++i) a[B][i][u] = *(const u4*)(wr[i] + k);
            xb[B][u] = *(const u4*)(xr + k);
            if constexpr (NORM) nb[B][u] = *(const u4*)(p.nw + 8 * g + k);
        }
    };
    f32x4_t acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) acc[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
    auto batch = [&](auto B, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u < s1) {
                u4 b = xb[B][u];
                if constexpr (NORM) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x0 = few_value<DT>(b[e], 0), x1 = few_value<DT>(b[e], 1);
                        ss = fmaf(x0, x0, ss);
                        ss = fmaf(x1, x1, ss);
                        b[e] = few_pair<DT>(x0 * few_value<DT>(nb[B][u][e], 0), x1 * few_value<DT>(nb[B][u][e], 1));
                    }
                }
#pragma unroll
                for (int i = 0; i < TILES; ++i)
                    acc[i] = few_mfma<DT>(__builtin_bit_cast(uint4, a[B][i][u]), __builtin_bit_cast(uint4, b), acc[i]);
            }
        }
        if (s + 2 * U < s1) load(B, s + 2 * U);
    };
    if (s0 < s1) load(std::integral_constant<int, 0>{}, s0);
    if (s0 + U < s1) load(std::integral_constant<int, 1>{}, s0 + U);
    for (int s = s0; s < s1; s += 2 * U) {
        batch(std::integral_constant<int, 0>{}, s);
        if (s + U < s1) batch(std::integral_constant<int, 1>{}, s + U);
    }
#pragma unroll
    for (int i = 0; i < TILES; ++i) s_sum[wave][i][lane] = acc[i];
    if constexpr (NORM) s_ss[wave][lane] = ss;
    __syncthreads();
    // Thread (token c, row r) of the tile: lane 16 (r / 4) + c of each wave's sums holds it; the
    // token's squares are in lanes 16 j + c.
    const int c = (tid >> 4) & 15, r = tid & 15;
    float rs = 1.f;
    if constexpr (NORM) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < FL_WAVES; ++w)
#pragma unroll
            for (int j = 0; j < 4; ++j) t += s_ss[w][16 * j + c];
        rs = rsqrtf(t / (float)p.K + p.eps);
        if (p.h) __syncthreads();  // s_ss takes the factors below
    }
    float y[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        y[i] = 0.f;
#pragma unroll
        for (int w = 0; w < FL_WAVES; ++w) y[i] += ((const float*)&s_sum[w][i][16 * (r >> 2) + c])[r & 3];
        if constexpr (NORM) y[i] *= rs;
    }
#pragma unroll
    for (int i = 0; i < ROWS / 16; ++i) {
        const int row = row0 + 16 * i + r;
        if (row >= p.N || c >= p.n || tid >= 256) break;
        float o = y[i];
        if constexpr (MODE == FEW_GATE) o = silu(y[0]) * y[TILES - 1];
        if constexpr (MODE == FEW_ADD) o += load_f(p.res, (int64_t)c * p.r_s0 + row, DT);
        store_f(p.out, (int64_t)c * p.o_s0 + row, DT, o);
    }
    if constexpr (NORM) {
        if (p.h) {  // every workgroup writes its share of the normalised rows, 8 values a thread
            if (r == 0 && tid < 256) s_ss[0][c] = rs;
            __syncthreads();
            const int per = p.K >> 3, total = p.n * per;
            const int share = (total + (int)gridDim.x - 1) / (int)gridDim.x, i0 = share * (int)blockIdx.x;
            for (int i = i0 + tid; i < min(i0 + share, total); i += 64 * FL_WAVES) {
                const int t = i / per, k = 8 * (i - t * per);
                float x[8], w[8];
                load8_f(p.x, (int64_t)t * p.x_s0 + k, DT, x);
                load8_f(p.nw, k, DT, w);
                const float q = s_ss[0][t];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] *= q * w[e];
                store8(p.h, (int64_t)t * p.K + k, DT, x);
            }
        }
    }
}

// Two tiles of rows a workgroup where that still is two workgroups a CU: x is read again by every
// workgroup, at 16 tokens and K = 4096 as many bytes as a tile's weights. One tile, two tiles:
// 32,000 rows 59.1, 57.2 us at one token and 82.9, 73.8 at 16; 12,288 rows 26.9, 29.5 and 35.3, 36.3.
constexpr int FEW_WIDE_N = 16384;

const void* few_pick(int dt, int mode, bool norm, bool wide) {
    if (mode == FEW_GATE) return (const void*)&few_linear_kernel<STARKV_BF16, FEW_GATE, true, 2>;
    if (norm)
        return wide ? (const void*)&few_linear_kernel<STARKV_BF16, FEW_PLAIN, true, 2>
                    : (const void*)&few_linear_kernel<STARKV_BF16, FEW_PLAIN, true, 1>;
    if (mode == FEW_ADD)
        return dt == STARKV_BF16 ? (const void*)&few_linear_kernel<STARKV_BF16, FEW_ADD, false, 1>
                                 : (const void*)&few_linear_kernel<STARKV_F16, FEW_ADD, false, 1>;
    if (wide)
        return dt == STARKV_BF16 ? (const void*)&few_linear_kernel<STARKV_BF16, FEW_PLAIN, false, 2>
                                 : (const void*)&few_linear_kernel<STARKV_F16, FEW_PLAIN, false, 2>;
    return dt == STARKV_BF16 ? (const void*)&few_linear_kernel<STARKV_BF16, FEW_PLAIN, false, 1>
                             : (const void*)&few_linear_kernel<STARKV_F16, FEW_PLAIN, false, 1>;
}

}  // namespace

}  // namespace starkv

using namespace starkv;

extern "C" {

int starkv_rope_qkv(void* stream, const void* q, int64_t q_s0, int64_t q_s1, const void* k, int64_t k_s0, int64_t k_s1,
                    const void* v, int64_t v_s0, int64_t v_s1, int dtype, int num_tokens, int num_heads,
                    int num_kv_heads, const void* positions, int pos_bits, const void* cos_sin, int64_t cs_s0,
                    int cs_dtype, int64_t cs_rows, void* q_out, void* k_out, void* k_cache, void* v_cache, int64_t c_s0,
                    int64_t c_s1, int64_t c_s2, int block_size, int64_t num_blocks, const void* slot_mapping,
                    int slot_bits, void* k_half, void* v_half) {
    clear_error();
    SKV_CHECK(num_tokens >= 0 && num_heads > 0 && num_kv_heads >= 0, "rope_qkv: bad sizes");
    SKV_CHECK(dtype >= STARKV_F32 && dtype <= STARKV_BF16 && cs_dtype >= STARKV_F32 && cs_dtype <= STARKV_BF16,
              "rope_qkv: bf16, fp16 or fp32");
    SKV_CHECK((pos_bits == 32 || pos_bits == 64) && (!k_cache || slot_bits == 32 || slot_bits == 64),
              "rope_qkv: positions and slots must be int32 or int64");
    if (num_tokens == 0) return STARKV_OK;
    SKV_CHECK(q && q_out && positions && cos_sin && cs_rows > 0, "rope_qkv: null pointer");
    SKV_CHECK((!v || k) && (!k_cache || (v && v_cache && slot_mapping && block_size > 0)) && (!v_half || v) &&
                  (!k_half || k) && (!k || k_out || k_cache || k_half),
              "rope_qkv: K and V go together");
    const int al = dtype == STARKV_F32 ? 4 : 8, cal = cs_dtype == STARKV_F32 ? 4 : 8;
    SKV_CHECK(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)cos_sin | (uintptr_t)q_out | (uintptr_t)k_out |
               (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)k_half | (uintptr_t)v_half) % 16 == 0 &&
                  (q_s0 | q_s1 | k_s0 | k_s1 | v_s0 | v_s1 | c_s0 | c_s1 | c_s2) % al == 0 && cs_s0 % cal == 0,
              "rope_qkv: rows must be 16-byte aligned");
    RopeParams p;
    p.q = q; p.q_s0 = q_s0; p.q_s1 = q_s1;
    p.k = k; p.k_s0 = k_s0; p.k_s1 = k_s1;
    p.v = v; p.v_s0 = v_s0; p.v_s1 = v_s1;
    p.dt = dtype; p.H = num_heads; p.Hkv = num_kv_heads;
    p.pos = positions; p.pos64 = pos_bits == 64;
    p.cs = cos_sin; p.cs_s0 = cs_s0; p.cs_dt = cs_dtype; p.cs_rows = cs_rows;
    p.q_out = q_out; p.k_out = k_out;
    p.kc = k_cache; p.vc = v_cache; p.c_s0 = c_s0; p.c_s1 = c_s1; p.c_s2 = c_s2;
    p.block_size = block_size; p.num_blocks = num_blocks;
    p.slots = slot_mapping; p.slot64 = slot_bits == 64;
    p.k16 = (uint16_t*)k_half; p.v16 = (uint16_t*)v_half;
    const int rows = num_heads + (k ? num_kv_heads : 0) + (v ? num_kv_heads : 0);
    hipLaunchKernelGGL(rope_qkv_kernel, dim3(num_tokens, (8 * rows + 255) / 256), dim3(256), 0, (hipStream_t)stream, p);
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

int starkv_decode_slots(void* stream, const void* block_table, int64_t bt_s0, int64_t bt_s1, int bt_bits, int width,
                        const int64_t* positions, int n, int block_size, int64_t* slots, int32_t* seq_lens) {
    clear_error();
    SKV_CHECK(n >= 0 && width > 0 && block_size > 0 && (bt_bits == 32 || bt_bits == 64), "decode_slots: bad sizes");
    if (n == 0) return STARKV_OK;
    SKV_CHECK(block_table && positions && slots && seq_lens, "decode_slots: null pointer");
    if (bt_bits == 32)
        hipLaunchKernelGGL(decode_slots_kernel<int32_t>, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           (const int32_t*)block_table, bt_s0, bt_s1, width, positions, n, block_size, slots, seq_lens);
    else
        hipLaunchKernelGGL(decode_slots_kernel<int64_t>, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           (const int64_t*)block_table, bt_s0, bt_s1, width, positions, n, block_size, slots, seq_lens);
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

int starkv_greedy_step(void* stream, const void* logits, int64_t s0, int dtype, int n, int width, int64_t* tokens,
                       int64_t* positions) {
    clear_error();
    SKV_CHECK(n >= 0 && width > 0, "greedy_step: bad sizes");
    SKV_CHECK(dtype >= STARKV_F32 && dtype <= STARKV_BF16, "greedy_step: bf16, fp16 or fp32 logits");
    if (n == 0) return STARKV_OK;
    SKV_CHECK(logits && tokens && positions, "greedy_step: null pointer");
    SKV_CHECK((uintptr_t)logits % 16 == 0 && s0 % 8 == 0, "greedy_step: rows must be 16-byte aligned");
    if (dtype == STARKV_BF16)
        hipLaunchKernelGGL(greedy_kernel<STARKV_BF16>, dim3(n), dim3(1024), 0, (hipStream_t)stream, logits, s0, width,
                           tokens, positions);
    else if (dtype == STARKV_F16)
        hipLaunchKernelGGL(greedy_kernel<STARKV_F16>, dim3(n), dim3(1024), 0, (hipStream_t)stream, logits, s0, width,
                           tokens, positions);
    else
        hipLaunchKernelGGL(greedy_kernel<STARKV_F32>, dim3(n), dim3(1024), 0, (hipStream_t)stream, logits, s0, width,
                           tokens, positions);
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

int starkv_silu_mul(void* stream, const void* gate_up, int64_t s0, int dtype, int num_tokens, int width, void* out) {
    clear_error();
    SKV_CHECK(num_tokens >= 0 && width >= 0, "silu_mul: bad sizes");
    SKV_CHECK(dtype == STARKV_F16 || dtype == STARKV_BF16, "silu_mul: bf16 or fp16");
    if (num_tokens == 0 || width == 0) return STARKV_OK;
    SKV_CHECK(gate_up && out, "silu_mul: null pointer");
    SKV_CHECK(width % 8 == 0 && s0 % 8 == 0 && ((uintptr_t)gate_up | (uintptr_t)out) % 16 == 0,
              "silu_mul: rows must be 16-byte aligned");
    const dim3 grid(num_tokens, (width + 2047) / 2048);
    if (dtype == STARKV_BF16)
        hipLaunchKernelGGL(silu_mul_kernel<STARKV_BF16>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)gate_up,
                           s0, (uint16_t*)out, width);
    else
        hipLaunchKernelGGL(silu_mul_kernel<STARKV_F16>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)gate_up,
                           s0, (uint16_t*)out, width);
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

int starkv_few_linear_fits(int n, int K) {
    return n >= 1 && n <= 16 && K >= 32 && K % 32 == 0;
}

int starkv_few_linear(void* stream, const void* x, int64_t x_s0, const void* w, int64_t w_s0, int dtype, int n, int N,
                      int K, const void* norm_weight, float eps, void* h_out, int mode, const void* residual,
                      int64_t r_s0, void* out, int64_t o_s0) {
    clear_error();
    SKV_CHECK(dtype == STARKV_F16 || dtype == STARKV_BF16, "few_linear: bf16 or fp16");
    SKV_CHECK(N > 0 && starkv_few_linear_fits(n, K), "few_linear: %d tokens, K %d", n, K);
    SKV_CHECK(!norm_weight || dtype == STARKV_BF16, "few_linear: fp16 rows times the norm's weight may pass fp16's range");
    SKV_CHECK(mode >= FEW_PLAIN && mode <= FEW_GATE && (mode != FEW_GATE || norm_weight) && (mode != FEW_ADD || !norm_weight),
              "few_linear: the gate takes normalised rows, the sum plain ones");
    SKV_CHECK(x && w && out && (mode != FEW_ADD || residual) && (!h_out || norm_weight), "few_linear: null pointer");
    SKV_CHECK(((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_weight | (uintptr_t)h_out) % 16 == 0 && x_s0 % 8 == 0 &&
                  w_s0 % 8 == 0,
              "few_linear: rows must be 16-byte aligned");
    FewParams p;
    p.x = (const uint16_t*)x; p.x_s0 = x_s0; p.w = (const uint16_t*)w; p.w_s0 = w_s0;
    p.nw = (const uint16_t*)norm_weight; p.eps = eps; p.h = (uint16_t*)h_out;
    p.res = (const uint16_t*)residual; p.r_s0 = r_s0; p.out = (uint16_t*)out; p.o_s0 = o_s0;
    p.n = n; p.N = N; p.K = K;
    const bool wide = mode == FEW_PLAIN && N >= FEW_WIDE_N;
    const void* fn = few_pick(dtype, mode, norm_weight != nullptr, wide);
    const int rows = wide ? 32 : 16;
    void* args[] = {(void*)&p};
    SKV_HIP(hipLaunchKernel(fn, dim3((N + rows - 1) / rows), dim3(64 * FL_WAVES), args, 0, (hipStream_t)stream));
    return STARKV_OK;
}

}  // extern "C"
