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
// decode step. ROPE_FIGURES
//
// silu_mul_kernel: silu(gate) * up, the gate rounded to the model dtype before the product as the
// two elementwise kernels did. SILU_FIGURES
//
// few_linear_kernel: y[n][N] = x[n][K] W[N][K]^T for n <= 16 tokens on v_mfma_f32_16x16x32 (M = 16
// rows of W, N = the tokens, K = 32 a step). A decode step reads every weight once, so the bound is
// HBM: a workgroup of 8 waves takes 16 rows of W (GATE: 16 of the gate's and the same 16 of the
// up projection's) and splits K over its waves, each with 16 steps of loads (1 KB each) in flight
// before the first is used; the waves' sums meet in LDS. NORM: x is first normalised, its rows read
// before the weights' and formed while those arrive, kept in LDS in the model dtype. Epilogues:
// silu(gate) * up in fp32, or the residual row added, one rounding to the model dtype.
// FEW_FIGURES
#include <type_traits>

#include "decode_pages.hpp"

namespace starkv {

namespace {

// ---------------------------------------------------------------------------
// RoPE, cache write, fp16 rows
// ---------------------------------------------------------------------------
struct RopeParams {
    const void* q; int64_t q_s0, q_s1;  // elements; v null: q only, or q and k
    const void* k; int64_t k_s0, k_s1;
    const void* v; int64_t v_s0, v_s1;
    int dt, H, Hkv, T;
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
        if (pos < 0) pos += p.cs_rows;  // as an index counts from the end
        float c[8], s[8];
        if (pos >= 0 && pos < p.cs_rows) {
            load8_f(p.cs, pos * p.cs_s0 + d, p.cs_dt, c);
            load8_f(p.cs, pos * p.cs_s0 + 64 + d, p.cs_dt, s);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) c[e] = s[e] = __builtin_nanf("");
        }
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

template <int DT, int MODE, bool NORM>
__global__ __launch_bounds__(64 * FL_WAVES, 4) void few_linear_kernel(const FewParams p) {
    constexpr int TILES = MODE == FEW_GATE ? 2 : 1;
    constexpr int U = 4;  // steps of 32 per batch of loads, two batches in flight
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) uint8_t s_x[];  // NORM: [n][K] and 16 bytes a row
    __shared__ f32x4_t s_sum[FL_WAVES][TILES][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = rfl(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16;
    const int steps = p.K >> 5;
    const int s0 = steps * wave / FL_WAVES, s1 = steps * (wave + 1) / FL_WAVES;
    const uint16_t* wr[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) wr[i] = p.w + (int64_t)(min(row0 + m, p.N - 1) + i * p.N) * p.w_s0 + 8 * g;
    const uint16_t* xr = p.x + (int64_t)min(m, p.n - 1) * p.x_s0 + 8 * g;

    u4 a[2][TILES][U], xb[2][NORM ? 1 : U];
    auto load = [&](auto B, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 32 * min(s + u, s1 - 1);
#pragma unroll
            for (int i = 0; i < TILES; ++i) a[B][i][u] = *(const u4*)(wr[i] + k);
            if constexpr (!NORM) xb[B][u] = *(const u4*)(xr + k);
        }
    };
    const int xs = 2 * p.K + 16;  // bytes of a normalised row
    auto first = [&]() {
        if (s0 < s1) load(std::integral_constant<int, 0>{}, s0);
        if (s0 + U < s1) load(std::integral_constant<int, 1>{}, s0 + U);
    };
    if constexpr (NORM) {
        constexpr int XR = 4;  // 16-byte pieces of x a lane in flight
        // The rows of x before the weights: the wait for them leaves the weights in flight.
        for (int r = wave; r < p.n; r += FL_WAVES) {
            uint8_t* row = s_x + r * xs;
            const uint16_t* src = p.x + (int64_t)r * p.x_s0;
            float ss = 0.f;
            for (int c0 = 8 * lane; c0 < p.K; c0 += 512 * XR) {
                u4 v[XR];
#pragma unroll
                for (int i = 0; i < XR; ++i) v[i] = *(const u4*)(src + min(c0 + 512 * i, p.K - 8));
                if (r == wave && c0 == 8 * lane) first();
#pragma unroll
                for (int i = 0; i < XR; ++i) {
                    const int c = c0 + 512 * i;
                    if (c >= p.K) break;
                    *(u4*)(row + 2 * c) = v[i];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float x = few_value<DT>(v[i][e >> 1], e);
                        ss = fmaf(x, x, ss);
                    }
                }
            }
            const float rs = rsqrtf(wave_sum(ss) / (float)p.K + p.eps);
            for (int c = 8 * lane; c < p.K; c += 512) {  // the lane's own pieces
                const u4 v = *(const u4*)(row + 2 * c);
                float w[8], y[8];
                load8_f(p.nw, c, DT, w);
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = few_value<DT>(v[e >> 1], e) * rs * w[e];
                store8(row, c, DT, y);
                if (p.h && blockIdx.x == 0) store8(p.h, (int64_t)r * p.K + c, DT, y);
            }
        }
        if (wave >= p.n) first();
        __syncthreads();
    } else {
        first();
    }

    f32x4_t acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) acc[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const uint8_t* xl = s_x + min(m, p.n - 1) * xs + 16 * g;
    auto batch = [&](auto B, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u < s1) {
                u4 b;
                if constexpr (NORM) b = *(const u4*)(xl + 64 * (s + u)); else b = xb[B][u];
#pragma unroll
                for (int i = 0; i < TILES; ++i)
                    acc[i] = few_mfma<DT>(__builtin_bit_cast(uint4, a[B][i][u]), __builtin_bit_cast(uint4, b), acc[i]);
            }
        }
        if (s + 2 * U < s1) load(B, s + 2 * U);
    };
    for (int s = s0; s < s1; s += 2 * U) {
        batch(std::integral_constant<int, 0>{}, s);
        if (s + U < s1) batch(std::integral_constant<int, 1>{}, s + U);
    }
#pragma unroll
    for (int i = 0; i < TILES; ++i) s_sum[wave][i][lane] = acc[i];
    __syncthreads();
    // Thread (token c, row r) of the tile: lane 16 (r / 4) + c of each wave's sums holds it.
    const int c = tid >> 4, r = tid & 15;
    if (c < p.n && row0 + r < p.N) {
        float y[TILES];
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            y[i] = 0.f;
#pragma unroll
            for (int w = 0; w < FL_WAVES; ++w) y[i] += ((const float*)&s_sum[w][i][16 * (r >> 2) + c])[r & 3];
        }
        float o = y[0];
        if constexpr (MODE == FEW_GATE) o = silu(y[0]) * y[TILES - 1];
        if constexpr (MODE == FEW_ADD) o += load_f(p.res, (int64_t)c * p.r_s0 + row0 + r, DT);
        store_f(p.out, (int64_t)c * p.o_s0 + row0 + r, DT, o);
    }
}

template <int DT>
const void* few_pick(int mode, bool norm) {
    if (mode == FEW_GATE) return (const void*)&few_linear_kernel<DT, FEW_GATE, true>;
    if (mode == FEW_ADD) return (const void*)&few_linear_kernel<DT, FEW_ADD, false>;
    return norm ? (const void*)&few_linear_kernel<DT, FEW_PLAIN, true> : (const void*)&few_linear_kernel<DT, FEW_PLAIN, false>;
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
    p.dt = dtype; p.H = num_heads; p.Hkv = num_kv_heads; p.T = num_tokens;
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

constexpr int FEW_LDS = (160 - 16) * 1024;  // dynamic, beside up to 16 KB of sums

int starkv_few_linear_fits(int n, int K, int norm) {
    return n >= 1 && n <= 16 && K >= 32 && K % 32 == 0 &&
           (!norm || (int64_t)n * (2 * K + 16) <= FEW_LDS);
}

int starkv_few_linear(void* stream, const void* x, int64_t x_s0, const void* w, int64_t w_s0, int dtype, int n, int N,
                      int K, const void* norm_weight, float eps, void* h_out, int mode, const void* residual,
                      int64_t r_s0, void* out, int64_t o_s0) {
    clear_error();
    SKV_CHECK(dtype == STARKV_F16 || dtype == STARKV_BF16, "few_linear: bf16 or fp16");
    SKV_CHECK(N > 0 && starkv_few_linear_fits(n, K, norm_weight != nullptr), "few_linear: %d tokens, K %d", n, K);
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
    const bool norm = norm_weight != nullptr;
    const void* fn = dtype == STARKV_BF16 ? few_pick<STARKV_BF16>(mode, norm) : few_pick<STARKV_F16>(mode, norm);
    const int lds = norm ? n * (2 * K + 16) : 0;
    if (lds > 32 * 1024) SKV_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, FEW_LDS));
    void* args[] = {(void*)&p};
    SKV_HIP(hipLaunchKernel(fn, dim3((N + 15) / 16), dim3(64 * FL_WAVES), args, (size_t)lds, (hipStream_t)stream));
    return STARKV_OK;
}

}  // extern "C"
