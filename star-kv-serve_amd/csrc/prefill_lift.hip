// The lift of a prompt's codes for the dense prefill (the reference lifts every KV head in one
// batched fp32 product and rotates it, attention.py:219-241): K[t, h] = RoPE(codes[t, head h]
// @ U_h) at the token's position in its prompt, formed in fp32 and rounded once to fp16, and
// the V codes in fp16, the left operand of V's lift.
//
// prefill_lift_kernel: one wave per (32 tokens, KV head), on v_mfma_f32_32x32x2_f32: D[d][token]
// with M = 32 head dimensions in each of 4 blocks, N = the 32 tokens, K = 2 ranks a step. Row i
// of block b stands for dimension 4 i + b, so a lane's A operands of the four blocks are one
// 16-byte load of a row of the fp32 U as it lies in memory, and it ends up with runs of 16
// dimensions of one token, d and its rotation partner d + 64 both among them. B = the codes,
// converted in registers. A sum is one fp32 chain whose ranks go by eights in the order
// 0 2 4 6 1 3 5 7 (two codes a 32-bit word: a lane takes the low, then the high halves of its
// two words), and the rotation's products and sums are rounded one by one (no contraction):
// bit for bit the keys of the batched fp32 product and elementwise rotation it replaced. The
// rows go through 8 KB of LDS per wave and out as whole 256-byte rows.
// The work is 2 T W 128 operations, 6 us of the fp32 matrix rate at 4096 tokens of W = 880, and
// the bound is that and the latency of a wave's few dependent loads.
// At 32 heads and W = 880, traced: 4096 tokens 31 us where those launches (a gather, conversions, a
// transposed copy, the product, six elementwise kernels, a concatenation) took 233; 6368 tokens in
// 7 prompts 39 us against 366. With the cos/sin values read after the products (96 registers, five
// waves a SIMD instead of two) 26 and 36 us.
// The V planes (grid.y past the head groups) convert the V codes of 32 tokens.
#include "decode_pages.hpp"

namespace starkv {

namespace {

constexpr int LIFT_TOK = 32;
constexpr int LIFT_WAVES = 4;
constexpr int LIFT_VWG = 4;      // workgroups converting the V codes of 32 tokens

struct LiftParams {
    const void* k; int64_t k_s0;       // elements
    const void* v; int64_t v_s0;
    int T, H, P;
    const int32_t* cu;
    const float* u; int64_t u_s0;      // [W][128]
    const int32_t* offs; const int32_t* widths;
    const void* cs; int64_t cs_s0;
    uint8_t* ko;                       // fp16 [T][H][128]
    uint16_t* vo; int v_rank;          // fp16 [T][v_rank]
    int hplanes;
};

// 16 bytes at any 2-byte boundary (a row of codes is as long as its ranks add up to).
struct __attribute__((packed, aligned(2))) Unaligned16 {
    uint32_t w[4];
};
// 16 consecutive cos or sin values, read as they are and converted where used.
template <int CDT>
struct LiftTrig {
    uint32_t w[CDT == STARKV_F32 ? 16 : 8];
    __device__ __forceinline__ void load(const void* p, int64_t i) {
        struct __attribute__((packed, aligned(CDT == STARKV_F32 ? 4 : 2))) Raw {
            uint32_t w[4];
        };
        const Raw* r = (const Raw*)((const uint8_t*)p + i * (CDT == STARKV_F32 ? 4 : 2));
#pragma unroll
        for (int k = 0; k < (CDT == STARKV_F32 ? 4 : 2); ++k) {
            const Raw x = r[k];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * k + e] = x.w[e];
        }
    }
    __device__ __forceinline__ float at(int e) const {
        if (CDT == STARKV_F32) return __uint_as_float(w[e]);
        if (CDT == STARKV_F16) return (float)as_h2(w[e >> 1])[e & 1];
        return e & 1 ? __uint_as_float(w[e >> 1] & 0xffff0000u) : __uint_as_float(w[e >> 1] << 16);
    }
};

// The rank of step s (of 8) and lane half hh among 16.
__device__ __forceinline__ int lift_rank(int s, int hh) { return 8 * (s >> 2) + 4 * (s & 1) + ((s >> 1) & 1) + 2 * hh; }

// Ranks [r0, r0 + 16) of a head (zeros from rank `width` on) as the B operands of 8 steps:
// x[s] is rank r0 + lift_rank(s, hh).
template <int DT>
__device__ __forceinline__ void lift_codes(const void* k, int64_t i, int r0, int width, int hh, float* x) {
    if (DT != STARKV_F32 && r0 + 16 <= width) {
        const Unaligned16* p = (const Unaligned16*)((const uint16_t*)k + i + r0);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const Unaligned16 a = p[g];
            const uint32_t w[2] = {hh ? a.w[1] : a.w[0], hh ? a.w[3] : a.w[2]};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t v = w[s & 1];
                if (DT == STARKV_BF16)
                    x[4 * g + s] = s < 2 ? __uint_as_float(v << 16) : __uint_as_float(v & 0xffff0000u);
                else
                    x[4 * g + s] = (float)as_h2(v)[s >> 1];
            }
        }
        return;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int r = r0 + lift_rank(s, hh);
        x[s] = r < width ? load_f(k, i + r, DT) : 0.f;
    }
}

// The V codes' elements [e0, e1) of the fp16 rows laid end to end, 8 a lane (e0 a multiple of 8).
template <int DT>
__device__ __forceinline__ void lift_v(const LiftParams& p, int64_t e0, int64_t e1) {
    for (int64_t e = e0 + 8 * (int)threadIdx.x; e < e1; e += 8 * 64 * LIFT_WAVES) {
        int64_t t = e / p.v_rank;
        int c = (int)(e - t * p.v_rank);
        half8_t o;
        if (DT != STARKV_F32 && c + 8 <= p.v_rank) {
            const Unaligned16 x = *(const Unaligned16*)((const uint16_t*)p.v + t * p.v_s0 + c);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[2 * i] = (_Float16)__uint_as_float(x.w[i] << 16);
                o[2 * i + 1] = (_Float16)__uint_as_float(x.w[i] & 0xffff0000u);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                o[i] = t < p.T ? (_Float16)load_f(p.v, t * p.v_s0 + c, DT) : (_Float16)0.f;
                if (++c == p.v_rank) {
                    c = 0;
                    ++t;
                }
            }
        }
        if (e + 8 <= e1)
            *(half8_t*)(p.vo + e) = o;
        else
            for (int i = 0; i < (int)(e1 - e); ++i) ((_Float16*)p.vo)[e + i] = o[i];
    }
}

__device__ __forceinline__ float2 lift_rotate(float x1, float x2, float c, float s) {
#pragma clang fp contract(off)
    return make_float2(x1 * c - x2 * s, x2 * c + x1 * s);
}

template <int DT, int CDT>
__global__ __launch_bounds__(64 * LIFT_WAVES, CDT == STARKV_F32 ? 3 : 4) void prefill_lift_kernel(const LiftParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t s_rows[LIFT_WAVES][LIFT_TOK * 256];
    const int lane = threadIdx.x & 63, wave = rfl(threadIdx.x >> 6);
    const int t0 = blockIdx.x * LIFT_TOK;
    if ((int)blockIdx.y >= p.hplanes) {
        // 32 rows are a multiple of 8 elements: every piece but the tensor's last is whole.
        const int64_t n8 = (int64_t)LIFT_TOK * p.v_rank / 8, j = (int)blockIdx.y - p.hplanes;
        const int64_t base = (int64_t)t0 * p.v_rank, end = (int64_t)p.T * p.v_rank;
        lift_v<DT>(p, base + 8 * (n8 * j / LIFT_VWG), min(base + 8 * (n8 * (j + 1) / LIFT_VWG), end));
        return;
    }
    const int h = (int)blockIdx.y * LIFT_WAVES + wave;
    if (h >= p.H) return;
    const int n = lane & 31, hh = lane >> 5;
    const int t = min(t0 + n, p.T - 1);
    const int off = rfl(p.offs[h]), width = rfl(p.widths[h]);

    // The token's position in its prompt: the last cu[i] <= t (empty prompts repeat a start).
    int lo = 0, hi = p.P - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (p.cu[mid] <= t) lo = mid; else hi = mid - 1;
    }
    const int64_t row = (int64_t)(t - p.cu[lo]) * p.cs_s0 + 16 * hh;
    const int64_t code = (int64_t)t * p.k_s0 + off;
    const float* u = p.u + (int64_t)off * p.u_s0 + 4 * n;
    f32x16_t z[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) z[b] = (f32x16_t){};
#pragma unroll 1
    for (int r0 = 0; r0 < width; r0 += 16) {
        float x[8];
        lift_codes<DT>(p.k, code, r0, width, hh, x);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            float4 a[4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
                a[s] = *(const float4*)(u + (int64_t)min(r0 + lift_rank(4 * g + s, hh), width - 1) * p.u_s0);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                z[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s].x, x[4 * g + s], z[0], 0, 0, 0);
                z[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s].y, x[4 * g + s], z[1], 0, 0, 0);
                z[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s].z, x[4 * g + s], z[2], 0, 0, 0);
                z[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s].w, x[4 * g + s], z[3], 0, 0, 0);
            }
        }
    }
    LiftTrig<CDT> cs[2], sn[2];  // dimensions 32 j + 16 hh .. + 15
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        cs[j].load(p.cs, row + 32 * j);
        sn[j].load(p.cs, row + 64 + 32 * j);
    }
    // z[b][4 j + e] is dimension 32 j + 16 hh + 4 e + b of token n; j + 2 holds the partners.
    uint8_t* rows = s_rows[wave];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int half = 0; half < 2; ++half) {  // 8 dimensions: one 16-byte granule, swizzled by the token
            half8_t x1, x2;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int e = 2 * half + (i >> 2), b = i & 3;
                const float k1 = z[b][4 * j + e], k2 = z[b][4 * (j + 2) + e];
                const float c = cs[j].at(4 * e + b), s = sn[j].at(4 * e + b);
                const float2 r = lift_rotate(k1, k2, c, s);
                x1[i] = (_Float16)r.x;
                x2[i] = (_Float16)r.y;
            }
            const int g = 4 * j + 2 * hh + half;
            *(half8_t*)(rows + n * 256 + ((g ^ (n & 15)) << 4)) = x1;
            *(half8_t*)(rows + n * 256 + (((g + 8) ^ (n & 15)) << 4)) = x2;
        }
    // The wave's own rows (LDS operations of a wave stay in order): 4 rows a store.
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < LIFT_TOK / 4; ++i) {
        const int r = 4 * i + (lane >> 4), g = lane & 15;
        const uint4 v = *(const uint4*)(rows + r * 256 + ((g ^ (r & 15)) << 4));
        if (t0 + r < p.T) *(uint4*)(p.ko + ((int64_t)(t0 + r) * p.H + h) * 256 + 16 * g) = v;
    }
}

template <int DT>
const void* lift_pick(int cdt) {
    if (cdt == STARKV_F32) return (const void*)&prefill_lift_kernel<DT, STARKV_F32>;
    if (cdt == STARKV_F16) return (const void*)&prefill_lift_kernel<DT, STARKV_F16>;
    return (const void*)&prefill_lift_kernel<DT, STARKV_BF16>;
}

}  // namespace

}  // namespace starkv

using namespace starkv;

extern "C" {

int starkv_prefill_lift(void* stream, const void* k_codes, int64_t k_s0, const void* v_codes, int64_t v_s0,
                        int code_dtype, int num_tokens, const int32_t* cu_seqlens, int num_prompts, const float* k_up,
                        int64_t u_s0, const int32_t* k_offsets, const int32_t* k_widths, int num_kv_heads,
                        const void* cos_sin, int64_t cs_s0, int cs_dtype, void* key, void* v_out, int v_rank) {
    clear_error();
    SKV_CHECK(num_tokens >= 0 && num_prompts >= 0 && num_kv_heads > 0, "prefill_lift: bad sizes");
    if (num_tokens == 0) return STARKV_OK;
    SKV_CHECK(num_prompts > 0, "prefill_lift: tokens without a prompt");
    SKV_CHECK(k_codes && cu_seqlens && k_up && k_offsets && k_widths && cos_sin && key, "prefill_lift: null pointer");
    SKV_CHECK(code_dtype >= STARKV_F32 && code_dtype <= STARKV_BF16 && cs_dtype >= STARKV_F32 && cs_dtype <= STARKV_BF16,
              "prefill_lift: codes and cos/sin must be bf16, fp16 or fp32");
    SKV_CHECK(((uintptr_t)key % 16) == 0 && ((uintptr_t)k_up % 16) == 0 && u_s0 % 4 == 0,
              "prefill_lift: K and the rows of U must be 16-byte aligned");
    if (v_out) {
        SKV_CHECK(v_codes && v_rank > 0, "prefill_lift: no V codes");
        SKV_CHECK(code_dtype != STARKV_F16, "prefill_lift: fp16 V codes need no conversion");
        SKV_CHECK(((uintptr_t)v_out % 16) == 0, "prefill_lift: V rows must be 16-byte aligned");
    }
    LiftParams p;
    p.k = k_codes; p.k_s0 = k_s0;
    p.v = v_codes; p.v_s0 = v_s0;
    p.T = num_tokens; p.H = num_kv_heads; p.P = num_prompts;
    p.cu = cu_seqlens;
    p.u = k_up; p.u_s0 = u_s0; p.offs = k_offsets; p.widths = k_widths;
    p.cs = cos_sin; p.cs_s0 = cs_s0;
    p.ko = (uint8_t*)key;
    p.vo = (uint16_t*)v_out; p.v_rank = v_rank;
    p.hplanes = (num_kv_heads + LIFT_WAVES - 1) / LIFT_WAVES;
    const dim3 grid((num_tokens + LIFT_TOK - 1) / LIFT_TOK, p.hplanes + (v_out ? LIFT_VWG : 0));
    const void* fn = code_dtype == STARKV_BF16  ? lift_pick<STARKV_BF16>(cs_dtype)
                     : code_dtype == STARKV_F16 ? lift_pick<STARKV_F16>(cs_dtype)
                                                : lift_pick<STARKV_F32>(cs_dtype);
    void* args[] = {(void*)&p};
    SKV_HIP(hipLaunchKernel(fn, grid, dim3(64 * LIFT_WAVES), args, 0, (hipStream_t)stream));
    return STARKV_OK;
}

}  // extern "C"
