// Cache write path: the bf16/fp16 code scatter and the 3.2-bit quantize + scatter
// (the quantizer and the row packing are in pack_rows.hpp). One wave quantizes one
// (token, KV head) block, or the token's V latent.
#include <stdarg.h>
#include <stdio.h>

#include "kv_gemm.hpp"
#include "pack_rows.hpp"

namespace starkv {

static thread_local char g_err[512];

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

void clear_error() { g_err[0] = 0; }

// ---------------------------------------------------------------------------
// bf16/fp16 codes: one wave copies a token's K and V codes to its slot in pieces of G bytes
// (16, or 4 or 2 over a whole workgroup: the widest that both sides' rows, strides and widths
// are multiples of), four pieces a lane in flight. The bound is the two copies of the rows in
// HBM, or the latency of a slot and a row at few tokens. 2160 codes a token, replayed from a
// graph, against a workgroup a token copying single codes: 6368 tokens 22.3 -> 10.3 us, 4096
// 13.8 -> 6.8, 64 3.96 -> 3.11, one 3.68 -> 2.73.
// ---------------------------------------------------------------------------
struct WriteCodesParams {
    const uint8_t* k; int64_t k_s0;  // bytes
    const uint8_t* v; int64_t v_s0;
    uint8_t* cache; int64_t c_s0, c_s1;
    int block_size; int64_t num_blocks;
    const void* slots; int slot_bits;
    int n, k_pieces, pieces;         // pieces of a row, of its K part
};

template <int G>
struct WritePiece;
template <>
struct WritePiece<16> { typedef uint32_t T __attribute__((ext_vector_type(4))); };
template <>
struct WritePiece<4> { typedef uint32_t T; };
template <>
struct WritePiece<2> { typedef uint16_t T; };

template <int G>
__global__ __launch_bounds__(256) void write_codes_kernel(const WriteCodesParams p) {
    typedef typename WritePiece<G>::T T;
    constexpr int U = 4, L = G == 16 ? 64 : 256;  // pieces a lane in flight, lanes of a token
    const int i = blockIdx.x * (256 / L) + (int)threadIdx.x / L, lane = (int)threadIdx.x % L;
    if (i >= p.n) return;
    const int64_t slot = load_slot(p.slots, p.slot_bits, i);
    if (slot >= p.num_blocks * p.block_size) return;
    const T* ks = (const T*)(p.k + (int64_t)i * p.k_s0);
    const T* vs = (const T*)(p.v + (int64_t)i * p.v_s0) - p.k_pieces;
    T* dst = (T*)(p.cache + (slot / p.block_size) * p.c_s0 + (slot % p.block_size) * p.c_s1);
    for (int c0 = 0; c0 < p.pieces; c0 += L * U) {
        T x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = min(c0 + L * u + lane, p.pieces - 1);
            x[u] = *(c < p.k_pieces ? ks + c : vs + c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + L * u + lane;
            if (c < p.pieces) dst[c] = x[u];
        }
    }
}

// Codes of another dtype than the cache's (or fp32), converted: one workgroup per token.
__global__ __launch_bounds__(256) void convert_codes_kernel(const void* __restrict__ k, int64_t k_s0,
                                                            const void* __restrict__ v, int64_t v_s0, int in_dt,
                                                            void* __restrict__ cache, int64_t c_s0, int64_t c_s1,
                                                            int cache_dt, int block_size, int64_t num_blocks,
                                                            const void* __restrict__ slots, int slot_bits,
                                                            int k_width, int v_rank) {
    const int i = blockIdx.x;
    const int64_t slot = load_slot(slots, slot_bits, i);
    if (slot >= num_blocks * block_size) return;
    const int64_t row = (slot / block_size) * c_s0 + (slot % block_size) * c_s1;
    const int width = k_width + v_rank;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        float x = c < k_width ? load_f(k, (int64_t)i * k_s0 + c, in_dt) : load_f(v, (int64_t)i * v_s0 + c - k_width, in_dt);
        store_f(cache, row + c, cache_dt, x);
    }
}

// ---------------------------------------------------------------------------
// 3.2-bit pack straight from memory, for rows of codes too long for LDS. Grid (n tokens,
// ceil((H + 1) / 4)); wave u of the token quantizes KV head u (u < H) or the V latent (u == H).
// ---------------------------------------------------------------------------
struct PackParams {
    const void* k; int64_t k_s0;
    const void* v; int64_t v_s0;
    int dt;
    uint8_t* cache; int64_t c_s0, c_s1;
    int block_size;
    int64_t num_blocks;
    const void* slots; int slot_bits;
    int H;
    const int32_t* ranks; const int32_t* offsets; const int32_t* nouts;
    int k_width, v_rank, v_nout, v_nbo, v_bytes;
    int ks_off, vs_off, vq_off, row_bytes;
};

__global__ __launch_bounds__(256) void pack_kv_kernel(const PackParams p) {
    const int i = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int u = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (u > p.H) return;
    const int64_t slot = load_slot(p.slots, p.slot_bits, i);
    if (slot >= p.num_blocks * p.block_size) return;
    uint8_t* row = p.cache + (slot / p.block_size) * p.c_s0 + (slot % p.block_size) * p.c_s1;

    if (u < p.H) {
        const int64_t base = (int64_t)i * p.k_s0 + p.offsets[u];
        pack_k_block([&](int l) { return load_f(p.k, base + l, p.dt); }, p.ranks[u], p.nouts[u], p.offsets[u], u,
                     p.ks_off, row, lane);
        return;
    }
    const int64_t base = (int64_t)i * p.v_s0;
    pack_v_block([&](int c) { return load_f(p.v, base + c, p.dt); }, p.v_rank, p.v_nout, p.v_nbo, p.v_bytes, p.vq_off,
                 p.vs_off, p.row_bytes, row, lane);
}

// ---------------------------------------------------------------------------
// 3.2-bit pack: one workgroup of 4 waves per token. The row's codes are read once
// with 16-byte loads into LDS; a 16-lane row takes a KV head (16 heads at a time: the maxima are
// reductions inside the row, a lane packs every 16th byte), all lanes the V latent; the finished
// row, assembled in LDS, goes out in whole 4-byte words. Against one wave per (token, head), whose
// 64 lanes met heads of 16 to 48 codes and stored single bytes (32 heads, W 880, V rank 1290,
// replayed from a graph): 4096 tokens 64.6 -> 20.5 us, 256 13.4 -> 5.9, one 10.2 -> 5.4. The
// bound is the instructions of the quantizer.
// ---------------------------------------------------------------------------
template <int DT>
struct PackElem { typedef uint16_t T; };
template <>
struct PackElem<STARKV_F32> { typedef float T; };

struct __attribute__((packed, aligned(2))) PackLoad16 {
    uint32_t w[4];
};

// Elements [i, i + n) of src into LDS at dst (16-byte aligned), 16 bytes a lane.
template <int DT>
__device__ __forceinline__ void pack_stage(const void* src, int64_t i, int n, typename PackElem<DT>::T* dst) {
    typedef typename PackElem<DT>::T T;
    constexpr int E = 16 / (int)sizeof(T);
    const T* s = (const T*)src + i;
    for (int c = E * (int)threadIdx.x; c < n; c += E * 256) {
        if (c + E <= n) {
            const PackLoad16 x = *(const PackLoad16*)(s + c);
            *(uint4*)(dst + c) = make_uint4(x.w[0], x.w[1], x.w[2], x.w[3]);
        } else {
            for (int k = c; k < n; ++k) dst[k] = s[k];
        }
    }
}

template <int DT>
__global__ __launch_bounds__(256) void pack_rows_kernel(const PackParams p) {
    typedef typename PackElem<DT>::T T;
    extern __shared__ __attribute__((aligned(16))) uint8_t s_mem[];
    __shared__ float s_max[8];
    uint8_t* s_row = s_mem;                          // row_bytes (a multiple of 16)
    T* s_k = (T*)(s_mem + p.row_bytes);              // k_width (a multiple of 16) codes, then V
    T* s_v = s_k + p.k_width;
    const int i = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = tid >> 4, l16 = tid & 15;
    const int64_t slot = load_slot(p.slots, p.slot_bits, i);
    if (slot >= p.num_blocks * p.block_size) return;  // the whole workgroup
    uint8_t* row = p.cache + (slot / p.block_size) * p.c_s0 + (slot % p.block_size) * p.c_s1;
    const auto val = [](T x) { return DT == STARKV_F32 ? (float)x : code_value_rt(__builtin_bit_cast(uint16_t, (uint16_t)x), DT); };

    // Bytes of K lanes that no head holds stay as they are in the cache.
    int held = 0;
    for (int u = lane; u < p.H; u += 64) held += (p.ranks[u] + 15) & ~15;
    const bool whole = wave_sum((float)held) == (float)p.k_width;
    pack_stage<DT>(p.k, (int64_t)i * p.k_s0, p.k_width, s_k);
    pack_stage<DT>(p.v, (int64_t)i * p.v_s0, p.v_rank, s_v);
    if (!whole)
        for (int j = 4 * tid; j < p.ks_off; j += 4 * 256) *(uint32_t*)(s_row + j) = *(const uint32_t*)(row + j);
    int rank = 0, nout = 0, off = 0;  // of the row's next head, read a round ahead
    const auto head = [&](int u) {
        if (u < p.H) {
            rank = p.ranks[u];
            nout = p.nouts[u];
            off = p.offsets[u];
        }
    };
    head(r16);
    __syncthreads();

    for (int u = r16; u < p.H; u += 16) {
        const int wh = (rank + 15) & ~15, no = nout, o = off;
        head(u + 16);
        float a_out = 0.f, a_in = 0.f;
        for (int l = l16; l < wh; l += 16) {
            const float x = fabsf(val(s_k[o + l]));
            if (l < no) a_out = fmaxf(a_out, x); else a_in = fmaxf(a_in, x);
        }
        const VScales s = v_scales(row16_max(a_out), row16_max(a_in));
        for (int kb = l16; 2 * kb < wh; kb += 16) {
            const int l = 2 * kb;
            const float x0 = val(s_k[o + l]), x1 = val(s_k[o + l + 1]);
            const int n0 = quant_code_of(x0, l < no, s), n1 = quant_code_of(x1, l + 1 < no, s);
            s_row[o / 2 + kb] = (uint8_t)(n0 | (n1 << 4));
        }
        if (l16 == 0) {
            const uint16_t so = f32_to_bf16_rne(no > 0 ? s.s_out : 1.0f), si = f32_to_bf16_rne(s.s_in);
            *(uint32_t*)(s_row + p.ks_off + 4 * u) = (uint32_t)so | ((uint32_t)si << 16);
        }
    }
    float a_out = 0.f, a_in = 0.f;
    for (int c = tid; c < p.v_rank; c += 256) {
        const float x = fabsf(val(s_v[c]));
        if (c < p.v_nout) a_out = fmaxf(a_out, x); else a_in = fmaxf(a_in, x);
    }
    a_out = wave_max(a_out);
    a_in = wave_max(a_in);
    if (lane == 0) {
        s_max[wave] = a_out;
        s_max[4 + wave] = a_in;
    }
    __syncthreads();
    const VScales s = v_scales(fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3])),
                               fmaxf(fmaxf(s_max[4], s_max[5]), fmaxf(s_max[6], s_max[7])));
    for (int j = tid; j < p.v_bytes; j += 256)
        s_row[p.vq_off + j] = pack_v_byte([&](int c) { return val(s_v[c]); }, j, p.v_rank, p.v_nout, p.v_nbo, s);
    if (wave == 0) pack_v_tail(s, p.v_nout, p.v_bytes, p.vq_off, p.vs_off, p.row_bytes, s_row, lane);
    __syncthreads();
    for (int j = 4 * tid; j < p.row_bytes; j += 4 * 256) *(uint32_t*)(row + j) = *(const uint32_t*)(s_row + j);
}

}  // namespace starkv

using namespace starkv;

extern "C" {

int starkv_abi_version(void) { return 7; }

const char* starkv_last_error(void) { return g_err; }

int starkv_write_codes(void* stream, const void* k_codes, int64_t k_s0, const void* v_codes, int64_t v_s0,
                       int in_dtype, void* cache, int64_t c_s0, int64_t c_s1, int cache_dtype, int block_size,
                       int64_t num_blocks, const void* slot_mapping, int slot_bits, int n, int k_width,
                       int v_rank) {
    clear_error();
    if (const int rc = flush_pending_write()) return rc;  // a deferred write goes first
    SKV_CHECK(n >= 0 && k_width >= 0 && v_rank >= 0, "write_codes: negative size");
    SKV_CHECK(block_size > 0, "write_codes: block_size must be positive");
    SKV_CHECK(slot_bits == 32 || slot_bits == 64, "write_codes: slot_mapping must be int32 or int64");
    SKV_CHECK(in_dtype >= 0 && in_dtype <= 2 && cache_dtype >= 0 && cache_dtype <= 2, "write_codes: bad dtype");
    if (n == 0) return STARKV_OK;
    SKV_CHECK(k_codes && v_codes && cache && slot_mapping, "write_codes: null pointer");
    if (in_dtype == cache_dtype && in_dtype != STARKV_F32) {
        if (k_width + v_rank == 0) return STARKV_OK;
        WriteCodesParams p;
        p.k = (const uint8_t*)k_codes; p.k_s0 = 2 * k_s0;
        p.v = (const uint8_t*)v_codes; p.v_s0 = 2 * v_s0;
        p.cache = (uint8_t*)cache; p.c_s0 = 2 * c_s0; p.c_s1 = 2 * c_s1;
        p.block_size = block_size; p.num_blocks = num_blocks; p.slots = slot_mapping; p.slot_bits = slot_bits;
        p.n = n;
        const int64_t all = (int64_t)(uintptr_t)k_codes | (int64_t)(uintptr_t)v_codes | (int64_t)(uintptr_t)cache | p.k_s0 |
                            p.v_s0 | p.c_s0 | p.c_s1 | (2 * (int64_t)k_width) | (2 * (int64_t)v_rank);
        const int g = all % 16 == 0 ? 16 : all % 4 == 0 ? 4 : 2;
        p.k_pieces = 2 * k_width / g;
        p.pieces = 2 * (k_width + v_rank) / g;
        const dim3 grid(g == 16 ? (n + 3) / 4 : n);
        if (g == 16)
            hipLaunchKernelGGL(write_codes_kernel<16>, grid, dim3(256), 0, (hipStream_t)stream, p);
        else if (g == 4)
            hipLaunchKernelGGL(write_codes_kernel<4>, grid, dim3(256), 0, (hipStream_t)stream, p);
        else
            hipLaunchKernelGGL(write_codes_kernel<2>, grid, dim3(256), 0, (hipStream_t)stream, p);
    } else {
        hipLaunchKernelGGL(convert_codes_kernel, dim3(n), dim3(256), 0, (hipStream_t)stream, k_codes, k_s0, v_codes,
                           v_s0, in_dtype, cache, c_s0, c_s1, cache_dtype, block_size, num_blocks, slot_mapping,
                           slot_bits, k_width, v_rank);
    }
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

int starkv_pack_kv(void* stream, const void* k_codes, int64_t k_s0, const void* v_codes, int64_t v_s0,
                   int code_dtype, uint8_t* cache, int64_t c_s0, int64_t c_s1, int block_size, int64_t num_blocks,
                   const void* slot_mapping, int slot_bits, int n, int num_kv_heads, const int32_t* k_ranks,
                   const int32_t* k_offsets, const int32_t* k_nouts, int k_width, int v_rank, int row_bytes) {
    clear_error();
    if (const int rc = flush_pending_write()) return rc;  // a deferred write goes first
    SKV_CHECK(n >= 0 && num_kv_heads > 0 && k_width > 0 && v_rank > 0, "pack_kv: bad sizes");
    SKV_CHECK(k_width % 16 == 0, "pack_kv: k_width must be a multiple of 16 (head widths are)");
    SKV_CHECK(block_size > 0, "pack_kv: block_size must be positive");
    SKV_CHECK(slot_bits == 32 || slot_bits == 64, "pack_kv: slot_mapping must be int32 or int64");
    SKV_CHECK(code_dtype >= 0 && code_dtype <= 2, "pack_kv: bad dtype");
    PackParams p;
    p.k = k_codes; p.k_s0 = k_s0; p.v = v_codes; p.v_s0 = v_s0; p.dt = code_dtype;
    SKV_CHECK(c_s0 % 4 == 0 && c_s1 % 4 == 0 && ((uintptr_t)cache % 4) == 0,
              "pack_kv: cache base and byte strides must be multiples of 4");
    p.cache = cache; p.c_s0 = c_s0; p.c_s1 = c_s1; p.block_size = block_size; p.num_blocks = num_blocks;
    p.slots = slot_mapping; p.slot_bits = slot_bits; p.H = num_kv_heads;
    p.ranks = k_ranks; p.offsets = k_offsets; p.nouts = k_nouts;
    p.k_width = k_width; p.v_rank = v_rank;
    const RowLayout rl = row_layout_host(k_width, num_kv_heads, v_rank);
    p.v_nout = rl.v_nout;
    p.v_nbo = rl.v_nbo;
    p.v_bytes = rl.v_bytes;
    p.ks_off = rl.ks_off;
    p.vs_off = rl.vs_off;
    p.vq_off = rl.vq_off;
    p.row_bytes = rl.nbytes;
    SKV_CHECK(row_bytes == p.row_bytes, "pack_kv: row_bytes %d != QuantRow.nbytes %d", row_bytes, p.row_bytes);
    if (n == 0) return STARKV_OK;
    SKV_CHECK(k_codes && v_codes && cache && slot_mapping && k_ranks && k_offsets && k_nouts, "pack_kv: null pointer");
    // One workgroup's LDS without raising its limit: 64 KB.
    const int64_t lds = (int64_t)row_bytes + (int64_t)(k_width + v_rank) * (code_dtype == STARKV_F32 ? 4 : 2);
    if (lds <= 60 * 1024) {
        if (code_dtype == STARKV_BF16)
            hipLaunchKernelGGL(pack_rows_kernel<STARKV_BF16>, dim3(n), dim3(256), (size_t)lds, (hipStream_t)stream, p);
        else if (code_dtype == STARKV_F16)
            hipLaunchKernelGGL(pack_rows_kernel<STARKV_F16>, dim3(n), dim3(256), (size_t)lds, (hipStream_t)stream, p);
        else
            hipLaunchKernelGGL(pack_rows_kernel<STARKV_F32>, dim3(n), dim3(256), (size_t)lds, (hipStream_t)stream, p);
    } else {
        hipLaunchKernelGGL(pack_kv_kernel, dim3(n, (num_kv_heads + 1 + 3) / 4), dim3(256), 0, (hipStream_t)stream, p);
    }
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

}  // extern "C"
