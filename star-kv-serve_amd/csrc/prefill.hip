// Dense causal prefill attention of the STAR-KV attention layer (the reference runs it on
// vLLM's FlashAttention: attention.py:219-251 lifts K and V from the step's codes, then
// flash_attn_varlen_func(causal=True) over the prompts). Every prompt attends to itself
// only (no cached context): out[t, h] = softmax(scale q[t, h] . K[s .. t, h / G]) V[s .. t,
// h / G] for token t of the prompt starting at s.
//
// Inputs: q [T, Hq, 128] (bf16, fp16 or fp32; converted to fp16 on load), K and V
// [T, Hkv, 128] fp16 (the lifted keys and values, rounded once to fp16), cu_seqlens
// [P + 1] (the prompts' first tokens), and a block list: per workgroup row, (prompt,
// 128-row query block) (starkv_prefill_block_list writes it on the host).
//
// prefill_kernel: one workgroup of 4 waves per (query block of 128 rows, query head); wave
// w takes query rows 32 w .. 32 w + 31 of the block. Keys go by tiles of 64, K and V of a
// tile copied global->LDS by all waves (buffer loads that write LDS, bounded to the
// prompt's rows), the next tile in flight while one is used. The block list puts the
// blocks with the most keys first. Per tile and wave, on v_mfma_f32_32x32x16_f16:
//   S^T = K Q^T: M = 32 keys (two blocks per tile), N = the wave's 32 queries, K = the 128
//     head dimensions (8 steps); A = a K row's 8 dimensions (ds_read_b128), B = Q
//     in registers for the whole kernel.
//   Each lane then holds 32 scores of one query (column n = lane % 32) and its partner lane
//     (lane ^ 32) the other 32: causal and prompt-end masking, an online softmax in the
//     log2 domain with a lazy reference max (it moves only when a score exceeds it by
//     2^8), one lane swap per tile for the max.
//   O^T += V^T P^T: M = 32 head dimensions (4 blocks), N = the queries, K = 16 keys (4
//     steps). The lane's P values of one step are already the B operand if the K index
//     8 h + e (h = lane / 32) stands for key 4 h + e (e < 4) or 8 + 4 h + e - 4; A = V^T with
//     the same key order, read with ds_read_b64_tr_b16 (4 key rows x 16 dimensions per
//     16-lane group, lane i receiving dimension i).
// K runs a tile ahead of V: the scores of tile t + 1 are formed beside the exponentials of tile
// t, so a wave's matrix and vector instructions alternate without waiting for each other (a tile
// is 32 matrix instructions of 32 cycles and about 1000 cycles of softmax per wave). The bound is
// the matrix unit with its power: 64 % busy, 983 TFLOP/s at one 16,384-token prompt of 32 heads
// where a large bf16 product of the library reaches 1242. Scores, softmax and P @ V one after the
// other, a swizzle whose V reads met in one bank quarter, and heads spread over the XCDs took
// 3214 us there against 2237 now, on one box; 4096 tokens 291 against 158, 2048 tokens 82 against 53.
// At the end the two halves of each query's sum are added and O / l is written.
#include <algorithm>
#include <array>
#include <type_traits>
#include <vector>

#include "decode_pages.hpp"

namespace starkv {

namespace {

constexpr int PF_WAVES = 4;
constexpr int PF_THR = PF_WAVES * 64;
constexpr int PF_QB = 32 * PF_WAVES;      // query rows per workgroup
constexpr int PF_KT = 64;                 // keys per tile
constexpr int PF_TILE = PF_KT * 256;      // bytes of K (or V) per tile: 64 rows x 128 fp16
constexpr int PF_LDS = 4 * PF_TILE;       // two K and two V tiles: the next lands while one is used
constexpr int PF_CPW = 16 / PF_WAVES;     // 1 KB copies per wave per K (or V) tile
constexpr float PF_LAZY = 8.f;            // log2 headroom of the reference max

typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct PrefillParams {
    const void* q; int64_t q_s0, q_s1; int q_dt;
    const uint8_t* k; const uint8_t* v; int64_t kv_s0, kv_s1;  // bytes
    const int32_t* cu;                                        // [P + 1]
    const int32_t* blocks; int nblocks;                       // [nblocks][2]: prompt, query block
    int Hq, G;
    float sc;                                                 // scale * log2(e)
    void* out; int64_t o_s0, o_s1; int out_dt;                // elements
};

// A row's granules (16 bytes, 16 a row) lie XOR-swizzled by its low 4 bits, their two halves
// exchanged: 16 consecutive rows put one granule into 16 places (K's reads), and 4 consecutive
// rows put a run of 4 granules into the 4 different quarters of a row (V's transposing reads,
// 64 bytes of 8 rows each; swizzled by the row's bits as they are, 4 rows met in one quarter and
// bank conflicts took 60 % of the LDS unit's cycles, 16,384 tokens 2600 us against 2262).
__device__ __forceinline__ int pf_swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// Physical byte of (row, granule g) in a K or V tile.
__device__ __forceinline__ uint32_t pf_addr(int row, int g) { return (uint32_t)(row * 256 + ((g ^ pf_swz(row)) << 4)); }

// 8 query dimensions times scale * log2(e), as fp16 (zeros past the prompt).
template <int QDT>
__device__ __forceinline__ half8_t pf_load_q(const PrefillParams& p, int64_t tok, int hq, int d0, bool ok) {
    half8_t r;
    if (!ok) {
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = (_Float16)0.f;
        return r;
    }
    const int64_t off = tok * p.q_s0 + (int64_t)hq * p.q_s1 + d0;
    float f[8];
    if (QDT == STARKV_F16) {
        const half8_t x = *(const half8_t*)((const _Float16*)p.q + off);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (float)x[e];
    } else if (QDT == STARKV_BF16) {
        const uint4 w = *(const uint4*)((const uint16_t*)p.q + off);
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            f[2 * k] = __uint_as_float(ws[k] << 16);
            f[2 * k + 1] = __uint_as_float(ws[k] & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = ((const float*)p.q)[off + e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (_Float16)(f[e] * p.sc);
    return r;
}

// 4 transposed 16-bit elements (see the file comment).
__device__ __forceinline__ uint2 pf_tr(uint32_t addr) {
    typedef short s4_t __attribute__((ext_vector_type(4)));
    const s4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4_t*)(uintptr_t)addr);
    return __builtin_bit_cast(uint2, r);
}

// The work of one workgroup: a (prompt, query block) entry of the list and a query head. Where
// the heads divide over the 8 XCDs (workgroups are dealt to them round-robin), an XCD takes the
// blocks of its own heads in list order, block by block: its L2 then streams an eighth of the K
// and V tiles instead of every head's passing through all eight. Head by head instead, the first
// head's last, short blocks no longer fill the tail: 2048 tokens 52 -> 66 us, 4096 156 -> 174.
__device__ __forceinline__ void pf_work(const PrefillParams& p, int& entry, int& hq) {
    const int id = blockIdx.x;
    if (p.Hq % 8 == 0) {
        const int hx = p.Hq / 8, pos = id >> 3;
        hq = (id & 7) * hx + pos % hx;
        entry = pos / hx;
    } else {
        hq = id / p.nblocks;
        entry = id % p.nblocks;
    }
}

template <int QDT, int ODT>
__global__ __launch_bounds__(PF_THR) __attribute__((amdgpu_waves_per_eu(2))) void prefill_kernel(const PrefillParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_kv[];  // K tiles 0, 1, V tiles 0, 1
    const int tid = threadIdx.x, lane = tid & 63, wave = rfl(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int entry, hq;
    pf_work(p, entry, hq);
    // Wave-uniform (readfirstlane): the copy descriptors built from them live in SGPRs.
    const int pr = rfl(p.blocks[2 * entry]), qblk = rfl(p.blocks[2 * entry + 1]);
    const int s = rfl(p.cu[pr]), L = rfl(p.cu[pr + 1]) - s;
    const int hk = hq / p.G;
    const int q0 = qblk * PF_QB;
    const int qw = q0 + 32 * wave;          // the wave's first query (prompt-relative)
    const int nq = min(32, L - qw);         // its rows (<= 0: none)
    const int qi = qw + n;                  // this lane's query
    const int kend = min(L, q0 + PF_QB);    // keys the workgroup needs: [0, kend)
    const int ntile = (kend + PF_KT - 1) / PF_KT;
    const int last = nq > 0 ? (qw + nq - 1) / PF_KT : -1;  // the wave's last tile with a visible key

    // Copies: a K or V tile is 16 KB, 16 copies of 1 KB, PF_CPW per wave. Copy c of wave w moves
    // LDS bytes [1024 (PF_WAVES c + w), + 1024): rows 4 (PF_WAVES c + w) .. + 3; lane j writes
    // physical granule j % 16 of row (j / 16) of them, i.e. logical granule (j % 16) ^ pf_swz(row).
    const uint32_t base = lds_addr(s_kv);
    uint32_t coff[PF_CPW];
#pragma unroll
    for (int c = 0; c < PF_CPW; ++c) {
        const int row = (PF_WAVES * c + wave) * 4 + (lane >> 4);
        coff[c] = (uint32_t)(row * p.kv_s0 + 16 * ((lane & 15) ^ pf_swz(row)));
    }
    const int64_t kv0 = (int64_t)s * p.kv_s0 + (int64_t)hk * p.kv_s1;
    // Tile t of K (or V) into its buffer at LDS address dst.
    auto issue = [&](const uint8_t* src, int t, uint32_t dst) {
        const int r0 = t * PF_KT;
        const int rows = max(0, min(PF_KT, L - r0));
        int4v_t rs = buffer_rsrc(src + kv0 + (int64_t)r0 * p.kv_s0, (int)(rows * p.kv_s0));
#pragma unroll
        for (int e = 0; e < 4; ++e) rs[e] = rfl(rs[e]);  // uniform by construction; the copies take them in SGPRs
#pragma unroll
        for (int c = 0; c < PF_CPW; ++c) lds_copy16(rs, dst + (uint32_t)(PF_WAVES * c + wave) * 1024u, coff[c]);
    };
    issue(p.k, 0, base);

    // Q as the B operand of S^T = K Q^T: query n, dimensions 16 ks + 8 h .. + 7.
    half8_t qb[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qb[ks] = pf_load_q<QDT>(p, (int64_t)s + qi, hq, 16 * ks + 8 * h, qi < L);

    // Per-lane LDS addresses of buffer 0; the other buffer and the row blocks are immediates.
    // A of S^T: key row 32 mb + n, granule 2 ks + h (block mb = 1 is 32 rows further: the same
    // swizzle, + 8 KB).
    uint32_t ka[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) ka[ks] = vgpr_pin(base + pf_addr(n, 2 * ks + h));
    // A of O^T: 16-lane group q reads key rows 16 ks + 4 (q >> 1) + i / 4 (and + 8) at dimensions
    // 32 md + 16 (q & 1) + 4 (i % 4). Step ks is 16 rows (4 KB) further with the same swizzle.
    const int qg = lane >> 4, li = lane & 15;
    uint32_t va[4][2];
#pragma unroll
    for (int md = 0; md < 4; ++md)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int row = 8 * half + 4 * (qg >> 1) + (li >> 2);
            const int dim = 32 * md + 16 * (qg & 1) + 4 * (li & 3);
            va[md][half] = vgpr_pin(base + 2 * PF_TILE + pf_addr(row, dim >> 3) + 2 * (dim & 7));
        }

    f32x16_t o[4], sa[2], sb[2];  // scores of the even and the odd tiles
#pragma unroll
    for (int md = 0; md < 4; ++md) o[md] = (f32x16_t){};
    float m = -INFINITY, l = 0.f;

    // S^T of the tile in K buffer B.
    auto scores = [&](auto B, f32x16_t* x) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) x[mb] = (f32x16_t){};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
                x[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_ld<half8_t>(ka[ks] + (uint32_t)(B * PF_TILE + 8192 * mb)),
                                                               qb[ks], x[mb], 0, 0, 0);
    };
    // Tile t, its scores in sc, its V in buffer B; the next tile's scores (NEXT, into nx) are formed
    // beside the exponentials: matrix and vector work of one wave with no dependence between them.
    auto tile = [&](auto B, int t, f32x16_t* sc, f32x16_t* nx) {
        const int k0 = t * PF_KT;
        // Scores of this lane's query (already scaled through q): key k0 + 32 mb + 8 (r / 4) +
        // 4 h + r % 4. Only a tile that reaches past the wave's first query or the prompt's
        // end needs the causal / end mask.
        if (k0 + PF_KT - 1 > qw || k0 + PF_KT > L) {
            const int lim = min(qi, L - 1) - k0 - 4 * h;  // the last visible key, from the lane's first
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (32 * mb + 8 * (r >> 2) + (r & 3) > lim) sc[mb][r] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[mb][r]);
        {  // with the partner lane's half: x[0] holds lane l % 32's value, x[1] lane 32 + l % 32's
            const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
        }
        if (__builtin_amdgcn_ballot_w64(mx > m + PF_LAZY) != 0) {
            const float mn = fmaxf(m, mx);
            const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int md = 0; md < 4; ++md)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[md][r] *= alpha;
        }
        const float mr = m == -INFINITY ? 0.f : m;  // no finite score yet: exp2(-inf - 0) = 0
        scores(std::integral_constant<int, 1 - B>{}, nx);
        // P in fp16 as the B operand of each 16-key step: elements 8 (ks % 2) .. + 7 of block ks / 2.
        half8_t pb[4];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float e0 = __builtin_amdgcn_exp2f(sc[mb][r] - mr), e1 = __builtin_amdgcn_exp2f(sc[mb][r + 1] - mr);
                l += e0;
                l += e1;
                const half2_t hh = cvt_h2(e0, e1);
                pb[2 * mb + (r >> 3)][r & 7] = hh[0];
                pb[2 * mb + (r >> 3)][(r & 7) + 1] = hh[1];
            }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int md = 0; md < 4; ++md) {
                const uint32_t at = (uint32_t)(B * PF_TILE + 4096 * ks);
                const uint2 a0 = pf_tr(va[md][0] + at), a1 = pf_tr(va[md][1] + at);
                const half8_t av = __builtin_bit_cast(half8_t, make_uint4(a0.x, a0.y, a1.x, a1.y));
                o[md] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, pb[ks], o[md], 0, 0, 0);
            }
        // The order of the block: LDS reads a few matrix instructions ahead of their use, the
        // softmax's vector instructions between the matrix ones of the scores and of the first half
        // of P @ V (which needs the first half of P only).
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 5, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (i < 13) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (i < 8) __builtin_amdgcn_sched_group_barrier(0x402, 5, 0);
        }
    };
    auto step = [&](auto B, int t, f32x16_t* sc, f32x16_t* nx) {
        SKV_WAIT_VM_LGKM0(0);  // V tile t and K tile t + 1 have landed (this wave's copies)
        lds_barrier();         // every wave's copies; every wave done with K tile t and V tile t - 1
        if (t + 2 < ntile) issue(p.k, t + 2, base + (uint32_t)(B * PF_TILE));
        if (t + 1 < ntile) issue(p.v, t + 1, base + (uint32_t)((3 - B) * PF_TILE));
        if (t <= last) tile(B, t, sc, nx);
    };
    // Two workgroups share a CU (64 KB of LDS each).
    SKV_WAIT_VM_LGKM0(0);
    lds_barrier();
    issue(p.v, 0, base + 2 * PF_TILE);
    if (ntile > 1) issue(p.k, 1, base + PF_TILE);
    if (last >= 0) scores(std::integral_constant<int, 0>{}, sa);
    for (int t = 0; t < ntile; t += 2) {
        step(std::integral_constant<int, 0>{}, t, sa, sb);
        if (t + 1 < ntile) step(std::integral_constant<int, 1>{}, t + 1, sb, sa);
    }
    // The query's sum over both halves, then O / l: dimensions 32 md + 8 (r / 4) + 4 h + r % 4.
    {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
        l = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    }
    if (qi < L && nq > 0) {
        const float inv = 1.f / l;
        const int64_t ob = ((int64_t)s + qi) * p.o_s0 + (int64_t)hq * p.o_s1;
#pragma unroll
        for (int md = 0; md < 4; ++md)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int d = 32 * md + 8 * j + 4 * h;
                const float v0 = o[md][4 * j] * inv, v1 = o[md][4 * j + 1] * inv;
                const float v2 = o[md][4 * j + 2] * inv, v3 = o[md][4 * j + 3] * inv;
                if (ODT == STARKV_F32) {
                    *(float4*)((float*)p.out + ob + d) = make_float4(v0, v1, v2, v3);
                } else if (ODT == STARKV_F16) {
                    const half2_t a = cvt_h2(v0, v1), b = cvt_h2(v2, v3);
                    *(uint2*)((_Float16*)p.out + ob + d) = make_uint2(h2_bits(a), h2_bits(b));
                } else {
                    const uint32_t a = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v0) |
                                       ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v1) << 16);
                    const uint32_t b = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v2) |
                                       ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v3) << 16);
                    *(uint2*)((uint16_t*)p.out + ob + d) = make_uint2(a, b);
                }
            }
    }
    SKV_WAIT_VM_LGKM0(0);  // no copy may land after the workgroup ends
}

// ---------------------------------------------------------------------------
// K and V of bf16 or fp32 as the fp16 rows that prefill_kernel reads: one launch, 8 values a
// lane from rows at any strides, contiguous out. The bound is HBM (4 bytes read and written per
// bf16 value). 16,384 tokens of 32 heads: 83 us where two conversions of torch took 314.
// ---------------------------------------------------------------------------
struct ToHalfParams {
    const void* src[2]; int64_t s0[2], s1[2];  // elements: K, V
    uint16_t* dst[2];                          // [T][H][128]
    int H;
    int64_t pieces;                            // of 8 values per tensor
    int wide;                                  // every piece 16-byte aligned
};

template <int DT>
__global__ __launch_bounds__(256) void to_half_kernel(const ToHalfParams p) {
    const int z = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < p.pieces; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i >> 4, t = row / p.H;
        const int h = (int)(row - t * p.H);
        const int64_t at = t * p.s0[z] + h * p.s1[z] + 8 * (i & 15);
        float x[8];
        if (p.wide) {
            load8_f(p.src[z], at, DT, x);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = load_f(p.src[z], at + e, DT);
        }
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)x[e];
        *(half8_t*)(p.dst[z] + 8 * i) = o;
    }
}

template <int QDT>
const void* pf_pick(int odt) {
    if (odt == STARKV_F32) return (const void*)&prefill_kernel<QDT, STARKV_F32>;
    if (odt == STARKV_F16) return (const void*)&prefill_kernel<QDT, STARKV_F16>;
    return (const void*)&prefill_kernel<QDT, STARKV_BF16>;
}

}  // namespace

}  // namespace starkv

using namespace starkv;

extern "C" {

int starkv_prefill_block_list(const int32_t* cu_seqlens, int num_prompts, int32_t* blocks, int capacity) {
    // (keys, prompt, block) of every 128-row query block, the most keys first (ties in
    // prompt then block order): the longest causal rows start first and the short ones
    // fill the tail.
    if (!cu_seqlens || num_prompts < 0) return -1;
    std::vector<std::array<int, 3>> all;
    for (int i = 0; i < num_prompts; ++i) {
        const int L = cu_seqlens[i + 1] - cu_seqlens[i];
        if (L < 0) return -1;
        for (int b = 0; b * PF_QB < L; ++b) all.push_back({std::min(L, PF_QB * (b + 1)), i, b});
    }
    std::stable_sort(all.begin(), all.end(), [](const std::array<int, 3>& x, const std::array<int, 3>& y) {
        return x[0] > y[0];
    });
    if (blocks)
        for (int k = 0; k < (int)all.size() && k < capacity; ++k) {
            blocks[2 * k] = all[k][1];
            blocks[2 * k + 1] = all[k][2];
        }
    return (int)all.size();
}

int starkv_prefill_attention(void* stream, const void* query, int64_t q_s0, int64_t q_s1, int q_dtype,
                             const void* key, const void* value, int64_t kv_s0, int64_t kv_s1, int kv_dtype,
                             const int32_t* cu_seqlens, const int32_t* blocks, int num_blocks, int num_heads,
                             int num_kv_heads, int head_size, float scale, void* out, int64_t o_s0, int64_t o_s1,
                             int out_dtype) {
    clear_error();
    SKV_CHECK(num_blocks >= 0, "prefill: num_blocks=%d", num_blocks);
    if (num_blocks == 0) return STARKV_OK;
    SKV_CHECK(query && key && value && cu_seqlens && blocks && out, "prefill: null pointer");
    SKV_CHECK(head_size == 128, "prefill: head_size %d (128 only)", head_size);
    SKV_CHECK(num_kv_heads >= 1 && num_heads >= 1 && num_heads % num_kv_heads == 0,
              "prefill: num_heads %% num_kv_heads != 0");
    SKV_CHECK(kv_dtype == STARKV_F16, "prefill: K and V must be fp16");
    SKV_CHECK(q_dtype >= STARKV_F32 && q_dtype <= STARKV_BF16 && out_dtype >= STARKV_F32 && out_dtype <= STARKV_BF16,
              "prefill: query and output dtypes must be bf16, fp16 or fp32");
    SKV_CHECK(((uintptr_t)key % 16) == 0 && ((uintptr_t)value % 16) == 0 && kv_s0 % 8 == 0 && kv_s1 % 8 == 0,
              "prefill: K and V rows must be 16-byte aligned");
    SKV_CHECK(kv_s0 * 2 * 64 < ((int64_t)1 << 31), "prefill: K / V row stride too large");
    const int qal = q_dtype == STARKV_F32 ? 4 : 8;
    SKV_CHECK(((uintptr_t)query % 16) == 0 && q_s0 % qal == 0 && q_s1 % qal == 0,
              "prefill: query rows must be 16-byte aligned");
    SKV_CHECK(o_s0 % 4 == 0 && o_s1 % 4 == 0 && ((uintptr_t)out % 16) == 0, "prefill: output rows must be aligned");
    PrefillParams p;
    p.q = query; p.q_s0 = q_s0; p.q_s1 = q_s1; p.q_dt = q_dtype;
    p.k = (const uint8_t*)key; p.v = (const uint8_t*)value;
    p.kv_s0 = kv_s0 * 2; p.kv_s1 = kv_s1 * 2;
    p.cu = cu_seqlens; p.blocks = blocks; p.nblocks = num_blocks;
    p.Hq = num_heads; p.G = num_heads / num_kv_heads;
    p.sc = scale * 1.4426950408889634f;
    p.out = out; p.o_s0 = o_s0; p.o_s1 = o_s1; p.out_dt = out_dtype;
    const void* fn = q_dtype == STARKV_F32 ? pf_pick<STARKV_F32>(out_dtype)
                     : q_dtype == STARKV_F16 ? pf_pick<STARKV_F16>(out_dtype)
                                             : pf_pick<STARKV_BF16>(out_dtype);
    const int lds = PF_LDS;
    static const void* raised[16];
    static int nraised = 0;
    bool seen = false;
    for (int i = 0; i < nraised; ++i) seen = seen || raised[i] == fn;
    if (!seen) {
        SKV_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        if (nraised < 16) raised[nraised++] = fn;
    }
    void* args[] = {(void*)&p};
    SKV_HIP(hipLaunchKernel(fn, dim3((unsigned)(num_blocks * num_heads)), dim3(PF_THR), args, (size_t)lds, (hipStream_t)stream));
    return STARKV_OK;
}

int starkv_prefill_to_half(void* stream, const void* key, int64_t k_s0, int64_t k_s1, void* key_out, const void* value,
                           int64_t v_s0, int64_t v_s1, void* value_out, int dtype, int num_tokens, int num_kv_heads) {
    clear_error();
    SKV_CHECK(num_tokens >= 0 && num_kv_heads > 0, "prefill_to_half: bad sizes");
    SKV_CHECK(dtype == STARKV_BF16 || dtype == STARKV_F32, "prefill_to_half: bf16 or fp32 rows");
    SKV_CHECK(((uintptr_t)key_out % 16) == 0 && ((uintptr_t)value_out % 16) == 0,
              "prefill_to_half: the results must be 16-byte aligned");
    if (num_tokens == 0) return STARKV_OK;
    SKV_CHECK(key && value && key_out && value_out, "prefill_to_half: null pointer");
    ToHalfParams p;
    p.src[0] = key; p.s0[0] = k_s0; p.s1[0] = k_s1; p.dst[0] = (uint16_t*)key_out;
    p.src[1] = value; p.s0[1] = v_s0; p.s1[1] = v_s1; p.dst[1] = (uint16_t*)value_out;
    p.H = num_kv_heads;
    p.pieces = (int64_t)num_tokens * num_kv_heads * 16;
    p.wide = 1;
    const int al = dtype == STARKV_F32 ? 4 : 8;
    for (int z = 0; z < 2; ++z)
        if (((uintptr_t)p.src[z] % 16) != 0 || p.s0[z] % al != 0 || p.s1[z] % al != 0) p.wide = 0;
    const dim3 grid((unsigned)std::min<int64_t>((p.pieces + 255) / 256, 4096), 2);
    if (dtype == STARKV_BF16)
        hipLaunchKernelGGL(to_half_kernel<STARKV_BF16>, grid, dim3(256), 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(to_half_kernel<STARKV_F32>, grid, dim3(256), 0, (hipStream_t)stream, p);
    SKV_HIP(hipGetLastError());
    return STARKV_OK;
}

}  // extern "C"
