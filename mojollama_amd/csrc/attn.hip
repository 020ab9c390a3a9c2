// attn.hip — decode attention over a KV cache held contiguously or in
// pages, the KV append of a new token, RoPE, and the host-side page table.
//
// A decode step reads every cached K and V row once: the work is streaming
// 2 * seq * n_kv_head * head_dim * 4 bytes, and what decides its rate is how
// many of those bytes are in flight.  So the unit of work is one wave on one
// 64-position chunk of one KV head, which requests 64 elements of every K row
// (the whole row up to head_dim 64) or a 64-element block of every V row before
// it uses any of it and serves all n_head / n_kv_head query heads that share the
// rows (GQA).  Both reference softmaxes need the maximum over all positions
// before any weight (gqa_attention.c's exp_ps_simd is not an exponential, so
// the online rescaling of flash decoding would not reproduce it), hence three
// launches:
//   k_attn_scores : scores and per-chunk maxima
//   k_attn_values : global maximum, weights, and per group of four chunks the
//                   weight sums and weighted V sums
//   k_attn_combine: out = (sum of group V sums) * 1 / (sum of weights [+ 1e-10])
#include <math.h>
#include <algorithm>
#include <type_traits>
#include <vector>
#include "decode.h"
#include "gemv.h"
#include "moe.h"

namespace {

constexpr int kChunk = 64;        // positions per wave (one per lane)
constexpr int kGroup = 4;         // chunks per workgroup of k_attn_values
constexpr int kMaxHD = 256;
constexpr int kMaxRep = 16;       // query heads per KV head

struct attn_args {
    const float *q;               // [B][NH*HD]
    mllm_kv_view kv;
    const int *seq_lens;          // [B]
    int max_seq, n_chunks, n_groups;   // ceil(max_seq / kChunk), ceil(n_chunks / kGroup)
    int NH, NKH, HD, mode;
    int hpw, nhg;                 // query heads per workgroup, workgroups per KV head's group of heads
    float *scores;                // [B][NH][max_seq]
    float *pmax;                  // [B][NH][n_chunks]
    float *psum;                  // [B][NH][n_groups]
    float *pout;                  // [B][NH][n_groups][HD]
    float *out;                   // [B][NH*HD]
};

// Row s of sequence b, KV head j (nullptr past a page table's reach: the
// row then reads as zeros).
__device__ __forceinline__ const float *kv_row(const float *base, const mllm_kv_view &kv, int b, int s, int NKH, int HD,
                                               int j)
{
    const long rs = (long)NKH * HD;
    if (!kv.block_tables) return base + b * kv.seq_stride + (long)s * rs + (long)j * HD;
    const int blk = s / kv.page_size;
    if (blk >= kv.max_blocks) return nullptr;
    const int page = kv.block_tables[(long)b * kv.max_blocks + blk];
    if (page < 0 || page >= kv.n_pages) return nullptr;
    return base + ((long)page * kv.page_size + s % kv.page_size) * rs + (long)j * HD;
}

// Offset (floats from the pool base) of position s0 + lane's row for KV head
// j, -1 past the sequence (lane >= rows) or on an unmapped page.
__device__ __forceinline__ long chunk_row(const mllm_kv_view &kv, int b, int s0, int lane, int rows, int NKH, int HD,
                                          int j)
{
    if (lane >= rows) return -1;
    const float *r = kv_row(kv.k, kv, b, s0 + lane, NKH, HD, j);
    return r ? r - kv.k : -1;
}

__device__ __forceinline__ int seq_len_of(const attn_args &a, int b)
{
    const int n = a.seq_lens[b];
    return n < 0 ? 0 : n > a.max_seq ? a.max_seq : n;
}

// Reductions by DPP steps within the 16-lane rows (a step is a few cycles; a
// ds_bpermute step waits on LDS, and these chains are on every workgroup's
// critical path), then over the rows' results.  row_max / wave_max: the largest
// of the values that are numbers, -inf where none is.
#define ROW_STEP(op, ctrl) v = op(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp( \
        __builtin_bit_cast(int, v), __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false)))
__device__ __forceinline__ float fadd2(float a, float b) { return a + b; }
__device__ __forceinline__ float lane_of(float v, int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float row_max(float v)
{
    v = v > -INFINITY ? v : -INFINITY;
    ROW_STEP(fmaxf, 0x128);   // row_ror:8, 4, 2, 1
    ROW_STEP(fmaxf, 0x124);
    ROW_STEP(fmaxf, 0x122);
    ROW_STEP(fmaxf, 0x121);
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
    v = row_max(v);
    return fmaxf(fmaxf(lane_of(v, 0), lane_of(v, 16)), fmaxf(lane_of(v, 32), lane_of(v, 48)));
}
__device__ __forceinline__ float wave_sum(float v)
{
    ROW_STEP(fadd2, 0x128);
    ROW_STEP(fadd2, 0x124);
    ROW_STEP(fadd2, 0x122);
    ROW_STEP(fadd2, 0x121);
    return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}
#undef ROW_STEP

// exp_ps_simd (gqa_attention.c:32-48) on one lane, as the source writes it:
// t = x log2e, n = rne(t + 0.5), f = t - n, an FMA chain that starts from 1
// and adds the coefficients in ascending order, times 2^n from the clamped
// biased exponent.  (Not an exponential: it gives 0.0013 at 0 and negative
// values below; the reference's weights are these values.)
__device__ __forceinline__ float exp_ps_simd_lane(float x)
{
    const float t = x * 1.4426950408889634f;
    const float nf = rintf(t + 0.5f);
    const float f = t - nf;
    float p = 1.0f;
    p = fmaf(p, f, 0.6931471805599453f);
    p = fmaf(p, f, 0.2402265069591007f);
    p = fmaf(p, f, 0.0555041086648216f);
    p = fmaf(p, f, 0.0096181291076285f);
    p = fmaf(p, f, 0.0013333558146428f);
    int biased = (int)nf + 127;
    biased = biased < 0 ? 0 : biased > 255 ? 255 : biased;
    return p * __uint_as_float((uint32_t)biased << 23);
}

// acc = fma(q[i], k[i], acc) for i = 0..7 (HI: 8..15) in order, q[i] from lane i of each
// 16-lane row of q (row_newbcast: the row's lanes all hold elements of one q vector), for one
// head or two interleaved (a chain's FMAs are 8 cycles apart).
#define AT1(i, r) "v_fmac_f32_dpp %0, %1, %" #r " row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n"
#define AT2(i, r) "v_fmac_f32_dpp %0, %2, %" #r " row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n" \
                  "v_fmac_f32_dpp %1, %3, %" #r " row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n"
template <bool HI> __device__ __forceinline__ void dot8(float &acc, float q, const float4 &x, const float4 &y)
{
    if constexpr (!HI)
        asm("s_nop 1\n" AT1(0, 2) AT1(1, 3) AT1(2, 4) AT1(3, 5) AT1(4, 6) AT1(5, 7) AT1(6, 8) AT1(7, 9)
            : "+v"(acc) : "v"(q), "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(y.x), "v"(y.y), "v"(y.z), "v"(y.w));
    else
        asm("s_nop 1\n" AT1(8, 2) AT1(9, 3) AT1(10, 4) AT1(11, 5) AT1(12, 6) AT1(13, 7) AT1(14, 8) AT1(15, 9)
            : "+v"(acc) : "v"(q), "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(y.x), "v"(y.y), "v"(y.z), "v"(y.w));
}
template <bool HI>
__device__ __forceinline__ void dot8x2(float &a0, float &a1, float q0, float q1, const float4 &x, const float4 &y)
{
    if constexpr (!HI)
        asm("s_nop 1\n" AT2(0, 4) AT2(1, 5) AT2(2, 6) AT2(3, 7) AT2(4, 8) AT2(5, 9) AT2(6, 10) AT2(7, 11)
            : "+v"(a0), "+v"(a1)
            : "v"(q0), "v"(q1), "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(y.x), "v"(y.y), "v"(y.z), "v"(y.w));
    else
        asm("s_nop 1\n" AT2(8, 4) AT2(9, 5) AT2(10, 6) AT2(11, 7) AT2(12, 8) AT2(13, 9) AT2(14, 10) AT2(15, 11)
            : "+v"(a0), "+v"(a1)
            : "v"(q0), "v"(q1), "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(y.x), "v"(y.y), "v"(y.z), "v"(y.w));
}
#undef AT1
#undef AT2

// scores[b][h][s] = (q_h . k_s) * (1 / sqrtf(HD)) for the chunk's positions,
// and the chunk's maximum per head.  grid (n_groups, NKH, B), wave w of four on
// chunk 4 * group + w, lane = position.  The chunk's K rows arrive 32 elements
// (one 128-byte line of every row) at a time, two such segments in flight (16 KB
// a wave, 16 waves a CU), and pass through LDS from the coalesced order of the
// loads to a row per lane (rows padded by 16 bytes: the lanes' 16-byte reads
// fall on distinct banks).  The FMAs of GT heads (>= G) then take k from the
// lane's registers and q from a DPP row broadcast, so per 16 elements and head
// the LDS serves one 4-byte read.  Each dot stays one fp32 FMA chain in element
// order (elements past HD, up to a multiple of 16, are zeros on both sides).
// Eight sequences of 2048..4096 on 64-row pages, 64 / 8 heads of 64: 32.6 ->
// 18.9 us (the chunk staged by four waves, an LDS read of q and one of k for every
// FMA; q as 16-byte LDS broadcasts 20.5, q from scalar loads 31.0).
constexpr int kSeg = 32;          // elements of a row per segment
constexpr int kSegLd = kSeg + 4;  // LDS row stride (floats)
template <int GT>
__global__ __launch_bounds__(256, 4) void k_attn_scores(attn_args a)
{
    __shared__ __attribute__((aligned(16))) float ks[kGroup][kChunk * kSegLd];
    extern __shared__ __attribute__((aligned(16))) float qs[];      // [GT][hdp], zeros from HD on
    const int j = blockIdx.y / a.nhg, g0 = (blockIdx.y - j * a.nhg) * a.hpw, b = blockIdx.z, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int len = seq_len_of(a, b), c = blockIdx.x * kGroup + w, s0 = c * kChunk;
    if ((int)blockIdx.x * kGroup * kChunk >= len) return;
    const int HD = a.HD, Gall = a.NH / a.NKH, G = min(a.hpw, Gall - g0), hdp = (HD + 15) / 16 * 16;
    const int rows = min(kChunk, len - s0);        // <= 0: a wave past the end
    const long ro = chunk_row(a.kv, b, s0, lane, rows, a.NKH, HD, j);
    const bool all = __all(ro >= 0);
    // load k of a segment: row 8 k + lane / 8 (its address from that row's lane), 16-byte piece lane % 8
    const int pc = lane & 7, nseg = (HD + kSeg - 1) / kSeg;
    const uint64_t addr = (uint64_t)(uintptr_t)(a.kv.k + (ro >= 0 ? ro : 0));
    float4 v[2][8];
    auto load = [&](int s, float4 (&d)[8]) __attribute__((always_inline)) {
        const int e = 4 * min(s * kSeg + 4 * pc, HD - 4);   // past the row: its last piece (stored as zeros)
#pragma unroll
        for (int k = 0; k < 8; k++)
            d[k] = *reinterpret_cast<const float4 *>((uintptr_t)__shfl(addr, 8 * k + (lane >> 3), 64) + e);
    };
    load(0, v[0]);
    load(1, v[1]);
    {
        const float *qb = a.q + ((long)b * a.NH + (long)j * Gall + g0) * HD;
        for (int g = w; g < GT; g += kGroup)   // rows past G: zeros (their dots are not stored)
            for (int d = lane; d < hdp; d += 64) qs[g * hdp + d] = d < HD && g < G ? qb[g * HD + d] : 0.0f;
    }
    __syncthreads();
    float dot[GT];
#pragma unroll
    for (int g = 0; g < GT; g++) dot[g] = 0.0f;
    float *kw = ks[w];
    // one copy of the code for all segments (the next one's registers move down): the
    // workgroup runs it once, so its fetch counts
#pragma unroll 1
    for (int s = 0; s < nseg; s++) {
        const int n = HD - s * kSeg;   // elements left (a segment's pieces past them are zeros)
        if (!all || n < kSeg) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                // with every lane active: lanes past the row's end hold offsets that the others read
                const bool miss = __shfl(ro, 8 * k + (lane >> 3), 64) < 0;
                if (miss || 4 * pc >= n) v[0][k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) *reinterpret_cast<float4 *>(kw + (8 * k + (lane >> 3)) * kSegLd + 4 * pc) = v[0][k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int nblk = n >= kSeg ? 2 : (n + 15) / 16;
#pragma unroll 1
        for (int i = 0; i < nblk; i++) {
            const float4 *kr = reinterpret_cast<const float4 *>(kw + lane * kSegLd + 16 * i);
            const float4 x0 = kr[0], x1 = kr[1], x2 = kr[2], x3 = kr[3];
            float q[GT];
#pragma unroll
            for (int g = 0; g < GT; g++) q[g] = qs[g * hdp + s * kSeg + 16 * i + (lane & 15)];
            if constexpr (GT == 1) {
                dot8<false>(dot[0], q[0], x0, x1);
                dot8<true>(dot[0], q[0], x2, x3);
            } else {
#pragma unroll
                for (int g = 0; g < GT; g += 2) {
                    dot8x2<false>(dot[g], dot[g + 1], q[g], q[g + 1], x0, x1);
                    dot8x2<true>(dot[g], dot[g + 1], q[g], q[g + 1], x2, x3);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 8; k++) v[0][k] = v[1][k];
        if (s + 2 < nseg) load(s + 2, v[1]);
    }
    if (rows <= 0) return;
    const float scale = 1.0f / sqrtf((float)HD);
#pragma unroll
    for (int g = 0; g < GT; g++) {
        const float sc = dot[g] * scale;                      // CE:152 dot *= inv; sgemm's alpha
        const int h = j * Gall + g0 + g;
        const float m = wave_max(lane < rows ? sc : -INFINITY);
        if (g < G && lane < rows) a.scores[((long)b * a.NH + h) * a.max_seq + s0 + lane] = sc;
        if (g < G && lane == 0) a.pmax[((long)b * a.NH + h) * a.n_chunks + c] = m;
    }
}

// Weights of the positions from the maximum over all chunks, their sum, and
// the weighted V sum per head, over a group of kGroup chunks.
//   mode 0 (CE:141-158): w = expf(s - max)
//   mode 1 (gqa_attention.c:50-88): positions below floor(len/8)*8 take
//     exp_ps_simd(clamp(s - max, -80, 80)), the rest expf(s - max) capped at 1e38
// The maximum starts from -1e30 (CE:146, gqa_attention.c:53).
// grid (n_groups * ceil(HD / 64), NKH, B), wave w of four on chunk 4 * group + w
// and a block of 64 elements.  A wave requests its scores (straight into LDS),
// the chunk maxima and all 64 V rows (load k: row 4 k + lane / 16, 16-byte piece
// lane % 16: 16 KB in flight) at once, forms the weights in LDS, and multiplies
// on v_mfma_f32_16x16x4_f32: A = the weights of 16 heads x rows 4 k .. 4 k + 3,
// B = component c of load k as it lies in the registers (columns n = elements
// 4 n + c).  The matrix cores do the FMAs in fp32 and the sum over the four lane
// groups' rows; what counts as much here is the code's size (a workgroup runs
// it once, and instruction fetch was most of an unrolled VALU form's 42 us).
// The waves' sums meet in LDS, so a quarter of the partial sums goes to memory.
// With one group (max_seq <= 256) the result is finished here and the combine
// launch saved.  Shape as above: 39.9 -> 18.1 us, the combine 4.8 -> 4.6 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kWld = 68;          // floats per head in LDS: A reads of 16 heads x 4 rows hit distinct banks
__global__ __launch_bounds__(256, 4) void k_attn_values(attn_args a)
{
    __shared__ __attribute__((aligned(16))) float wt[kGroup][kMaxRep * kWld];   // weights, then V sums
    __shared__ float mx[kMaxRep], sm[kGroup][kMaxRep];
    const int j = blockIdx.y / a.nhg, g0 = (blockIdx.y - j * a.nhg) * a.hpw, b = blockIdx.z, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int HD = a.HD, Gall = a.NH / a.NKH, G = min(a.hpw, Gall - g0), nd = (HD + 63) >> 6;
    const int grp = blockIdx.x / nd, di = blockIdx.x - grp * nd;   // chunk group, block of 64 elements
    const int len = seq_len_of(a, b), c = grp * kGroup + w, s0 = c * kChunk;
    if (grp * kGroup * kChunk >= len) {
        // an empty sequence gives zeros (the reference's products over no positions)
        if (len == 0 && a.n_groups == 1 && di == 0)
            for (int i = threadIdx.x; i < G * HD; i += 256) a.out[((long)b * a.NH + j * Gall + g0) * HD + i] = 0.0f;
        return;
    }
    const int rows = min(kChunk, len - s0), nc = (len + kChunk - 1) / kChunk;   // rows <= 0: a wave past the end
    const long hb = (long)b * a.NH + (long)j * Gall + g0;
    float *wl = wt[w];
    // positions past the end read the last score (their weight is 0)
    for (int g = 0; g < G; g++)
        __builtin_amdgcn_global_load_lds((const void *)(a.scores + (hb + g) * a.max_seq + min(s0 + lane, len - 1)),
                                         (__attribute__((address_space(3))) void *)(wl + g * kWld), 4, 0, 0);
    const long ro = chunk_row(a.kv, b, s0, lane, rows, a.NKH, HD, j);
    const bool all = __all(ro >= 0);
    const int n = lane & 15, rg = lane >> 4;
    const uint64_t addr = (uint64_t)(uintptr_t)(a.kv.v + (ro >= 0 ? ro : 0));
    float4 v[16];
    {
        const int e = 4 * min(64 * di + 4 * n, HD - 4);
#pragma unroll
        for (int k = 0; k < 16; k++)
            v[k] = *reinterpret_cast<const float4 *>((uintptr_t)__shfl(addr, 4 * k + rg, 64) + e);
    }
    // maxima of heads w + 4 rg, sixteen lanes each
    {
        const float *pm = a.pmax + (hb + min(w + kGroup * rg, G - 1)) * a.n_chunks;
        float m = -INFINITY;
        for (int k = n; k < nc; k += 64) {
#pragma unroll
            for (int u = 0; u < 4; u++) m = fmaxf(m, pm[min(k + 16 * u, nc - 1)]);
        }
        m = fmaxf(row_max(m), -1e30f);
        if (n == 0) mx[w + kGroup * rg] = m;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the scores are in LDS
    __syncthreads();
    const int vec_end = a.mode == 1 ? len / 8 * 8 : 0;
    // positions of the vector loop (mode 1), the exponentials, or (one chunk) both
    const bool vec = s0 < vec_end, scalar = s0 + rows > vec_end;
    for (int g = 0; g < G; g++) {
        const float z = wl[g * kWld + lane] - mx[g];
        float e = 0.0f;
        if (scalar) {
            e = expf(z);
            if (a.mode == 1 && e > 1e38f) e = 1e38f;
        }
        if (vec) {
            float y = z > -80.0f ? z : -80.0f;
            y = exp_ps_simd_lane(y < 80.0f ? y : 80.0f);
            e = s0 + lane < vec_end ? y : e;
        }
        if (lane >= rows) e = 0.0f;
        wl[g * kWld + lane] = e;
        const float sum = wave_sum(e);
        if (lane == 0) sm[w][g] = sum;
    }
    // rows past the end or on unmapped pages are zeros (what was read there may be anything)
    if (!all) {
#pragma unroll
        for (int k = 0; k < 16; k++)
            if (__shfl(ro, 4 * k + rg, 64) < 0) v[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    f32x4 acc[4] = {};
    const float *wa = wl + min(n, G - 1) * kWld + rg;   // heads past G repeat the last one's and are not stored
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const float q = wa[4 * k];
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, v[k].x, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, v[k].y, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, v[k].z, acc[2], 0, 0, 0);
        acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, v[k].w, acc[3], 0, 0, 0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // lane (n, rg) holds heads 4 rg + r, elements 4 n + c: over the wave's own weights
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4 *>(wl + (4 * rg + r) * kWld + 4 * n) =
            make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
    __syncthreads();
    const int d = 64 * di + lane;
    if (d >= HD) return;
    for (int g = w; g < G; g += kGroup) {
        float o = 0.0f, s = 0.0f;
#pragma unroll
        for (int x = 0; x < kGroup; x++) {
            o += wt[x][g * kWld + lane];
            s += sm[x][g];
        }
        if (a.n_groups == 1) {
            a.out[(hb + g) * HD + d] = o * (a.mode == 1 ? 1.0f / (s + 1e-10f) : 1.0f / s);
        } else {
            const long at = (hb + g) * a.n_groups + grp;
            a.pout[at * HD + d] = o;
            if (d == 0) a.psum[at] = s;
        }
    }
}

// out[b][h][d] = sum_c pout * 1 / (sum_c psum [+ 1e-10 in mode 1]); an empty
// sequence gives zeros (the reference's products over no positions).
// grid (NH, B), 256 threads: 256 / HD groups of HD lanes each take every
// ng-th group of chunks (four loads in flight per lane), then group 0 adds the groups.
__global__ __launch_bounds__(256) void k_attn_combine(attn_args a)
{
    __shared__ float part[256], spart[256];
    const int h = blockIdx.x, b = blockIdx.y, HD = a.HD, ng = 256 / HD;
    const int gi = threadIdx.x / HD, d = threadIdx.x - gi * HD;
    const int len = seq_len_of(a, b), nc = (len + kGroup * kChunk - 1) / (kGroup * kChunk);
    const float *ps = a.psum + ((long)b * a.NH + h) * a.n_groups;
    const float *po = a.pout + ((long)b * a.NH + h) * a.n_groups * HD + d;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (gi < ng) {
        int c = gi;
        for (; c + 3 * ng < nc; c += 4 * ng) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                acc[u] += po[(long)(c + u * ng) * HD];
                sum[u] += ps[c + u * ng];
            }
        }
        for (; c < nc; c += ng) { acc[0] += po[(long)c * HD]; sum[0] += ps[c]; }
        part[threadIdx.x] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        spart[threadIdx.x] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    }
    __syncthreads();
    if (gi != 0) return;
    float o = 0.0f, s = 0.0f;
    for (int g = 0; g < ng; g++) { o += part[g * HD + d]; s += spart[g * HD + d]; }
    const float inv = a.mode == 1 ? 1.0f / (s + 1e-10f) : 1.0f / s;
    a.out[((long)b * a.NH + h) * HD + d] = len == 0 ? 0.0f : o * inv;
}

// New K/V rows: token b's k/v [NKH*HD] to row pos[b] of its cache (CE:1363-1381,
// GO:158-161).  A position whose page is unmapped or past the table is skipped.
__global__ void k_kv_append(mllm_kv_view kv, const int *pos, const float *k_new, const float *v_new, int NKH, int HD)
{
    const int b = blockIdx.y, n = NKH * HD;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int s = pos[b];
    if (s < 0) return;
    const int j = i / HD, d = i - j * HD;
    const float *kr = kv_row(kv.k, kv, b, s, NKH, HD, j);
    if (!kr) return;
    const long off = kr - kv.k;
    kv.k[off + d] = k_new[(long)b * n + i];
    kv.v[off + d] = v_new[(long)b * n + i];
}

// rope_apply (GO:37-51, CE's rope_apply): per head the pairs (j, j + r/2),
// r = rope_dim (head_dim when <= 0), rotated by cos/sin rows [pos][r/2].
// grid (T), threads over NH * r/2; buf [T][NH*HD], pos [T].
__global__ void k_rope(float *buf, int NH, int HD, const int *pos, const float *cos_t, const float *sin_t, int r)
{
    const int t = blockIdx.x, hd2 = r / 2;
    const long p = pos[t];
    for (int i = threadIdx.x; i < NH * hd2; i += blockDim.x) {
        const int h = i / hd2, jj = i - h * hd2;
        float *bh = buf + ((long)t * NH + h) * HD;
        const float a0 = bh[jj], a1 = bh[jj + hd2];
        const float cs = cos_t[p * hd2 + jj], sn = sin_t[p * hd2 + jj];
        bh[jj] = a0 * cs - a1 * sn;
        bh[jj + hd2] = a1 * cs + a0 * sn;
    }
}

// mllm_rope_append: grid (NH + 2 NKH) heads, one wave each.  One launch of a decode step's
// layer instead of two (4.1 and 2.3 us, latency).
__global__ __launch_bounds__(64) void k_rope_append(float *qkv, int NH, int NKH, int HD, const int *pos,
                                                    const float *cos_t, const float *sin_t, int r, mllm_kv_view kv,
                                                    const int *kv_pos)
{
    const int h = blockIdx.x, hd2 = r / 2;
    const float *src = qkv + (long)h * HD;
    float *dst = qkv + (long)h * HD;
    if (h >= NH) {
        const int j = (h - NH) % NKH, s = kv_pos[0];
        const float *row = s < 0 ? nullptr : kv_row(kv.k, kv, 0, s, NKH, HD, j);
        if (!row) return;
        dst = (h < NH + NKH ? kv.k : kv.v) + (row - kv.k);
    }
    if (h >= NH + NKH) {
        for (int i = threadIdx.x; i < HD; i += 64) dst[i] = src[i];
        return;
    }
    const long p = pos[0];
    for (int i = threadIdx.x; i < hd2; i += 64) {
        const float a0 = src[i], a1 = src[i + hd2];
        const float cs = cos_t[p * hd2 + i], sn = sin_t[p * hd2 + i];
        dst[i] = a0 * cs - a1 * sn;
        dst[i + hd2] = a1 * cs + a0 * sn;
    }
    if (h >= NH)
        for (int i = r + threadIdx.x; i < HD; i += 64) dst[i] = src[i];
}

long a256(long n) { return (n + 255) / 256 * 256; }

// Workspace carve-up of mllm_gqa_decode.
long attn_ws(int B, int NH, int HD, int max_seq, attn_args *a, uint8_t *base)
{
    const int nc = (max_seq + kChunk - 1) / kChunk, ng = (nc + kGroup - 1) / kGroup;
    long o = 0;
    auto take = [&](long bytes) { long at = o; o += a256(bytes); return base ? (float *)(base + at) : nullptr; };
    float *scores = take((long)B * NH * max_seq * 4);
    float *pmax = take((long)B * NH * nc * 4);
    float *psum = take((long)B * NH * ng * 4);
    float *pout = take((long)B * NH * ng * HD * 4);
    if (a) { a->scores = scores; a->pmax = pmax; a->psum = psum; a->pout = pout; a->n_chunks = nc; a->n_groups = ng; }
    return o > 0 ? o : 256;
}

bool attn_shape_ok(int NH, int NKH, int HD)
{
    return NH > 0 && NKH > 0 && NH % NKH == 0 && NH / NKH <= kMaxRep && HD > 0 && HD <= kMaxHD && HD % 4 == 0;
}

} // namespace

extern "C" {

MLLM_API long mllm_gqa_workspace_size(int B, int NH, int HD, int max_seq)
{
    if (B <= 0 || NH <= 0 || HD <= 0 || max_seq <= 0) return 256;
    return attn_ws(B, NH, HD, max_seq, nullptr, nullptr);
}

MLLM_API int mllm_gqa_decode(int mode, const float *q, const mllm_kv_view *kv, const int *seq_lens, int max_seq, int B,
                             int NH, int NKH, int HD, float *out, void *workspace, long ws_bytes, void *stream)
{
    if ((mode != 0 && mode != 1) || !q || !kv || !kv->k || !kv->v || !seq_lens || !out || B <= 0 || max_seq < 0 ||
        !attn_shape_ok(NH, NKH, HD)) {
        mllm_set_error("mllm_gqa_decode: bad arguments (mode 0/1, NH % NKH == 0, NH/NKH <= 16, HD <= 256 and a "
                       "multiple of 4)");
        return -1;
    }
    if (((uintptr_t)kv->k | (uintptr_t)kv->v) & 15) {
        mllm_set_error("mllm_gqa_decode: K and V must be 16-byte aligned");
        return -1;
    }
    if (kv->block_tables && (kv->page_size <= 0 || kv->max_blocks <= 0 || kv->n_pages <= 0)) {
        mllm_set_error("mllm_gqa_decode: a paged view needs page_size, max_blocks and n_pages > 0");
        return -1;
    }
    // contiguous rows are read as float4 from b * seq_stride + s * NKH * HD: the
    // stride keeps that 16-byte aligned and, with several sequences, past the
    // max_seq rows of the previous one
    if (!kv->block_tables && (kv->seq_stride < 0 || kv->seq_stride % 4 ||
                              (B > 1 && kv->seq_stride < (long)max_seq * NKH * HD))) {
        mllm_set_error("mllm_gqa_decode: seq_stride must be a non-negative multiple of 4 floats and, for B > 1, at "
                       "least max_seq * NKH * HD");
        return -1;
    }
    hipStream_t st = (hipStream_t)stream;
    attn_args a{};
    a.q = q; a.kv = *kv; a.seq_lens = seq_lens; a.max_seq = max_seq > 0 ? max_seq : 1;
    a.NH = NH; a.NKH = NKH; a.HD = HD; a.mode = mode; a.out = out;
    if (ws_bytes < attn_ws(B, NH, HD, a.max_seq, nullptr, nullptr)) {
        mllm_set_error("mllm_gqa_decode: workspace below mllm_gqa_workspace_size");
        return -1;
    }
    attn_ws(B, NH, HD, a.max_seq, &a, (uint8_t *)workspace);
    const int G = NH / NKH;
    // Heads per workgroup: all that share the KV head, each K and V row then read once; where
    // that leaves CUs idle, two (the rows' further readers hit L2, and a wave's chain of work is
    // shorter).  64 / 8 heads of 64, all / two: one sequence of 1024 (32 workgroups) 16.3 / 13.1 us,
    // of 4096 (128) 18.8 / 18.7, two of 4096 (256) 22.6 / 25.9, eight (1024) 46.4 / 69.2; eight of
    // 300 on 16-row pages (128) 18.6 / 20.7.
    const dim3 wg(64 * kGroup);
    a.hpw = (long)a.n_groups * NKH * B < 128 ? std::min(G, 2) : G;
    a.nhg = (G + a.hpw - 1) / a.hpw;
    const unsigned gy = (unsigned)(NKH * a.nhg);
    auto go = [&](auto gt_c) {
        constexpr int GT = decltype(gt_c)::value;
        hipLaunchKernelGGL(k_attn_scores<GT>, dim3(a.n_groups, gy, B), wg, (size_t)GT * ((HD + 15) / 16 * 16) * 4, st, a);
    };
    // heads taken together (the registers of a wave): the next power of two
    if (a.hpw == 1) go(std::integral_constant<int, 1>{});
    else if (a.hpw == 2) go(std::integral_constant<int, 2>{});
    else if (a.hpw <= 4) go(std::integral_constant<int, 4>{});
    else if (a.hpw <= 8) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, 16>{});
    hipLaunchKernelGGL(k_attn_values, dim3(a.n_groups * ((HD + 63) / 64), gy, B), wg, 0, st, a);
    if (a.n_groups > 1) hipLaunchKernelGGL(k_attn_combine, dim3(NH, B), dim3(256), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

MLLM_API int mllm_kv_append(const mllm_kv_view *kv, const int *pos, const float *k_new, const float *v_new, int B,
                            int NKH, int HD, void *stream)
{
    if (!kv || !kv->k || !kv->v || !pos || !k_new || !v_new || B <= 0 || NKH <= 0 || HD <= 0 ||
        (kv->block_tables && (kv->page_size <= 0 || kv->max_blocks <= 0 || kv->n_pages <= 0))) {
        mllm_set_error("mllm_kv_append: bad arguments");
        return -1;
    }
    const int n = NKH * HD;
    if (!kv->block_tables && (kv->seq_stride < 0 || (B > 1 && kv->seq_stride < n))) {
        mllm_set_error("mllm_kv_append: seq_stride must be >= 0 and, for B > 1, at least NKH * HD");
        return -1;
    }
    hipLaunchKernelGGL(k_kv_append, dim3((n + 255) / 256, B), dim3(256), 0, (hipStream_t)stream, *kv, pos, k_new,
                       v_new, NKH, HD);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

MLLM_API int mllm_rope(float *buf, int T, int NH, int HD, const int *pos, const float *cos_t, const float *sin_t,
                       int rope_dim, void *stream)
{
    const int r = rope_dim <= 0 ? HD : rope_dim;
    if (!buf || !pos || !cos_t || !sin_t || T <= 0 || NH <= 0 || HD <= 0 || r > HD || (r & 1)) {
        mllm_set_error("mllm_rope: bad arguments (rope_dim even and <= head_dim)");
        return -1;
    }
    hipLaunchKernelGGL(k_rope, dim3(T), dim3(256), 0, (hipStream_t)stream, buf, NH, HD, pos, cos_t, sin_t, r);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

} // extern "C"

int mllm_rope_append(float *qkv, int NH, int NKH, int HD, const int *pos, const float *cos_t, const float *sin_t,
                     int rope_dim, const mllm_kv_view *kv, const int *kv_pos, hipStream_t st)
{
    const int r = rope_dim <= 0 ? HD : rope_dim;
    if (!qkv || !pos || !cos_t || !sin_t || !kv || !kv->k || !kv->v || !kv_pos || NH <= 0 || NKH <= 0 || HD <= 0 ||
        r > HD || (r & 1)) {
        mllm_set_error("mllm_rope_append: bad arguments");
        return -1;
    }
    hipLaunchKernelGGL(k_rope_append, dim3(NH + 2 * NKH), dim3(64), 0, st, qkv, NH, NKH, HD, pos, cos_t, sin_t, r, *kv,
                       kv_pos);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" {

// ------------------------------------------------------------ page table
// CE:160-201: a free list initialised so that allocation hands out pages
// 0, 1, 2, ... in order, and a logical -> physical table of 1024 entries
// (MAX_BLOCKS, CE:23), -1 when unmapped.
struct mllm_page_table {
    int page_size, n_pages, free_count;
    std::vector<int> table, free_pages;
};

MLLM_API mllm_page_table *mllm_page_table_create(int max_pages, int page_size)
{
    if (max_pages <= 0 || page_size <= 0) return nullptr;
    mllm_page_table *pt = new mllm_page_table;
    pt->page_size = page_size;
    pt->n_pages = max_pages;
    pt->table.assign(MLLM_PAGE_TABLE_BLOCKS, -1);
    pt->free_pages.resize(max_pages);
    for (int i = 0; i < max_pages; i++) pt->free_pages[i] = max_pages - 1 - i;
    pt->free_count = max_pages;
    return pt;
}

MLLM_API void mllm_page_table_destroy(mllm_page_table *pt) { delete pt; }

MLLM_API int mllm_page_table_alloc(mllm_page_table *pt)
{
    if (!pt || pt->free_count <= 0) return -1;
    return pt->free_pages[--pt->free_count];
}

MLLM_API void mllm_page_table_free(mllm_page_table *pt, int page_id)
{
    if (pt && pt->free_count < pt->n_pages) pt->free_pages[pt->free_count++] = page_id;
}

MLLM_API void mllm_page_table_map(mllm_page_table *pt, int logical_page, int physical_page)
{
    if (pt && logical_page >= 0 && logical_page < MLLM_PAGE_TABLE_BLOCKS) pt->table[logical_page] = physical_page;
}

MLLM_API const int *mllm_page_table_entries(const mllm_page_table *pt) { return pt ? pt->table.data() : nullptr; }

MLLM_API int mllm_page_table_lookup(const mllm_page_table *pt, int logical_page)
{
    return pt && logical_page >= 0 && logical_page < MLLM_PAGE_TABLE_BLOCKS ? pt->table[logical_page] : -1;
}

} // extern "C"
