// Attention of MLA.forward for few new tokens per sequence (a decode step; reference: inference/model.py:480-497): the
// query is folded through wkv_b (wkv_b_absorb.hip, side Q), so that every head works on the latent cache itself, the
// weighted sum of latents is folded through its value half (side V).  Between the two, here:
//   attend   split over the positions: scores, softmax and weighted sum of one range of positions, for 128 (token, head)
//            rows of a sequence that share the range's latents; binary32 partial sums
//   combine  the ranges' partial sums to the bf16 latent of each row
// and, in front of the query projection, latent: both RMS norms, the cache rows, the query's quantisation.
// Roundings are those of the tensor operations they replace, with the scores and exponentials' sums in binary32
// throughout; exponentials go to bf16 in front of the value product.
#include "mla.hpp"

namespace dsv3 {
namespace {

typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4bf* lds_v4bf;

constexpr int kC = 512, kRope = 64, kNope = 128, kQd = kNope + kRope;
constexpr int kTile = 32;                               // positions per tile
constexpr int kStages = 4;                              // tiles in LDS: one computed, three on their way
constexpr int kRopeOff = kTile * kC * 2;                // a stage: 32 rows of 1 KiB latents, then 32 rows of 128 B rotary keys
constexpr int kStage = kRopeOff + kTile * kRope * 2;
constexpr int kAhead = 6;                               // operands read from LDS ahead of the MFMA that takes them
constexpr int kRows = 128;                              // rows per workgroup: 4 wavefronts x 32
constexpr int kPartFloats = kRows * kC;                 // partial sums of a workgroup, in its registers' order

struct DecodeArgs {
    const uint16_t* ql;                                 // folded queries [batch][rows][512], rows = tokens * heads
    const uint16_t* q;                                  // queries [batch][rows][192]: their rotary part is read here
    const v2f* freqs;                                   // [tokens][32] (cos, sin)
    const uint16_t* kv; int64_t kv_bs;                  // latent cache, batch stride in elements
    const uint16_t* pe; int64_t pe_bs;
    const void* mask;                                   // [tokens][positions]
    float* part; v2f* ml;                               // [batch][row block][split]: kPartFloats floats; kRows x (maximum, sum)
    uint16_t* out;                                      // bf16 [batch][rows][512]
    int batch, rows, heads, positions, tiles, blocks, splits, per;
    float unit, scale, inv_scale;                       // score_unit's unit and rest, and the rest's reciprocal; without a mask 1 and the scale
};

// Chunks of 16 bytes of a latent row r are stored at chunk position c ^ swz(r) (low four bits).  Sixteen rows read at
// the same c (the score product) then hit sixteen different 16-byte columns, and the four consecutive rows of a
// transposed read (the value product: 64 bytes of each) four different 64-byte ones.
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// v *= a on accumulators that stay in the accumulation registers: as an ordinary product the compiler moves all 256 of them
// to and fro and spills.  At least 36 MFMAs with other results lie between the last write of v and this (the S products).
__device__ __forceinline__ void scale_agprs(v16f& v, float a) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        float x = v[e], y;
        asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1" : "+a"(x), "=&v"(y) : "v"(a));
        v[e] = x;
    }
}

// Four wavefronts with all 512 registers of their SIMD lane each: a wavefront holds 32 rows' queries as MFMA operands (144
// registers) and their 32 x 512 weighted sums (256).  Per tile of 32 positions (36 KiB, copied into
// LDS three tiles ahead): S^T = K Q^T (36 MFMAs), exponentials in registers, O^T += V^T P^T (32 MFMAs).  The
// transposed products leave a row in one lane (and the lane 32 further), and S^T's accumulators already are P^T's operand
// (position 16 u + 8 a + 4 g + r of a tile in register 8 u + 4 a + r of lane half g, slot 4 a + r of K step u).  Keys and
// values are the same 32 x 512 block: the keys are read as rows, the values through the LDS's transposing reads, four
// positions of one feature per lane.
// Bound: per tile 68 MFMAs of 32 cycles; with one wavefront per SIMD its exponentials and barriers stand beside them.  32
// sequences at 4096 positions (16 tiles a workgroup): 53 .. 58 us, 70 with each LDS read next to its MFMA; 12 us of it are the 67 MB
// of partial sums at the end, and one tile alone (a short context) takes 12 us in all.  The tensor operations in its place
// took 250 us (58 us in the products, the rest in passes over the scores).
enum { kNoMask, kMaskBf16, kMaskF32 };
template <int MASK>
__global__ __launch_bounds__(256, 1) void mla_decode_kernel(DecodeArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 31, g = lane >> 5;
    const int split = blockIdx.x, b = blockIdx.y, blk = blockIdx.z;
    const int t0 = split * p.per, t1 = min(p.tiles, t0 + p.per);
    const int row0 = blk * kRows + wave * 32;
    const int row = min(row0 + i, p.rows - 1);          // rows past the end repeat the last one; combine leaves them out

    const uint16_t* kvb = p.kv + b * p.kv_bs;
    const uint16_t* peb = p.pe + b * p.pe_bs;
    const uint32_t lds0 = lds_addr_of(lds);
    auto issue = [&](int t, int st) {
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int r = wave * 8 + n;
            const int pos = min(t * kTile + r, p.positions - 1);
            copy16(kvb + (int64_t)pos * kC, (uint32_t)((lane ^ swz(r)) << 4), lds0 + st * kStage + r * 1024);
        }
        // eight rows of 128 bytes; chunk c of row r at c ^ (r / 2 & 7)
        const int r = wave * 8 + (lane >> 3);
        const int pos = min(t * kTile + r, p.positions - 1);
        copy16(peb, (uint32_t)pos * (kRope * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4), lds0 + st * kStage + kRopeOff + wave * 1024);
    };
#pragma unroll
    for (int n = 0; n < kStages - 1; ++n)
        if (t0 + n < t1) issue(t0 + n, n);

    // lane (row i, half g) holds elements 16 s + 8 g .. + 7; the last four steps are rotated here
    v4u Q[36];
    {
        const uint16_t* src = p.ql + ((int64_t)b * p.rows + row) * kC + 8 * g;
#pragma unroll
        for (int s = 0; s < 32; ++s) Q[s] = *(const v4u*)(src + 16 * s);
        const uint16_t* rsrc = p.q + ((int64_t)b * p.rows + row) * kQd + kNope + 8 * g;
        const v2f* fr = p.freqs + (int64_t)(row / p.heads) * (kRope / 2) + 4 * g;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            Q[32 + s] = *(const v4u*)(rsrc + 16 * s);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const v2f cs = fr[8 * s + e];
                const float re = bf16lo_to_f32(Q[32 + s][e]), im = bf16hi_to_f32(Q[32 + s][e]);
                Q[32 + s][e] = pack_bf16(re * cs.x - im * cs.y, re * cs.y + im * cs.x);
            }
        }
    }

    const uint32_t kaddr = i * 1024 + ((g ^ swz(i)) << 4);                      // ^ (2 s mod 16) << 4
    const uint32_t raddr = kRopeOff + i * 128 + ((g ^ ((i >> 1) & 7)) << 4);    // ^ 2 s << 4
    // transposed reads: lane group q of 16 takes features 16 q .. of the 32, its lane l fetches four features of row l / 4
    const int l15 = lane & 15, q2 = (lane >> 4) & 1;
    const uint32_t vaddr = (4 * g + (l15 >> 2)) * 1024 + ((((2 * q2 + ((l15 & 3) >> 1)) ^ g) | ((l15 >> 2) << 2)) << 4) + 8 * (l15 & 1);

    v16f O[16] = {};
    float m = -__builtin_inff(), l = 0.f;               // running maximum of the scores, this lane's share of the sum
    const float scale2 = p.scale * 1.44269504088896340736f;
    int st = 0;
    for (int t = t0; t < t1; ++t) {
        // this wavefront's nine copies of the tile: those of the tiles behind it stay in flight
        if (t + 2 < t1)      __builtin_amdgcn_s_waitcnt(0x0f70 | (18 & 15) | (18 >> 4) << 14);      // vmcnt(18)
        else if (t + 1 < t1) __builtin_amdgcn_s_waitcnt(0x0f70 | 9);
        else                 __builtin_amdgcn_s_waitcnt(0x0f70);
        barrier_no_fence();                             // everybody's, and the stage of the tile before is free
        if (t + kStages - 1 < t1) issue(t + kStages - 1, (st + kStages - 1) % kStages);
        const uint8_t* base = lds + st * kStage;
        v16f T[1] = {};
        v16f& S = T[0];
        // operands kAhead steps ahead; the barriers keep this order (the scheduler puts each read next to its use and waits)
        v4u ring[kAhead];
        auto key = [&](int s) -> v4u {
            return s < 32 ? *(const v4u*)(base + (kaddr ^ ((s & 7) << 5)) + (s >> 3) * 256) : *(const v4u*)(base + (raddr ^ ((s - 32) << 5)));
        };
#pragma unroll
        for (int s = 0; s < kAhead; ++s) ring[s] = key(s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 36; ++s) {
            S = mfma32(ring[s % kAhead], Q[s], S);
            if (s + kAhead < 36) ring[s % kAhead] = key(s + kAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MASK != kNoMask) {
            const int64_t mrow = (int64_t)(row / p.heads) * p.positions;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t at = mrow + min(t * kTile + 8 * (e >> 2) + 4 * g + (e & 3), p.positions - 1);
                S[e] = __builtin_fmaf(S[e], p.unit, mask_at<MASK == kMaskF32>(p.mask, at) * p.inv_scale);
            }
        }
        if ((t + 1) * kTile > p.positions) {            // the last tile may reach past the end
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (t * kTile + 8 * (e >> 2) + 4 * g + (e & 3) >= p.positions) S[e] = -__builtin_inff();
        }
        float mx = S[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = __builtin_elementwise_maximum(mx, S[e]);
        mx = fmaxf(mx, xor32(mx));
        // The maximum is only raised when it grows by more than 2^64: exponentials and sums have room for that in binary32
        // and bf16, and so the 256 multiplications are needed in the rarest of cases.
        const bool raise = (mx - m) * scale2 > 64.f || (m == -__builtin_inff() && mx > m);
        if (__any(raise)) {
            const float mn = fmaxf(m, mx);
            const float a = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m - mn) * scale2);
            l *= a;
            m = mn;
            if (t > t0) {
#pragma unroll
                for (int d = 0; d < 16; ++d) scale_agprs(O[d], a);
                asm volatile("s_nop 7" ::: "memory");
            }
        }
        const float off = softmax_offset(T, m, scale2);
        const uint32_t vbase = lds0 + st * kStage + vaddr;      // stages are multiples of 1 KiB: the xors below stay inside a row
        auto value = [&](int s) -> v4u {                        // positions 16 (s / 16) .. of features 32 (s % 16) ..
            const uint32_t at = (vbase ^ ((s & 3) << 6)) + (s >> 4) * 16384 + ((s & 15) >> 2) * 256;
            const v2u lo = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf)(uintptr_t)at));
            const v2u hi = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf)(uintptr_t)((at ^ 32) + 8192)));
            return v4u{ lo[0], lo[1], hi[0], hi[1] };
        };
#pragma unroll
        for (int s = 0; s < kAhead; ++s) ring[s] = value(s);    // on their way during the exponentials
        __builtin_amdgcn_sched_barrier(0);
        float sum = 0.f;
        v4u P[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int e = 8 * u + 2 * q;
                const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e], scale2, -off));
                const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e + 1], scale2, -off));
                sum += x + y;
                P[u][q] = pack_bf16(x, y);
            }
        l += sum;
#pragma unroll
        for (int s = 0; s < 32; ++s) {
            O[s & 15] = mfma32(ring[s % kAhead], P[s >> 4], O[s & 15]);
            if (s + kAhead < 32) ring[s % kAhead] = value(s + kAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
        st = (st + 1) % kStages;
    }

    l += xor32(l);
    const int64_t unit = ((int64_t)b * p.blocks + blk) * p.splits + split;
    if (g == 0) p.ml[unit * kRows + wave * 32 + i] = v2f{ m, l };
    v4f* dst = (v4f*)(p.part + unit * kPartFloats) + wave * 64 * 64 + lane;
#pragma unroll
    for (int d = 0; d < 16; ++d)
#pragma unroll
        for (int a = 0; a < 4; ++a) dst[(d * 4 + a) * 64] = v4f{ O[d][4 * a], O[d][4 * a + 1], O[d][4 * a + 2], O[d][4 * a + 3] };
}

// One workgroup: 32 features of 32 rows.  Wavefront w takes splits w, w + 4, .. with a running maximum of its own, the four
// meet in LDS.  Reads 1 KiB per instruction in the order attend wrote it: bound by those reads (67 MB at 256 attend
// workgroups: 12.4 us, 5.4 TB/s, mostly out of the last-level cache).
__global__ __launch_bounds__(256) void mla_combine_kernel(DecodeArgs p) {
    __shared__ v4f acc_s[4][4][64];
    __shared__ v2f ml_s[4][32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 31, g = lane >> 5;
    const int d = blockIdx.x & 15, wv = blockIdx.x >> 4, b = blockIdx.y, blk = blockIdx.z;
    const int row = blk * kRows + wv * 32 + i;
    if (blk * kRows + wv * 32 >= p.rows) return;
    const int64_t unit0 = ((int64_t)b * p.blocks + blk) * p.splits;
    const v4f* src = (const v4f*)(p.part + unit0 * kPartFloats) + (wv * 64 + d * 4) * 64 + lane;
    const v2f* mls = p.ml + unit0 * kRows + wv * 32 + i;
    const float scale2 = p.scale * 1.44269504088896340736f;
    auto weight = [&](float from, float to) { return from == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((from - to) * scale2); };
    float m = -__builtin_inff(), l = 0.f;
    v4f acc[4] = {};
#pragma unroll 2
    for (int s = wave; s < p.splits; s += 4) {
        const v2f x = mls[(int64_t)s * kRows];
        v4f o[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) o[a] = src[(int64_t)s * (kPartFloats / 4) + a * 64];
        const float mn = fmaxf(m, x.x), wa = weight(m, mn), wb = weight(x.x, mn);
        l = l * wa + x.y * wb;
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[a] = acc[a] * wa + o[a] * wb;
        m = mn;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) acc_s[wave][a][lane] = acc[a];
    if (g == 0) ml_s[wave][i] = v2f{ m, l };
    __syncthreads();
    float mm = ml_s[0][i].x;
#pragma unroll
    for (int w = 1; w < 4; ++w) mm = fmaxf(mm, ml_s[w][i].x);
    float ll = 0.f;
    v4f r = {};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float k = weight(ml_s[w][i].x, mm);
        ll += ml_s[w][i].y * k;
        r += acc_s[w][wave][lane] * k;
    }
    r *= 1.0f / ll;                                     // a row without any position: 0 * inf, NaN as softmax gives
    if (row < p.rows)
        *(v2u*)(p.out + ((int64_t)b * p.rows + row) * kC + 32 * d + 8 * wave + 4 * g) = v2u{ pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]) };
}

struct LatentArgs {
    const uint16_t* a; int64_t a_stride;                // bf16 rows [q_rank | 512 | 64], stride in elements
    const uint16_t* q_w; const uint16_t* kv_w;          // norm weights
    const v2f* freqs;                                   // [tokens][32]
    uint16_t* kv; int64_t kv_bs;                        // cache rows of the first new token, batch strides in elements
    uint16_t* pe; int64_t pe_bs;
    uint8_t* y; float* ys;                              // e4m3 [rows][q_rank], scales [rows][q_rank / 128]
    int tokens, q_rank;
    float q_eps, kv_eps;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}
__device__ __forceinline__ void unpack8(v4u p, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) { f[2 * e] = bf16lo_to_f32(p[e]); f[2 * e + 1] = bf16hi_to_f32(p[e]); }
}
__device__ __forceinline__ float sum_sq8(const float (&f)[8]) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += f[e] * f[e];
    return s;
}

// What follows the two low-rank projections of a token, one workgroup per token: wavefronts 0 .. 3 the query latent (RMS
// norm, rounded to bf16, quantised per 128 values = 16 lanes for the next projection), wavefront 4 the cache row (RMS norm
// of the 512 latents, rotation of the 64-wide key).  Eight values per lane, one pass.  Bound by its launch up to some
// hundred tokens; at 4096 it reads 17 MB and writes 11 MB in 14 us.  In its place stood
// twelve launches of tensor operations (90 us at 4096 tokens).
__global__ __launch_bounds__(320) void mla_latent_kernel(LatentArgs p) {
    __shared__ float part[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t row = blockIdx.x;
    const int b = (int)(row / p.tokens), tok = (int)(row - (int64_t)b * p.tokens);
    const uint16_t* src = p.a + row * p.a_stride;
    float x[8], w[8];
    if (wave == 4) {
        unpack8(*(const v4u*)(src + p.q_rank + lane * 8), x);
        unpack8(*(const v4u*)(p.kv_w + lane * 8), w);
        const uint32_t key = lane < 32 ? *(const uint32_t*)(src + p.q_rank + kC + lane * 2) : 0u;
        const float r = 1.0f / __builtin_sqrtf(wave_sum(sum_sq8(x)) * (1.0f / kC) + p.kv_eps);
        v4u o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = pack_bf16(x[2 * e] * r * w[2 * e], x[2 * e + 1] * r * w[2 * e + 1]);
        *(v4u*)(p.kv + b * p.kv_bs + (int64_t)tok * kC + lane * 8) = o;
        if (lane < 32) {
            const v2f cs = p.freqs[(int64_t)tok * (kRope / 2) + lane];
            const float re = bf16lo_to_f32(key), im = bf16hi_to_f32(key);
            *(uint32_t*)(p.pe + b * p.pe_bs + (int64_t)tok * kRope + lane * 2) = pack_bf16(re * cs.x - im * cs.y, re * cs.y + im * cs.x);
        }
    } else {
        const int c = threadIdx.x * 8;
        const bool live = c < p.q_rank;                 // whole 16-lane groups: q_rank is a multiple of 128
        v4u raw = {}, wr = {};
        if (live) { raw = *(const v4u*)(src + c); wr = *(const v4u*)(p.q_w + c); }
        unpack8(raw, x);
        unpack8(wr, w);
        const float sum = wave_sum(sum_sq8(x));
        if (lane == 0) part[wave] = sum;
    }
    __syncthreads();
    if (wave == 4) return;
    const int c = threadIdx.x * 8;
    const float r = 1.0f / __builtin_sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)p.q_rank + p.q_eps);
    uint32_t abits = 0u;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        x[e] = round_bf16(x[e] * r * w[e]);
        abits = umax_u32(abits, abs_bits(x[e]));
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) abits = umax_u32(abits, (uint32_t)__shfl_xor((int)abits, d));
    const float sc = block_scale(abits, false), rs = 1.0f / sc;
    const bool fast = block_is_finite(abits);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = block_quotient(x[e], sc, rs, fast);
    if (c < p.q_rank) {
        *(v2u*)(p.y + row * p.q_rank + c) = v2u{ pack_fp8x4(v[0], v[1], v[2], v[3]), pack_fp8x4(v[4], v[5], v[6], v[7]) };
        if ((lane & 15) == 0) p.ys[row * (p.q_rank / 128) + c / 128] = sc;
    }
}

inline int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// How the positions of a step are split: one attend workgroup per compute unit (its LDS and registers take a whole one; fewer
// leave units idle, more write more partial sums), a tile each at least.
void decode_plan(DecodeArgs& a, int64_t batch, int64_t rows, int64_t positions) {
    a.batch = (int)batch; a.rows = (int)rows; a.positions = (int)positions;
    a.tiles = (int)((positions + kTile - 1) / kTile);
    a.blocks = (int)((rows + kRows - 1) / kRows);
    const int64_t base = batch * a.blocks;
    int64_t splits = 256 / base;
    splits = splits < 1 ? 1 : splits > a.tiles ? a.tiles : splits;
    a.per = (int)((a.tiles + splits - 1) / splits);
    a.splits = (a.tiles + a.per - 1) / a.per;
}

}  // namespace

size_t mla_decode_workspace_bytes(int64_t batch, int64_t tokens, int64_t positions, int heads) {
    DecodeArgs a;
    decode_plan(a, batch, tokens * heads, positions);
    const int64_t units = batch * a.blocks * a.splits;
    return (size_t)(2 * align256(batch * a.rows * kC * 2) + units * (kPartFloats * 4 + kRows * 8));
}

int launch_mla_decode(const void* q, const void* freqs, const void* kv, int64_t kv_bs, const void* pe, int64_t pe_bs,
                      const void* w, const float* ws, const void* mask, bool mask_f32, void* y, int64_t batch, int64_t tokens,
                      int64_t positions, int heads, float scale, void* workspace, hipStream_t st) {
    DecodeArgs a;
    if (tokens * heads > 0x7fffffff / kRows) return DSV3_ERR_BAD_SHAPE;
    decode_plan(a, batch, tokens * heads, positions);
    if (a.blocks > 65535) return DSV3_ERR_BAD_SHAPE;
    uint8_t* wsp = (uint8_t*)workspace;
    const int64_t lat = align256(batch * a.rows * kC * 2), units = batch * a.blocks * a.splits;
    uint16_t* ql = (uint16_t*)wsp;
    a.out = (uint16_t*)(wsp + lat);
    a.part = (float*)(wsp + 2 * lat);
    a.ml = (v2f*)(a.part + units * kPartFloats);
    a.ql = ql; a.q = (const uint16_t*)q; a.freqs = (const v2f*)freqs;
    a.kv = (const uint16_t*)kv; a.kv_bs = kv_bs; a.pe = (const uint16_t*)pe; a.pe_bs = pe_bs;
    a.mask = mask; a.heads = heads;
    const ScoreUnit u = mask ? score_unit(scale) : ScoreUnit{ 1.f, scale };
    a.unit = u.unit; a.scale = u.rest; a.inv_scale = 1.0f / u.rest;
    int rc = launch_wkv_b_absorb(q, (int64_t)heads * kQd, kQd, w, ws, ql, DSV3_ABSORB_Q, batch * tokens, heads, kNope, kNope, kC, st);
    if (rc != DSV3_OK) return rc;
    const int which = !mask ? kNoMask : mask_f32 ? kMaskF32 : kMaskBf16;
    void (*const kernel)(DecodeArgs) = !mask ? mla_decode_kernel<kNoMask> : mask_f32 ? mla_decode_kernel<kMaskF32> : mla_decode_kernel<kMaskBf16>;
    static LdsGrant grant[3];
    if (!grant[which].ensure((const void*)kernel, kStages * kStage)) return DSV3_ERR_LAUNCH;
    hipLaunchKernelGGL(kernel, dim3(a.splits, (unsigned)batch, a.blocks), dim3(256), kStages * kStage, st, a);
    hipLaunchKernelGGL(mla_combine_kernel, dim3(64, (unsigned)batch, a.blocks), dim3(256), 0, st, a);
    if ((rc = launch_status()) != DSV3_OK) return rc;
    return launch_wkv_b_absorb(a.out, (int64_t)heads * kC, kC, w, ws, y, DSV3_ABSORB_V, batch * tokens, heads, kNope, kNope, kC, st);
}

int launch_mla_latent(const void* a, int64_t a_stride, const void* q_w, const void* kv_w, const void* freqs, void* kv,
                      int64_t kv_bs, void* pe, int64_t pe_bs, void* y, float* ys, int64_t batch, int64_t tokens, int q_rank,
                      float q_eps, float kv_eps, hipStream_t st) {
    LatentArgs p;
    p.a = (const uint16_t*)a; p.a_stride = a_stride;
    p.q_w = (const uint16_t*)q_w; p.kv_w = (const uint16_t*)kv_w; p.freqs = (const v2f*)freqs;
    p.kv = (uint16_t*)kv; p.kv_bs = kv_bs; p.pe = (uint16_t*)pe; p.pe_bs = pe_bs;
    p.y = (uint8_t*)y; p.ys = ys; p.tokens = (int)tokens; p.q_rank = q_rank;
    p.q_eps = q_eps; p.kv_eps = kv_eps;
    hipLaunchKernelGGL(mla_latent_kernel, dim3((unsigned)(batch * tokens)), dim3(320), 0, st, p);
    return launch_status();
}

}  // namespace dsv3
