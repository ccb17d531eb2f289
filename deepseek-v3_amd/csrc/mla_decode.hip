// Attention of MLA.forward for few new tokens per sequence (a decode step; reference: inference/model.py:480-497): the
// query is folded through wkv_b (wkv_b_absorb.hip, side Q), so that every head works on the latent cache itself, the
// weighted sum of latents through its value half.  Here, behind the query's fold:
//   attend   split over the positions: scores, softmax and weighted sum of one range of positions, for 128 (token, head)
//            rows of a sequence that share the range's latents; binary32 partial sums
//   fold     the ranges' partial sums to the bf16 latent of each row, its product with the value half of wkv_b and, where the
//            output projection takes it so, the quantisation of the result
// and, in front of the query projection, latent: both RMS norms, the cache rows, the query's quantisation.
// Roundings are those of the tensor operations they replace, with the scores and exponentials' sums in binary32
// throughout; exponentials go to bf16 in front of the value product.
#include <type_traits>

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
constexpr int kPartFloats = kRows * kC;                 // partial sums of a workgroup

struct DecodeArgs {
    const void* ql;                                     // folded queries [batch][rows][512], rows = tokens * heads, or in operand order
    const uint16_t* q;                                  // queries [batch][rows][192]: their rotary part is read here
    const v2f* freqs;                                   // [tokens][32] (cos, sin)
    const uint16_t* kv; int64_t kv_bs;                  // latent cache, batch stride in elements
    const uint16_t* pe; int64_t pe_bs;
    const void* mask;                                   // [tokens][positions]
    float* part;                                        // [batch][row block][split][row][512]
    v2f* ml;                                            // [batch][row block][row][split] (maximum, sum)
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
// of partial sums at the end, and one tile alone (a short context) takes 10.7 us in all, 12.7 without PACK.  The tensor operations in its place
// took 250 us (58 us in the products, the rest in passes over the scores).
// PACK: the folded queries come in operand order (launch_wkv_b_absorb_q_packed), a KiB of consecutive bytes per load; as rows a
// load touches 32 of them and takes 64 cycles of the compute unit's load path, 3.8 us for the workgroup's 128.
enum { kNoMask, kMaskBf16, kMaskF32 };
template <int MASK, bool PACK>
__global__ __launch_bounds__(256, 1) void mla_decode_kernel(DecodeArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 31, g = lane >> 5;
    const int split = blockIdx.x, b = blockIdx.y, blk = blockIdx.z;
    const int t0 = split * p.per, t1 = min(p.tiles, t0 + p.per);
    const int row0 = blk * kRows + wave * 32;
    const int row = min(row0 + i, p.rows - 1);          // rows past the end repeat the last one; fold leaves them out

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
        // (packed, a last block's missing rows hold anything; nobody reads their results)
        const v4u* src = (const v4u*)p.ql + (PACK ? (((int64_t)b * p.blocks + blk) * 4 + wave) * (kC / 16) * 64 + lane : ((int64_t)b * p.rows + row) * (kC / 8) + g);
#pragma unroll
        for (int s = 0; s < 32; ++s) Q[s] = src[s * (PACK ? 64 : 2)];
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
        // (Rows past the end, whose queries are whatever the scratch held, do not ask for it: the others' roundings would follow.)
        const bool raise = row0 + i < p.rows && ((mx - m) * scale2 > 64.f || (m == -__builtin_inff() && mx > m));
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
    const int64_t bb = (int64_t)b * p.blocks + blk;
    if (g == 0) p.ml[(bb * kRows + wave * 32 + i) * p.splits + split] = v2f{ m, l };
    // The sums leave as rows, which fold reads whole: 64 features of 32 rows at a time through LDS (16-byte chunks xor-ed with
    // the row), so that a store writes four pieces of 256 bytes; straight from the registers it would be 32 of 32.
    barrier_no_fence();                                 // everybody has read the last tile
    uint8_t* stg = lds + wave * 16384;                  // two buffers: the next 64 features are written while these are read
    float* dst = p.part + (bb * p.splits + split) * kPartFloats + (wave * 32 + (lane >> 4)) * kC + (lane & 15) * 4;
    auto put = [&](int d2) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const v16f& o = O[2 * d2 + (c >> 2)];
            const int e = 4 * (c & 3);
            *(v4f*)(stg + (d2 & 1) * 8192 + i * 256 + (((2 * c + g) ^ (i & 15)) << 4)) = v4f{ o[e], o[e + 1], o[e + 2], o[e + 3] };
        }
    };
    put(0);
#pragma unroll
    for (int d2 = 0; d2 < 8; ++d2) {
        v4f x[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int r = 4 * n + (lane >> 4);
            x[n] = *(const v4f*)(stg + (d2 & 1) * 8192 + r * 256 + (((lane & 15) ^ (r & 15)) << 4));
        }
        if (d2 < 7) put(d2 + 1);
#pragma unroll
        for (int n = 0; n < 8; ++n) *(v4f*)(dst + n * 4 * kC + d2 * 64) = x[n];
    }
}

struct FoldArgs {
    const float* part; const v2f* ml;                   // as DecodeArgs
    const uint8_t* w; const float* ws;                  // wkv_b fp8 [heads * 256, 512] and its block scales
    void* y; float* ys;                                 // bf16 [tokens][heads][128], or e4m3 and scales [tokens][heads]
    int tokens, per_seq, heads, blocks, splits, group;  // tokens of all sequences and of one; tokens at a time, up to 16
    float scale;
};

// One workgroup: a head and up to 16 tokens at a time.  The wavefronts first form the tokens' latents from the ranges' partial sums
// (a wavefront a token and 2 KiB a range, several wavefronts a token where there are fewer than eight) and leave them in
// LDS as bf16, then multiply: wavefront (kb, dh) holds K block kb of the 64 features dh of the head's value weights and
// the four K blocks' results meet in LDS (absorb_v_ksplit_kernel's maps, wkv_b_absorb.hip).  The 128 features
// of a (token, head) are one quantisation block of the output projection's input.
// Three launches were in its place (combine 5 .. 13.7 us, the product 4.5 .. 7.5, act_quant 4.2).
template <bool QUANT>
__global__ __launch_bounds__(512, 4) void mla_fold_kernel(FoldArgs p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lat[16 * 1024];   // chunk c of row r at c ^ r (low four bits)
    __shared__ v4f sums[8][4][64];                                      // products' partial results; before, latents' partial sums
    __shared__ float norm[8];
    __shared__ uint32_t amax[8][16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4, kb = wave & 3, dh = wave >> 2, h = blockIdx.x;

    // The weights are loaded behind the latents, whose sums need the registers, but their lines (64 KiB, one a thread) are
    // brought into the L2 beside them.
    uint32_t touched = *(const uint32_t*)(p.w + ((int64_t)h * 256 + 128 + (threadIdx.x >> 2)) * kC + (threadIdx.x & 3) * 128);
    const float scale2 = p.scale * 1.44269504088896340736f;
    for (int ms = blockIdx.z * p.group; ms < p.tokens; ms += gridDim.z * p.group) {
        const int n = min(p.group, p.tokens - ms);
        const int per = n == 1 ? 8 : n == 2 ? 4 : n <= 4 ? 2 : 1, sub = wave & (per - 1);       // wavefronts of a token
        auto put = [&](int k, int f, v4f x) {           // features f .. f + 3 of token k
            *(v2u*)(lat + k * 1024 + (((f >> 3) ^ k) << 4) + (f & 4) * 2) = v2u{ pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]) };
        };
        for (int k = wave / per; k < n; k += 8 / per) {
            const int t = ms + k, b = t / p.per_seq, row = (t - b * p.per_seq) * p.heads + h;
            const int64_t bb = (int64_t)b * p.blocks + row / kRows;
            const v2f* ml = p.ml + (bb * kRows + row % kRows) * p.splits;
            const float* src = p.part + bb * p.splits * kPartFloats + (row % kRows) * kC + lane * 4;
            // a chunk of 64 ranges, a lane each; up to six ranges' sums are requested before the first is added
            const v2f none = { -__builtin_inff(), 0.f };
            v2f x = lane < p.splits ? ml[lane] : none;
            float m = x.x, l = 0.f;
            for (int s = 64 + lane; s < p.splits; s += 64) m = fmaxf(m, ml[s].x);
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
            v4f a0 = {}, a1 = {};
            for (int s0 = 0; s0 < p.splits; s0 += 64) {
                if (s0 > 0) x = s0 + lane < p.splits ? ml[s0 + lane] : none;
                const float wt = x.x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((x.x - m) * scale2);
                l += x.y * wt;
                const int end = min(64, p.splits - s0);
                auto add = [&](auto count, int s) {     // ranges s, s + per, ..
                    constexpr int U = decltype(count)::value;
                    v4f o[U][2];
                    const float* at = src + (int64_t)(s0 + s) * kPartFloats;
#pragma unroll
                    for (int u = 0; u < U; ++u, at += (int64_t)per * kPartFloats) { o[u][0] = *(const v4f*)at; o[u][1] = *(const v4f*)(at + kC / 2); }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const float k2 = u32_as_f32((uint32_t)__builtin_amdgcn_readlane((int)f32_as_u32(wt), s + u * per));
                        a0 += o[u][0] * k2;
                        a1 += o[u][1] * k2;
                    }
                };
                int s = sub;
                for (; s + 5 * per < end; s += 6 * per) add(std::integral_constant<int, 6>(), s);
                if (s + 3 * per < end) { add(std::integral_constant<int, 4>(), s); s += 4 * per; }
                if (s + per < end) { add(std::integral_constant<int, 2>(), s); s += 2 * per; }
                if (s < end) add(std::integral_constant<int, 1>(), s);
            }
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) l += __shfl_xor(l, d);
            const float rl = 1.0f / l;                  // a row without any position: 0 * inf, NaN as softmax gives
            if (per == 1) {
                put(k, lane * 4, a0 * rl);
                put(k, kC / 2 + lane * 4, a1 * rl);
            } else {
                v4f* dst = (v4f*)sums + wave * 128 + lane;
                dst[0] = a0;
                dst[64] = a1;
                if (lane == 0) norm[wave] = rl;
            }
        }
        if (per > 1) {
            __syncthreads();
            const int k = threadIdx.x >> 7, f4 = threadIdx.x & 127;
            if (k < n) {
                v4f x = ((const v4f*)sums)[k * per * 128 + f4];
                for (int w = 1; w < per; ++w) x += ((const v4f*)sums)[(k * per + w) * 128 + f4];
                put(k, f4 * 4, x * norm[k * per]);
            }
        }
        asm volatile("" :: "v"(touched));
        v4u raw[4][2];
        float sc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int64_t r = (int64_t)h * 256 + 128 + dh * 64 + (i >> 2) * 16 + t * 4 + (i & 3);
            sc[t] = p.ws[(r >> 7) * (kC / 128) + kb];
            const v4u* src = (const v4u*)(p.w + r * kC + kb * 128 + g * 32);
            raw[t][0] = src[0];
            raw[t][1] = src[1];
        }
        barrier_no_fence();                             // the latents are there, and the partial sums have been read
        v4f acc[4] = {};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const v4u x = *(const v4u*)(lat + i * 1024 + ((kb * 16 + ((g * 4 + s) ^ i)) << 4));
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t lo = raw[t][s >> 1][2 * (s & 1)], hi = raw[t][s >> 1][2 * (s & 1) + 1];
                const v2f x0 = fp8x2_lo_to_f32(lo), x1 = fp8x2_hi_to_f32(lo), x2 = fp8x2_lo_to_f32(hi), x3 = fp8x2_hi_to_f32(hi);
                const v4u A = { pack_bf16(x0.x * sc[t], x0.y * sc[t]), pack_bf16(x1.x * sc[t], x1.y * sc[t]),
                                pack_bf16(x2.x * sc[t], x2.y * sc[t]), pack_bf16(x3.x * sc[t], x3.y * sc[t]) };
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, A), __builtin_bit_cast(v8bf, x), acc[t], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);          // (no more operands at a time than registers)
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) sums[wave][t][lane] = acc[t];
        __syncthreads();
        // the lane's token is i, its features dh 64 + g 16 + kb 4 + [0, 4)
        v4f r = sums[dh * 4][kb][lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) r += sums[dh * 4 + w][kb][lane];
        const int64_t out = (int64_t)(ms + i) * p.heads + h;
        const int f = dh * 64 + g * 16 + kb * 4;
        if constexpr (QUANT) {
            uint32_t abits = 0u;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r[e] = round_bf16(r[e]);
                abits = umax_u32(abits, abs_bits(r[e]));
            }
            abits = umax_u32(abits, (uint32_t)__shfl_xor((int)abits, 16));
            abits = umax_u32(abits, (uint32_t)__shfl_xor((int)abits, 32));
            if (g == 0) amax[wave][i] = abits;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < 8; ++w) abits = umax_u32(abits, amax[w][i]);
            const float bs = block_scale(abits, false), rs = 1.0f / bs;
            const bool fast = block_is_finite(abits);
            if (i < n) {
                *(uint32_t*)((uint8_t*)p.y + out * 128 + f) = pack_fp8x4(block_quotient(r[0], bs, rs, fast), block_quotient(r[1], bs, rs, fast),
                                                                         block_quotient(r[2], bs, rs, fast), block_quotient(r[3], bs, rs, fast));
                if (wave == 0 && g == 0) p.ys[out] = bs;
            }
        } else if (i < n) {
            *(v2u*)((uint16_t*)p.y + out * 128 + f) = v2u{ pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]) };
        }
        __syncthreads();                                // everybody is done with this group's sums
    }
}

struct LatentArgs {
    const uint16_t* a; int64_t a_stride;                // bf16 rows [q_rank | 512 | 64], stride in elements
    const float* parts; int num_parts; int64_t part;    // or that many binary32 slabs of them, `part` elements each, to be added
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
// PARTS: the projections come as the slabs of their K slices, added here in order and rounded to bf16 as the reduction that
// would stand between the two launches does (4 us of a decode step of 3 to 64 sequences).
template <bool PARTS>
__global__ __launch_bounds__(320) void mla_latent_kernel(LatentArgs p) {
    __shared__ float part[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t row = blockIdx.x;
    const int b = (int)(row / p.tokens), tok = (int)(row - (int64_t)b * p.tokens);
    const uint16_t* src = p.a + row * p.a_stride;
    const float* psrc = p.parts + row * p.a_stride;
    auto eight = [&](int c) -> v4u {                    // elements c .. c + 7 of the row
        if constexpr (!PARTS) return *(const v4u*)(src + c);
        constexpr int U = 8;
        v4f v[2] = {};
        for (int s = 0; s < p.num_parts; s += U) {      // slabs past the last are requested again from it and left out
            v4f t[U][2];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float* at = psrc + (int64_t)min(s + u, p.num_parts - 1) * p.part + c;
                t[u][0] = *(const v4f*)at;
                t[u][1] = *(const v4f*)(at + 4);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) v[h] = s + u < p.num_parts ? v[h] + t[u][h] : v[h];
        }
        return v4u{ pack_bf16(v[0][0], v[0][1]), pack_bf16(v[0][2], v[0][3]), pack_bf16(v[1][0], v[1][1]), pack_bf16(v[1][2], v[1][3]) };
    };
    auto two = [&](int c) -> uint32_t {
        if constexpr (!PARTS) return *(const uint32_t*)(src + c);
        constexpr int U = 8;
        v2f v = {};
        for (int s = 0; s < p.num_parts; s += U) {
            v2f t[U];
#pragma unroll
            for (int u = 0; u < U; ++u) t[u] = *(const v2f*)(psrc + (int64_t)min(s + u, p.num_parts - 1) * p.part + c);
#pragma unroll
            for (int u = 0; u < U; ++u) v = s + u < p.num_parts ? v + t[u] : v;
        }
        return pack_bf16(v[0], v[1]);
    };
    float x[8], w[8];
    if (wave == 4) {
        const uint32_t key = lane < 32 ? two(p.q_rank + kC + lane * 2) : 0u;
        unpack8(eight(p.q_rank + lane * 8), x);
        unpack8(*(const v4u*)(p.kv_w + lane * 8), w);
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
        if (live) { raw = eight(c); wr = *(const v4u*)(p.q_w + c); }
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
    return (size_t)(batch * a.blocks * (kRows * kC * 2) + units * (kPartFloats * 4 + kRows * 8));
}

int launch_mla_decode(const void* q, const void* freqs, const void* kv, int64_t kv_bs, const void* pe, int64_t pe_bs,
                      const void* w, const float* ws, const void* mask, bool mask_f32, void* y, float* ys, int64_t batch,
                      int64_t tokens, int64_t positions, int heads, float scale, void* workspace, hipStream_t st) {
    DecodeArgs a;
    if (tokens * heads > 0x7fffffff / kRows || batch * tokens > 0x7fffffff - 16) return DSV3_ERR_BAD_SHAPE;
    decode_plan(a, batch, tokens * heads, positions);
    if (a.blocks > 65535) return DSV3_ERR_BAD_SHAPE;
    uint8_t* wsp = (uint8_t*)workspace;
    const int64_t units = batch * a.blocks * a.splits;
    a.part = (float*)(wsp + batch * a.blocks * (kRows * kC * 2));
    a.ml = (v2f*)(a.part + units * kPartFloats);
    a.ql = wsp; a.q = (const uint16_t*)q; a.freqs = (const v2f*)freqs;
    a.kv = (const uint16_t*)kv; a.kv_bs = kv_bs; a.pe = (const uint16_t*)pe; a.pe_bs = pe_bs;
    a.mask = mask; a.heads = heads;
    const ScoreUnit u = mask ? score_unit(scale) : ScoreUnit{ 1.f, scale };
    a.unit = u.unit; a.scale = u.rest; a.inv_scale = 1.0f / u.rest;
    // Operand order up to 16 tokens in all: the attention gains 2 us (1 at 700: 12.7 -> 10.7, 3 at 200: 12.4 -> 10.3, 8 at 2000: 24.2 ->
    // 22.2), the fold's scattered stores cost it 0.4.  With more they cost 1 to 1.7 us (32 tokens 5.1 -> 6.1, 64 6.2 -> 7.8), the gain
    // disappears behind the tiles (32 at 4096: 56.7 -> 56.4, 64 at 1000: 39.7 -> 39.6).
    const bool pack = batch * tokens <= 16;
    const int rc = pack ? launch_wkv_b_absorb_q_packed(q, (int64_t)heads * kQd, kQd, w, ws, wsp, batch, tokens, a.blocks, heads, kNope, kNope, st)
                        : launch_wkv_b_absorb(q, (int64_t)heads * kQd, kQd, w, ws, wsp, DSV3_ABSORB_Q, batch * tokens, heads, kNope, kNope, kC, st);
    if (rc != DSV3_OK) return rc;
    const int which = (!mask ? kNoMask : mask_f32 ? kMaskF32 : kMaskBf16) * 2 + pack;
    static void (*const kernels[6])(DecodeArgs) = { mla_decode_kernel<kNoMask, false>, mla_decode_kernel<kNoMask, true>,
                                                    mla_decode_kernel<kMaskBf16, false>, mla_decode_kernel<kMaskBf16, true>,
                                                    mla_decode_kernel<kMaskF32, false>, mla_decode_kernel<kMaskF32, true> };
    static LdsGrant grant[6];
    if (!grant[which].ensure((const void*)kernels[which], kStages * kStage)) return DSV3_ERR_LAUNCH;
    hipLaunchKernelGGL(kernels[which], dim3(a.splits, (unsigned)batch, a.blocks), dim3(256), kStages * kStage, st, a);
    FoldArgs f;
    f.part = a.part; f.ml = a.ml; f.w = (const uint8_t*)w; f.ws = ws; f.y = y; f.ys = ys;
    f.tokens = (int)(batch * tokens); f.per_seq = (int)tokens; f.heads = heads; f.blocks = a.blocks; f.splits = a.splits;
    f.scale = a.scale;
    // A head and four, eight or 16 tokens a workgroup, as few as leave a workgroup a compute unit (8 sequences at
    // 2000 positions: 19.5 us with eight tokens in 128 workgroups, 17.0 with four in 256, 18.3 with two in 512; 32 at 4096: 16.5 with
    // 16 in 256, 17.3 with eight in 512); then the groups are dealt over at most 1024.
    f.group = 4;
    while (f.group < 16 && (batch * tokens + f.group - 1) / f.group * heads > 256) f.group *= 2;
    int64_t gz = (batch * tokens + f.group - 1) / f.group, most = 1024 / heads;
    most = most < 1 ? 1 : most;
    gz = gz > most ? most : gz;
    const dim3 grid(heads, 1, (unsigned)gz);
    if (ys) hipLaunchKernelGGL(mla_fold_kernel<true>, grid, dim3(512), 0, st, f);
    else hipLaunchKernelGGL(mla_fold_kernel<false>, grid, dim3(512), 0, st, f);
    return launch_status();
}

int launch_mla_latent(const void* a, int64_t a_stride, const float* parts, int num_parts, const void* q_w, const void* kv_w, const void* freqs, void* kv,
                      int64_t kv_bs, void* pe, int64_t pe_bs, void* y, float* ys, int64_t batch, int64_t tokens, int q_rank,
                      float q_eps, float kv_eps, hipStream_t st) {
    LatentArgs p;
    p.a = (const uint16_t*)a; p.a_stride = a_stride;
    p.parts = parts; p.num_parts = num_parts; p.part = batch * tokens * a_stride;
    p.q_w = (const uint16_t*)q_w; p.kv_w = (const uint16_t*)kv_w; p.freqs = (const v2f*)freqs;
    p.kv = (uint16_t*)kv; p.kv_bs = kv_bs; p.pe = (uint16_t*)pe; p.pe_bs = pe_bs;
    p.y = (uint8_t*)y; p.ys = ys; p.tokens = (int)tokens; p.q_rank = q_rank;
    p.q_eps = q_eps; p.kv_eps = kv_eps;
    const dim3 grid((unsigned)(batch * tokens));
    if (num_parts > 0) hipLaunchKernelGGL(mla_latent_kernel<true>, grid, dim3(320), 0, st, p);
    else hipLaunchKernelGGL(mla_latent_kernel<false>, grid, dim3(320), 0, st, p);
    return launch_status();
}

}  // namespace dsv3
