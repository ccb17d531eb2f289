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
constexpr int kStages = 4;                              // tiles in LDS, computed or on their way
constexpr int kRopeOff = kTile * kC * 2;                // a stage: 32 rows of 1 KiB latents, then 32 rows of 128 B rotary keys
constexpr int kStage = kRopeOff + kTile * kRope * 2;
constexpr int kAhead = 6;                               // operands read from LDS ahead of the MFMA that takes them
constexpr int kSync = 28;                               // the value step behind which a tile's stage is free and the next tile's keys are read

struct DecodeArgs {
    const void* ql;                                     // folded queries [batch][rows][512], rows = tokens * heads, or in operand order
    const uint16_t* q;                                  // queries [batch][rows][192]: their rotary part is read here
    const v2f* freqs;                                   // [tokens][32] (cos, sin)
    const uint16_t* kv; int64_t kv_bs;                  // latent cache, batch stride in elements
    const uint16_t* pe; int64_t pe_bs;
    const void* mask;                                   // [tokens][positions]
    float* part;                                        // [batch][row block][split][row][512]
    v2f* ml;                                            // [batch][row block][row][split] (maximum, sum)
    int rows, heads, positions, tiles, groups, side, blocks, splits, per;   // groups: of 32 rows, in whole 128s; side: tiles that a workgroup takes side by side (G)
    uint32_t blocks_magic, splits_magic;                // for quotient()
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

// mfma32 with its result in ordinary registers: the compiler would put it into accumulation registers, which are all taken, and move 16 sums
// out and back per tile.  It does not know that these are MFMAs, so what it would keep apart stands here: two wait states in front
// (an ordinary instruction may have written an operand); behind the last one, before its result is read, scores_ready.
__device__ __forceinline__ void mfma32_first(v16f& d, v4u a, v4u b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma32_next(v16f& d, v4u a, v4u b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void scores_ready(v16f& d) { asm volatile("s_nop 15" : "+v"(d)); }

// n / d by a multiplication: magic is 2^32 / d rounded up, exact as long as n d < 2^32, or 0 where that does not hold (a division in front of
// everything else costs a quarter of a microsecond)
__device__ __forceinline__ int quotient(int n, int d, uint32_t magic) { return d == 1 ? n : magic ? (int)__umulhi((uint32_t)n, magic) : n / d; }
inline uint32_t magic_of(int64_t most, int64_t d) { return d > 1 && most * d < (1ll << 32) ? (uint32_t)(((1ll << 32) + d - 1) / d) : 0u; }

// Four wavefronts with all 512 registers of their SIMD lane each: a wavefront holds 32 rows' queries as MFMA operands (144
// registers) and their 32 x 512 weighted sums (256).  Per tile of 32 positions (36 KiB in LDS): S^T = K Q^T (36 MFMAs), exponentials in
// registers, O^T += V^T P^T (32 MFMAs).  The
// transposed products leave a row in one lane (and the lane 32 further), and S^T's accumulators already are P^T's operand
// (position 16 u + 8 a + 4 g + r of a tile in register 8 u + 4 a + r of lane half g, slot 4 a + r of K step u).  Keys and
// values are the same 32 x 512 block: the keys are read as rows, the values through the LDS's transposing reads, four
// positions of one feature per lane.
// G tiles side by side: 4 / G groups of 32 rows share a tile, the G wavefronts of a group take every G-th tile of the range and add their
// sums in LDS at the end.  The partial sums that leave (2 KiB a row and range) and that fold reads again are a G-th, the latents that the
// workgroups copy G times as many (from the XCD's L2, the row blocks of a range are neighbours there), and the four stages hold three
// tiles ahead (G = 1), one (2) or none (4).
// Bound: per tile 68 MFMAs of 32 cycles (2180), 1250 + 1190 cycles with their operands' reads, 700 of exponentials, of which the second half stand
// beside the first half's products; a tile takes 3800 in all (4630 with the copies in a row in front and every exponential between the products),
// of which the clock takes back half (1.97 against 2.07 GHz at 32 x 4096).  What a range costs besides: at 256 workgroups and G = 1 67 MB of partial sums, 12 us
// to write and as long to read.  Attention with the query's fold and mla_fold_kernel (us, before: G = 1): 8 sequences at 2000 positions 41.9 ->
// 30.0 (G = 4), 16 at 2000 48.7 -> 34.8 (4), 32 at 1000 50.0 -> 38.3 (4), 64 at 1000 62.6 -> 53.4 (2), 32 at 4096 78.7 -> 68.7 (2).
// PACK: the folded queries come in operand order (launch_wkv_b_absorb_q_packed), a KiB of consecutive bytes per load; as rows a
// load touches 32 of them and takes 64 cycles of the compute unit's load path, 3.8 us for the workgroup's 128.
enum { kNoMask, kMaskBf16, kMaskF32 };
template <int MASK, bool PACK, int G>
__global__ __launch_bounds__(256, 1) void mla_decode_kernel(DecodeArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    constexpr int RB = 4 / G, R = kStages / G;          // row groups of a workgroup; steps that the stages hold
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 31, g = lane >> 5, rg = wave % RB, par = wave / RB;
    // a contiguous run of workgroups per XCD, the row blocks of a range next to each other: its latents are in the XCD's L2
    int unit = blockIdx.x;
    {
        const int T = gridDim.x, q = T / 8, r = T % 8, x = unit % 8;
        unit = x * q + min(x, r) + unit / 8;
    }
    const int range = quotient(unit, p.blocks, p.blocks_magic), blk = unit - range * p.blocks;
    const int b = quotient(range, p.splits, p.splits_magic), split = range - b * p.splits;
    const int t0 = split * p.per, t1 = min(p.tiles, t0 + p.per), limit = min(p.positions, t1 * kTile);
    const int row0 = blk * (RB * 32) + rg * 32;
    const int row = min(row0 + i, p.rows - 1);          // rows past the end repeat the last one; fold leaves them out

    // A tile is a buffer of the positions that it has: rows past the end, and all of a tile past the range, read as zeros without a
    // request, so that every tile is as many copies, whose outstanding ones can be counted.
    const uint32_t lds0 = lds_addr_of(lds);
    const uint16_t* kvb = p.kv + b * p.kv_bs;
    const uint16_t* peb = p.pe + b * p.pe_bs;
    struct Source { v4i kv, pe; uint32_t at; };
    auto source = [&](int t, int st) -> Source {
        const int rows = t < t1 ? min(p.positions - t * kTile, kTile) : 0;
        return { buffer_of(kvb + (int64_t)t * (kTile * kC), rows * (kC * 2)), buffer_of(peb + (int64_t)t * (kTile * kRope), rows * (kRope * 2)), lds0 + st * kStage };
    };
    // G < 4: all wavefronts copy a tile, nine copies each: rows 4 w .. and 16 + 4 w .. of the latents (whose swizzles differ in constants only)
    // and eight rotary rows.  G = 4: a wavefront its own tile, 36 copies.
    const uint32_t kvoff = G < 4 ? wave * 4096 + ((lane ^ wave) << 4) : lane << 4;      // row 0 of the wavefront's; row r has chunk c at c ^ swz(r)
    const int w2 = G < 4 ? (wave & 1) << 2 : 0;
    const uint32_t peoff = (G < 4 ? wave * 1024 : 0) + (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 4) & 3 | w2)) << 4);   // row r has chunk c at c ^ (r / 2 & 7)
    const uint32_t kv_add = G < 4 ? wave * 4096 : 0, pe_add = kRopeOff + (G < 4 ? wave * 1024 : 0);
    auto issue = [&](const Source& s, auto which) {
        constexpr int n = decltype(which)::value;
        if constexpr (G < 4) {
            if constexpr (n < 8) copy16_buffer<(n & 3) * 1024 + (n >> 2) * 16384>(s.kv, kvoff ^ ((n & 3) * 0x440 + (n >> 2) * 16384), s.at + kv_add);
            else copy16_buffer<0>(s.pe, peoff, s.at + pe_add);
        } else {
            uint32_t off = n < 32 ? kvoff : peoff;
            asm volatile("" : "+v"(off));               // (nor for 36 copies' offsets)
            if constexpr (n < 32) copy16_buffer<n * 1024>(s.kv, off ^ (n * 1024 + (((n & 3) << 2 | (n >> 2 & 3)) << 4)), s.at);
            else copy16_buffer<(n - 32) * 1024>(s.pe, off ^ ((n - 32) * 1024 + ((n & 1) << 6)), s.at + pe_add);
        }
    };
    if constexpr (G < 4) {
        for (int n = 0; n < (R - 1) * G && (G > 1 || t0 + n < t1); ++n) {
            const Source s = source(t0 + n, n);
            unrolled<9>([&](auto k) { issue(s, k); });
        }
    } else if (t0 + par < t1) {
        const Source s = source(t0 + par, par);
        unrolled<36>([&](auto k) { issue(s, k); });
    }

    // lane (row i, half g) holds elements 16 s + 8 g .. + 7; the last four steps are rotated here
    v4u Q[36];
    {
        // (packed, a last block's missing rows hold anything; nobody reads their results)
        const v4u* src = (const v4u*)p.ql + (PACK ? ((int64_t)b * p.groups + row0 / 32) * (kC / 16) * 64 + lane : ((int64_t)b * p.rows + row) * (kC / 8) + g);
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
    // Operands are read kAhead MFMAs ahead of use; the sched_barriers keep the order that is written here (left alone, the scheduler puts each read
    // next to its MFMA and waits).  The ring goes from the keys to the values and on to the next tile's keys; as it makes no whole
    // number of turns in the 32 value steps, the first two keys have registers of their own.
    v4u ring[kAhead], first[2];
    auto key = [&](const uint8_t* base, int s) -> v4u {
        return s < 32 ? *(const v4u*)(base + (kaddr ^ ((s & 7) << 5)) + (s >> 3) * 256) : *(const v4u*)(base + (raddr ^ ((s - 32) << 5)));
    };
    auto first_keys = [&](const uint8_t* base) {
        first[0] = key(base, 0);
        first[1] = key(base, 1);
#pragma unroll
        for (int s = 2; s < kAhead + 2; ++s) ring[s % kAhead] = key(base, s);
    };
    // the next step's tiles are there, once this wavefront's copies of them are (G = 1: those of the two behind it stay in flight) and everybody's
    auto arrived = [&] {
        constexpr int left = R > 2 ? (R - 2) * 9 * G : 0;
        __builtin_amdgcn_s_waitcnt(0x0f70 | (left & 15) | (left >> 4) << 14);   // vmcnt
        barrier_no_fence();
    };

    // One tile.  qk_copy and pv_copy: copies beside the MFMA just issued.  The last value steps read the next tile's first keys (G < 4).
    auto tile = [&](int t, const uint8_t* base, const uint8_t* next, auto qk_copy, auto pv_copy) {
        const uint32_t vbase = lds_addr_of(base) + vaddr;       // stages are multiples of 1 KiB: the xors below stay inside a row
        auto value = [&](int s) -> v4u {                        // positions 16 (s / 16) .. of features 32 (s % 16) ..
            const uint32_t at = (vbase ^ ((s & 3) << 6)) + (s >> 4) * 16384 + ((s & 15) >> 2) * 256;
            const v2u lo = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf)(uintptr_t)at));
            const v2u hi = __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf)(uintptr_t)((at ^ 32) + 8192)));
            return v4u{ lo[0], lo[1], hi[0], hi[1] };
        };
        v16f T[1];
        v16f& S = T[0];
        __builtin_amdgcn_sched_barrier(0);
        unrolled<36>([&](auto step) {
            constexpr int s = decltype(step)::value;
            if constexpr (s == 0) mfma32_first(S, first[0], Q[0]);
            else mfma32_next(S, s < 2 ? first[s] : ring[s % kAhead], Q[s]);
            if constexpr (s >= 2) ring[s % kAhead] = s + kAhead < 36 ? key(base, s + kAhead) : value(s + kAhead - 36);
            qk_copy(step);
            __builtin_amdgcn_sched_barrier(0);
        });
        scores_ready(S);
        if constexpr (MASK != kNoMask) {
            int tok = row / p.heads;
            asm volatile("" : "+v"(tok));               // (the addresses are formed here: there are no registers to keep them in)
            const int64_t mrow = (int64_t)tok * p.positions;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t at = mrow + min(t * kTile + 8 * (e >> 2) + 4 * g + (e & 3), p.positions - 1);
                S[e] = __builtin_fmaf(S[e], p.unit, mask_at<MASK == kMaskF32>(p.mask, at) * p.inv_scale);
            }
        }
        if ((t + 1) * kTile > limit) {                  // the last tile may reach past the end, a step's tiles past the range
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (t * kTile + 8 * (e >> 2) + 4 * g + (e & 3) >= limit) S[e] = -__builtin_inff();
        }
        float mx = S[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = __builtin_elementwise_maximum(mx, S[e]);
        const v2f both = halves32(mx);
        mx = fmaxf(both.x, both.y);
        // The maximum is only raised when it grows by more than 2^64: exponentials and sums have room for that in binary32
        // and bf16, and so the 256 multiplications are needed in the rarest of cases.
        // (Rows past the end, whose queries are whatever the scratch held, do not ask for it: the others' roundings would follow.)
        const bool raise = row0 + i < p.rows && ((mx - m) * scale2 > 64.f || (m == -__builtin_inff() && mx > m));
        if (__any(raise)) {
            const float mn = fmaxf(m, mx);
            const float a = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m - mn) * scale2);
            l *= a;
            m = mn;
            if (t >= t0 + G) {
#pragma unroll
                for (int d = 0; d < 16; ++d) scale_agprs(O[d], a);
                asm volatile("s_nop 7" ::: "memory");
            }
        }
        const float off = softmax_offset(T, m, scale2);
        float sum = 0.f;
        v4u P[2];
        auto weights = [&](int u, int q) {              // two positions' exponentials
            const int e = 8 * u + 2 * q;
            const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e], scale2, -off));
            const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e + 1], scale2, -off));
            sum += x + y;
            P[u][q] = pack_bf16(x, y);
        };
#pragma unroll
        for (int q = 0; q < 4; ++q) weights(0, q);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<32>([&](auto step) {
            constexpr int s = decltype(step)::value;
            O[s & 15] = mfma32(ring[s % kAhead], P[s >> 4], O[s & 15]);
            if constexpr (s + kAhead < 32) ring[s % kAhead] = value(s + kAhead);
            if constexpr (s < 12 && s % 3 == 2) weights(1, s / 3);      // the second half's, beside the first half's products
            pv_copy(step);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G < 4 && s == kSync) {                        // this tile's last operands are in registers: its stage is free behind the barrier
                arrived();
                first[0] = key(next, 0);
                first[1] = key(next, 1);
#pragma unroll
                for (int f = 2; f <= kSync - 24; ++f) ring[f] = key(next, f);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (G < 4 && s > kSync) {
                ring[s % kAhead] = key(next, s - 24);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        l += sum;
#pragma unroll
        for (int d = 0; d < 16; ++d) asm volatile("" : "+a"(O[d]));     // (the sums stay where they are)
    };
    auto no_copy = [](auto) {};

    if constexpr (G < 4) {
        if (t0 + (R - 1) * G > t1) __builtin_amdgcn_s_waitcnt(0x0f70);  // (fewer copies than are counted)
        arrived();
        first_keys(lds + par * kStage);
        int st = 0;
        for (int t = t0; t < t1; t += G) {
            const int st_next = (st + 1) % R, st_free = (st + R - 1) % R;
            // A copy beside every fourth (second) MFMA into the stage of the step before, which is free: the four wavefronts take turns on
            // the compute unit's load path while the matrix cores are busy; nine in a row keep each of them for a thousand cycles.
            Source ahead[G];
#pragma unroll
            for (int j = 0; j < G; ++j) ahead[j] = source(t + (R - 1) * G + j, st_free * G + j);
            tile(t + par, lds + (st * G + par) * kStage, lds + (st_next * G + par) * kStage, [&](auto step) {
                constexpr int s = decltype(step)::value, E = 4 / G;
                if constexpr (s % E == E - 1) issue(ahead[s / E / 9], std::integral_constant<int, s / E % 9>());
            }, no_copy);
            st = st_next;
        }
    } else {
        for (int t = t0 + par; t < t1; t += G) {
            int at = par * kStage;                      // one stage a wavefront, nobody else's
            asm volatile("" : "+s"(at));                // (its addresses are formed in the loop: there are no registers to keep them in)
            const uint8_t* own = lds + at;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            first_keys(own);
            // the next tile comes where this one's rows have been read: the rotary rows behind the scores, the first 16 positions' beside the
            // second half's products
            const Source ahead = source(t + G, par);
            tile(t, own, own, no_copy, [&](auto step) {
                constexpr int s = decltype(step)::value;
                if constexpr (s >= 1 && s <= 4) issue(ahead, std::integral_constant<int, 31 + s>());
                if constexpr (s >= 16) issue(ahead, std::integral_constant<int, s - 16>());
            });
            unrolled<16>([&](auto k) { issue(ahead, std::integral_constant<int, decltype(k)::value + 16>()); });
        }
    }

    const v2f parts = halves32(l);
    l = parts.x + parts.y;
    const int64_t bb = (int64_t)b * p.blocks + blk;
    __builtin_amdgcn_s_waitcnt(0x0f70);                 // (copies of the tiles past the range still write zeros)
    barrier_no_fence();
    // The sums leave as rows, which fold reads whole: 64 features of 32 rows at a time through LDS (16-byte chunks xor-ed with
    // the row), so that a store writes four pieces of 256 bytes; straight from the registers it would be 32 of 32.  The G wavefronts of
    // a row group first add theirs, each for 32 / G of the rows.
    v2f* const table = (v2f*)(lds + 65536);             // (maximum, sum) [wavefront][row]
    constexpr int N = 8 / G;
    float wt[N][G];
    if constexpr (G == 1) {
        if (g == 0) p.ml[(bb * (RB * 32) + rg * 32 + i) * p.splits + split] = v2f{ m, l };
    } else {
        if (g == 0) table[wave * 32 + i] = v2f{ m, l };
        barrier_no_fence();
        auto weigh = [&](int r, float (&w)[G]) -> v2f { // row r's weights; its maximum and sum
            v2f x[G];
            float top = -__builtin_inff(), sum = 0.f;
#pragma unroll
            for (int j = 0; j < G; ++j) { x[j] = table[(rg + RB * j) * 32 + r]; top = fmaxf(top, x[j].x); }
#pragma unroll
            for (int j = 0; j < G; ++j) {
                w[j] = x[j].x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((x[j].x - top) * scale2);
                sum += x[j].y * w[j];
            }
            return v2f{ top, sum };
        };
#pragma unroll
        for (int n = 0; n < N; ++n) weigh(4 * (par * N + n) + (lane >> 4), wt[n]);
        if (par == 0) {
            float w[G];
            const v2f ml = weigh(i, w);
            if (g == 0) p.ml[(bb * (RB * 32) + rg * 32 + i) * p.splits + split] = ml;
        }
    }
    float* dst = p.part + ((bb * p.splits + split) * (RB * 32) + rg * 32 + par * (4 * N) + (lane >> 4)) * kC + (lane & 15) * 4;
    auto put = [&](int d2) {                            // two buffers a wavefront: the next 64 features are written while these are read
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const v16f& o = O[2 * d2 + (c >> 2)];
            const int e = 4 * (c & 3);
            *(v4f*)(lds + wave * 16384 + (d2 & 1) * 8192 + i * 256 + (((2 * c + g) ^ (i & 15)) << 4)) = v4f{ o[e], o[e + 1], o[e + 2], o[e + 3] };
        }
    };
    put(0);
#pragma unroll
    for (int d2 = 0; d2 < 8; ++d2) {
        if constexpr (G > 1) barrier_no_fence();        // everybody's are there, and the buffers written next have been read
        v4f x[N][G];
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const int r = 4 * (par * N + n) + (lane >> 4);
                x[n][j] = *(const v4f*)(lds + (rg + RB * j) * 16384 + (d2 & 1) * 8192 + r * 256 + (((lane & 15) ^ (r & 15)) << 4));
            }
        if (d2 < 7) put(d2 + 1);
#pragma unroll
        for (int n = 0; n < N; ++n) {
            v4f v = x[n][0];
            if constexpr (G > 1) {
                v = v * wt[n][0];
#pragma unroll
                for (int j = 1; j < G; ++j) v += x[n][j] * wt[n][j];
            }
            *(v4f*)(dst + n * 4 * kC + d2 * 64) = v;
        }
    }
}

struct FoldArgs {
    const float* part; const v2f* ml;                   // as DecodeArgs
    const uint8_t* w; const float* ws;                  // wkv_b fp8 [heads * 256, 512] and its block scales
    void* y; float* ys;                                 // bf16 [tokens][heads][128], or e4m3 and scales [tokens][heads]
    int tokens, per_seq, heads, rows, blocks, splits, group;    // tokens of all sequences and of one; rows of an attention workgroup and its blocks; tokens at a time, up to 16
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
            const int64_t bb = (int64_t)b * p.blocks + row / p.rows, part = (int64_t)p.rows * kC;
            const v2f* ml = p.ml + (bb * p.rows + row % p.rows) * p.splits;
            const float* src = p.part + bb * p.splits * part + (row % p.rows) * kC + lane * 4;
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
                    const float* at = src + (s0 + s) * part;
#pragma unroll
                    for (int u = 0; u < U; ++u, at += per * part) { o[u][0] = *(const v4f*)at; o[u][1] = *(const v4f*)(at + kC / 2); }
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
// leave units idle, more write more partial sums), a tile a wavefront each at least; and how many tiles a workgroup takes side by side: what
// costs least by the measured costs (us) of a wavefront's tiles one after another (2.3; 2.65 and 3.4 where two and four at a time leave less or no room for
// the next ones), of the partial sums (8 to 12 us for those of 256 workgroups of 128 rows) and of adding the wavefronts' sums (0.5 for two, 1.0 for four).
// Where a wavefront has one tile, copies, barrier and sum stand beside nothing (0.8 for two, 1.2 for four, 0.3 where a context of one or two tiles leaves half of
// these without any), and of the partial sums those of rows that there are cost most, with 0.01 for each range that a row has.  The layer, us for one /
// two / four, three layers' weights in turn: 1 sequence of 128 heads at 300 positions 65.5 / 66.1 / 66.6, at 700 65.9 / 65.4 / 65.6, at 2000 69.2 / 68.2 / 67.4, 8 at 64
// 69.8 / 69.5 / 68.7; attention with the query's fold and mla_fold_kernel: 8 at 2000 45.1 / 36.0 / 34.7, 32 at 4096 84.8 / 80.5 / 93.5, 64 at 4096 125 / 129 / 152, 4 of 16
// heads at 64 19.9 / 21.0 / 20.3.  Over 759 shapes of one tile a wavefront (8 .. 128 heads, 1 .. 128 sequences, 1 .. 5 tokens, 32 .. 4000 positions) the rule is 0.4 %
// from the best of the three on average and 1.06 x faster than one everywhere, at worst 2 % slower (with the costs of several tiles 1.3 % from the
// best, at worst 14 % slower than one); in the layer 0.10 us from the best on average over 47 of them, 0.27 before.
// A wavefront has the tiles that one of G = 1 has: longer ranges would round more exponentials (a range's largest is exactly one).
void decode_plan(DecodeArgs& a, int64_t batch, int64_t rows, int64_t positions) {
    a.rows = (int)rows; a.positions = (int)positions;
    a.tiles = (int)((positions + kTile - 1) / kTile);
    a.groups = (int)((rows + 127) / 128 * 4);
    double best = 0;
    bool one_tile = false;                              // a wavefront has one tile
    for (int side = 1; side <= 4; side *= 2) {
        const int64_t blocks = (rows + 128 / side - 1) / (128 / side), base = batch * blocks, steps = (a.tiles + side - 1) / side;
        int64_t splits = 256 / base;
        splits = splits < 1 ? 1 : splits > steps ? steps : splits;
        const int64_t n = (steps + splits - 1) / splits;
        splits = (steps + n - 1) / n;
        if (side == 1) one_tile = n == 1;
        const int64_t units = base * splits, rounds = (units + 255) / 256;
        double us = rounds * (2.3 + (n - 1) * (side == 1 ? 2.3 : side == 2 ? 2.65 : 3.4)) + (rounds - 1) * 3;
        if (one_tile) us += units * (128 / side) * 0.0001 + batch * rows * splits * 0.0004 + splits * 0.01 + (side == 1 ? 0 : side == 2 ? 0.8 : a.tiles <= 2 ? 0.3 : 1.2);
        else us += units * (128 / side) * 0.00049 + (side == 1 ? 0 : side == 2 ? 0.5 : 1.0);
        if (side > 1 && us >= best) continue;
        best = us;
        a.side = side; a.blocks = (int)blocks; a.per = (int)(n * side); a.splits = (int)splits;
    }
}
size_t decode_bytes(const DecodeArgs& a, int64_t batch) {
    const int64_t units = batch * a.blocks * a.splits, rows = 128 / a.side;
    return (size_t)(batch * a.groups * (32 * kC * 2) + units * rows * (kC * 4 + 8));
}

template <int G> int launch_attend(const DecodeArgs& a, int which, unsigned grid, hipStream_t st) {
    static void (*const kernels[6])(DecodeArgs) = { mla_decode_kernel<kNoMask, false, G>, mla_decode_kernel<kNoMask, true, G>,
                                                    mla_decode_kernel<kMaskBf16, false, G>, mla_decode_kernel<kMaskBf16, true, G>,
                                                    mla_decode_kernel<kMaskF32, false, G>, mla_decode_kernel<kMaskF32, true, G> };
    static LdsGrant grant[6];
    if (!grant[which].ensure((const void*)kernels[which], kStages * kStage)) return DSV3_ERR_LAUNCH;
    hipLaunchKernelGGL(kernels[which], dim3(grid), dim3(256), kStages * kStage, st, a);
    return DSV3_OK;
}

}  // namespace

int mla_decode_side(int64_t batch, int64_t tokens, int64_t positions, int heads) {
    DecodeArgs a;
    decode_plan(a, batch, tokens * heads, positions);
    return a.side;
}

size_t mla_decode_workspace_bytes(int64_t batch, int64_t tokens, int64_t positions, int heads) {
    DecodeArgs a;
    decode_plan(a, batch, tokens * heads, positions);
    return decode_bytes(a, batch);
}

int launch_mla_decode(const void* q, const void* freqs, const void* kv, int64_t kv_bs, const void* pe, int64_t pe_bs,
                      const void* w, const float* ws, const void* mask, bool mask_f32, void* y, float* ys, int64_t batch,
                      int64_t tokens, int64_t positions, int heads, float scale, void* workspace, hipStream_t st) {
    DecodeArgs a;
    if (tokens * heads > 0x7fffffff / 128 || batch * tokens > 0x7fffffff - 16) return DSV3_ERR_BAD_SHAPE;
    decode_plan(a, batch, tokens * heads, positions);
    const int64_t rows = 128 / a.side, units = batch * a.blocks * a.splits;
    if (a.groups / 4 > 65535 || batch > 65535 || units > 0x7fffffff) return DSV3_ERR_BAD_SHAPE;
    a.blocks_magic = magic_of(units, a.blocks);
    a.splits_magic = magic_of(units, a.splits);
    uint8_t* wsp = (uint8_t*)workspace;
    a.part = (float*)(wsp + batch * a.groups * (32 * kC * 2));
    a.ml = (v2f*)(a.part + units * rows * kC);
    a.ql = wsp; a.q = (const uint16_t*)q; a.freqs = (const v2f*)freqs;
    a.kv = (const uint16_t*)kv; a.kv_bs = kv_bs; a.pe = (const uint16_t*)pe; a.pe_bs = pe_bs;
    a.mask = mask; a.heads = heads;
    const ScoreUnit u = mask ? score_unit(scale) : ScoreUnit{ 1.f, scale };
    a.unit = u.unit; a.scale = u.rest; a.inv_scale = 1.0f / u.rest;
    // Operand order up to 16 tokens in all, which is what the kernel that writes it takes (a sub-tile of 16 tokens): query's fold, attention and
    // mla_fold_kernel of 128 heads at 100 / 700 / 4096 positions, rows against operand order, 1 sequence 25.1 / 27.4 / 31.0 -> 23.1 / 25.8 / 28.4 us, 4 26.8 / 30.2 / 37.0 ->
    // 25.3 / 28.0 / 34.6, 16 29.6 / 35.5 / 54.7 -> 27.9 / 33.7 / 52.9.  With more tokens, tried with one tile at a time, the fold's scattered stores cost 1 to 1.7 us
    // (32 tokens 5.1 -> 6.1, 64 6.2 -> 7.8) and the gain disappears behind the tiles.
    const bool pack = batch * tokens <= 16;
    const int rc = pack ? launch_wkv_b_absorb_q_packed(q, (int64_t)heads * kQd, kQd, w, ws, wsp, batch, tokens, a.groups / 4, heads, kNope, kNope, st)
                        : launch_wkv_b_absorb(q, (int64_t)heads * kQd, kQd, w, ws, wsp, DSV3_ABSORB_Q, batch * tokens, heads, kNope, kNope, kC, st);
    if (rc != DSV3_OK) return rc;
    const int which = (!mask ? kNoMask : mask_f32 ? kMaskF32 : kMaskBf16) * 2 + pack;
    const int launched = a.side == 1 ? launch_attend<1>(a, which, (unsigned)units, st) : a.side == 2 ? launch_attend<2>(a, which, (unsigned)units, st)
                                                                                                     : launch_attend<4>(a, which, (unsigned)units, st);
    if (launched != DSV3_OK) return launched;
    FoldArgs f;
    f.part = a.part; f.ml = a.ml; f.w = (const uint8_t*)w; f.ws = ws; f.y = y; f.ys = ys;
    f.tokens = (int)(batch * tokens); f.per_seq = (int)tokens; f.heads = heads; f.rows = (int)rows; f.blocks = a.blocks; f.splits = a.splits;
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
