// Attention of MLA.forward for many new tokens per sequence (reference: inference/model.py:470-497), from the query
// projection and the latent cache to the FP8 input of the output projection, without a score matrix in memory.
//
// The latent cache holds one 512-wide latent and one 64-wide rotary key per position; the key of head h is
// [W_k[h] latent | rotary key] (128 + 64 wide), its value W_v[h] latent (128 wide), W = wkv_b.  The absorbed form
// folds W_k into the query and W_v into the output, which costs nothing per position but makes every query-key pair
// a 576-wide and every weighted sum a 512-wide product; here the keys and values are formed first (2 * 512 * 256
// operations per head and position) and a pair costs 192 + 128.  With as many new tokens as positions that is 3.4 x
// less work in front of the matrix cores; where few tokens meet many positions the absorbed form wins (mla_decode.hip;
// MLA._explicit_pays weighs the two).
// Roundings: keys and values to bf16 (the absorbed form rounds the folded query and the latent sum instead), exponentials
// to bf16 in front of the value product, scores and sums in binary32, the result to bf16 and then quantised.
//
// Two launches: expand (keys and values, and the rotary keys, in the order in which the attention kernel's wavefronts
// read their operands, and which tiles of the mask are all zero or all -inf) and attend.
// At 4096 tokens, 128 heads, causal mask (kernel trace): expand 140 .. 149 us, attend 735 .. 770 us on a cool card (0.9 PFLOP/s
// of the pairs the mask leaves) and more on a warm one, whose clock falls to 1.8 GHz under it; the layer 1.53 ms where the
// absorbed form as tensor operations took 20.1 ms (2 x 2.5 ms score products, 1.6 ms value product and 12 ms of passes over
// the 4.3 GB score matrix).
#include <type_traits>

#include "mla.hpp"

namespace dsv3 {
namespace {

constexpr int kC = 512, kRope = 64, kNope = 128, kV = 128, kQd = kNope + kRope;
constexpr int kTile = 64;                       // positions per tile
constexpr int kAhead = 6;                       // operands read from LDS ahead of the MFMA that takes them
// One tile's operands, bytes.  Keys: [position half][16-wide K step][lane][16]; the same for the rotary keys; values:
// [32 features][16 positions][lane][16].  A wavefront's operand of one MFMA is 1 KiB, lane l's piece at 16 l.
constexpr int kKeyBytes = kTile * kNope * 2, kValBytes = kTile * kV * 2, kRopeBytes = kTile * kRope * 2;
constexpr int kHeadTile = kKeyBytes + kValBytes;
constexpr int kQTile = 128;                     // query rows per workgroup: 4 wavefronts x 32
constexpr int kQGroup = 256;                    // query rows whose mask flags are one word

// ----------------------------------------------------------------------------------------------------------- flags

enum : uint8_t { kClear = 0, kMixed = 1, kSkip = 2 };
enum MaskKind { kNoMask = 0, kMaskBF16 = 1, kMaskF32 = 2 };

// flags[q / 256][tile][q / 32 % 8]: what the mask does to 32 query rows x 64 positions (all zero, anything, all -inf or no
// row).  An attend workgroup's eight (or four) flags of a tile are one 64-bit word (or half of it), its tiles follow one another.
// A wavefront looks at one such block and requests all of it before it looks at any: 16 bytes per lane where rows are whole
// 16-byte pieces (`wide`) and the block has all its rows and positions, else one element per lane and row.  The wavefronts of the expand
// kernel do this while their weights are on their way (a launch of its own took 5 us at 200 tokens, 12 at 4096).
template <bool F32>
__device__ __forceinline__ uint8_t mask_flag(const void* mask, int rows, int positions, int wide, int q32, int tile, int lane) {
    const int p0 = tile * kTile;
    uint32_t not_zero = 0u, not_ninf = 0u;              // bits in which a value differs from +-0, from -inf
    if (wide && q32 * 32 + 32 <= rows && p0 + kTile <= positions) {
        constexpr int kPer = F32 ? 4 : 8, kChunks = kTile / kPer, kRowsAt = 64 / kChunks, kLoads = 32 / kRowsAt;
        constexpr int kSize = F32 ? 4 : 2;
        const uint8_t* src = (const uint8_t*)mask + ((int64_t)(q32 * 32 + lane / kChunks) * positions + p0 + lane % kChunks * kPer) * kSize;
        v4u v[kLoads];
#pragma unroll
        for (int n = 0; n < kLoads; ++n) v[n] = *(const v4u*)(src + (int64_t)n * kRowsAt * positions * kSize);
#pragma unroll
        for (int n = 0; n < kLoads; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                not_zero |= v[n][e] & (F32 ? 0x7fffffffu : 0x7fff7fffu);
                not_ninf |= v[n][e] ^ (F32 ? 0xff800000u : 0xff80ff80u);
            }
    } else if (p0 + lane < positions) {
        float v[32];
        int q = q32 * 32;
        asm("" : "+v"(q));                              // (32 rows' addresses do not fit the scalar registers)
#pragma unroll
        for (int r = 0; r < 32; ++r) v[r] = mask_at<F32>(mask, (int64_t)min(q + r, rows - 1) * positions + p0 + lane);
#pragma unroll
        for (int r = 0; r < 32; ++r)
            if (q32 * 32 + r < rows) {
                not_zero |= f32_as_u32(v[r]) & 0x7fffffffu;
                not_ninf |= f32_as_u32(v[r]) ^ 0xff800000u;
            }
    }
    return __all(not_ninf == 0u) ? kSkip : __all(not_zero == 0u) ? kClear : kMixed;
}

// ---------------------------------------------------------------------------------------------------------- expand

struct ExpandArgs {
    const uint16_t* kv; int64_t kv_bs;          // latents [batch][positions][512], batch stride in elements
    const uint16_t* pe; int64_t pe_bs;          // rotary keys [batch][positions][64]
    const uint8_t* w; const float* ws;          // wkv_b fp8 [heads * 256, 512] and its block scales
    uint8_t* img;                               // [batch][heads][tiles][kHeadTile]
    uint8_t* rope;                              // [batch][tiles][kRopeBytes]
    int batch, heads, positions, tiles;
    const void* mask; uint8_t* flags;           // [rows][positions] / [qgroups][tiles][8]
    int rows, qgroups, wide;                    // qgroups: 256 query rows each
};

// A workgroup owns one head: wavefronts 0-3 hold 32 key features each, 4-7 32 value features, as bf16 MFMA operands
// (32 features x 512 = 128 registers, dequantised once), and stream 32-position sub-tiles of the latents past them
// (32 KiB each, through LDS, one sub-tile ahead).  Key features are issued as the A operand and positions as B, value
// features the other way round, so that in both cases a lane ends up with 16-byte pieces of the attention kernel's
// operand order and a store instruction writes 1 KiB of consecutive bytes: MFMA row 8j + 4g + r of a key wavefront is
// feature 16 (j / 2) + 8 g + 4 (j % 2) + r; a value lane's accumulator registers 8u .. 8u + 7 are, in order, the
// eight positions that the attention kernel's K step u has in that lane.
// Measured at 4096 positions, 128 heads: 219 us with each LDS read next to its MFMA, 136 .. 156 with six on their way (up to 1
// PFLOP/s; MFMAs 60 % of the cycles, the 268 MB of results alone would take 57 us).  What bounds it: every operand read from LDS feeds one
// MFMA.  Four wavefronts of 64 features, where it feeds two, have their weights in accumulation registers, which the compiler
// copies back and forth: 168 us.
template <int MASK> __global__ __launch_bounds__(512, 2) void mla_expand_kernel(ExpandArgs p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * 32 * 1024];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 31, g = lane >> 5;
    const int h = blockIdx.x;
    const int subs = p.batch * p.tiles * 2;                 // 32-position sub-tiles, batch-major
    const int per = (subs + gridDim.y - 1) / gridDim.y;
    const int s0 = blockIdx.y * per, s1 = min(subs, s0 + per);
    auto look_at_mask = [&]() {
        if constexpr (MASK != kNoMask) {
            const int tasks = p.qgroups * p.tiles * 8, stride = gridDim.x * gridDim.y * 8;
            for (int n = (blockIdx.y * gridDim.x + blockIdx.x) * 8 + wave; n < tasks; n += stride) {
                const int grp = n / (p.tiles * 8), in = n - grp * p.tiles * 8;
                const uint8_t f = mask_flag<MASK == kMaskF32>(p.mask, p.rows, p.positions, p.wide, grp * 8 + (in & 7), in >> 3, lane);
                if (lane == 0) p.flags[n] = f;
            }
        }
    };
    if (s0 >= s1) { look_at_mask(); return; }

    if (h == p.heads) {                                     // the rotary keys, shared by all heads: only re-ordered
        for (int sub = s0 + wave; sub < s1; sub += 8) {
            const int b = sub / (p.tiles * 2), sb = sub - b * p.tiles * 2;
            const int pos = min(sb * 32 + i, p.positions - 1);
            const uint16_t* src = p.pe + b * p.pe_bs + (int64_t)pos * kRope + g * 8;
            v4u* dst = (v4u*)(p.rope + (int64_t)sub * (kRopeBytes / 2)) + lane;
#pragma unroll
            for (int s = 0; s < 4; ++s) dst[s * 64] = *(const v4u*)(src + s * 16);
        }
        look_at_mask();
        return;
    }

    // sub-tile rows: 1 KiB each, 16-byte chunk c stored at c ^ (row & 15): 16 rows read at the same c hit 16 distinct
    // 16-byte columns
    const uint32_t lds0 = lds_addr_of(lds);
    auto issue = [&](int sub, int st) {
        sub = min(sub, s1 - 1);
        const int b = sub / (p.tiles * 2), sb = sub - b * p.tiles * 2;
        const uint16_t* base = p.kv + b * p.kv_bs;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int row = wave * 4 + n;
            const int pos = min(sb * 32 + row, p.positions - 1);
            copy16(base + (int64_t)pos * kC, (uint32_t)((lane ^ (row & 15)) << 4), lds0 + st * 32768 + row * 1024);
        }
    };
    issue(s0, 0);

    const bool keys = wave < 4;
    v4u W[32];
    {
        const int j = i >> 3, g2 = (i >> 2) & 1, r = i & 3;
        const int f = keys ? 16 * (j >> 1) + 8 * g2 + 4 * (j & 1) + r : i;
        const int64_t row = (int64_t)h * (kNope + kV) + (keys ? 0 : kNope) + 32 * (wave & 3) + f;
        const uint8_t* src = p.w + row * kC + 16 * g;
        const float* sc = p.ws + (row >> 7) * (kC / 128);
        v4u raw[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) raw[s] = *(const v4u*)(src + 32 * s);
        look_at_mask();                         // while the weights are on their way
#pragma unroll
        for (int s = 0; s < 32; ++s) {
            const uint32_t lo = raw[s / 2][2 * (s & 1)], hi = raw[s / 2][2 * (s & 1) + 1];
            const float k = sc[s / 8];
            const v2f a = fp8x2_lo_to_f32(lo), b = fp8x2_hi_to_f32(lo), c = fp8x2_lo_to_f32(hi), d = fp8x2_hi_to_f32(hi);
            W[s] = v4u{ pack_bf16(a.x * k, a.y * k), pack_bf16(b.x * k, b.y * k), pack_bf16(c.x * k, c.y * k), pack_bf16(d.x * k, d.y * k) };
        }
    }
    // K steps 2 s' and 2 s' + 1 take elements 32 s' + 16 g + 0 .. 7 and + 8 .. 15: a lane reads 16 bytes of its weight row at a time
    const uint32_t frag = i * 1024 + (((2 * g) ^ (i & 15)) << 4);  // chunk 4 s' + 2 g + (s & 1) of row i
    int st = 0;
    for (int sub = s0; sub < s1; ++sub, st ^= 1) {
        if (sub == s0) __builtin_amdgcn_s_waitcnt(0x0f70);          // vmcnt(0)
        else           __builtin_amdgcn_s_waitcnt(0x0f70 | 2);      // vmcnt(2): the two stores of the sub-tile before are younger
        barrier_no_fence();
        issue(sub + 1, st ^ 1);
        v16f acc = {};
        const uint8_t* t = lds + st * 32768;
        // latents kAhead steps ahead; the barriers keep this order
        auto chunk = [&](int s) -> v4u { return *(const v4u*)(t + (frag ^ ((((s >> 1) & 3) * 4 + (s & 1)) << 4)) + (s >> 3) * 256); };
        v4u ring[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) ring[s] = chunk(s);
        __builtin_amdgcn_sched_barrier(0);
        auto products = [&](auto is_key) {
#pragma unroll
            for (int s = 0; s < 32; ++s) {
                acc = is_key ? mfma32(W[s], ring[s % kAhead], acc) : mfma32(ring[s % kAhead], W[s], acc);
                if (s + kAhead < 32) ring[s % kAhead] = chunk(s + kAhead);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (keys) products(std::true_type());
        else products(std::false_type());
        const int b = sub / (p.tiles * 2), sb = sub - b * p.tiles * 2;
        uint8_t* tile = p.img + (((int64_t)b * p.heads + h) * p.tiles + (sb >> 1)) * kHeadTile;
        v4u o[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) o[u][q] = pack_bf16(acc[8 * u + 2 * q], acc[8 * u + 2 * q + 1]);
        // keys: K steps 2 wave + u of position half sb & 1; values: positions 16 (2 (sb & 1) + u) of features 32 (wave - 4)
        v4u* dst = keys ? (v4u*)(tile + ((sb & 1) * 8 + 2 * wave) * 1024) : (v4u*)(tile + kKeyBytes + ((wave & 3) * 4 + 2 * (sb & 1)) * 1024);
        dst[lane] = o[0];
        dst[64 + lane] = o[1];
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);         // the repeated copies of the last iteration still write LDS
}

// ---------------------------------------------------------------------------------------------------------- attend

struct AttendArgs {
    const uint16_t* q;                          // [batch][rows][heads][192], rotary part not yet rotated
    const v2f* freqs;                           // [rows][32] (cos, sin)
    const uint8_t* img; const uint8_t* rope;
    const void* mask; const uint32_t* flags;    // [rows][positions] / [query groups][tiles][2], or null
    uint8_t* y; float* ys;                      // fp8 [batch][rows][heads * 128], scales [batch][rows][heads]
    int batch, heads, rows, positions, tiles, qtiles, per_head;     // per_head: workgroups of a head
    int mask4;                                  // four positions' mask values are one aligned load
    float unit, scale, inv_scale;               // score_unit's unit and rest, and the rest's reciprocal
};

// One workgroup: 128 query rows of one head; wavefront w rows 32 w .. 32 w + 31.  Per tile of 64 positions (40 KiB of
// operands, copied into LDS while the tile before is computed) a wavefront forms S^T = K Q^T (24 MFMAs),
// exponentials in registers, and O^T += V^T P^T (16 MFMAs).  The transposed products leave a query row in one lane
// (and the lane 32 further), so maxima and sums need one exchange, the rescale factor is one value per lane, and the
// accumulator layout of S^T already is the B operand of the second product: position 16 u + 8 a + 4 g + r of a tile sits
// in register 8 u' + 4 a + r of lane half g, which is slot 4 a + r of K step u, and the values were written in that
// order.  The running maximum is only raised when it grows by more than 2^8 (exponentials then stay below 2^8, and most
// tiles skip the 64 multiplications of the rescale).
// Two workgroups share a compute unit, each with two stages of 40 KiB and one wavefront per SIMD: one does matrix products while the
// other does exponentials, waits for its queries or writes its results, and nothing makes them wait for each other; the exponentials and
// the products beside them go first (layer at 800 / 4096: 282 -> 279, 1520 -> 1508 us; with the score product first instead about as much, with
// all products half).  As one workgroup of 256 rows (eight wavefronts in two groups half a tile apart, three stages) the copies of a tile
// served twice the rows, but the steps of the causal diagonal, a ragged last tile and each start and end kept the whole unit: us at
// 200 / 800 / 4096 rows of 128 heads 21.6 / 92 / 785, now 16.5 / 69 / 735; with queries' loads behind the first tile's copies and four
// mask values a load (each was one of its own: 32 lines a load, 2000 cycles of a unit's load path for every block on the diagonal).
template <bool MF32>
__global__ __launch_bounds__(kQTile * 2, 2) void mla_attend_kernel(AttendArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    constexpr int kStage = kHeadTile + kRopeBytes, NW = kQTile / 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 31, g = lane >> 5;
    // heads are dealt over the XCDs (whose L2 then holds a head's keys and values for all its query tiles), the query
    // tiles of a head run last to first: with a causal mask the long ones start first
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int bh = xcd + 8 * (idx / p.per_head), part = idx % p.per_head;
    if (bh >= p.batch * p.heads) return;
    const int b = bh / p.heads, h = bh - b * p.heads;
    const uint8_t* himg = p.img + (int64_t)bh * p.tiles * kHeadTile;
    const uint8_t* rimg = p.rope + (int64_t)b * p.tiles * kRopeBytes;
    const uint32_t lds0 = lds_addr_of(lds), lane16 = lane * 16;
    const float scale2 = p.scale * 1.44269504088896340736f;

#pragma unroll 1
    for (int qt = p.qtiles - 1 - part;;) {
    const int q0 = qt * kQTile + wave * 32;
    const int row = min(q0 + i, p.rows - 1);

    auto issue = [&](int t, int st) {
        const uint8_t* src = himg + (int64_t)t * kHeadTile + wave * 1024;
        const uint8_t* rsrc = rimg + (int64_t)t * kRopeBytes + wave * 1024;
        const uint32_t to = lds0 + st * kStage + wave * 1024;
#pragma unroll 1
        for (int n = 0; n < kHeadTile; n += NW * 1024) copy16(src + n, lane16, to + n);
#pragma unroll 1
        for (int n = 0; n < kRopeBytes; n += NW * 1024) copy16(rsrc + n, lane16, to + kHeadTile + n);
    };
    // Flags of 64 tiles at a time, one word per lane, as three masks: tiles that somebody needs, this wavefront's mixed and
    // skipped ones.  (A look at memory per tile stood in the way of every tile and of each one behind a causal diagonal.)
    constexpr uint32_t kAllSkip = 0x02020202u;
    int window = 0;
    uint64_t act, mix, skip;
    auto look = [&]() {
        uint32_t f = kAllSkip;
        if (window + lane < p.tiles) f = p.flags ? p.flags[((int64_t)(qt >> 1) * p.tiles + window + lane) * 2 + (qt & 1)] : 0u;
        const uint8_t mine = (uint8_t)(f >> (8 * wave));
        act = __ballot(f != kAllSkip);
        mix = __ballot(mine == kMixed);
        skip = __ballot(mine == kSkip);
    };
    auto next_tile = [&](int t, uint8_t& flag) {        // the first tile from t on that somebody needs, and this wavefront's flag
        for (;;) {
            if (t >= window + 64) { window += 64; if (window >= p.tiles) return p.tiles; look(); }
            const uint64_t rest = act >> (t - window);
            if (rest != 0) {
                t += __builtin_ctzll(rest);
                flag = (skip >> (t - window)) & 1 ? kSkip : (mix >> (t - window)) & 1 ? kMixed : kClear;
                return t;
            }
            t = window + 64;
        }
    };

    v16f O[4] = {};
    float m = -__builtin_inff(), l = 0.f;           // running maximum of the scores, this lane's share of the sum
    look();
    uint8_t flag = kSkip, flag_n = kSkip;           // of this tile and the next one
    int t = next_tile(0, flag), st = 0;
    if (t < p.tiles) issue(t, 0);

    // query operands, in the scores' unit: lane (row i, half g) holds elements 16 s + 8 g .. + 7; the last four steps are
    // rotated here
    v4u Q[12];
    {
        int gl = g;
        asm volatile("" : "+v"(gl));       // (addresses kept over both query tiles would spill)
        const uint16_t* src = p.q + (((int64_t)b * p.rows + row) * p.heads + h) * kQd + 8 * gl;
#pragma unroll
        for (int s = 0; s < 12; ++s) Q[s] = *(const v4u*)(src + 16 * s);
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) Q[s][e] = pack_bf16(bf16lo_to_f32(Q[s][e]) * p.unit, bf16hi_to_f32(Q[s][e]) * p.unit);
        const v2f* fr = p.freqs + (int64_t)row * (kRope / 2) + 4 * gl;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const v2f cs = fr[8 * s + e];
                const float re = bf16lo_to_f32(Q[8 + s][e]), im = bf16hi_to_f32(Q[8 + s][e]);
                Q[8 + s][e] = pack_bf16((re * cs.x - im * cs.y) * p.unit, (re * cs.y + im * cs.x) * p.unit);
            }
    }
    while (t < p.tiles) {
        const int tn = next_tile(t + 1, flag_n);
        __builtin_amdgcn_s_waitcnt(0x0f70);             // this tile has landed, everybody is done with the one before
        barrier_no_fence();
        if (tn < p.tiles) issue(tn, st ^ 1);
        const uint8_t* base = lds + st * kStage + lane16;
        v4u ring[kAhead];
        v16f S[2] = {};
        // a mixed block's mask values, requested in front of the score product: lane (row i, half g) positions 32 k + 8 a + 4 g .. + 3
        using MaskVec = typename std::conditional<MF32, v4f, v2u>::type;
        MaskVec M[8];
        const int64_t mrow = (int64_t)row * p.positions;
        auto mask_values = [&]() {
#pragma unroll
            for (int n = 0; n < 8; ++n)
                M[n] = *(const MaskVec*)((const uint8_t*)p.mask + (mrow + min(t * kTile + 8 * n + 4 * g, p.positions - 4)) * (MF32 ? 4 : 2));
        };
        if (!MF32 && flag == kMixed && p.mask4) mask_values();
        if (flag != kSkip) {
            // operands are read kAhead steps ahead; the barriers keep this order (left to itself the scheduler reads two ahead
            // and waits for most of them)
            auto key = [&](int n) -> v4u {              // step n: K step n / 2 of position half n & 1
                return *(const v4u*)(base + (n < 16 ? (n & 1) * 8 + (n >> 1) : kHeadTile / 1024 + (n & 1) * 4 + (n >> 1) - 8) * 1024);
            };
#pragma unroll
            for (int n = 0; n < kAhead; ++n) ring[n] = key(n);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < 24; ++n) {
                S[n & 1] = mfma32(ring[n % kAhead], Q[n >> 1], S[n & 1]);
                if (n + kAhead < 24) ring[n % kAhead] = key(n + kAhead);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (flag != kSkip) {
            if (flag == kMixed && p.mask4) {
                if (MF32) mask_values();        // (32 registers, which the score product does not leave)
#pragma unroll
                for (int n = 0; n < 8; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float v;
                        if constexpr (MF32) v = M[n][r];
                        else v = r & 1 ? bf16hi_to_f32(M[n][r >> 1]) : bf16lo_to_f32(M[n][r >> 1]);
                        S[n >> 2][4 * (n & 3) + r] += v * p.inv_scale;
                    }
            } else if (flag == kMixed) {
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int pos = t * kTile + 32 * k + 8 * (e >> 2) + 4 * g + (e & 3);
                        S[k][e] += mask_at<MF32>(p.mask, mrow + min(pos, p.positions - 1)) * p.inv_scale;
                    }
            }
            if ((t + 1) * kTile > p.positions) {            // the last tile may reach past the end
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int pos = t * kTile + 32 * k + 8 * (e >> 2) + 4 * g + (e & 3);
                        if (pos >= p.positions) S[k][e] = -__builtin_inff();
                    }
            }
            __builtin_amdgcn_s_setprio(1);          // (the other workgroup's matrix products can wait)
            float mx = S[0][0];
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = __builtin_elementwise_maximum(mx, S[k][e]);
            mx = fmaxf(mx, xor32(mx));
            const bool raise = (mx - m) * scale2 > 8.f || (m == -__builtin_inff() && mx > m);
            if (__any(raise)) {
                const float mn = fmaxf(m, mx);
                const float a = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m - mn) * scale2);
                l *= a;
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int e = 0; e < 16; ++e) O[d][e] *= a;
                m = mn;
            }
            const float off = softmax_offset(S, m, scale2);
            auto value = [&](int n) -> v4u { return *(const v4u*)(base + kKeyBytes + ((n & 3) * 4 + (n >> 2)) * 1024); };
#pragma unroll
            for (int n = 0; n < kAhead; ++n) ring[n] = value(n);
            __builtin_amdgcn_sched_barrier(0);
            float sum = 0.f;
            v4u P[4];
            auto expo = [&](int u, int q) {
                const int e = 8 * (u & 1) + 2 * q;
                const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(S[u >> 1][e], scale2, -off));
                const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(S[u >> 1][e + 1], scale2, -off));
                sum += x + y;
                P[u][q] = pack_bf16(x, y);
            };
#pragma unroll
            for (int q = 0; q < 4; ++q) expo(0, q);
#pragma unroll
            for (int n = 0; n < 16; ++n) {              // step n: positions 16 (n / 4), features 32 (n & 3); beside it exponentials of the next positions
                const int u = n >> 2, d = n & 3;
                O[d] = mfma32(ring[n % kAhead], P[u], O[d]);
                if (n + kAhead < 16) ring[n % kAhead] = value(n + kAhead);
                if (u < 3) expo(u + 1, d);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            l += sum;
        }
        st ^= 1;
        t = tn;
        flag = flag_n;
    }

    // O / l to bf16, then the 128 values of a (token, head) as one quantisation block of the output projection's input
    l += xor32(l);
    const float rl = 1.0f / l;
    uint32_t abits = 0u;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            O[d][e] = round_bf16(O[d][e] * rl);
            abits = umax_u32(abits, abs_bits(O[d][e]));
        }
    abits = umax_u32(abits, (uint32_t)__shfl_xor((int)abits, 32));
    const float sc = block_scale(abits, false), rs = 1.0f / sc;
    const bool fast = block_is_finite(abits);
    const bool live = q0 + i < p.rows;
    const int64_t out = (((int64_t)b * p.rows + row) * p.heads + h);
    uint8_t* dst = p.y + out * kV;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            uint32_t by[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = block_quotient(O[d][8 * a + 4 * k + r], sc, rs, fast);
                by[k] = pack_fp8x4(v[0], v[1], v[2], v[3]);
            }
            // by[k]: features 32 d + 16 a + 8 k + 4 g ..; after the exchange lane half g holds 16 a + 8 g .. + 7
            const uint32_t give = g ? by[0] : by[1];
            const uint32_t got = (uint32_t)__shfl_xor((int)give, 32);
            const v2u o = g ? v2u{ got, by[1] } : v2u{ by[0], got };
            if (live) *(v2u*)(dst + 32 * d + 16 * a + 8 * g) = o;
        }
    if (live && g == 0) p.ys[out] = sc;

    // the head's other query tile, if this workgroup has two
    if (p.per_head == p.qtiles || qt <= part) return;
    qt = part;
    barrier_no_fence();                                 // everybody has read the last tiles
    }
}

inline int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

}  // namespace

// Two query tiles a workgroup, the j-th last and the j-th first, where that still makes two workgroups per compute unit:
// under a causal mask every workgroup then has the same work.  Layer, paired against one tile each (us): 800 rows 277 / 282, 1024
// 338 / 352, 4096 1527 / 1557; below the line 400 rows 188 / 169.
bool mla_prefill_paired(int64_t batch, int64_t rows, int heads) {
    return batch * heads * (((rows + kQTile - 1) / kQTile + 1) / 2) >= 512;
}

size_t mla_prefill_workspace_bytes(int64_t batch, int64_t rows, int64_t positions, int heads) {
    const int64_t tiles = (positions + kTile - 1) / kTile, groups = (rows + kQGroup - 1) / kQGroup * 8;
    return (size_t)(align256(batch * heads * tiles * kHeadTile) + align256(batch * tiles * kRopeBytes) + align256(tiles * groups));
}

int launch_mla_prefill(const void* q, const void* freqs, const void* kv, int64_t kv_bs, const void* pe, int64_t pe_bs,
                       const void* w, const float* ws, const void* mask, bool mask_f32, void* y, float* ys, int64_t batch,
                       int64_t rows, int64_t positions, int heads, float scale, void* workspace, hipStream_t st) {
    const int64_t tiles = (positions + kTile - 1) / kTile, qgroups = (rows + kQGroup - 1) / kQGroup;
    const int64_t qtiles = (rows + kQTile - 1) / kQTile;
    const int64_t heads8 = (batch * heads + 7) / 8 * 8;
    const int64_t per_head = mla_prefill_paired(batch, rows, heads) ? (qtiles + 1) / 2 : qtiles;
    const int64_t wgs = heads8 * per_head;
    if (wgs > 0x7fffffff || batch * tiles * 2 > 0x7fffffff || qgroups > 65535) return DSV3_ERR_BAD_SHAPE;
    ExpandArgs e;
    e.kv = (const uint16_t*)kv; e.kv_bs = kv_bs; e.pe = (const uint16_t*)pe; e.pe_bs = pe_bs;
    e.w = (const uint8_t*)w; e.ws = ws;
    e.img = (uint8_t*)workspace;
    e.rope = e.img + align256(batch * heads * tiles * kHeadTile);
    e.batch = (int)batch; e.heads = heads; e.positions = (int)positions; e.tiles = (int)tiles;
    uint8_t* flags = e.rope + align256(batch * tiles * kRopeBytes);
    // one workgroup per compute unit: more ranges of positions would only convert the weights more often (4096 positions
    // and 128 heads: 2 ranges, against 4 ranges in two rounds)
    const int64_t subs = batch * tiles * 2;
    int64_t gy = heads < 256 ? 256 / heads : 1;
    gy = gy > subs ? subs : gy;
    e.mask = mask; e.flags = flags; e.rows = (int)rows; e.qgroups = (int)qgroups;
    const int mask_size = mask_f32 ? 4 : 2;
    e.wide = (uintptr_t)mask % 16 == 0 && positions * mask_size % 16 == 0;
    const auto expand = !mask ? mla_expand_kernel<kNoMask> : mask_f32 ? mla_expand_kernel<kMaskF32> : mla_expand_kernel<kMaskBF16>;
    hipLaunchKernelGGL(expand, dim3(heads + 1, (unsigned)gy), dim3(512), 0, st, e);

    AttendArgs a;
    a.q = (const uint16_t*)q; a.freqs = (const v2f*)freqs; a.img = e.img; a.rope = e.rope;
    a.mask = mask; a.flags = mask ? (const uint32_t*)flags : nullptr;
    a.y = (uint8_t*)y; a.ys = ys;
    a.batch = (int)batch; a.heads = heads; a.rows = (int)rows; a.positions = (int)positions;
    a.tiles = (int)tiles; a.qtiles = (int)qtiles; a.per_head = (int)per_head;
    const ScoreUnit u = score_unit(scale);
    a.unit = u.unit; a.scale = u.rest; a.inv_scale = 1.0f / u.rest;
    a.mask4 = positions % 4 == 0 && (uintptr_t)mask % (4 * mask_size) == 0;
    const bool f32 = mask && mask_f32;
    const auto attend = f32 ? mla_attend_kernel<true> : mla_attend_kernel<false>;
    constexpr int bytes = 2 * (kHeadTile + kRopeBytes);
    static LdsGrant grant[2];
    if (!grant[f32].ensure((const void*)attend, bytes)) return DSV3_ERR_LAUNCH;
    hipLaunchKernelGGL(attend, dim3((unsigned)wgs), dim3(kQTile * 2), bytes, st, a);
    return launch_status();
}

}  // namespace dsv3
