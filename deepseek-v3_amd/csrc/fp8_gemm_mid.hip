// fp8_gemm for 33 rows and more where whole 256-column tiles leave compute units without work: up to 256 rows of wide weights, up to
// a few thousand of narrow ones, 8192 where these have 128 columns or fewer
// (reference arithmetic: inference/kernel.py:118-172).
//
// A tile of 16 MT rows x 16 SN WN columns per workgroup: eight wavefronts, WM along the rows (16-row sub-tiles dealt round-robin) x
// WN = 8 / WM along the columns (SN strips of 16 each), v_mfma_f32_16x16x128_f8f6f4 with the weights as its A operand.  The large-M
// kernel (fp8_gemm_prefill.hip) has 256 columns per tile and 128 or 256 rows: 7168 -> 36864 at 65 .. 224 rows is 144 such tiles on 256
// compute units (or 288 in more than one round), 7168 -> 1536 is 6 per row tile, cut into up to eight K slices.  Here the columns are
// chosen so that one round fills the chip, mostly without slices.
//
// K blocks of A and B are copied global -> LDS (1 KiB a copy: 8 rows x 128 bytes, chunks xor-ed with the row), S blocks in a ring.  One
// barrier per block, two sub-tiles before its end: the operands that the block still needs are in registers then, its stage is refilled up to the
// next barrier, and the next block's first operands are read while its last MFMAs run.  Each MFMA is followed by the
// FMAs of the one before the last.  Loads and copies are the compiler's own, whose counting sees all of them; it keeps to the
// counted wait in front of the barrier.
// Scales: a row's a_s are K / 128 values apart, so that a copy of 64 rows' scales of one K block is 64 lines, which takes a compute unit's
// load path as long as 4 KiB of tile and, when all units ask, 59 ns.  So four K blocks' are copied at a time, 16 bytes a row; in the
// other three blocks a copy of one line that nobody reads keeps the counts.  (7168 -> 36864 at 128 rows: 70 -> 61 us.)
//
// Measured against the large-M kernel (us, weights from HBM): 7168 -> 36864 at 65 / 128 / 160 / 224 rows 68.5 / 79.3 / 86.0 / 97.1 -> 57.8 / 64.6 /
// 71.1 / 82.7 (a 128-row tile takes 1.07 us per K block, 4.4 TB/s of weights; each row adds: its copies and the weights' share the load
// path); 1536 -> 24576 at 65 / 128 rows 17.2 / 17.6 -> 13.6 / 15.5; the narrow ones at the rule below.
// A wavefront whose last sub-tile lies past the rows leaves it out, and every other column group deals from the other end, so that a SIMD's two
// wavefronts share the rest evenly; copies spread over the whole block.  With the quantisation in front, without / with both: 130 rows 75.5 / 69.5, 160 76.6 /
// 74.3, 193 89.0 / 82.1, 224 92.5 / 85.8.  What bounds it then: at 128 rows the copies (L2 to LDS 8 TB/s of weights and activations, the arithmetic costs 1 us of
// 67), at 224 both sides cost 1.2 .. 1.3 us a block of 1.4 by themselves (1.3 without LDS reads, 1.2 without copies).
// Not used elsewhere: with both dimensions in whole rounds of 256 x 256 tiles the two-phase kernel is up to 25 % faster.
#include <cstdlib>
#include <type_traits>
#include "common.hpp"

namespace dsv3 {
namespace mid {

constexpr int NW = 8;

__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }
__device__ __forceinline__ v8i join(v4i lo, v4i hi) {
    v8i r = { lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3] };
    return r;
}
typedef __attribute__((address_space(3))) void* lptr_t;

template <int MT, int WM, int SN, int S> struct Geo {
    static constexpr int WN = NW / WM, JM = (MT + WM - 1) / WM;         // JM: sub-tiles of a wavefront
    static constexpr int TM = 16 * MT, BN = 16 * SN * WN;
    static constexpr int LA = (2 * MT + NW - 1) / NW, LB = (2 * SN * WN + NW - 1) / NW;   // 1 KiB copies per wavefront and K block
    static constexpr int PER = LA + LB + 1;                             // ... and one of scales
    static constexpr int A_STAGE = TM * 128, B_STAGE = BN * 128, SCW = (TM + 63) / 64;
    // scales of four K blocks: 16 bytes per row in copies of 64 rows, then one of the weights' (from lane 0 on, the tile's 128-column
    // blocks); two buffers, and a KiB that takes the copies nobody reads
    static constexpr int SC_BUF = (SCW + 1) * 1024, LDS_B = S * A_STAGE, LDS_SC = LDS_B + S * B_STAGE, LDS_DUMP = LDS_SC + 2 * SC_BUF;
    static constexpr int LDS = LDS_DUMP + 1024;
    // S <= 4: a group's buffer is requested anew S blocks ahead, which is behind the last block of the group that it held
    static_assert(JM >= 2 && SCW < NW && S >= 2 && S <= 4 && (S - 1) * PER <= 63 && LDS <= 160 * 1024, "tile");
};

// K a multiple of 512, a_s and b_s 16-byte aligned, nkb (K blocks per slice, blockIdx.y) a multiple of four.
template <int MT, int WM, int SN, int S>
__global__ __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void fp8_gemm_mid_kernel(
        const uint8_t* __restrict__ a, const float* __restrict__ a_s, const uint8_t* __restrict__ b, const float* __restrict__ b_s,
        void* __restrict__ out, int out_dtype,      // F32 slabs [gridDim.y][M][N] when gridDim.y > 1, else c
        int M, int N, int K, int tiles_m, int tiles_n, int nkb) {
#ifdef __HIP_DEVICE_COMPILE__               // (the buffer builtins have no host form)
    using G = Geo<MT, WM, SN, S>;
    constexpr int JM = G::JM, LA = G::LA, LB = G::LB, WN = G::WN;
    constexpr bool ONE = 8 % SN == 0;           // a wavefront's columns lie in one 128-column block of weight scales
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (every other column group deals its sub-tiles from the other end: where some wavefronts have one more, they are not on one SIMD)
    const int fr = lane & 15, fq = lane >> 4, wn = wave / WM, wm = wn & 1 ? WM - 1 - wave % WM : wave % WM;

    // a contiguous run of tiles per XCD, the row tiles of a column tile next to each other
    int pid = blockIdx.x;
    {
        const int T = tiles_m * tiles_n, q = T / 8, r = T % 8, x = pid % 8;
        pid = x * q + (x < r ? x : r) + pid / 8;
    }
    const int tn = pid / tiles_m, tm = pid - tn * tiles_m;
    const int m0 = tm * G::TM, rows_here = min(G::TM, M - m0), n0 = tn * G::BN;
    const int KBT = K >> 7, kb0 = blockIdx.y * nkb, KB = min(nkb, KBT - kb0);

    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a, 0, (uint32_t)M * (uint32_t)K, 0x00027000),
                                 b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)b, 0, (uint32_t)N * (uint32_t)K, 0x00027000);
    // copy t of a block: unit u = rows 8 u .. 8 u + 7 of the tile's A or B; past the last one it is repeated
    uint32_t off[LA + LB];
    int dst[LA + LB];
#pragma unroll
    for (int t = 0; t < LA + LB; ++t) {
        const bool is_a = t < LA;
        const int u = min((is_a ? t : t - LA) * NW + wave, is_a ? 2 * MT - 1 : 2 * SN * WN - 1), row = u * 8 + (lane >> 3);
        const int r = is_a ? m0 + min(row, rows_here - 1) : min(n0 + row, N - 1);
        off[t] = (uint32_t)r * (uint32_t)K + (((lane & 7) ^ swz(row)) * 16);
        dst[t] = (is_a ? 0 : G::LDS_B) + u * 1024;
    }
    // scales: wavefronts 0 .. SCW - 1 the activations', SCW the weights', the others none
    const int nb0 = n0 >> 7, nb_last = (N - 1) >> 7;
    const bool sc_live = wave <= G::SCW;
    const uint32_t s_off = wave < G::SCW ? (uint32_t)(m0 + min(wave * 64 + lane, rows_here - 1)) * (uint32_t)KBT * 4u
                                         : (uint32_t)min(nb0 + (wave == G::SCW ? min(lane, 7) : 0), nb_last) * (uint32_t)KBT * 4u;
    const __amdgpu_buffer_rsrc_t s_rsrc = wave < G::SCW ? __builtin_amdgcn_make_buffer_rsrc((void*)a_s, 0, (uint32_t)M * (uint32_t)KBT * 4u, 0x00027000)
                                                        : __builtin_amdgcn_make_buffer_rsrc((void*)b_s, 0, (uint32_t)(nb_last + 1) * (uint32_t)KBT * 4u, 0x00027000);
    const uint32_t s_one = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_off);
    // copy t of K block kb_ (the last one again past the end) into stage st
    auto copy = [&](int t, int kb_, int st) {
        const int kb = kb0 + min(kb_, KB - 1);
        if (t < LA) __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lptr_t)(lds + dst[t] + st * G::A_STAGE), 16, off[t], kb * 128, 0, 0);
        else if (t < LA + LB) __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lptr_t)(lds + dst[t] + st * G::B_STAGE), 16, off[t], kb * 128, 0, 0);
        else {          // (past the end: the last group again, into the buffer not in use)
            const bool real = sc_live && (kb_ & 3) == 0;
            const int grp = min(kb_ >> 2, (KB - 1) >> 2);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, (lptr_t)(lds + (real ? G::LDS_SC + ((kb_ >> 2) & 1) * G::SC_BUF + wave * 1024 : G::LDS_DUMP)),
                                                     16, real ? s_off : s_one, real ? (kb0 + grp * 4) * 4 : 0, 0, 0);
        }
    };
    const int fx = swz(fr);
    const int c0 = fr * 128 + (((2 * fq) ^ fx) * 16), c1 = fr * 128 + (((2 * fq + 1) ^ fx) * 16);
    // sub-tile j of the wavefront: rows 16 (j WM + wm); one past the tile's last one is repeated and its results dropped
    auto a_sub = [&](int j) { return (j + 1) * WM <= MT ? j * WM + wm : min(j * WM + wm, MT - 1); };
    auto frag_a = [&](int j, int st) {
        const uint8_t* p = lds + st * G::A_STAGE + a_sub(j) * 2048;
        return join(*(const v4i*)(p + c0), *(const v4i*)(p + c1));
    };
    auto frag_b = [&](int s, int st) {
        const uint8_t* p = lds + G::LDS_B + st * G::B_STAGE + (wn * SN + s) * 2048;
        return join(*(const v4i*)(p + c0), *(const v4i*)(p + c1));
    };
    auto scale_a = [&](int j, int kb) { return *(const float*)(lds + G::LDS_SC + ((kb >> 2) & 1) * G::SC_BUF + (a_sub(j) * 16 + fr) * 16 + (kb & 3) * 4); };
    constexpr int NB = ONE ? 1 : SN;
    int bs_at[NB];
#pragma unroll
    for (int s = 0; s < NB; ++s) bs_at[s] = G::LDS_SC + G::SCW * 1024 + (min(n0 + (wn * SN + s) * 16, N - 1) / 128 - nb0) * 16;
    auto scale_b = [&](int s, int kb) { return *(const float*)(lds + bs_at[s] + ((kb >> 2) & 1) * G::SC_BUF + (kb & 3) * 4); };

    // JA: the wavefront's sub-tiles, JM or, where the rows end, JM - 1
    auto run = [&](auto ja_tag) {
    constexpr int JA = decltype(ja_tag)::value, Q = JA * SN, SYNC = JA - 2;
    // The copies into a freed stage are spread over the MFMAs from one barrier to the next, copy t beside MFMA t Q / PER behind the barrier: a
    // compute unit's load path takes 20 cycles a copy and the wavefront that issues one waits for it.  So the last copies of block S - 1
    // are requested in front of the first barrier.
    auto slot_of = [](int t) { return t * Q / G::PER; };
    constexpr int LATE = [] {
        int n = 0;
        for (int t = 0; t < G::PER; ++t) n += t * Q / G::PER < Q - SYNC * SN;
        return n;
    }();
#pragma unroll
    for (int p = 0; p < S; ++p)
#pragma unroll
        for (int t = 0; t < G::PER; ++t)
            if (p < S - 1 || t < LATE) copy(t, p, p);

    v4f acc[JA][SN];
#pragma unroll
    for (int j = 0; j < JA; ++j)
#pragma unroll
        for (int s = 0; s < SN; ++s) acc[j][s] = (v4f){0.f, 0.f, 0.f, 0.f};

    v8i bf[SN], af[2];
    float sa[JA], sa_next[JA], bs[NB], bs_next[NB];
    constexpr int FIRST = (S - 2) * G::PER + LATE;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (FIRST & 15) | ((FIRST >> 4) << 14));       // vmcnt: block 0 has landed
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int s = 0; s < NB; ++s) bs_next[s] = scale_b(s, 0);
#pragma unroll
    for (int s = 0; s < SN; ++s) bf[s] = frag_b(s, 0);
    af[0] = frag_a(0, 0); af[1] = frag_a(1, 0);
#pragma unroll
    for (int j = 0; j < JA; ++j) sa_next[j] = scale_a(j, 0);
    v4f pend[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};         // raw products of the last two MFMAs
    float pend_sc[2] = {0.f, 0.f};
    int st = 0;

    for (int kb = 0; kb < KB; ++kb) {
        const int st_next = st == S - 1 ? 0 : st + 1, st_prev = st == 0 ? S - 1 : st - 1;
        float prev_sc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) prev_sc[h] = pend_sc[h];
#pragma unroll
        for (int j = 0; j < JA; ++j) sa[j] = ONE ? sa_next[j] * bs_next[0] : sa_next[j];
#pragma unroll
        for (int s = 0; s < NB; ++s) bs[s] = bs_next[s];
        auto factor = [&](int q) { return ONE ? sa[q / SN] : sa[q / SN] * bs[q % NB]; };
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int j = q / SN, s = q % SN;
            if (q == SYNC * SN) {
                // this block's last operands are in registers; the next block has landed
                constexpr int LEFT = (S - 2) * G::PER;
                __builtin_amdgcn_s_waitcnt(0x0f70 | (LEFT & 15) | ((LEFT >> 4) << 14));
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int s2 = 0; s2 < NB; ++s2) bs_next[s2] = scale_b(s2, kb + 1);
#pragma unroll
                for (int j2 = 0; j2 < JA; ++j2) sa_next[j2] = scale_a(j2, kb + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            const v4f z = {0.f, 0.f, 0.f, 0.f};
            const v4f r = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[s], af[j & 1], z, 0, 0, 0, 0, 0, 0);
            const int p = q - 2;                // the MFMA before the last one
            const int pq = p >= 0 ? p : Q + p;
            const float f = p >= 0 ? factor(p) : prev_sc[p + 2];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[pq / SN][pq % SN][e] = __builtin_fmaf(pend[q & 1][e], f, acc[pq / SN][pq % SN][e]);
            pend[q & 1] = r;
            if (j == JA - 1) bf[s] = frag_b(s, st_next);
            if (s == SN - 1) af[j & 1] = j + 2 < JA ? frag_a(j + 2, st) : frag_a(j + 2 - JA, st_next);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
            __builtin_amdgcn_sched_barrier(0);
            // refill: behind the barrier of this block's stage, in front of it the rest of the stage of the block before
#pragma unroll
            for (int t = 0; t < G::PER; ++t)
                if (slot_of(t) == (q + Q - SYNC * SN) % Q) {
                    if (q >= SYNC * SN) copy(t, kb + S, st);
                    else copy(t, kb - 1 + S, st_prev);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        // (Q odd: the two results in flight change places)
        if (Q & 1) { const v4f x = pend[0]; pend[0] = pend[1]; pend[1] = x; }
        pend_sc[0] = factor(Q - 2); pend_sc[1] = factor(Q - 1);
        if (JA & 1) { const v8i x = af[0]; af[0] = af[1]; af[1] = x; }      // (and so do the two fragments read ahead)
        st = st_next;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v4f& x = acc[(Q - 2 + h) / SN][(Q - 2 + h) % SN];
            x[e] = __builtin_fmaf(pend[h][e], pend_sc[h], x[e]);
        }
    __builtin_amdgcn_s_waitcnt(0x0f70);         // the repeated requests of the last block still write LDS

    // lane holds c[m][n .. n + 3] for every (j, s)
    const size_t slab = (size_t)blockIdx.y * M * N;
#pragma unroll
    for (int j = 0; j < JA; ++j) {
        const int r = (j * WM + wm) * 16 + fr;
        if (r >= rows_here) continue;
        const int m = m0 + r;
#pragma unroll
        for (int s = 0; s < SN; ++s) {
            const int n = n0 + (wn * SN + s) * 16 + fq * 4;
            const size_t idx = slab + (size_t)m * N + n;
            if ((N & 3) == 0 && n + 3 < N) {
                if (out_dtype == DSV3_F32)       *(v4f*)((float*)out + idx) = acc[j][s];
                else if (out_dtype == DSV3_BF16) *(v2u*)((uint16_t*)out + idx) = v2u{ pack_bf16(acc[j][s][0], acc[j][s][1]), pack_bf16(acc[j][s][2], acc[j][s][3]) };
                else                             *(v2u*)((uint16_t*)out + idx) = v2u{ pack_f16(acc[j][s][0], acc[j][s][1]), pack_f16(acc[j][s][2], acc[j][s][3]) };
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e >= N) break;
                if (out_dtype == DSV3_F32)       ((float*)out)[idx + e] = acc[j][s][e];
                else if (out_dtype == DSV3_BF16) ((uint16_t*)out)[idx + e] = cvt_out<DSV3_BF16>(acc[j][s][e]);
                else                             ((uint16_t*)out)[idx + e] = cvt_out<DSV3_F16>(acc[j][s][e]);
            }
        }
    }
    };
    if constexpr (JM > 2) {
        if (((JM - 1) * WM + wm) * 16 < rows_here) run(std::integral_constant<int, JM>());
        else run(std::integral_constant<int, JM - 1>());
    } else run(std::integral_constant<int, JM>());
#endif
}

// Five windows in which the large-M kernel's tiles fit the chip badly.  Power-of-two scales take the same kernel (accumulating in the
// matrix core was equal to 4 % faster here).
struct Plan { int mt, wm, sn, splits, nkb; bool tall; };       // mt == 0: not for this kernel; tall: more than 256 rows of narrow weights
// The variables that pin how the large-M kernel runs its dense tiles (one K slice, a tile height, a schedule) pin that kernel too.
inline bool large_m_pinned() {
    static const bool v = [] {
        for (const char* name : { "DSV3_PREFILL_TILE", "DSV3_PREFILL_NOSPLIT", "DSV3_PREFILL_NOPP", "DSV3_PREFILL_NOPP128" })
            if (std::getenv(name)) return true;
        return false;
    }();
    return v;
}
inline Plan make_plan(int64_t m, int64_t n, int64_t k) {
    Plan p{};
    const int64_t kb = k / 128;
    if (m <= 32 || k % 512 || m * k >= (1ll << 32) || n * k >= (1ll << 32) || large_m_pinned()) return p;
    p.splits = 1;
    p.nkb = (int)kb;
    // Weights of 96 MiB and more, of more columns than 128 of the large-M kernel's tiles and at most 256 tiles of 160: one round here, with
    // one row tile.  65 .. 224 rows of 7168 -> 36864 (231 tiles).  Measured with the quantisation in front over 32769 .. 40960 columns and K
    // of 2560 .. 16384, (large-M kernel's time) / (time here): 1.05 .. 1.30 up to 192 rows, 1.02 .. 1.23 at 193 and 224.  What is left out:
    // 32768 columns and fewer, where 128-row tiles of the large-M kernel, two a column tile or in two K slices, are one full round
    // (7168 -> 31744 at 65 / 160 / 193 rows 0.93 / 0.88 / 0.84); K of 32768 (0.81 .. 1.50, 0.92 .. 0.96 at 193 rows); from 193 rows on,
    // whose ring has three stages, fewer than 212 tiles or 32 K blocks (16384 -> 32769 0.94, 2560 -> 40960 0.98); 225 rows and more, whose
    // ring would have two.  33 .. 64 rows of such weights are the large-M kernel's otherwise, too (fp8_gemm_tile.hip): 7168 -> 36864 at 33 / 64 rows, the product alone, 61.2 /
    // 66.7 us there, 53.5 / 56.9 here, over 32769 .. 40960 columns and K of 2560 .. 16384 1.05 .. 1.21.  Nor two row tiles of 116 for 7168 -> 18432 (129 .. 224 rows, 48.4 us there, 53.5 here at 193): that one 128- or
    // 256-row tile of the large-M kernel reads the weights once.
    const int64_t t160 = (n + 159) / 160, rows = (m + 15) / 16;
    if (n * k >= (96ll << 20) && n > 32768 && t160 <= 256 && kb <= 128 && rows <= (t160 < 212 || kb < 32 ? 12 : 14)) {
        p.wm = 4; p.sn = 5;
        p.mt = rows <= 6 ? 6 : rows <= 8 ? 8 : rows <= 10 ? 10 : rows <= 12 ? 12 : 14;
        return p;
    }
    // Up to 128 rows of a weight of 176 to 256 tiles of 128 columns, in one round where 256 columns make half a round: over 22401 .. 32768
    // columns and K of 1536 .. 16384, measured as above, 0.98 .. 1.77, 1536 -> 24576 1.23 .. 1.14.  Not below 12 K blocks (512 -> 32768: equal to
    // 12 % more time), nor above 128 (32768 -> 28672 at 128 rows 0.98).  33 .. 64 rows on 28 to 80 K blocks: 1.00 .. 1.17 over 23 sizes, 1.07 on average;
    // on fewer 0.99 .. 1.01 (2560 -> 24704 at 48 rows 20.0 / 20.0 us), on more 0.87 .. 1.03 (12288 -> 23424 at 35 rows 73.4 / 84.0 us: two K slices of as many tiles
    // of the large-M kernel fill the chip as well, and their slabs cost little beside that many blocks).
    const int64_t t128 = (n + 127) / 128;
    if (m <= 128 && t128 >= 176 && t128 <= 256 && (m <= 64 ? kb >= 28 && kb <= 80 : kb >= 12 && kb <= 128)) {
        p.mt = 8; p.wm = 4; p.sn = 4;
        return p;
    }
    // 129 .. 256 rows of 32 to 128 tiles of 128 columns, in as many K slices as one round takes, where slices and columns fill it (240 of 256 units, 220 with
    // slices of 24 blocks): the large-M kernel's tile has 128 or 256 rows and two stages, one of these as many rows as there are and three.  Up to
    // 160 rows, and above on slices of 32 blocks and more (three or four, nearly equal) of a K range up to 18432: 16384 -> 7168 at 129 / 193 / 224 / 256 rows 1.15 / 1.04 / 1.08 / 1.10,
    // 18432 -> 7168 1.05 / 1.02 / 1.04 / 1.04, 16384 -> 8192 1.06 .. 1.11, 7168 -> 16384 at 129 / 160 1.15 / 1.06 times the speed with the quantisation in front;
    // over 125 drawn and listed sizes 0.98 .. 1.48, 1.05 on average (power-of-two scales 1.04).  Left out: 7168 -> 12288 (192 units) 0.92 .. 1.01 at 16384, 20480 -> 9216
    // 0.91, 11264 -> 7168 at 193 rows 0.96 (slices of 24), 7168 -> 7168 at 159 0.96 (of 16), and slices of eight blocks with a shorter last one, which are a slab more
    // than the large-M kernel's for nothing (1536 -> 15488 at 139 rows, one slice there, 19.1 us, two here 24.7; 3584 -> 8064 at 159 25.3 / 26.0, 5632 -> 5376 at 159
    // equal; 2048 -> 16000 at 147, two even ones, 29.0 / 25.5).
    if (m > 128 && m <= 256 && t128 >= 32 && t128 <= 128 && kb <= 144) {
        const int64_t sl = 256 / t128, nkb = ((kb + sl - 1) / sl + 3) / 4 * 4, splits = (kb + nkb - 1) / nkb, units = t128 * splits;
        if ((nkb > 8 || (nkb == 8 && kb % 8 == 0)) && (units >= 240 || (units >= 220 && nkb >= 24)) && (m <= 160 || (nkb >= 32 && splits >= 3 && nkb * splits - kb <= 8))) {
            p.nkb = (int)nkb;
            p.splits = (int)splits;
            p.wm = 4; p.sn = 4;
            p.mt = rows <= 10 ? 10 : rows <= 12 ? 12 : rows <= 14 ? 14 : 16;
            return p;
        }
    }
    // Narrow weights on a long K range: tiles of 64 x 128 as far as they are one round, in as many K slices as that leaves room for (up to
    // seven), while a slice is at most 20 blocks: a tile here takes 0.6 times the time per block that one of the large-M kernel's with four
    // times the columns does, which pays only as long as the round is short.  Behind the quantisation (us, large-M kernel / here), slices of
    // 8 .. 20 blocks: 7168 -> 1536 at 128 / 256 / 448 rows 19.8 / 23.0 / 23.7 -> 16.3 / 18.9 / 22.7, 7168 -> 576 at 256 / 1024 19.5 / 25.0 ->
    // 16.3 / 23.8, 7168 -> 2112 at 128 / 320 20.3 / 22.7 -> 17.2 / 21.6, 4096 -> 1024 at 900 25.5 -> 20.8; of 28: 7168 -> 1536 at 449 24.0 ->
    // 24.8, 7168 -> 2112 at 321 22.9 -> 24.0; of 44: 16384 -> 2304 at 300 30.8 -> 38.0; of 56: 7168 -> 1536 at 777 29.3 -> 33.7.
    // Over 1 .. 2304 columns and K of 4096 .. 16384, 65 rows up to the last one taken (1 .. 128 columns: 8192 at K of 4096, 5440 at 7168;
    // 300: 2688; 576: 1600), measured as above: 0.99 .. 1.51, at the last ones 1.01 .. 1.28.
    const int64_t tiles = (m + 63) / 64 * t128;
    if (m > 64 && n <= 2304 && kb >= 32 && tiles <= 256) {
        int64_t s = 256 / tiles;
        s = s > 7 ? 7 : s;
        int64_t nkb = ((kb + s - 1) / s + 3) / 4 * 4;
        nkb = nkb < 8 ? 8 : nkb;
        if (nkb <= 20) {
            p.nkb = (int)nkb;
            p.splits = (int)((kb + nkb - 1) / nkb);
            p.mt = 4; p.wm = 2; p.sn = 2;
            return p;
        }
    }
    // More rows of them: tiles of 128 rows (112 where that pads less) x 128 columns in one round, without slices or in three and more: the large-M kernel has
    // 256-column tiles in up to eight slices, twice the slabs and more, or fewer tiles than units.  Behind the quantisation (us, large-M kernel / here): 7168 -> 1536 at
    // 512 / 640 / 896 rows 27.3 / 29.0 / 33.0 -> 25.5 / 28.0 / 31.8, at 777 30.7 .. 35.4 from process to process -> 31.2 .. 31.7, 7168 -> 2112 at 350 / 640 / 1800 26.1 / 32.7 / 57.8
    // -> 24.8 / 30.6 / 52.0; power-of-two scales alike.  Over 81 drawn and listed sizes of 256 .. 2304 columns and K of 4096 .. 16384 0.98 .. 1.36, 1.07 on average.
    // A slice of at most 24 blocks: with 28 and more the large-M kernel's twice as many slices were up to 7 % faster on one card and up to 5 % slower on another (9728 -> 1408 at
    // 817 rows 34.3 .. 39.6 / 37.0 .. 37.6), 16384 -> 1408 at 398 33.0 / 34.8 on both.  Without slices up to 56 blocks in tiles of 128 rows that fill 216 units: 7168 -> 1536 at 1800 rows
    // (204) 48.4 / 50.5, at 2400 (228) 56.5 / 54.7, 11776 -> 1792 at 1948 (tiles of 112) 72.8 / 80.5, 16384 -> 1024 at 2886 97.3 / 111.5, 8192 -> 2304 at 1600 56.0 / 57.0.
    // Both lines only where columns are whole fours: the large-M kernel sums other slabs value by value (4096 -> 1453 at 1844 rows 50.1 / 36.9, 13312 -> 2187 at 423
    // 53.5 / 48.5).  Left out, too: two slices (7168 -> 1536 at 930 / 1280 rows 0.94 / 0.97, 8192 -> 381 at 4757 0.94; 16384 -> 1707 at 1060 would be 1.16) and rounds
    // with more units idle (7168 -> 2112 at 400, 204 of 256: 0.96), and up to 640 columns on a K range up to 8192 (7168 -> 576 at 1700 .. 2048 0.99 .. 1.06, with
    // power-of-two scales 0.94 .. 1.00).
    if (m > 256 && n <= 2304 && kb >= 32 && (t128 >= 6 || kb > 64)) {
        for (int mt : {8, 7}) {
            const int64_t tm = (m + 16 * mt - 1) / (16 * mt), s = 256 / (tm * t128 > 0 ? tm * t128 : 1);
            if (s < 1 || (mt == 7 && tm * 112 >= (m + 127) / 128 * 128)) continue;
            int64_t nkb = ((kb + s - 1) / s + 3) / 4 * 4;
            nkb = nkb < 8 ? 8 : nkb;
            const int64_t splits = (kb + nkb - 1) / nkb;
            const bool whole = n % 4 == 0;
            if (splits == 2 || tm * t128 * splits < (splits == 1 && !whole ? 200 : 216) || (p.mt && nkb > p.nkb)) continue;
            if (whole && (splits > 1 ? nkb > 24 : mt == 7 || kb > 56)) continue;
            p.mt = mt; p.wm = 4; p.sn = 4;
            p.nkb = (int)nkb; p.splits = (int)splits; p.tall = true;
        }
    }
    return p;
}

template <int MT, int WM, int SN, int S>
int launch_cfg(const Plan& p, const void* a, const float* a_s, const void* b, const float* b_s, void* out, int od, int m, int n, int k, hipStream_t st) {
    using G = Geo<MT, WM, SN, S>;
    void (*const kern)(const uint8_t*, const float*, const uint8_t*, const float*, void*, int, int, int, int, int, int, int) = fp8_gemm_mid_kernel<MT, WM, SN, S>;
    static LdsGrant grant;
    if (!grant.ensure((const void*)kern, G::LDS)) return DSV3_ERR_LAUNCH;
    const int tm = (m + G::TM - 1) / G::TM, tn = (n + G::BN - 1) / G::BN;
    hipLaunchKernelGGL(kern, dim3((unsigned)(tm * tn), (unsigned)p.splits), dim3(NW * kWave), G::LDS, st, (const uint8_t*)a, a_s,
                       (const uint8_t*)b, b_s, out, od, m, n, k, tm, tn, p.nkb);
    return launch_status();
}

}  // namespace mid

bool mid_supported(int64_t m, int64_t n, int64_t k) {
    const mid::Plan p = mid::make_plan(m, n, k);
    return m > 64 && p.mt != 0 && !p.tall;
}
bool mid_takes(int64_t m, int64_t n, int64_t k) { return mid::make_plan(m, n, k).mt != 0; }

size_t mid_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    const mid::Plan p = mid::make_plan(m, n, k);
    return p.mt != 0 && p.splits > 1 ? (size_t)p.splits * (size_t)m * (size_t)n * sizeof(float) : 0;
}

// As launch_stream.  The scale rows are copied in 16-byte pieces: a_s and b_s that are not 16-byte aligned are for another kernel.
bool mid_takes_scales(const float* a_s, const float* b_s) { return (((uintptr_t)a_s | (uintptr_t)b_s) & 15) == 0; }

int launch_mid(const void* a, const float* a_s, const void* b, const float* b_s, void* c, int c_dtype, int64_t m, int64_t n, int64_t k,
               void* ws, int* splits_out, hipStream_t st) {
    using namespace mid;
    const Plan p = make_plan(m, n, k);
    if (p.mt == 0) return DSV3_ERR_BAD_SHAPE;
    if (p.splits > 1 && !ws) return DSV3_ERR_WORKSPACE;
    void* out = p.splits > 1 ? ws : c;
    const int od = p.splits > 1 ? (int)DSV3_F32 : c_dtype;
    *splits_out = p.splits;
    switch (p.mt * 10 + p.sn) {
        case 65:  return launch_cfg<6, 4, 5, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 85:  return launch_cfg<8, 4, 5, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 105: return launch_cfg<10, 4, 5, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 125: return launch_cfg<12, 4, 5, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 145: return launch_cfg<14, 4, 5, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 84:  return launch_cfg<8, 4, 4, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 74:  return launch_cfg<7, 4, 4, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 104: return launch_cfg<10, 4, 4, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 124: return launch_cfg<12, 4, 4, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 144: return launch_cfg<14, 4, 4, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 164: return launch_cfg<16, 4, 4, 3>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        case 42:  return launch_cfg<4, 2, 2, 4>(p, a, a_s, b, b_s, out, od, (int)m, (int)n, (int)k, st);
        default: return DSV3_ERR_BAD_SHAPE;
    }
}

}  // namespace dsv3
