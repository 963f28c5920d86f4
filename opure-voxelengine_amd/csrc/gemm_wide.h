// ============================================================================
//  gemm_wide.h -- the GEMV for more than 16 activation rows (a batch of
//  sequences times K+1 rows, up to 256, or a prompt's, up to 2,048): a thin
//  GEMM on the matrix cores.
//
//  The same tiled weights and the same MFMA operand mapping as the K+1-row
//  kernel (gemv_kernel.h): y^T = W X^T in 16 x 16 tiles, A = 16 weight rows
//  x 32 k, B = 32 k x 16 columns of X.
//
//  Work split.  A workgroup owns 8 consecutive 16-row weight tiles (a row
//  group), up to 8 16-column tiles of X (a column group) and one range of K
//  blocks (a split; shapes with few row groups split K so the CUs fill).  A
//  set of 4 waves covers the row group (more than 64 rows of X): wave w multiplies
//  tiles 2w, 2w + 1 by all of the group's column tiles, so it keeps 16 accumulator
//  tiles, loads each weight byte once and reads each B fragment once per block for
//  two MFMAs.  Fewer rows take one weight tile a wave, an int8 prompt's of more
//  than 256 rows four on a 2 x 2 wave grid (WideShape).  Weights go straight from
//  HBM into registers: every wave loads its own tiles' 16 bytes a lane per block,
//  in static register slots DW steps ahead.  X goes through LDS: per block the
//  set loads its column group's fragments into registers DX steps ahead and
//  writes them into a two-stage ring laid out fragment by fragment, 16 bytes a
//  lane.  One barrier per step (one block, or two at one weight tile a wave)
//  separates a stage's writes from its reads and the reads of two steps back
//  from the next writes.  Up to 256 rows the int8 kernel runs two such sets on
//  alternate K blocks (KH = 2, two waves a SIMD) and adds them at the end.
//
//  The budget per block of a workgroup is L2 -> CU traffic (8 KB of weights
//  and 16 KB of X at 128 columns), which is why a wave owns whole weight
//  tiles (no two waves load the same weights) and X loads cover whole
//  128-byte lines.
//
//  With one split the epilogue runs here; with several, each split writes
//  its raw accumulators and k_wide_reduce adds the splits in split order and
//  runs the epilogue (k_wide_reduce_norm for a residual that feeds an
//  rmsnorm: it also writes the normalised rows).  Each (row, column) sums its
//  blocks in a fixed order, so runs are reproducible.  For 17 to 256 rows the
//  split count depends on the weight shape only and every kernel shape has the
//  same order (each wave set's blocks in order, then the sets added), so a row's
//  result does not depend on how many rows share the call.  A prompt's step of
//  more rows takes its splits from the row count and, in int8, adds all blocks of
//  a split in one chain: a row's last bits then depend on the step's rows.
// ============================================================================
#pragma once

#include "gemv_kernel.h"

namespace opure_gemv {

constexpr uint32_t WIDE_RT = 8;       // weight tiles of the plan's row groups (the K splits follow from these)
constexpr uint32_t WIDE_CG = 8;       // column tiles per workgroup at most

// The wave grid: a set of 4 waves is 4 / WC wave rows x WC wave columns, each
// wave TA weight tiles x TB column tiles.  CT = WC * TB column tiles a
// workgroup; RT = (4 / WC) * TA weight tiles.
//   CT 8: the general shape (128 x 128 outputs a workgroup)
//   CT 4, 2: a batch of at most 64 / 32 rows, which is bound by the weight
//     stream: no matrix work on column tiles that are not there, and at one
//     tile a wave twice the workgroups (8B o_proj, 4 splits: 128 -> 256), so
//     every CU loads: uint4 gate/up 28,672 x 4,096 at 24 rows 77.5 -> 26.3 us.
// KH = 2 runs two sets of 4 waves on alternate K blocks (two waves a SIMD: one
// issues MFMAs while the other waits); the uint4 kernel's registers leave room
// for one.
template <uint32_t TA_, uint32_t TB_, uint32_t WC_, uint32_t KH_> struct WideShape {
    static constexpr uint32_t TA = TA_, TB = TB_, WC = WC_, KH = KH_, RT = (4u / WC_) * TA_, CT = WC_ * TB_, NTH = 256u * KH_;
};

// The software pipeline goes SB blocks a step (one barrier and one LDS stage a
// step), DW steps of weights and DX of X in flight in registers; the K loop is
// unrolled by U steps so slots and stages are compile-time.  At one weight
// tile a wave a block is 8 or 16 MFMAs behind a barrier, an LDS round trip and
// the X staging, so two blocks share those; X two steps ahead because loads
// return in order and a wait for X waits for the weights issued before it (8B layer,
// 24 rows: 131.3 -> 128.5 us).  Eight blocks of weights and four of X in flight
// were slower (139 us, the loop unrolled eight times), two weight tiles a wave
// too (1B gate/up at 24 rows 8.8 -> 10.2 us).
template <int WF, class SH> struct WideDepth {
    static constexpr bool FEW = SH::TA == 1u, I8 = WF == OPURE_W_I8PC;
    static constexpr uint32_t SB = FEW ? 2 : 1, DW = !FEW && I8 && SH::KH == 2u ? 4 : 2,
                              DX = I8 || SH::CT < 8u ? 2 : 1, U = DW > DX ? DW : DX;
};
// the plan's splits are multiples of this many blocks
constexpr uint32_t wide_split_unit(uint32_t wf) { return wf == OPURE_W_I8PC ? 4u : 2u; }

struct WParams {
    KParams p;        // shape, pointers, epilogue
    uint32_t mt;      // 16-column tiles of X
    uint32_t nrg;     // row groups (the kernel shape's RT tiles each)
    uint32_t ncg;     // column groups
    uint32_t cgs;     // column tiles per group (<= WIDE_CG)
    uint32_t splits;  // K splits
    uint32_t bps;     // blocks per split
    uint32_t part_rows;  // splits > 1: 0 = accumulators [split][tile][mt][64] lanes, 1 = [split][M][out] rows
    f4_t* part;       // splits > 1: the splits' accumulators
    uint32_t prompt;  // host: more than OPURE_MAX_BATCH_ROWS rows (a prompt's step)
};

// Workgroup -> (split, row group, column group).  Workgroups are dispatched
// to the 8 XCDs round robin; the remap gives each XCD a contiguous range of
// the work list, so the column groups of one row group (the same weights)
// run on one XCD and share its L2.
__device__ __forceinline__ void wide_coords(const WParams& wp, uint32_t& split, uint32_t& rg, uint32_t& cg)
{
    const uint32_t G = gridDim.x, i = blockIdx.x;
    const uint32_t xcd = i & 7u, j = i >> 3, q = G >> 3, r = G & 7u;
    const uint32_t L = xcd < r ? xcd * (q + 1u) + j : r * (q + 1u) + (xcd - r) * q + j;
    cg = L % wp.ncg;
    const uint32_t rest = L / wp.ncg;
    rg = rest % wp.nrg;
    split = rest / wp.nrg;
}

template <int WF, int AF, int EPI, class SH>
__global__ __launch_bounds__(SH::NTH) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_wide(WParams wp)
{
    static_assert(WF == OPURE_W_I8PC || WF == OPURE_W_I4G128, "the wide GEMV reads quantised weights");
    constexpr uint32_t KB = Fmt<WF>::KB;
    constexpr uint32_t NMF = KB / 32u;             // MFMAs (16-byte B fragments) per block per tile pair
    constexpr uint32_t CH = KB / 8u;               // 16-byte X chunks per row per block
    constexpr uint32_t TA = SH::TA, TB = SH::TB, WC = SH::WC, RT = SH::RT, CT = SH::CT;
    constexpr uint32_t XR = CT * 16u * CH / 256u;  // X chunks a thread stages per block
    constexpr uint32_t STAGE = CT * NMF * 64u;     // u4_t per LDS stage
    using WD = WideDepth<WF, SH>;
    constexpr uint32_t SB = WD::SB, DW = WD::DW, DX = WD::DX, U = WD::U, KH = SH::KH;
    static_assert(U % 2 == 0 && U % DX == 0 && U % DW == 0, "static slots and stages");
    constexpr bool GS = WF == OPURE_W_I4G128;      // group sums of X
    static_assert(XR >= 1 && TB % 2 == 0, "whole chunks a thread; the halves exchange half of the tiles");
    static_assert(KH == 1 || 4u * TA * TB * 64u <= KH * 2u * STAGE, "the halves' exchange reuses the X stages");
    static_assert(!GS || CH == 16u, "a DPP row of lanes stages one X row's group");
    __shared__ u4_t xl[KH * 2 * SB * STAGE];
    __shared__ float xsl[GS ? 2 * SB : 1][GS ? CT * 16u : 1u];   // uint4: each block's group sums of X
    const KParams& p = wp.p;
    const uint32_t tid = threadIdx.x & 255u, lane = tid & 63u, g4 = lane >> 4, r16 = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t kh = wave >> 2, w4 = wave & 3u;            // K half, wave within the half
    const uint32_t wr = w4 / WC, wc = w4 % WC;
    const uint32_t nblk = p.nblk, G = p.in / 128u;
    uint32_t split, rg, cg;
    wide_coords(wp, split, rg, cg);
    const uint32_t ct0 = cg * wp.cgs;
    const uint32_t cn = min(wp.cgs, wp.mt - ct0);            // column tiles of this group; of this wave: TB wc + j
    const uint32_t tile0 = rg * RT + wr * TA;
    const uint32_t b_begin = split * wp.bps, b_end = min(nblk, b_begin + wp.bps);
    u4_t* xh = xl + kh * 2u * SB * STAGE;                     // this half's two stages of SB blocks

    // X chunk u of this thread: row rr of local column tile ctl, 16-byte chunk c of the block (a
    // wave's load covers 8 rows x 128 contiguous bytes).  In LDS, chunk c of row rr sits at row
    // slot rr ^ c of its fragment: the 8 chunks of a row land in 8 bank groups, and a fragment
    // read (lane (g4, r16) takes chunk NMF g4 + q of row r16) still reads 16 distinct slots.
    // Rows past M (or past the group's column tiles) read row M - 1 again: their columns are
    // computed and never stored.  Two wave sets of two weight tiles (int8 past 64 rows) put
    // zeros in their place: products of zeros run faster than the row's again (LM head 128,256
    // x 2,048 at 65 rows 84.9 -> 81.6 us, gate/up 16,384 x 2,048 at 144 21.2 -> 20.9; with no
    // row past M the selects cost up to 1%).  The other shapes lose more by the selects (int8
    // gate/up at 48 rows 10.1 -> 10.8, uint4 down 4,096 x 14,336 at 128 54.1 -> 56.5).
    constexpr bool XZ = KH == 2u && TA == 2u;
    uint64_t xrow[XR];
    uint32_t xdst[XR];
    bool xzero[XR];
#pragma unroll
    for (uint32_t u = 0; u < XR; ++u)
    {
        const uint32_t e = u * 256u + tid;
        const uint32_t c = e % CH, rr = (e / CH) & 15u, ctl = e / (16u * CH);
        const uint32_t m = 16u * (ct0 + ctl) + rr;
        xzero[u] = XZ && (ctl >= cn || m >= p.M);
        xrow[u] = (static_cast<uint64_t>(min(m, p.M - 1u)) * p.in + 8u * c) * 2u;
        xdst[u] = (ctl * NMF + c % NMF) * 64u + (c / NMF) * 16u + (rr ^ (c & 15u));
    }
    auto xload = [&](u4_t (&v)[XR], uint32_t b) {
        const uint64_t k0 = static_cast<uint64_t>(min(b, nblk - 1u)) * KB * 2u;
#pragma unroll
        for (uint32_t u = 0; u < XR; ++u) v[u] = *reinterpret_cast<const u4_t*>(p.x + xrow[u] + k0);
    };
    // uint4: the group's sum of X of a row, once a workgroup here instead of
    // in every wave beside its MFMAs (it was 38% of the loop's vector
    // instructions, which bound the loop; uint4 gate/up 28,672 x 4,096 at 256
    // rows 165 -> 95 us with the fresh group accumulators kept to one column
    // tile and out of the accumulation registers).  The 16 lanes of a DPP row stage one row: chunk c = 4 g +
    // q is MFMA q's share of lane group g; the sums over q in order, then
    // (g0 + g1) + (g2 + g3).
    auto xstore = [&](const u4_t (&v)[XR], uint32_t st) {
        float t[XR];
#pragma unroll
        for (uint32_t u = 0; u < XR; ++u)
        {
            xh[st * STAGE + xdst[u]] = xzero[u] ? u4_t{0u, 0u, 0u, 0u} : v[u];
            if constexpr (GS)
            {
                const float s = unit_sum<AF>(v[u][0], v[u][1], v[u][2], v[u][3]);
                t[u] = dpp_f<0x00>(s) + dpp_f<0x55>(s);
                t[u] += dpp_f<0xAA>(s);
                t[u] += dpp_f<0xFF>(s);
                t[u] += dpp_f<0x141>(t[u]);   // row_half_mirror: g ^ 1
                t[u] += dpp_f<0x140>(t[u]);   // row_mirror: the other pair
            }
        }
        if constexpr (GS)
        {
            if ((tid & 15u) == 0u)
#pragma unroll
                for (uint32_t u = 0; u < XR; ++u) xsl[st][u * 16u + (tid >> 4)] = t[u];
        }
    };

    // this wave's weight tiles (clamped for loads; the epilogue skips tiles past the end)
    const uint8_t* wbase[TA];
    const uint32_t* sbase[TA];
#pragma unroll
    for (uint32_t a = 0; a < TA; ++a)
    {
        const uint32_t lt = min(tile0 + a, p.tiles - 1u);
        wbase[a] = p.w + (static_cast<uint64_t>(lt) * nblk << 10) + (lane << 4);
        sbase[a] = static_cast<const uint32_t*>(p.sc) + static_cast<uint64_t>(lt) * G * 16u + 4u * g4;
    }
    auto wload = [&](u4_t (&w)[TA], u4_t (&s)[TA], uint32_t b) {
        const uint32_t bc = min(b, nblk - 1u);
#pragma unroll
        for (uint32_t a = 0; a < TA; ++a)
        {
            w[a] = *reinterpret_cast<const u4_t*>(wbase[a] + (static_cast<uint64_t>(bc) << 10));
            if constexpr (WF == OPURE_W_I4G128) s[a] = *reinterpret_cast<const u4_t*>(sbase[a] + bc * 16u);
        }
    };

    f4_t acc[TA][TB];
#pragma unroll
    for (uint32_t a = 0; a < TA; ++a)
#pragma unroll
        for (uint32_t j = 0; j < TB; ++j) acc[a][j] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    auto mma = [&](const u4_t& a, const u4_t& b, const f4_t& c) -> f4_t {
        if constexpr (AF == OPURE_A_F16)
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    };
    // one block: B fragments from LDS stage st, A decoded from the weight
    // registers.  Every wave runs all TB column slots (a slot past the group
    // is never stored): no branches between MFMAs.
    auto compute = [&](const u4_t (&w)[TA], const u4_t (&s)[TA], uint32_t st) {
        const u4_t* xb = xh + st * STAGE;
        auto frag = [&](uint32_t j, uint32_t q) {
            return xb[((TB * wc + j) * NMF + q) * 64u + g4 * 16u + (r16 ^ ((NMF * g4 + q) & 15u))];
        };
        if constexpr (!GS)
        {
#pragma unroll
            for (uint32_t q = 0; q < NMF; ++q)
            {
                u4_t bf[TB];
#pragma unroll
                for (uint32_t j = 0; j < TB; ++j) bf[j] = frag(j, q);
#pragma unroll
                for (uint32_t a = 0; a < TA; ++a)
                {
                    uint32_t o[4];
                    u8x4_to_f16(w[a][2u * q], o[0], o[1]);
                    u8x4_to_f16(w[a][2u * q + 1u], o[2], o[3]);
                    const u4_t af = {o[0], o[1], o[2], o[3]};
#pragma unroll
                    for (uint32_t j = 0; j < TB; ++j) acc[a][j] = mma(af, bf[j], acc[a][j]);
                }
            }
        }
        else
        {
            // a column tile at a time, so that the fresh group accumulators
            // take 4 TA registers instead of 4 TA TB
            u4_t af[TA][NMF];
            f4_t sc[TA], zo[TA];
#pragma unroll
            for (uint32_t a = 0; a < TA; ++a)
            {
#pragma unroll
                for (uint32_t q = 0; q < NMF; ++q)
                {
                    uint32_t o[4];
                    u4x8_pairs<AF>(w[a][q], o);
                    af[a][q] = u4_t{o[0], o[1], o[2], o[3]};
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    float c, z;
                    u4_group<AF>(s[a][i], c, z);
                    sc[a][i] = c;
                    zo[a][i] = z;
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < TB; ++j)
            {
                u4_t bf[NMF];
#pragma unroll
                for (uint32_t q = 0; q < NMF; ++q) bf[q] = frag(j, q);
                const float xs = xsl[st][16u * (TB * wc + j) + r16];
                f4_t bacc[TA];
#pragma unroll
                for (uint32_t a = 0; a < TA; ++a) bacc[a] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (uint32_t q = 0; q < NMF; ++q)
#pragma unroll
                    for (uint32_t a = 0; a < TA; ++a) bacc[a] = mma(af[a][q], bf[q], bacc[a]);
                // acc += (s / MUL) * (bacc - (OFF + MUL z) * xs), xs = the block's sum of X for this column (see U4)
#pragma unroll
                for (uint32_t a = 0; a < TA; ++a)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[a][j][i] = __fmaf_rn(sc[a][i], __fmaf_rn(-zo[a][i], xs, bacc[a][i]), acc[a][j][i]);
            }
        }
    };

    // the two halves share the epilogue by weight tiles where a wave has two, so
    // that a column group of 5 tiles is shared evenly too (by column tiles, 4 and
    // 1, int8 gate/up 16,384 x 2,048 at 80 rows takes 21.3 us instead of 20.1, at
    // 144 22.4 instead of 20.9), else by column tiles
    constexpr bool BYT = KH == 2u && TA % 2u == 0u;
    constexpr uint32_t FT = BYT ? TA / 2u : TA, FB = KH == 2u && !BYT ? TB / 2u : TB;   // tiles a wave finishes
    const uint32_t a0 = BYT ? kh * FT : 0u, j0 = KH == 2u && !BYT ? kh * FB : 0u;
    // int8 with one split: the row scales of the tiles this wave finishes, loaded
    // now rather than after the K loop (a round trip off the epilogue)
    f4_t scl[FT];
    if constexpr (WF == OPURE_W_I8PC)
    {
#pragma unroll
        for (uint32_t a = 0; a < FT; ++a)
        {
            const uint32_t t = min(tile0 + a0 + a, p.tiles - 1u);
#pragma unroll
            for (int i = 0; i < 4; ++i) scl[a][i] = f16_to_f32(static_cast<const uint16_t*>(p.sc)[t * 16u + 4u * g4 + i]);
        }
    }

    // Half kh takes blocks b_begin + kh, + kh + KH, ...; a step moves both
    // halves SB blocks on, with one barrier for the whole workgroup.
    const uint32_t steps = (b_end - b_begin + KH * SB - 1u) / (KH * SB);
    const uint32_t bh = b_begin + kh;
    u4_t xr[DX * SB][XR];
    u4_t wv[DW * SB][TA], sv[DW * SB][TA];
    // slot SB d + k: block k of the d-th step ahead, bh + KH (SB d + k)
#pragma unroll
    for (uint32_t d = 0; d < DX * SB; ++d) xload(xr[d], bh + KH * d);
#pragma unroll
    for (uint32_t d = 0; d < DW * SB; ++d) wload(wv[d], sv[d], bh + KH * d);
    for (uint32_t i0 = 0; i0 < steps; i0 += U)
    {
#pragma unroll
        for (uint32_t s = 0; s < U; ++s)
        {
            const uint32_t b = bh + KH * SB * (i0 + s), st = (s & 1u) * SB, xs = s % DX * SB, ws = s % DW * SB;
            if constexpr (SB == 1u && TA == 2u)
            {
                // the loops below over one block, written out: the compiler
                // schedules it better (int8 gate/up 28,672 x 4,096 at 256 rows
                // 69.5 -> 68.0 us; uint4 at 256 87.5 -> 86.2, LM head 317 -> 310;
                // a prompt's shapes of four weight tiles lose up to 1% by it)
                xstore(xr[xs], st);
                xload(xr[xs], b + KH * DX);
                __syncthreads();
                if (b < b_end) compute(wv[ws], sv[ws], st);
                wload(wv[ws], sv[ws], b + KH * DW);
            }
            else
            {
#pragma unroll
                for (uint32_t k = 0; k < SB; ++k) xstore(xr[xs + k], st + k);
#pragma unroll
                for (uint32_t k = 0; k < SB; ++k) xload(xr[xs + k], b + KH * (SB * DX + k));
                __syncthreads();
#pragma unroll
                for (uint32_t k = 0; k < SB; ++k)
                    if (b + KH * k < b_end) compute(wv[ws + k], sv[ws + k], st + k);
#pragma unroll
                for (uint32_t k = 0; k < SB; ++k) wload(wv[ws + k], sv[ws + k], b + KH * (SB * DW + k));
            }
        }
    }

    // a, j: the tile's index among the ones that this wave finishes
    auto finish = [&](uint32_t a, uint32_t j, const f4_t& tot) {
        const uint32_t tile = tile0 + a0 + a, cl = TB * wc + j0 + j;
        if (tile >= p.tiles || cl >= cn) return;
        const uint32_t ct = ct0 + cl;
        if (wp.splits == 1u)
        {
            float bv = 0.0f;
            int32_t bi = 0;
            epilogue<WF, EPI>(p, tile, 16u * ct + r16, g4, tot, bv, bi, WF == OPURE_W_I8PC ? &scl[a] : nullptr);
        }
        else if (wp.part_rows)
        {
            const uint32_t m = 16u * ct + r16;
            if (m < p.M)
                *reinterpret_cast<f4_t*>(reinterpret_cast<float*>(wp.part) +
                                         (static_cast<uint64_t>(split) * p.M + m) * p.out + 16u * tile + 4u * g4) = tot;
        }
        else
        {
            wp.part[((static_cast<uint64_t>(split) * p.tiles + tile) * wp.mt + ct) * 64u + lane] = tot;
        }
    };
    if constexpr (KH == 1)
    {
#pragma unroll
        for (uint32_t a = 0; a < TA; ++a)
#pragma unroll
            for (uint32_t j = 0; j < TB; ++j) finish(a, j, acc[a][j]);
    }
    else
    {
        // the halves add through LDS (the X stages are free): half 0 finishes
        // the first half of its wave's weight or column tiles, half 1 the others;
        // each sum is (even blocks) + (odd blocks)
        constexpr uint32_t UA = BYT ? FT : 0u, UB = BYT ? 0u : FB;   // from half 0's tiles to half 1's
        __syncthreads();
        u4_t* ex = xl + ((1u - kh) * 4u + w4) * (FT * FB * 64u);  // the other half's inbox for this wave
#pragma unroll
        for (uint32_t a = 0; a < FT; ++a)
#pragma unroll
            for (uint32_t j = 0; j < FB; ++j)
                ex[(a * FB + j) * 64u + lane] = __builtin_bit_cast(u4_t, kh == 0 ? acc[UA + a][UB + j] : acc[a][j]);
        __syncthreads();
        const u4_t* in = xl + (kh * 4u + w4) * (FT * FB * 64u);
#pragma unroll
        for (uint32_t a = 0; a < FT; ++a)
#pragma unroll
            for (uint32_t j = 0; j < FB; ++j)
            {
                const f4_t other = __builtin_bit_cast(f4_t, in[(a * FB + j) * 64u + lane]);
                const f4_t mine = kh == 0 ? acc[a][j] : acc[UA + a][UB + j];
                const f4_t even = kh == 0 ? mine : other, odd = kh == 0 ? other : mine;
                finish(a, j, even + odd);
            }
    }
}

// the K splits of one (tile, column tile) added in split order, then the epilogue
template <int WF, int EPI>
__global__ __launch_bounds__(256) void k_wide_reduce(WParams wp)
{
    const KParams& p = wp.p;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t id = blockIdx.x * 4u + wave;
    if (id >= p.tiles * wp.mt) return;
    const uint32_t tile = id / wp.mt, ct = id - tile * wp.mt;
    f4_t tot = wp.part[(static_cast<uint64_t>(tile) * wp.mt + ct) * 64u + lane];
    for (uint32_t s = 1; s < wp.splits; ++s)
        tot += wp.part[((static_cast<uint64_t>(s) * p.tiles + tile) * wp.mt + ct) * 64u + lane];
    float bv = 0.0f;
    int32_t bi = 0;
    epilogue<WF, EPI>(p, tile, 16u * ct + (lane & 15u), lane >> 4, tot, bv, bi);
}

// The residual GEMV's splits added (row-major accumulators) with the next
// consumer's rmsnorm fused in: one workgroup per row m.  Per 4 outputs
// (o = 4u .. 4u + 3: tile u / 4, lane group u % 4) the same operations as the
// residual epilogue after k_wide_reduce -- splits added in split order, the
// int8 scale, y += v, the 4-output fma chain of squares and the tile's sum
// (g0 + g1) + (g2 + g3) -- then inv_rms from the tile sums in inv_rms_wave's
// order and round(y * inv * gain) as k_rmsnorm_rows, so y, ss_out and the
// normalised rows equal the separate passes' bit for bit.
// RN_THREADS 1024 up to 128 rows, 256 past that: a few rows are one round trip
// of each thread's loads, so fewer a thread (8B layer, fp16, at 20 rows 95.5 ->
// 94.1 us, at 128 228.1 -> 226.9; at 160 and 256 rows within 1% either way).
constexpr uint32_t RN_SPLITS = 8;   // the plan splits K at most 8 ways
template <int WF, int AF, int UNITS, uint32_t RN_THREADS>
__global__ __launch_bounds__(RN_THREADS) void k_wide_reduce_norm(WParams wp, const float* gain, void* xn)
{
    const KParams& p = wp.p;
    const uint32_t m = blockIdx.x, tid = threadIdx.x, lane = tid & 63u;
    const uint32_t units = p.out / 4u;
    __shared__ float ss_t[RN_THREADS * UNITS / 4u];
    __shared__ float inv_s;
    float* y = static_cast<float*>(p.y) + static_cast<uint64_t>(m) * p.out;
    const float* part = reinterpret_cast<const float*>(wp.part);
    // every split's accumulators and the residual in one round trip
    f4_t ps[UNITS][RN_SPLITS], y0[UNITS];
#pragma unroll
    for (uint32_t j = 0; j < UNITS; ++j)
    {
        const uint32_t uc = min(tid + RN_THREADS * j, units - 1u);
#pragma unroll
        for (uint32_t s = 0; s < RN_SPLITS; ++s)
            ps[j][s] = *reinterpret_cast<const f4_t*>(part + (static_cast<uint64_t>(min(s, wp.splits - 1u)) * p.M + m) * p.out +
                                                      4u * uc);
        y0[j] = *reinterpret_cast<const f4_t*>(y + 4u * uc);
    }
    f4_t nv[UNITS];
#pragma unroll
    for (uint32_t j = 0; j < UNITS; ++j)
    {
        const uint32_t u = tid + RN_THREADS * j;
        const bool live = u < units;
        const uint32_t uc = live ? u : 0u;
        f4_t tot = ps[j][0];
#pragma unroll
        for (uint32_t s = 1; s < RN_SPLITS; ++s)
            if (s < wp.splits) tot += ps[j][s];
        float sq = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            float v = tot[i];
            if constexpr (WF == OPURE_W_I8PC) v = __fmul_rn(v, f16_to_f32(static_cast<const uint16_t*>(p.sc)[4u * uc + i]));
            nv[j][i] = __fadd_rn(y0[j][i], v);
            sq = __fmaf_rn(nv[j][i], nv[j][i], sq);
        }
        if (live) *reinterpret_cast<f4_t*>(y + 4u * uc) = nv[j];
        // the tile's 4 lane groups are 4 consecutive threads
        const float a = __fadd_rn(sq, __shfl_xor(sq, 1));
        const float t = __fadd_rn(a, __shfl_xor(a, 2));
        if (live && (u & 3u) == 0u)
        {
            ss_t[u >> 2] = t;
            if (p.ss_out) p.ss_out[static_cast<uint64_t>(u >> 2) * p.M + m] = t;
        }
    }
    __syncthreads();
    if (tid < 64u)
    {
        float ssum = 0.0f;
        for (uint32_t t = lane; t < p.tiles; t += 64u) ssum += ss_t[t];
        KParams q = p;
        q.in = p.out;                 // the rms is over this GEMV's outputs
        const float inv = inv_rms_finish(q, ssum);
        if (tid == 0) inv_s = inv;
    }
    __syncthreads();
    const float inv = inv_s;
    uint8_t* dst = static_cast<uint8_t*>(xn) + static_cast<uint64_t>(m) * p.out * 2u;
#pragma unroll
    for (uint32_t j = 0; j < UNITS; ++j)
    {
        const uint32_t u = tid + RN_THREADS * j;
        if (u >= units) continue;
        const f4_t g = *reinterpret_cast<const f4_t*>(gain + 4u * u);
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = __fmul_rn(__fmul_rn(nv[j][i], inv), g[i]);
        *reinterpret_cast<u2_t*>(dst + 8u * u) = u2_t{pack2<AF>(r[0], r[1]), pack2<AF>(r[2], r[3])};
    }
}

// outputs up to 2048 (2 units of 4 a thread of 256) or 4096 (4, or 1 of 1024)
template <int WF, int AF>
int launch_wide_reduce_norm(opure_dev* dev, const WParams& wp, const float* gain, void* xn)
{
    if (wp.p.M <= 128u)
        OPURE_LAUNCH(dev, (k_wide_reduce_norm<WF, AF, 1, 1024u>), dim3(wp.p.M), dim3(1024), 0, wp, gain, xn);
    else if (wp.p.out <= 2048u)
        OPURE_LAUNCH(dev, (k_wide_reduce_norm<WF, AF, 2, 256u>), dim3(wp.p.M), dim3(256), 0, wp, gain, xn);
    else
        OPURE_LAUNCH(dev, (k_wide_reduce_norm<WF, AF, 4, 256u>), dim3(wp.p.M), dim3(256), 0, wp, gain, xn);
    OPURE_LAUNCH_CHECK("k_wide_reduce_norm");
    return OPURE_OK;
}

template <int WF, int AF, int EPI>
int launch_wide_epi_only(opure_dev* dev, const WParams& wp)
{
    // the kernel shape by the column tiles a workgroup has
    auto go = [&](auto sh) {
        using SH = decltype(sh);
        WParams q = wp;
        q.nrg = (wp.p.tiles + SH::RT - 1u) / SH::RT;
        OPURE_LAUNCH(dev, (k_gemm_wide<WF, AF, EPI, SH>), dim3(q.nrg * q.ncg * q.splits),
                     dim3(SH::NTH), 0, q);
        OPURE_LAUNCH_CHECK("k_gemm_wide");
        return OPURE_OK;
    };
    constexpr uint32_t KH = WF == OPURE_W_I8PC ? 2u : 1u;
    // an int8 prompt's step: one set of waves a workgroup, each wave four weight
    // tiles by four column tiles, or two in column groups of half the size
    if constexpr (WF == OPURE_W_I8PC)
    {
        if (wp.prompt && wp.cgs <= 4u) return go(WideShape<4, 2, 2, 1>{});
        if (wp.prompt) return go(WideShape<4, 4, 2, 1>{});
    }
    // the shapes of 17 to 256 rows (and a longer uint4 prompt's): one order of
    // a row's blocks
    if (wp.cgs <= 2u) return go(WideShape<1, 2, 1, KH>{});
    if (wp.cgs <= 4u) return go(WideShape<1, 4, 1, KH>{});
    return go(WideShape<2, 8, 1, KH>{});
}

template <int WF, int AF, int EPI>
int launch_wide_epi(opure_dev* dev, const WParams& wp, uint32_t lds)
{
    (void)lds;
    const int rc0 = launch_wide_epi_only<WF, AF, EPI>(dev, wp);
    if (rc0) return rc0;
    if (wp.splits > 1u)
    {
        const uint32_t n = wp.p.tiles * wp.mt;
        OPURE_LAUNCH(dev, (k_wide_reduce<WF, EPI>), dim3((n + 3u) / 4u), dim3(256), 0, wp);
        OPURE_LAUNCH_CHECK("k_wide_reduce");
    }
    return OPURE_OK;
}

// every epilogue but the per-workgroup argmax partials (wide callers store
// fp32 logits and take the argmax over them); a residual with K splits and a
// fused rmsnorm (gain != null) adds its splits in k_wide_reduce_norm
template <int WF, int AF>
int launch_wide_format(opure_dev* dev, uint32_t epi, const WParams& wp, uint32_t lds, const float* gain = nullptr,
                       void* xn = nullptr)
{
    if (gain && epi == opure_hip::EPI_RESIDUAL && wp.splits > 1u)
    {
        const int rc = launch_wide_epi_only<WF, AF, opure_hip::EPI_RESIDUAL>(dev, wp);
        return rc ? rc : launch_wide_reduce_norm<WF, AF>(dev, wp, gain, xn);
    }
    using namespace opure_hip;
    switch (epi)
    {
    case EPI_STORE: return launch_wide_epi<WF, AF, EPI_STORE>(dev, wp, lds);
    case EPI_RESIDUAL: return launch_wide_epi<WF, AF, EPI_RESIDUAL>(dev, wp, lds);
    case EPI_SWIGLU: return launch_wide_epi<WF, AF, EPI_SWIGLU>(dev, wp, lds);
    case EPI_QKV: return launch_wide_epi<WF, AF, EPI_QKV>(dev, wp, lds);
    }
    return set_error(OPURE_E_INVALID, "gemv: epilogue %u is not built for more than %d rows", epi, OPURE_MAX_ROWS);
}

}  // namespace opure_gemv
