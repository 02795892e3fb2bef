#pragma once
// MFMA submanifold conv for grids too small to fill the chip: the LDS-staged conv of
// conv_halo_kernel.hpp with a tile's work cut into up to eight times as many units.
//
// A unit is RGW of a tile's four row groups (128 voxels each) x 64 NCG output channels, run by one
// workgroup of 8 waves. Every wave owns a whole 128-voxel x 64-channel block of accumulators, as in
// the large-grid kernel, so an operand read from LDS or L2 feeds as many MFMAs; the waves beyond
// the unit's RGW x NCG blocks share the taps of a slice instead: tap group tg of TG = 8 / (RGW NCG)
// runs taps tg, tg + TG, ... At the end the tap groups' partial sums are added in group order
// through LDS (deterministic). Per unit and slice the workgroup stages the tile's distinct rows
// once, as the large-grid kernel does for the whole tile.
//
// The order of an output's sum depends on TG alone: TG follows from (n, ci, co) and the kind of
// stores (conv_split_pick), never from the plan, so the conv with and without a stored plan, and
// over any range of a plan's tiles, gives the same bits.
//
// Measured (one MI355X, us a conv, against the large-grid kernel, whose 512-voxel x 128-channel
// units are too few here): 2.6 K voxels 64 -> 64 f16 26 -> 13; 1.2 K 512 -> 512 253 -> 49;
// 4.1 K 1024 -> 1024 508 -> 266; 15 K 128 -> 128 70 -> 21; 35 K 512 -> 512 (1.08 rounds there)
// 499 -> 418; the C2S block 256 -> 128 on 2.6 K 235 -> 80. What bounds it: the latency of a slice (rows,
// weights, the barrier) and the CUs left idle. 4.1 K 1024 -> 1024, 144 units: the matrix cores are busy 31 %
// of the chip's cycles, 56 % of those of the CUs in use, and the waves wait 39 % of theirs; the rest
// is a unit's fixed 5-6 us (plan, first slice, the partial sums). Left out, the slice pieces give
// 12-20 %, the spread of the weights' addresses 10 %. An issue priority alternating between the waves,
// which the large-grid kernel takes, costs 3-7 % here.
#include "conv_halo_kernel.hpp"

namespace tsp {
namespace {

// Taps of a slice that a tap group runs, and the steps of the weight ring they take: the ring has
// 4 slots (weights 3 steps ahead), so a group of 7 taps counts as 8 steps, the last one empty.
constexpr int SPLIT_SLOTS2 = 1024;     // most distinct rows of a tile staged 32 channels at a time
constexpr int SPLIT_BUF = 4 * (SPLIT_SLOTS2 + 1) * 8;   // uint16 of a slice buffer
static_assert(SPLIT_BUF >= 2 * HB_ROWS * 8, "16 channels of HB_SLOTS rows fit too");
constexpr int split_steps(int tg) { return (kTaps + tg - 1) / tg; }

template <bool BF16, int RGW, int NCG, int ODT, int EPI, bool PLANNED>
__global__ __launch_bounds__(512, 1) void k_conv_split(
    const uint16_t* __restrict__ feats, int64_t n, int ci, const int32_t* __restrict__ nbr, PlanView plan,
    const uint16_t* __restrict__ weight, const float* __restrict__ bias, int co, void* __restrict__ out,
    int64_t n_tiles, int n_ctiles, int64_t per_xcd, bool ctile_major, OctantScatter osc, SkipAdd skip, PadRow pad,
    RowNorm ln) {
    constexpr int NT = 512, RB = 4, CB = 2;
    constexpr int BN = 64 * NCG, RS = 4 / RGW;       // channels of a unit; units of a tile
    constexpr int TG = 8 / (RGW * NCG);              // tap groups
    constexpr int S = split_steps(TG);               // steps of a slice
    constexpr int SV = S % 4 == 3 ? S + 1 : S;       // ring steps of a slice
    static_assert(TG >= 2 && RGW * NCG * TG == 8 && (2 * SV) % 4 == 0, "8 waves, ring of 4 over slice pairs");
    // the two slice buffers: 16 channels of up to HB_SLOTS rows or 32 of up to SPLIT_SLOTS2, in planes
    // of 8 channels, each plane ending in a zero slot
    __shared__ __attribute__((aligned(16))) uint16_t sH0[SPLIT_BUF];
    __shared__ __attribute__((aligned(16))) uint16_t sH1[SPLIT_BUF];
    __shared__ __attribute__((aligned(16))) uint16_t sL[kTaps][4][32][4];
    __shared__ int sRed[2 * NT / 64];

    // Each XCD takes a contiguous range of units. Units in column-tile-major order keep an XCD on
    // few weight columns, in tile-major order on few feature rows: the caller picks by which is
    // larger, the weights or the features.
    constexpr bool OCT = EPI == 1 || EPI == 4 || EPI == 5;
    int64_t units = n_tiles * n_ctiles * RS;
    bool on_oct = false;
    if constexpr (EPI == 1 || EPI == 5) {
        if (!octant_side(osc, plan)) return;
        if (osc.oct) {   // (never more units than on the parents' plan)
            on_oct = true;
            units = (int64_t)osc.oct->total * (osc.cout / BN) * RS;
            per_xcd = (units + 7) / 8;
        }
    }
    const int64_t u = (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || u >= units) return;
    int64_t tile;
    int ct, rsub;
    if (on_oct) {
        // octant after octant in column-tile-major order; otherwise the octants take turns
        const int cpo = osc.cout / BN;               // column tiles of an octant
        rsub = (int)(u % RS);
        int oct, k, c;
        if (ctile_major) {
            int64_t v = u / RS;
            for (oct = 0; oct < 7 && v >= (int64_t)osc.oct->tiles[oct] * cpo; ++oct) v -= (int64_t)osc.oct->tiles[oct] * cpo;
            c = (int)(v / osc.oct->tiles[oct]);
            k = (int)(v % osc.oct->tiles[oct]);
        } else {
            c = (int)(u / RS % cpo);
            octant_turn(osc.oct, (int)(u / RS / cpo), oct, k);
        }
        tile = osc.oct->base[oct] + k;
        ct = oct * cpo + c;
    } else if (ctile_major) {
        const int64_t pc = n_tiles * RS;
        ct = (int)(u / pc);
        tile = (u % pc) / RS;
        rsub = (int)(u % RS);
    } else {
        tile = u / ((int64_t)n_ctiles * RS);
        const int k = (int)(u % ((int64_t)n_ctiles * RS));
        ct = k / RS;
        rsub = k % RS;
    }
    const int64_t row0 = tile * HB_M;

    const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rgl = wave % RGW, cg = (wave / RGW) % NCG, tg = wave / (RGW * NCG);
    const int rg = rsub * RGW + rgl;                 // row group of the tile
    const int co0 = ct * BN, c0 = co0 + cg * 64;
    const int nkc = ci / HB_KC;

    // a unit of the last tile may hold no voxel at all
    {
        bool any = false;
        if (tid < 128 * RGW) {
            const int p = 128 * RGW * rsub + tid;
            if constexpr (PLANNED) any = plan.vox[tile * HB_M + p] >= 0;
            else any = row0 + p < n;
        }
        if (!__syncthreads_or(any)) return;
    }

    // the padding row 0 * feats[0], and whether absent taps may be skipped (conv_halo_kernel.hpp)
    bool row0_bad = false;
    if (!pad.zero) {
        if (pad.row0) {
            for (int k = tid; k < ci; k += NT) row0_bad |= !__builtin_isfinite(pad.row0[k]);
        } else {
            for (int k = tid * 8; k < ci; k += NT * 8) {
                const u32x4_t v = *reinterpret_cast<const u32x4_t*>(feats + k);
                constexpr uint32_t kExp = BF16 ? 0x7F807F80u : 0x7C007C00u;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    row0_bad |= ((v[e] & kExp & 0xffffu) == (kExp & 0xffffu)) ||
                                ((v[e] & kExp & 0xffff0000u) == (kExp & 0xffff0000u));
            }
        }
    }
    row0_bad = __syncthreads_or(row0_bad);
    // act bits of this wave's taps: step s of tap group tg is tap s TG + tg, whose 4 block bits start
    // at bit 4 (s TG + tg); the words are shifted by 4 tg here, so that a step's place is static
    uint32_t ab[HB_ACT_WORDS];
    bool may_skip = false;
    if constexpr (PLANNED)
        may_skip = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(weight) +
                                                      (size_t)kTaps * ci * co * 2) == 0u;
    uint32_t ob = 0xffffffffu;                       // octant stores: blocks that keep the wave's octant
    const int oct = OCT ? c0 / osc.cout : 0;
    if constexpr (EPI == 1 || EPI == 4 || EPI == 5) {
        if (osc.blocks) {
            const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)osc.blocks[tile * 4 + rg]);
            ob = ((w >> (4 * oct)) & 15u) * 0x11111111u;
        }
    }
#pragma unroll
    for (int k = 0; k < HB_ACT_WORDS; ++k) {
        uint32_t v = ~0u;
        if (PLANNED && may_skip)
            v = (uint32_t)__builtin_amdgcn_readfirstlane((int)plan.act[(tile * 4 + rg) * HB_ACT_WORDS + k]);
        if (k == HB_ACT_WORDS - 1) v &= (1u << (4 * (kTaps - 8 * k))) - 1u;   // no tap past the last
        ab[k] = (v & ob) >> (4 * tg);
    }
    auto step_bits = [&](int s) -> uint32_t {
        uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)ab[(s * TG) >> 3]);
        asm volatile("" : "+s"(v));
        return (v >> ((4 * s * TG) & 31)) & 15u;
    };
    // tap of step s; past the last tap (all its bits clear) the last tap, whose operands are unused
    auto step_tap = [&](int s) { return (s + 1) * TG <= kTaps ? s * TG + tg : min(s * TG + tg, kTaps - 1); };

    // ---- the tile's slot table and the rows of this wave's slice pieces. A tile of at most
    // SPLIT_SLOTS2 distinct rows (98-100 % of the tiles of surface sets, in Morton order) stages 32
    // channels at a time: a lane quad loads 64 contiguous bytes of a row, so a piece touches 16 cache
    // lines where 16 channels at a time touch 32 for the same bytes, and a barrier serves two slices.
    // The taps still run slice by slice, so the sums' order does not depend on it.
    constexpr int PIECES = 8;
    int H;
    bool direct;
    if constexpr (PLANNED) {
        const int32_t* hdr = plan.hdr + tile * 4;
        const int32_t h0 = hdr[0], h1 = hdr[1];
        const char* src = reinterpret_cast<const char*>(plan.slots + tile * HB_SLOT_TABLE);
        for (int p = wave; p < HB_SLOT_TABLE * 2 / 1024; p += 8)   // 27 x 1 KiB
            __builtin_amdgcn_global_load_lds(
                src + p * 1024 + lane * 16,
                (__attribute__((address_space(3))) void*)(reinterpret_cast<char*>(&sL[0][0][0][0]) + p * 1024), 16, 0, 0);
        H = __builtin_amdgcn_readfirstlane(h0);
        direct = __builtin_amdgcn_readfirstlane(h1) != 0;
    } else {
        int hh;
        bool dd;
        tile_plan<NT>(nbr, n, row0, sL, reinterpret_cast<int32_t*>(sH0), reinterpret_cast<uint32_t*>(sH1), sRed, hh, dd);
        H = __builtin_amdgcn_readfirstlane(hh);
        direct = __builtin_amdgcn_readfirstlane((int)dd) != 0;
    }

    uint32_t boff[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        if constexpr (PLANNED) boff[cb] = (uint32_t)((((c0 >> 5) + cb) * nkc * kTaps * 64 + lane) * 16u);
        else boff[cb] = (uint32_t)(((uint32_t)(c0 + cb * 32 + r32) * (uint32_t)(kTaps * ci) + g * 8) * 2u);
    }
    auto load_b = [&](int t, int kc, u32x4_t* dst) {
        const char* wt;
        if constexpr (PLANNED) wt = reinterpret_cast<const char*>(weight) + ((int64_t)kc * kTaps + t) * 1024;
        else wt = reinterpret_cast<const char*>(weight + ((int64_t)t * ci + kc * HB_KC));
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            uint32_t o = boff[cb];
            asm volatile("" : "+v"(o));
            dst[cb] = *reinterpret_cast<const u32x4_t*>(wt + o);
        }
    };

    f32x16_t acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[rb][cb][j] = 0.f;

    // KS 16-channel slices a buffer
    auto staged = [&](auto ks_c) {
        constexpr int KS = decltype(ks_c)::value;
        constexpr int LPS = 2 * KS, SPP = 64 / LPS;  // lanes of a slot's piece, slots of a piece
        constexpr int ROWS = (KS == 2 ? SPLIT_SLOTS2 : HB_SLOTS) + 1;
        const int plane = lane % LPS;
        auto piece_slot = [&](int j) { return SPP * (wave + 8 * j) + lane / LPS; };
        const int np = min(PIECES, max(0, (H - SPP * wave + 8 * SPP - 1) / (8 * SPP)));   // this wave's pieces
        uint32_t poff[PIECES];
        {
            int32_t prow[PIECES];
            const int32_t* ro = PLANNED ? plan.rowof + tile * HB_SLOTS : reinterpret_cast<const int32_t*>(sH0);
#pragma unroll
            for (int j = 0; j < PIECES; ++j) prow[j] = ro[piece_slot(j)];
            if (!PLANNED) __syncthreads();           // sH0 is overwritten by the first slice below
#pragma unroll
            for (int j = 0; j < PIECES; ++j) {
                const int32_t r = (piece_slot(j) < H && (uint32_t)prow[j] < (uint32_t)n) ? prow[j] : 0;
                poff[j] = (uint32_t)r * (uint32_t)ci * 2u + plane * 16u;
                asm volatile("" : "+v"(poff[j]));
            }
        }
        // slot r of plane p
        auto at = [](int p, int r) { return (p * ROWS + r) * 8; };
        auto fetch_piece = [&](int kc, int j, u32x4_t& r) {
            r = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const char*>(feats) + poff[j] +
                                                  (uint32_t)kc * (HB_KC * 2));
        };
        auto put_piece = [&](uint16_t* dst, int j, const u32x4_t& r) {
            *reinterpret_cast<u32x4_t*>(dst + at(plane, piece_slot(j))) = r;
        };
        if (tid < 2 * LPS)   // the zero slots, past every staged one
            *reinterpret_cast<u32x4_t*>((tid < LPS ? sH0 : sH1) + at(tid % LPS, ROWS - 1)) = u32x4_t{0, 0, 0, 0};
        u32x4_t bR[4][CB];
#pragma unroll
        for (int s = 0; s < 3; ++s) load_b(step_tap(s), 0, bR[s]);
        u32x4_t stg[4];
        // first slices: pieces 0..3 together, then 4..7
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j = 4 * h; j < 4 * h + 4; ++j)
                if (j < np) fetch_piece(0, j, stg[j & 3]);
#pragma unroll
            for (int j = 4 * h; j < 4 * h + 4; ++j)
                if (j < np) put_piece(sH0, j, stg[j & 3]);
        }
        wait_vmcnt0();       // the slot table's direct-to-LDS loads
        __syncthreads();

        // When piece j of the next buffer is loaded and when it is written to LDS, in steps of this
        // buffer's KS S (all before its barrier); pieces j and j + 4 share their registers.
        constexpr int GS = KS * S;
        auto fetch_at = [](int j) -> int {
            if (GS >= 26) return 3 * j;                     // 28 steps
            if (GS >= 13) return j < 4 ? j : j + 1;         // 14
            if (GS >= 8) return j < 4 ? j / 2 : 3;          // 8
            if (GS >= 7) return j < 4 ? j / 2 : 4;          // 7
            return j < 4 ? 0 : 2;                           // 4
        };
        auto put_at = [](int j) -> int {
            if (GS >= 26) return 3 * j + 4;
            if (GS >= 13) return j < 4 ? j + 4 : j + 5;
            if (GS >= 8) return j < 4 ? 3 : 6;
            if (GS >= 7) return j < 4 ? 3 : 6;
            return j < 4 ? 2 : 3;
        };
        // The slots of a step's 4 blocks (absent taps: the zero slot of this layout). They are the same
        // in every slice: with few steps a slice (TG >= 4) a wave keeps them in registers, otherwise
        // they are read from LDS a step ahead of the operands.
        auto read_slots = [&](int s) {
            uint2 sl = *reinterpret_cast<const uint2*>(&sL[step_tap(s)][rg][r32][0]);
            if constexpr (KS == 2) {
                typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
                const u16x2_t z = {ROWS - 1, ROWS - 1};
                sl.x = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, sl.x), z));
                sl.y = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, sl.y), z));
            }
            return sl;
        };
        constexpr bool KEEP = TG >= 4;
        uint2 kept[KEEP ? S : 1];
        if constexpr (KEEP) {
#pragma unroll
            for (int s = 0; s < S; ++s) kept[s] = read_slots(s);
        }
        auto slots_of = [&](int s) {
            if constexpr (KEEP) {
                uint2 v = kept[s];
                asm volatile("" : "+v"(v.x), "+v"(v.y));   // the words, not the addresses made of them, stay live
                return v;
            } else {
                return read_slots(s);
            }
        };
        auto a_of = [&](const uint16_t* buf, int ps, uint32_t slot) {
            return *reinterpret_cast<const u32x4_t*>(buf + at(2 * ps + g, (int)slot));
        };
        u32x4_t aC[RB];      // the A operands of the next step
        uint2 slN{};         // the slots of the step after it (not KEEP)
        if constexpr (!KEEP) slN = read_slots(1);
        {
            const uint2 sl = slots_of(0);
            aC[0] = a_of(sH0, 0, sl.x & 0xffffu);
            aC[1] = a_of(sH0, 0, sl.x >> 16);
            aC[2] = a_of(sH0, 0, sl.y & 0xffffu);
            aC[3] = a_of(sH0, 0, sl.y >> 16);
        }
        // One buffer: this wave's taps of slices k0 .. k0 + KS - 1 on `cur` while slices kn .. stream
        // into `nxt`. r0: the weight ring's slot of the first step. The one barrier of a buffer comes
        // before its last step: by then every wave has written its pieces of `nxt` and read its last
        // operands of `cur`, so the last step's MFMAs run behind it while the next buffer's first
        // operands are read.
        auto run_buffer = [&](auto ring0, const uint16_t* cur, uint16_t* nxt, int k0, int kn) {
            u32x4_t aN[RB];
#pragma unroll
            for (int ps = 0; ps < KS; ++ps) {
#pragma unroll
                for (int s = 0; s < SV; ++s) {
                    const int R0 = (decltype(ring0)::value + ps * SV) % 4, G = ps * S + s;
                    // weights 3 ring steps ahead (the first steps of the next slice at the end)
                    {
                        const int q = s + 3;
                        if (q < S) load_b(step_tap(q), k0 + ps, bR[(R0 + q) % 4]);
                        else if (q >= SV) load_b(step_tap(q - SV), ps + 1 < KS ? k0 + ps + 1 : kn, bR[(R0 + q) % 4]);
                    }
                    if (s >= S) {                        // the empty ring step
                        __builtin_amdgcn_sched_barrier(0);
                        continue;
                    }
#pragma unroll
                    for (int j = 0; j < PIECES; ++j)
                        if (put_at(j) == G && j < np) put_piece(nxt, j, stg[j & 3]);
#pragma unroll
                    for (int j = 0; j < PIECES; ++j)
                        if (fetch_at(j) == G && j < np) fetch_piece(kn, j, stg[j & 3]);
                    const bool last = G == GS - 1;
                    if (last) __syncthreads();
                    // the next step's operands: of this slice, of the buffer's next slice, or of the
                    // next buffer
                    const uint16_t* src = last ? nxt : cur;
                    const int nps = s + 1 < S ? ps : last ? 0 : ps + 1;
                    const uint32_t on = step_bits(s);
                    auto mfma_block = [&](int rb) {
                        if (__builtin_expect((on >> rb) & 1u, 1)) {
#pragma unroll
                            for (int cb = 0; cb < CB; ++cb)
                                acc[rb][cb] = mfma32x32x16<BF16>(aC[rb], bR[(R0 + s) % 4][cb], acc[rb][cb]);
                        }
                    };
                    mfma_block(0);
                    uint2 sl;
                    if constexpr (KEEP) {
                        sl = slots_of(s + 1 < S ? s + 1 : 0);
                    } else {
                        sl = slN;
                        slN = read_slots((s + 2) % S);
                    }
                    mfma_block(1);
                    aN[0] = a_of(src, nps, sl.x & 0xffffu);
                    aN[1] = a_of(src, nps, sl.x >> 16);
                    mfma_block(2);
                    aN[2] = a_of(src, nps, sl.y & 0xffffu);
                    aN[3] = a_of(src, nps, sl.y >> 16);
                    mfma_block(3);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) aC[rb] = aN[rb];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) asm volatile("" ::"v"(acc[rb][cb]));
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, (KS * SV) % 4>;
        // the last buffer re-loads itself into the idle one, so there is no branch
        for (int kc = 0; kc < nkc; kc += 2 * KS) {
            const int k1 = kc + KS < nkc ? kc + KS : kc;
            run_buffer(I0{}, sH0, sH1, kc, k1);
            if (kc + KS < nkc) run_buffer(I1{}, sH1, sH0, kc + KS, kc + 2 * KS < nkc ? kc + 2 * KS : kc + KS);
        }
        __syncthreads();     // every wave is past its last read of the slice buffers
    };
    if (!direct) {
        if (H <= SPLIT_SLOTS2 && nkc % 2 == 0) staged(std::integral_constant<int, 2>{});
        else staged(std::integral_constant<int, 1>{});
    } else {
        // ---- direct path: A gathered from global memory
        for (int kc = 0; kc < nkc; ++kc)
            for (int t = tg; t < kTaps; t += TG) {
                u32x4_t bq[CB];
                load_b(t, kc, bq);
                u32x4_t a[RB];
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const int p = 128 * rg + 32 * rb + r32;   // tile position
                    int64_t i = row0 + p;
                    if constexpr (PLANNED) i = plan.vox[tile * HB_M + p];
                    const int32_t v = (i >= 0 && i < n) ? nbr[(int64_t)t * n + i] : (int32_t)n;
                    a[rb] = u32x4_t{0, 0, 0, 0};
                    if ((uint32_t)v < (uint32_t)n)
                        a[rb] = *reinterpret_cast<const u32x4_t*>(feats + (int64_t)v * ci + kc * HB_KC + g * 8);
                }
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb)
                        acc[rb][cb] = mfma32x32x16<BF16>(a[rb], bq[cb], acc[rb][cb]);
            }
        __syncthreads();     // (the planned slot table load may still be writing sL; nothing reads it)
    }

    // ---- partial sums through LDS, two phases of 64 rows per row group: TG x (64 RGW rows) x BN
    // channels f32 = 128 KiB, half of the tap groups in each slice buffer. Then a thread takes 8
    // channels of a row: the sum over the tap groups, + bias, and the stores.
    constexpr int PROWS = 64 * RGW;                  // rows of a phase
    constexpr int LPR = BN / 8;                      // lanes of a row
    constexpr int ITEMS = PROWS * LPR / NT;
    static_assert((TG / 2) * PROWS * BN * 4 <= (int)sizeof(sH0), "partials fit the slice buffers");
    static_assert(PROWS * LPR % NT == 0 && NT % LPR == 0, "whole items per thread");
    auto part = [&](int q) -> float* {               // tap group q's partials
        return reinterpret_cast<float*>(q < TG / 2 ? sH0 : sH1) + (q % (TG / 2)) * PROWS * BN;
    };
    const int ch = (tid % LPR) * 8;                  // this thread's channels of the unit
    float bv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bv[e] = bias[co0 + ch + e];
    // output rows of the thread's items, both phases
    int vrow[2][ITEMS];
#pragma unroll
    for (int ph = 0; ph < 2; ++ph)
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int r = (it * NT + tid) / LPR;
            const int p = 128 * (rsub * RGW + r / 64) + 64 * ph + r % 64;
            if constexpr (PLANNED) vrow[ph][it] = plan.vox[tile * HB_M + p];
            else vrow[ph][it] = row0 + p < n ? (int)(row0 + p) : -1;
        }
    float* mine = part(tg) + (64 * rgl) * BN + cg * 64 + r32;
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
        if (ph) __syncthreads();                     // the first phase's partials are read
#pragma unroll
        for (int rb2 = 0; rb2 < 2; ++rb2)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    mine[(32 * rb2 + 8 * (j / 4) + 4 * g + (j % 4)) * BN + cb * 32] = acc[2 * ph + rb2][cb][j];
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int r = (it * NT + tid) / LPR;
            const int64_t i = vrow[ph][it];
            float v[8];
#pragma unroll
            for (int q = 0; q < TG; ++q) {
                const float* src = part(q) + r * BN + ch;
                const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(src), hi = *reinterpret_cast<const f32x4_t*>(src + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = q ? v[e] + lo[e] : lo[e];
                    v[4 + e] = q ? v[4 + e] + hi[e] : hi[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += bv[e];
            // a row with an absent tap is NaN where row 0 is not finite (before or after a norm alike)
            bool nan_row = false;
            if (row0_bad && i >= 0)
                for (int t = 0; t < kTaps; ++t) nan_row |= nbr[(int64_t)t * n + i] == (int32_t)n;
            if constexpr (EPI == 3 || EPI == 4 || EPI == 5) {
                // the row's (EPI 4, 5: the child row's) LayerNorm over its BN channels
                float sum = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) sum += v[e];
                const float mean = group_sum<LPR>(sum) / (float)BN;
                float sq = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float d = v[e] - mean;
                    sq += d * d;
                }
                const float rstd = 1.0f / sqrtf(group_sum<LPR>(sq) / (float)BN + (EPI == 3 ? ln.eps : osc.norm_eps));
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v[e] = (v[e] - mean) * rstd;
                    if constexpr (EPI == 3) v[e] = v[e] * ln.w[ch + e] + ln.b[ch + e];
                    else v[e] = v[e] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[e]));
                }
            }
            if (nan_row) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = NAN;
            }
            // the stored row and its first channel
            bool keep = i >= 0;
            int64_t o = i * co + co0 + ch;
            if constexpr (EPI == 1 || EPI == 4 || EPI == 5) {
                int64_t child = -1;
                const int uo = co0 / osc.cout;       // the unit's octant
                if (keep) {
                    constexpr uint64_t kLow7 = 0x7f7f7f7f7f7f7f7full;
                    const uint64_t mw = *reinterpret_cast<const uint64_t*>(osc.mask + 8 * i);
                    const uint64_t kept = (((mw & kLow7) + kLow7) | mw) & ~kLow7;   // bit 8b+7: byte b != 0
                    if ((kept >> (8 * uo + 7)) & 1) child = osc.mstart[i] + __popcll(kept & ((1ull << (8 * uo)) - 1));
                }
                keep = child >= 0;
                o = child * osc.cout + (co0 - uo * osc.cout) + ch;
            }
            if (!keep) continue;
            if constexpr (EPI == 2) {
                // child row: + x[gidx / 8][(gidx % 8) K + c / R], 4 channels sharing an element
                const int gi = skip.gidx[i], kk = skip.cin / 8, rep_r = co / kk;
                const float* xr = skip.x + (int64_t)(gi >> 3) * skip.cin + (gi & 7) * kk;
                const float s0 = xr[(co0 + ch) / rep_r], s1 = xr[(co0 + ch + 4) / rep_r];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += e < 4 ? s0 : s1;
            }
            if constexpr (ODT == TSP_F32) {
                float* dst = reinterpret_cast<float*>(out) + o;
                *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{v[0], v[1], v[2], v[3]};
                *reinterpret_cast<f32x4_t*>(dst + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
            }
            auto pack = [&](bool bf) {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    w[e] = bf ? f32x2_to_bf16x2_bits(v[2 * e], v[2 * e + 1])
                              : f32_to_f16_bits(v[2 * e]) | ((uint32_t)f32_to_f16_bits(v[2 * e + 1]) << 16);
                return u32x4_t{w[0], w[1], w[2], w[3]};
            };
            if constexpr (EPI == 2) {
                if (skip.out16)   // (8-byte aligned)
                {
                    const u32x4_t w = pack(skip.out16_bf16);
                    uint2* dst = reinterpret_cast<uint2*>(static_cast<uint16_t*>(skip.out16) + o);
                    dst[0] = uint2{w[0], w[1]};
                    dst[1] = uint2{w[2], w[3]};
                }
            }
            if constexpr (ODT != TSP_F32)
                *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(out) + o) = pack(ODT == TSP_BF16);
        }
    }
}

// The launch over a plan's tiles [t0, t0 + nt) (all tiles without a plan).
template <bool BF16, int RGW, int NCG>
int split_launch(int odt, bool planned, const void* feats, int64_t n, int ci, const int32_t* nbr, const void* plan,
                 const void* weight, const float* bias, int co, void* out, hipStream_t s, OctantScatter osc,
                 SkipAdd skip, PadRow pad, RowNorm ln, TileRange tr) {
    constexpr int BN = 64 * NCG;
    constexpr int O16 = BF16 ? TSP_BF16 : TSP_F16;
    const int64_t all_tiles = ceil_div(n, HB_M);
    const int64_t t0 = planned ? tr.t0 : 0;
    const int64_t n_tiles = planned && tr.nt >= 0 ? tr.nt : all_tiles - t0;
    if (t0 < 0 || n_tiles < 0 || t0 + n_tiles > all_tiles) {
        set_error("MFMA conv: tiles [%lld, %lld) outside the plan's %lld", (long long)t0,
                  (long long)(t0 + n_tiles), (long long)all_tiles);
        return TSP_ERR_INVALID;
    }
    if (n_tiles == 0) return TSP_OK;
    const int n_ctiles = co / BN;
    const int64_t per_xcd = ceil_div(n_tiles * n_ctiles * (4 / RGW), 8);
    const bool ctile_major = n < (int64_t)kTaps * co;
    PlanView pv{};
    if (planned) {
        pv = carve_plan(const_cast<void*>(plan), all_tiles);
        pv.hdr += t0 * 4;
        pv.rowof += t0 * HB_SLOTS;
        pv.slots += t0 * HB_SLOT_TABLE;
        pv.vox += t0 * HB_M;
        pv.act += t0 * 4 * HB_ACT_WORDS;
    }
    if (osc.blocks) osc.blocks += t0 * 4;
    auto go = [&](auto odt_c, auto epi_c, auto planned_c) -> int {
        hipLaunchKernelGGL((k_conv_split<BF16, RGW, NCG, decltype(odt_c)::value, decltype(epi_c)::value,
                                         decltype(planned_c)::value>),
                           dim3((unsigned)(per_xcd * 8)), dim3(512), 0, s, reinterpret_cast<const uint16_t*>(feats), n,
                           ci, nbr, pv, reinterpret_cast<const uint16_t*>(weight), bias, co, out, n_tiles, n_ctiles,
                           per_xcd, ctile_major, osc, skip, pad, ln);
        TSP_CHECK_LAUNCH();
        return TSP_OK;
    };
    using std::integral_constant;
    using F = integral_constant<int, TSP_F32>;
    using H = integral_constant<int, O16>;
    using P = std::true_type;
    if constexpr (NCG == 2) {
        if (osc.norm_silu) return go(H{}, integral_constant<int, 5>{}, P{});
        return go(H{}, integral_constant<int, 3>{}, P{});
    } else {
        if (osc.cout) return osc.norm_silu ? go(H{}, integral_constant<int, 4>{}, P{}) : go(F{}, integral_constant<int, 1>{}, P{});
        if (skip.cin) return go(F{}, integral_constant<int, 2>{}, P{});
        if (ln.w) return go(H{}, integral_constant<int, 3>{}, P{});
        using I0 = integral_constant<int, 0>;
        if (odt == TSP_F32) return planned ? go(F{}, I0{}, P{}) : go(F{}, I0{}, std::false_type{});
        return planned ? go(H{}, I0{}, P{}) : go(H{}, I0{}, std::false_type{});
    }
}

}  // namespace
}  // namespace tsp
