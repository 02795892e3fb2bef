// The LDS-staged MFMA conv's entry points: weight packing and the dispatch to the kernel
// instantiations (conv_halo_kernel.hpp holds the kernel; conv_halo_{bf16,f16}_{128,64}.hip
// instantiate it, one translation unit per family so that they compile in parallel).
#include "conv_halo_kernel.hpp"

namespace tsp {
namespace {

// packed[((c32 * nkc + kc) * 27 + t) * 64 + lane][0..7] = W[32 c32 + lane%32][t][16 kc + 8 (lane/32) ..];
// *nonfinite (the first word of the trailer, cleared before) |= 1 where a weight is an Inf or a NaN.
__global__ void k_weight_pack(const uint16_t* __restrict__ w, int ci, int co, bool bf16,
                              uint16_t* __restrict__ packed, uint32_t* __restrict__ nonfinite) {
    const int nkc = ci / HB_KC;
    const int64_t blk = blockIdx.x;                    // (c32 * nkc + kc) * 27 + t
    const int t = (int)(blk % kTaps);
    const int64_t ck = blk / kTaps;
    const int kc = (int)(ck % nkc), c32 = (int)(ck / nkc);
    const int lane = threadIdx.x;
    const int col = c32 * 32 + (lane & 31);
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(
        w + ((int64_t)col * kTaps + t) * ci + kc * HB_KC + (lane >> 5) * 8);
    reinterpret_cast<u32x4_t*>(packed)[blk * 64 + lane] = v;
    const uint32_t e = bf16 ? 0x7F80u : 0x7C00u;     // exponent all ones: Inf or NaN
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) bad |= (v[k] & e) == e || ((v[k] >> 16) & e) == e;
    if (bad) atomicOr(nonfinite, 1u);
}

__global__ void k_pack_trailer_clear(uint32_t* __restrict__ trailer) {
    trailer[threadIdx.x] = 0u;
}

}  // namespace

bool halo_fits(int64_t n, int ci) { return n * (int64_t)ci * 2 < ((int64_t)1 << 32); }

int halo_weight_pack(const void* w, int wdt, int ci, int co, void* packed, hipStream_t s) {
    const int64_t blocks = (int64_t)(co / 32) * (ci / HB_KC) * kTaps;
    uint32_t* trailer = reinterpret_cast<uint32_t*>(static_cast<char*>(packed) + (size_t)kTaps * ci * co * 2);
    hipLaunchKernelGGL(k_pack_trailer_clear, dim3(1), dim3(HB_PACK_TRAILER / 4), 0, s, trailer);
    TSP_CHECK_LAUNCH();
    if (blocks == 0) return TSP_OK;
    hipLaunchKernelGGL(k_weight_pack, dim3((unsigned)blocks), dim3(64), 0, s,
                       reinterpret_cast<const uint16_t*>(w), ci, co, wdt == TSP_BF16,
                       reinterpret_cast<uint16_t*>(packed), trailer);
    TSP_CHECK_LAUNCH();
    return TSP_OK;
}

int64_t column_split_tiles(int64_t n_tiles, int nct, int cus) {
    if (n_tiles <= 0 || nct <= 0 || cus <= 0) return 0;
    // the planned grid at 128 channels a unit: cus / 8 workgroups per XCD rounded down to a
    // multiple of the nct column tiles, each XCD walking its contiguous share of the units a round
    // at a time
    const int64_t g128 = 8 * std::max<int64_t>(1, cus / 8 / nct) * nct;
    const int64_t rounds = n_tiles * nct / g128;
    if (rounds < 1) return 0;
    const int64_t t_split = rounds * (g128 / nct);   // whole rounds of every workgroup
    const int64_t left = n_tiles - t_split;
    if (left <= 0) return 0;
    // the last round's units as 64-channel units: worth it while they make one round of the
    // 64-channel grid (each unit half the products, at 0.64-0.83 of a 128-channel unit's time)
    const int64_t fit64 = std::max<int64_t>(1, cus / 8 / (2 * nct)) * (2 * nct);
    return ceil_div(left * 2 * nct, 8) <= fit64 ? t_split : 0;
}

int conv_cus() { return cu_count(); }

int conv_split_pick(int64_t n, int ci, int co, int ncg) {
    if (n <= 0 || co % (64 * ncg) != 0) return 0;
    const int64_t cus = cu_count(), nkc = ci / HB_KC, tiles = ceil_div(n, HB_M);
    // The kernels' times in us (fits to single convs of 1.2K-117K voxels, 64-1024 channels): a round
    // of units costs so much per 16-channel slice, plus a fixed part (the large-grid kernel's tiles
    // are pipelined and pay it once; a thin last round costs it 5.6 a slice, column_split_tiles).
    const int64_t big = tiles * (co % 128 == 0 ? co / 128 : co / 64);
    int64_t whole = ceil_div(big, cus);
    double per = co % 128 == 0 ? 9.3 : 4.6;
    // One round of the large-grid kernel runs faster on a part of the chip: 33.5 K and 45 K 256 -> 256, a
    // half and two thirds of a round, 137 and 146 us where a full one is 158.
    if (whole == 1) per *= 0.84 + 0.32 * std::max(0.0, (double)big / (double)cus - 0.5);
    double base = 9.0;
    if (ncg == 1 && co % 128 == 0 && column_split_tiles(tiles, co / 128, (int)cus) > 0) {
        whole -= 1;
        base += 5.6 * (double)nkc;
    }
    const double large = base + per * (double)(whole * nkc);
    // The units of a tile each stage its rows, and more of them on a plan of consecutive rows or without
    // a plan, which take the same kernel. Where those rows come from L2 (features of up to 8 MiB, or the
    // units that run together share few tiles) or are staged once a column tile, a twentieth less
    // time is enough; elsewhere a twelfth: 33.5 K 512 -> 256, in three rounds of units of two row groups, was
    // 243 us on a Morton plan (262 on the large-grid kernel), but 294 on rows (261) and 488 without a
    // plan (440).
    const bool in_l2 = n * (int64_t)ci * 2 <= ((int64_t)8 << 20);
    double best = large;
    int pick = 0;
    const int64_t full = n / HB_M, rem = n % HB_M;
    const int64_t last = rem ? std::min<int64_t>(4, ceil_div(rem, 32)) : 0;   // row groups of the last tile
    for (int rgw = 4 / ncg; rgw >= 1; rgw /= 2) {
        const int64_t units = (full * (4 / rgw) + ceil_div(last, rgw)) * (co / (64 * ncg));
        const int w = rgw * ncg;
        const int64_t rounds = ceil_div(units, cus);
        const double slice = w == 4 ? 4.6 : w == 2 ? (rounds == 1 ? 2.2 : in_l2 ? 2.255 : 2.45) : (rounds > 1 ? 1.6 : 1.45);
        const double cost = 4.0 + (double)rounds * (6.0 + slice * (double)nkc);
        const int64_t share = (4 / rgw) * (co / (64 * ncg));   // units of a tile
        const bool near = w == 4 || share >= 64 || (share >= 32 && whole == 1);
        if (cost < best && cost < (in_l2 ? 0.955 : near ? 0.95 : 0.92) * large) {
            best = cost;
            pick = rgw;
        }
    }
    return pick;
}

int halo_conv_launch(int fdt, int odt, const void* feats, int64_t n, int ci, const int32_t* nbr,
                     const void* plan, const void* weight, const float* bias, int co, void* out,
                     hipStream_t s, OctantScatter osc, SkipAdd skip, PadRow pad, RowNorm ln, TileRange tr) {
    const bool planned = plan != nullptr;
    const bool all_tiles = tr.t0 == 0 && tr.nt < 0;
    if (!all_tiles && !planned) {
        set_error("MFMA conv: a tile range needs a plan");
        return TSP_ERR_INVALID;
    }
    if (ln.w && (!planned || !(co == 64 || co == 128) || odt != fdt || osc.cout || skip.cin)) {
        set_error("MFMA conv: a row norm needs a plan, co = 64 or 128 and output in the feature type "
                  "(co=%d)", co);
        return TSP_ERR_UNSUPPORTED;
    }
    const bool bn128 = co % 128 == 0;
    if (osc.cout && (!planned || osc.cout % (bn128 ? 64 : 32) != 0 || (int64_t)osc.cout * 8 != co)) {
        set_error("MFMA conv: an octant scatter needs a plan, co = 8 * cout and cout %% %d == 0 "
                  "(co=%d cout=%d)", bn128 ? 64 : 32, co, osc.cout);
        return TSP_ERR_UNSUPPORTED;
    }
    if (osc.oct && (osc.cout % 128 != 0 || !osc.oct_plan || osc.side != OctantScatter::EITHER || !all_tiles)) {
        set_error("MFMA conv: an octant plan needs cout %% 128 == 0 (cout=%d) and is run whole", osc.cout);
        return TSP_ERR_UNSUPPORTED;
    }
    if (osc.norm_silu && (!bn128 || (osc.cout != 64 && osc.cout != 128) || odt != fdt)) {
        set_error("MFMA conv: octant stores with the child norm need cout = 64 or 128, co %% 128 == 0 and "
                  "output in the feature type (co=%d cout=%d)", co, osc.cout);
        return TSP_ERR_UNSUPPORTED;
    }
    if (skip.cin && (!planned || skip.cin % 8 != 0 || co % (skip.cin / 8) != 0 || (co / (skip.cin / 8)) % 4 != 0)) {
        set_error("MFMA conv: a skip add needs a plan, cin %% 8 == 0 and co / (cin / 8) a multiple of 4 "
                  "(cin=%d co=%d)", skip.cin, co);
        return TSP_ERR_UNSUPPORTED;
    }
    // the slice DMA addresses feature rows with 32-bit byte offsets
    if (!halo_fits(n, ci)) {
        set_error("MFMA conv: n * ci * 2 = %lld bytes of features exceed the 4 GiB the LDS-staged "
                  "kernel addresses", (long long)(n * ci * 2));
        return TSP_ERR_UNSUPPORTED;
    }
    // grids that leave most of the chip idle, or a costly last round, take the small-grid kernel
    const int ncg = (ln.w && co == 128) || (osc.norm_silu && osc.cout == 128) ? 2 : 1;
    if (const int rgw = conv_split_pick(n, ci, co, ncg)) {
        auto* split = fdt == TSP_BF16 ? (rgw == 1 ? split_launch_bf16_1 : rgw == 2 ? split_launch_bf16_2 : split_launch_bf16_4)
                                      : (rgw == 1 ? split_launch_f16_1 : rgw == 2 ? split_launch_f16_2 : split_launch_f16_4);
        return split(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln, tr, ncg);
    }
    auto* fn64 = fdt == TSP_BF16 ? halo_launch_bf16_64 : halo_launch_f16_64;
    auto* fn = bn128 ? (fdt == TSP_BF16 ? halo_launch_bf16_128 : halo_launch_f16_128) : fn64;
    // With a plan, whole rounds of 128-channel units and the tiles left over as 64-channel units
    // (kernels where either width runs: not the row norms, which need whole rows in a workgroup)
    if (!all_tiles) return fn(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln, tr);
    if (planned && bn128 && !ln.w && !osc.norm_silu) {
        const int64_t t_split = column_split_tiles(ceil_div(n, HB_M), co / 128, cu_count());
        if (t_split > 0) {
            if (osc.oct) {   // an octant plan takes no column split
                osc.side = OctantScatter::OCTANTS;
                if (int st = fn(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln,
                                TileRange{}))
                    return st;
                osc.side = OctantScatter::PARENTS;
            }
            if (int st = fn(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln,
                            TileRange{0, t_split}))
                return st;
            return fn64(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln,
                        TileRange{t_split, -1});
        }
    }
    return fn(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad, ln, TileRange{});
}

}  // namespace tsp
