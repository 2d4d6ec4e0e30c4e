// rf_tile_inst.hip -- k_adam8_tile, the step kernel of the leaves whose blocks
// are not 2048 elements (rf_tile.h), instantiated for one (APPLY, MSR, EXACT)
// combination, as rf_adam8_inst.hip does k_adam8.
#include "rf_device.h"

#if !defined(RFI_APPLY) || !defined(RFI_MSR) || !defined(RFI_EXACT)
#error "build with -DRFI_APPLY=0|1 -DRFI_MSR=0|1 -DRFI_EXACT=0|1"
#endif

#define RF_PICK_NAME2(a, m, e) rf_pick_tile_a##a##_m##m##_e##e
#define RF_PICK_NAME(a, m, e) RF_PICK_NAME2(a, m, e)

// Waves per SIMD the tile kernel is register-allocated for.
#ifndef RF_TILE_WAVES_PER_EU
#define RF_TILE_WAVES_PER_EU 3
#endif

namespace rf {

// The tile list: its leading KIND_QTEAM units a workgroup each, then a wave
// per unit in runs of h.run, as in k_adam8.
template <int32_t DT, bool APPLY, bool MSR, bool PSR, bool EXACT>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(RF_TILE_WAVES_PER_EU))) void k_adam8_tile(
    const rf_adam8_leaf* __restrict__ leaves, const Seg* __restrict__ segs, int64_t total_units, KHp h,
    const uint4* __restrict__ tables)
{
    constexpr int TJ = (int)(TILE_SPAN / 512);
    constexpr uint32_t LDS_TABLES = MSR ? SEARCH_BYTES : TABLE_BYTES;
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_TABLES];
    __shared__ uint32_t red[2 * WAVES_PER_WG];
    stage_tables<LDS_TABLES>(lds, tables);
    const int64_t wave = (int64_t)blockIdx.x * WAVES_PER_WG + uniform_u32(threadIdx.x / WAVE);
    const int64_t nwaves = (int64_t)gridDim.x * WAVES_PER_WG;
    if (gate_rejects(h)) {
        reject_units<APPLY>(leaves, segs, total_units, wave, nwaves);
        return;
    }
    UnitCtx c;
    c.lds = lds;
    c.wtab = nullptr;
    c.xbuf = nullptr;
    c.fed = (h.flags & RF_FED_BITS) != 0;
    c.packed = !c.fed && (h.flags & RF_PACKED_BITS) != 0;
    c.zero = false;
    c.mpart = nullptr;
    c.mbase = 0;
    clip_context(c, h);
    c.wd_mode = WD_OFF;
    c.kmu0 = c.kmu1 = c.knu0 = c.knu1 = c.kp0 = c.kp1 = 0;
    const bool nest = (h.flags & RF_NESTEROV) != 0;
    int32_t s = 0, cur_leaf = -1;
    const int32_t nseg = segs[0].nseg;
    const int64_t nlead = segs[0].lead;
    rf_adam8_leaf L;
    KHp hl = h;
    flr_setup(hl);
    // Makes unit u's segment current; units in the same segment as the last
    // one need no load.
    Seg sg{};
    int64_t seg_end = -1;
    auto seek = [&](int64_t u) {
        if (u < seg_end) return;
        s = seek_seg(segs, nseg, s, u);
        sg = segs[s];
        seg_end = segs[s + 1].unit_start;
        if (sg.leaf != cur_leaf) {
            cur_leaf = sg.leaf;
            L = leaves[cur_leaf];
            if (h.groups != nullptr) {
                group_hparams(hl, h, L);
                flr_setup(hl);
            }
            leaf_context<true>(c, L, hl, MSR, PSR);
        }
    };
    // Wave unit u of the current segment as a span.
    auto span = [&](int64_t u) {
        const int64_t idx = sg.first + (u - sg.unit_start);
        const int64_t bs = L.block_size;
        if (sg.kind != KIND_QTILE) return tile_span(L, idx * bs, idx * bs + bs, idx, 10);
        const int32_t lg = 31 - __builtin_clz((uint32_t)bs);
        const int64_t total = (max((int64_t)1, L.size) + bs - 1) >> lg << lg;
        return tile_span(L, idx * TILE_SPAN, min(total, idx * TILE_SPAN + TILE_SPAN), idx << (10 - lg), lg);
    };
    for (int64_t q = blockIdx.x; q < nlead; q += gridDim.x) {
        seek(q);
        TileSlot own[2];
        unit_tile<DT, APPLY, MSR, PSR, EXACT, false, TJ>(
            c, L, hl, nest, true, team_span(L, sg.first + (q - sg.unit_start)), own, false, TileSpan{}, red);
    }
    TileSlot sl[2];
    bool have0 = false;  // sl[0] holds chunk 0 of unit u
    const int64_t units = total_units - nlead;
    const int64_t run = h.run;
    const int64_t nruns = (units + run - 1) / run;
    for (int64_t r = wave; r < nruns; r += nwaves) {
        const int64_t u_end = min(r * run + run, units);
        for (int64_t u = r * run; u < u_end; ++u) {
            seek(nlead + u);
            const TileSpan sp = span(nlead + u);
            const bool whole = sp.rem == TILE_SPAN;
            // a whole next span of the same leaf is prefetched over a whole
            // span (not at runtime dtypes, whose slots would spill)
            const int64_t un = u + 1 < u_end ? u + 1 : (r + nwaves) * run;
            TileSpan next{};
            if (DT != DT_ANY && whole && un < units && nlead + un < seg_end) {
                next = span(nlead + un);
                if (next.rem < TILE_SPAN) next.len = 0;
            }
            const bool done =
                whole && unit_tile<DT, APPLY, MSR, PSR, EXACT, true, TJ>(c, L, hl, nest, false, sp, sl, have0, next, red);
            if (!done)  // a short span, or the codes of one with a slow block (the next one's chunk is loaded anew)
                unit_tile<DT, APPLY, MSR, PSR, EXACT, false, TJ>(c, L, hl, nest, false, sp, sl, false, TileSpan{}, red,
                                                                 whole);
            have0 = done && next.len > 0;
        }
    }
}

template <int32_t DT>
static adam_kernel_t pick(bool psr)
{
    constexpr bool A = RFI_APPLY != 0, M = RFI_MSR != 0, E = RFI_EXACT != 0;
    if constexpr (A) {
        if (psr) return &k_adam8_tile<DT, A, M, true, E>;
    }
    return &k_adam8_tile<DT, A, M, false, E>;
}

// bf16: every leaf of the list has bf16 params and grads
adam_kernel_t RF_PICK_NAME(RFI_APPLY, RFI_MSR, RFI_EXACT)(bool bf16, bool psr)
{
    return bf16 ? pick<RF_BF16>(psr) : pick<DT_ANY>(psr);
}

}  // namespace rf
