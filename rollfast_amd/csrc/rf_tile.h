// rf_tile.h -- the work units of quantization blocks of other sizes than 2048
// (adam8.py:243-391 takes any block_size; small blocks follow outliers more
// closely, large ones save scales), for k_adam8_tile (rf_tile_inst.hip), and
// of 2048-element blocks in lists too short for k_adam8 and leaves' partial
// last blocks, for the generic list.  Included by rf_device.h.
//
// Same execution model as k_adam8: a wave owns a span of up to
// TILE_SPAN = 1024 consecutive elements, lane l of chunk j the eight from
// j*512 + 8l, every access a 16-byte (params, grads) or 8-byte (codes) vector
// access, and the new moments stay in registers until the scales are known,
// so nothing is read twice.  Only the absmax reduction and the scales differ
// by block size:
//
//   KIND_QTILE  block sizes 8, 16, .. 512 (powers of two): a span holds
//               whole blocks, a block being 1 to 64 lanes of a chunk; one
//               scale per lane and chunk.
//   KIND_QWAVE  1024, and other multiples of 8 below it: a wave per block,
//               its last lanes idle.
//   KIND_QTEAM  multiples of 8 from 1032 to 4096: a workgroup per block, a
//               quarter of it per wave, the absmax meeting in LDS.  In the
//               generic list: blocks of up to 2048, one chunk per wave.
//
// Partial blocks (a leaf's last) take the same units, the lanes past the
// leaf's end masked.  The weight-decay mode and eps_root are resolved at run
// time by wave-uniform branches per chunk, and so are the dtypes in the
// instances with DT = DT_ANY; DT = RF_BF16 has bf16 params and grads (fewer
// registers and branches).
//
// Bound: HBM, with the latency of a wave's chunk next.  One GPU, a 202 M
// parameter bf16 layer (2.04 GB) in blocks of 256, nearest rounding: 435 us,
// 4.7 TB/s, 58 VALU instructions per element (the 2048-element kernel: 43;
// codes are scaled per element instead of through a per-block table, and the
// reduction and reciprocals come per chunk).  What led there: 6.63 ms with a
// workgroup per block, element accesses and two passes; 528 us with spans of
// 2048 elements without prefetch (747 us with it: the registers spill); 463
// us with spans of 1024, prefetch and the bf16 instance (545 us without
// that); 437 us with the mask-free WHOLE instance.
#pragma once

namespace rf {

// What a wave works on: code elements [base, base + len) of the leaf.
struct TileSpan {
    int64_t base;  // a multiple of 8
    int64_t blk0;  // the block of element base
    int32_t len;   // a multiple of 8, at most J chunks (0: nothing)
    int32_t rem;   // of these, elements of the leaf (the rest is padding)
    int32_t lg;    // log2 of the block size (3 .. 9) where the span holds whole blocks; 10: one block or a part of one
};

// One 512-element chunk in flight: codes, grads, params (16-byte words, the
// second of an array only for f32) and the old scales of the lane's block.
struct TileSlot {
    uint2 mc, vc;
    uint4 g[2], p[2];
    float sm, sv;
};

constexpr int32_t DT_ANY = -1;

// Element eo of the span at element `base` of an array of `size`-byte
// elements: a uniform base and a 32-bit lane offset.
template <typename T>
__device__ __forceinline__ RF_GLOBAL T* tile_ptr(const void* array, int64_t base, int32_t size, int32_t eo)
{
    return (RF_GLOBAL T*)((RF_GLOBAL uint8_t*)array + base * size + (uint32_t)(eo * size));
}

// Eight elements from eo (16-byte aligned).
__device__ __forceinline__ void tile_load8(uint4 (&w)[2], const void* array, int32_t dtype, int64_t base, int32_t eo)
{
    if (dtype == RF_F32) {
        const RF_GLOBAL uint4* q = tile_ptr<uint4>(array, base, 4, eo);
        w[0] = q[0];
        w[1] = q[1];
    } else {
        w[0] = ld_nt((const RF_GLOBAL uint4*)tile_ptr<uint4>(array, base, 2, eo));
    }
}

// The first nv (1 .. 7) of them; the others zero.
__device__ __forceinline__ void tile_load_some(uint4 (&w)[2], const void* base, int32_t dtype, int64_t e0, int32_t nv)
{
    uint32_t d[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (dtype == RF_F32) {
#pragma unroll
        for (int t = 0; t < 7; ++t)
            if (t < nv) d[t] = gld<uint32_t>(base, e0 + t);
    } else {
#pragma unroll
        for (int t = 0; t < 7; ++t)
            if (t < nv) d[t >> 1] |= (uint32_t)gld<uint16_t>(base, e0 + t) << (16 * (t & 1));
    }
    w[0] = make_uint4(d[0], d[1], d[2], d[3]);
    w[1] = make_uint4(d[4], d[5], d[6], d[7]);
}

__device__ __forceinline__ void tile_unpack8(const uint4 (&w)[2], int32_t dtype, float (&x)[8])
{
    if (dtype == RF_BF16) {
        raw8_unpack<uint16_t>(Raw8<uint16_t>{{w[0]}}, x);
    } else if (dtype == RF_F16) {
        raw8_unpack<_Float16>(Raw8<_Float16>{{w[0]}}, x);
    } else {
        raw8_unpack<float>(Raw8<float>{{w[0], w[1]}}, x);
    }
}

__device__ __forceinline__ void tile_clip8(const UnitCtx& c, int32_t dtype, float (&g)[8])
{
    if (dtype == RF_BF16) clip8<uint16_t>(c, g);
    else if (dtype == RF_F16) clip8<_Float16>(c, g);
    else clip8<float>(c, g);
}

// Issues chunk j's loads, unmasked where the chunk lies wholly inside the
// leaf (WHOLE: known to; else a wave-uniform test); otherwise lanes past the
// span or the leaf read as zero codes under a zero scale, zero grads and
// zero params.
template <int32_t DT, bool WHOLE>
__device__ __forceinline__ void tile_issue(TileSlot& s, const rf_adam8_leaf& L, const TileSpan& sp, int j, bool need_p)
{
    const int lane = threadIdx.x & (WAVE - 1);
    const int32_t eo = j * 512 + lane * 8;
    const int32_t pdt = DT == DT_ANY ? L.param_dtype : DT, gdt = DT == DT_ANY ? L.grad_dtype : DT;
    auto codes_and_scales = [&]() {
        s.mc = ld_nt((const RF_GLOBAL uint2*)tile_ptr<uint2>(L.mu, sp.base, 1, eo));
        s.vc = ld_nt((const RF_GLOBAL uint2*)tile_ptr<uint2>(L.nu, sp.base, 1, eo));
        const int64_t blk = sp.blk0 + (eo >> sp.lg);
        s.sm = load_scale(L.mu_scales, L.flags, blk);
        s.sv = load_scale(L.nu_scales, L.flags, blk);
    };
    if (WHOLE || sp.rem >= (j + 1) * 512) {
        codes_and_scales();
        tile_load8(s.g, L.grad, gdt, sp.base, eo);
        if (need_p) tile_load8(s.p, L.param, pdt, sp.base, eo);
        return;
    }
    s.mc = s.vc = make_uint2(0, 0);
    s.g[0] = s.g[1] = s.p[0] = s.p[1] = make_uint4(0, 0, 0, 0);
    s.sm = s.sv = 0.0f;
    if (eo < sp.len) codes_and_scales();
    const int32_t nv = sp.rem - eo;
    if (nv >= 8) {
        tile_load8(s.g, L.grad, gdt, sp.base, eo);
        if (need_p) tile_load8(s.p, L.param, pdt, sp.base, eo);
    } else if (nv > 0) {
        tile_load_some(s.g, L.grad, gdt, sp.base + eo, nv);
        if (need_p) tile_load_some(s.p, L.param, pdt, sp.base + eo, nv);
    }
}

// Max over the lanes of one block within a chunk: blocks of 2^lg elements
// are 2^(lg - 3) lanes (lg >= 9: the whole wave).  Every lane active; lg
// uniform.
__device__ __forceinline__ uint32_t tile_max(uint32_t x, int32_t lg)
{
    if (lg >= 4) x = max(x, dpp_u32<0xB1>(x));   // quad_perm [1,0,3,2]
    if (lg >= 5) x = max(x, dpp_u32<0x4E>(x));   // quad_perm [2,3,0,1]
    if (lg >= 6) x = max(x, dpp_u32<0x141>(x));  // row_half_mirror
    if (lg >= 7) x = max(x, dpp_u32<0x140>(x));  // row_mirror
    if (lg >= 8) {
        const uint32_t lo = max((uint32_t)__builtin_amdgcn_readlane(x, 0), (uint32_t)__builtin_amdgcn_readlane(x, 16));
        const uint32_t hi = max((uint32_t)__builtin_amdgcn_readlane(x, 32), (uint32_t)__builtin_amdgcn_readlane(x, 48));
        x = lg >= 9 ? max(lo, hi) : ((threadIdx.x & 32u) ? hi : lo);
    }
    return x;
}

// New params (or f32 updates) of a lane's eight elements; nv: how many exist.
__device__ __forceinline__ void tile_store8_f32(void* array, int64_t base, int32_t eo, int32_t nv,
                                                const float (&x)[8])
{
    if (nv >= 8) {
        RF_GLOBAL float4* q = tile_ptr<float4>(array, base, 4, eo);
        q[0] = make_float4(x[0], x[1], x[2], x[3]);
        q[1] = make_float4(x[4], x[5], x[6], x[7]);
    } else {
#pragma unroll
        for (int t = 0; t < 7; ++t)
            if (t < nv) gst<float>(array, base + eo + t, x[t]);
    }
}

__device__ __forceinline__ void tile_store8_h16(void* array, int64_t base, int32_t eo, int32_t nv,
                                                const uint32_t (&w)[4])
{
    if (nv >= 8) {
        st_nt(tile_ptr<uint4>(array, base, 2, eo), make_uint4(w[0], w[1], w[2], w[3]));
    } else {
#pragma unroll
        for (int t = 0; t < 7; ++t)
            if (t < nv) gst<uint16_t>(array, base + eo + t, (uint16_t)(w[t >> 1] >> (16 * (t & 1))));
    }
}

// Weight decay and learning rate of eight updates, the mode a uniform branch.
__device__ __forceinline__ void tile_decay8(const KHp& h, int32_t wd_mode, float (&u)[8], const float (&p)[8])
{
    if (wd_mode == WD_BF16) decay_and_scale8<WD_BF16>(h, u, p);
    else if (wd_mode == WD_F16) decay_and_scale8<WD_F16>(h, u, p);
    else if (wd_mode == WD_F32) decay_and_scale8<WD_F32>(h, u, p);
    else decay_and_scale8<WD_OFF>(h, u, p);
}

// The codes of one chunk's moments under scales sm, sv (fast range), nearest.
__device__ __forceinline__ void tile_code8(const uint8_t* lds, const float (&m)[8], const float (&v)[8], float sm,
                                           float sv, uint2& wm, uint2& wv)
{
    const float rsm = 1.0f / sm, rsv = 1.0f / sv;
    // batched phases, as in unit_qfast: 16 independent LDS reads in flight
    float nm[8], nv[8], tm[8], tv[8];
    uint32_t cm[8], cv[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        nm[t] = div_by_scale(m[t], sm, rsm);
        nv[t] = div_by_scale(v[t], sv, rsv);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        cm[t] = cand_signed(lds, nm[t]);
        cv[t] = cand_unsigned(lds, nv[t]);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        tm[t] = *(const float*)(lds + L_TS + cm[t] * 4u);
        tv[t] = *(const float*)(lds + L_TU + cv[t] * 4u);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        cm[t] += nm[t] >= tm[t] ? 1u : 0u;
        cv[t] += nv[t] >= tv[t] ? 1u : 0u;
    }
    wm.x = pack4_u8(cm[0], cm[1], cm[2], cm[3]);
    wm.y = pack4_u8(cm[4], cm[5], cm[6], cm[7]);
    wv.x = pack4_u8(cv[0], cv[1], cv[2], cv[3]);
    wv.y = pack4_u8(cv[4], cv[5], cv[6], cv[7]);
}

// The same with stochastic rounding from the packed source (unit_qfast's
// packed branch): main halves for four elements of both moments at a time,
// whole words where a draw stays open.
__device__ __forceinline__ void tile_code8_packed(const UnitCtx& c, uint64_t e0, const float (&m)[8],
                                                  const float (&v)[8], float sm, float sv, uint2& wm, uint2& wv)
{
    const float* cbs = (const float*)(c.lds + L_CBS);
    const float* cbu = (const float*)(c.lds + L_CBU);
    const float4* srs = (const float4*)(c.lds + L_SRS);
    const float4* sru = (const float4*)(c.lds + L_SRU);
    const float rsm = 1.0f / sm, rsv = 1.0f / sv;
    uint32_t pm2[2], pv2[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
        uint32_t ym[2], yv[2], um[4], uv[4], cm[4], cv[4];
        float nm[4], nv[4], pm[4], pv[4];
#pragma unroll
        for (int pr = 0; pr < 2; ++pr)
            packed_moment_block(c.kmu0, c.kmu1, e0 + 4 * hh + 2 * pr, false, ym[pr], yv[pr]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            nm[t] = div_by_scale(m[4 * hh + t], sm, rsm);
            nv[t] = div_by_scale(v[4 * hh + t], sv, rsv);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            um[t] = cand_signed(c.lds, nm[t]);
            uv[t] = cand_unsigned(c.lds, nv[t]);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            pm[t] = sr_upper(cbs, srs, um[t], nm[t]);
            pv[t] = sr_upper(cbu, sru, uv[t], nv[t]);
        }
        uint64_t open = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            cm[t] = packed_sr_main(um[t], pm[t], half16(ym[t >> 1], t), open);
            cv[t] = packed_sr_main(uv[t], pv[t], half16(yv[t >> 1], t), open);
        }
        if (__builtin_expect(open != 0, 0)) {
            uint32_t zm[2], zv[2];
#pragma unroll
            for (int pr = 0; pr < 2; ++pr)
                packed_moment_block(c.kmu0, c.kmu1, e0 + 4 * hh + 2 * pr, true, zm[pr], zv[pr]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                cm[t] = sr_decide(um[t], pm[t], (half16(ym[t >> 1], t) << 16) | half16(zm[t >> 1], t));
                cv[t] = sr_decide(uv[t], pv[t], (half16(yv[t >> 1], t) << 16) | half16(zv[t >> 1], t));
            }
        }
        pm2[hh] = pack4_u8(cm[0], cm[1], cm[2], cm[3]);
        pv2[hh] = pack4_u8(cv[0], cv[1], cv[2], cv[3]);
    }
    wm = make_uint2(pm2[0], pm2[1]);
    wv = make_uint2(pv2[0], pv2[1]);
}

// One moment's stochastically rounded codes from a stream of its own (fed
// words, or jax.random.bits under k0, k1).
template <bool SECOND>
__device__ __forceinline__ uint2 tile_code8_stream(const UnitCtx& c, const uint32_t* bits, int64_t e0,
                                                   const float (&x)[8], float s)
{
    const float* cb = (const float*)(c.lds + (SECOND ? L_CBU : L_CBS));
    const float4* rec = (const float4*)(c.lds + (SECOND ? L_SRU : L_SRS));
    const float rs = 1.0f / s;
    uint32_t b[8], cc[8];
    float n[8];
    if (c.fed) {
        load8_u32(bits, e0, b);
    } else {
        const uint32_t k0 = SECOND ? c.knu0 : c.kmu0, k1 = SECOND ? c.knu1 : c.kmu1;
#pragma unroll
        for (int t = 0; t < 8; ++t) b[t] = jax_bits(k0, k1, (uint64_t)(e0 + t));
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) n[t] = div_by_scale(x[t], s, rs);
#pragma unroll
    for (int t = 0; t < 8; ++t) cc[t] = SECOND ? cand_unsigned(c.lds, n[t]) : cand_signed(c.lds, n[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) cc[t] = sr_code(cb, rec, cc[t], n[t], b[t]);
    return make_uint2(pack4_u8(cc[0], cc[1], cc[2], cc[3]), pack4_u8(cc[4], cc[5], cc[6], cc[7]));
}

// One moment's codes by the literal search (code_literal), whatever the
// scale: the eight searches advance together, so a step of theirs is one LDS
// round trip; the draws are made one at a time, which keeps this rare path
// short.
template <bool MSR, bool SECOND>
__device__ __forceinline__ uint2 tile_code8_literal(const UnitCtx& c, const rf_adam8_leaf& L, int64_t e0,
                                                    const float (&x)[8], float s)
{
    const float* cb = (const float*)(c.lds + (SECOND ? L_CBU : L_CBS));
    uint32_t bits[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (MSR) {
#pragma unroll 1
        for (int t = 0; t < 8; ++t) {
#pragma unroll
            for (int k = 0; k < 7; ++k) bits[k] = bits[k + 1];
            bits[7] = SECOND ? nu_bits1(c, L, e0 + t) : mu_bits1(c, L, e0 + t);
        }
    }
    const float lo = cb[0], hi = cb[255];
    float n[8];
    uint32_t pos[8];
    bool nan[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        n[t] = x[t] / s;  // IEEE division
        nan[t] = n[t] != n[t];
        n[t] = n[t] < lo ? lo : n[t];
        n[t] = n[t] > hi ? hi : n[t];
        pos[t] = 0;
    }
#pragma unroll 1
    for (uint32_t step = 128; step >= 1; step >>= 1) {
#pragma unroll
        for (int t = 0; t < 8; ++t) pos[t] += cb[pos[t] + step - 1] < n[t] ? step : 0u;
    }
    uint32_t code[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const uint32_t ui = pos[t], li = ui > 0 ? ui - 1 : 0;
        const float lv = cb[li], uv = cb[ui];
        bool upper;
        if constexpr (MSR) {
            const float den = uv - lv;
            float p = den > 0.0f ? (n[t] - lv) / den : 0.0f;
            p = p < 0.0f ? 0.0f : (p > 1.0f ? 1.0f : p);
            upper = uniform_from_bits(bits[t]) < p;
        } else {
            upper = fabsf(uv - n[t]) < fabsf(n[t] - lv);
        }
        code[t] = nan[t] ? 254u : upper ? ui : li;
    }
    return make_uint2(pack4_u8(code[0], code[1], code[2], code[3]), pack4_u8(code[4], code[5], code[6], code[7]));
}

// Each block's absmax bits, from the lanes' own, in all of the block's lanes.
// `team`: the workgroup's four waves hold the parts of one block, whose bits
// meet in `red`; called by every wave.
template <bool WHOLE, int J>
__device__ __forceinline__ void tile_block_max(uint32_t (&am)[J], uint32_t (&av)[J], int32_t lg, bool team,
                                               uint32_t* red)
{
    if (lg < 10) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            am[j] = tile_max(am[j], lg);
            av[j] = tile_max(av[j], lg);
        }
        return;
    }
#pragma unroll
    for (int j = 1; j < J; ++j) {
        am[0] = max(am[0], am[j]);
        av[0] = max(av[0], av[j]);
    }
    am[0] = wave_max_u32(am[0]);
    av[0] = wave_max_u32(av[0]);
    if (!WHOLE && team) {
        const int w = (int)uniform_u32(threadIdx.x / WAVE);
        if ((threadIdx.x & (WAVE - 1)) == 0) {
            red[2 * w] = am[0];
            red[2 * w + 1] = av[0];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < WAVES_PER_WG; ++k) {
            am[0] = max(am[0], red[2 * k]);
            av[0] = max(av[0], red[2 * k + 1]);
        }
        __syncthreads();  // red is free again
    }
#pragma unroll
    for (int j = 1; j < J; ++j) {
        am[j] = am[0];
        av[j] = av[0];
    }
}

// The direction of eight elements, Nesterov's by a uniform branch.
template <bool EXACT>
__device__ __forceinline__ void tile_direction8(const KHp& h, bool nest, const float (&m)[8], const float (&v)[8],
                                                const float (&g)[8], float (&u)[8])
{
    if (nest) {
#pragma unroll
        for (int t = 0; t < 8; ++t) u[t] = adam_direction<true, EXACT>(h, m[t], v[t], g[t]);
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) u[t] = adam_direction<false, EXACT>(h, m[t], v[t], g[t]);
    }
}

// One span.  `team`: the workgroup's four waves hold the parts of one block
// (`red`: 8 words of LDS where their absmax bits meet); every wave calls it.
// `have0`: sl[0] already holds the span's chunk 0; `next`: the wave's next
// span, of the same leaf, whose chunk 0 is loaded into sl[0] while this one
// is requantized (len 0: none).  WHOLE: the span is TILE_SPAN elements of
// the leaf, and so is `next`.  That instance has no masks: every path through
// it issues the same number of memory operations, so the compiler's waits
// for a chunk's loads leave the later stores in flight.  Nor has it the
// literal search: it returns false for a span with a tiny, infinite or NaN
// scale, its params stored, codes and scales as they were, which the caller
// gives to the other instance with `codes_only` (true: the params or updates
// are not written again).
// J: the span's chunks at most.
template <int32_t DT, bool APPLY, bool MSR, bool PSR, bool EXACT, bool WHOLE, int J>
__device__ __forceinline__ bool unit_tile(const UnitCtx& c, const rf_adam8_leaf& L, const KHp& h, bool nest, bool team,
                                          const TileSpan& sp, TileSlot (&sl)[2], bool have0, const TileSpan& next,
                                          uint32_t* red, bool codes_only = false)
{
    const int lane = threadIdx.x & (WAVE - 1);
    const int32_t pdt = DT == DT_ANY ? L.param_dtype : DT, gdt = DT == DT_ANY ? L.grad_dtype : DT;
    const bool need_p = APPLY || c.wd_mode != WD_OFF;
    // The learning-rate-folded direction (flr_setup) under the same
    // conditions as in k_adam8.
    bool flr = false;
    if constexpr (APPLY && !EXACT)
        flr = !nest && h.flr && h.er2 == 0.0f && pdt == RF_BF16 && (c.wd_mode == WD_BF16 || c.wd_mode == WD_OFF);
    const float* cbs = (const float*)(c.lds + L_CBS);
    const float* cbu = (const float*)(c.lds + L_CBU);

    float m[J][8], v[J][8];
    uint32_t am[J], av[J];
    uint64_t odd = 0;  // lanes whose old scales are not finite
    if (!have0 && (WHOLE || sp.len > 0)) tile_issue<DT, WHOLE>(sl[0], L, sp, 0, need_p);
#pragma unroll
    for (int j = 0; j < J; ++j) {
        am[j] = av[j] = 0;
#pragma unroll
        for (int t = 0; t < 8; ++t) m[j][t] = v[j][t] = 0.0f;
        if (!WHOLE && j * 512 >= sp.len) continue;
        if (j + 1 < J && (WHOLE || (j + 1) * 512 < sp.len))
            tile_issue<DT, WHOLE>(sl[(j + 1) & 1], L, sp, j + 1, need_p);
        if (WHOLE && j + 1 == J && next.len > 0) tile_issue<DT, true>(sl[0], L, next, 0, need_p);  // slot 0 is free
        const TileSlot& s = sl[j & 1];
        const int32_t eo = j * 512 + lane * 8;
        const int64_t e0 = sp.base + eo;
        const int32_t nv = WHOLE ? 8 : sp.rem - eo;
        odd |= __builtin_amdgcn_ballot_w64((__float_as_uint(s.sm) & 0x7FFFFFFFu) >= 0x7F800000u ||
                                           (__float_as_uint(s.sv) & 0x7FFFFFFFu) >= 0x7F800000u);
        float g[8], p[8], u[8], sum[8];
        tile_unpack8(s.g, gdt, g);
        tile_clip8(c, gdt, g);
        if (need_p) {
            tile_unpack8(s.p, pdt, p);
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t) p[t] = 0.0f;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const uint32_t cm = ((t < 4 ? s.mc.x : s.mc.y) >> (8 * (t & 3))) & 0xFFu;
            const uint32_t cv = ((t < 4 ? s.vc.x : s.vc.y) >> (8 * (t & 3))) & 0xFFu;
            ema(h, cbs[cm] * s.sm, cbu[cv] * s.sv, g[t], m[j][t], v[j][t]);
        }
        if (!WHOLE && sp.rem < (j + 1) * 512) {
            // padding past the leaf's end has zero moments (adam8.py:137-141)
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if (t >= nv) m[j][t] = v[j][t] = 0.0f;
            }
        }
        float amf = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            amf = fmaxf(amf, fabsf(m[j][t]));
            av[j] = max(av[j], __float_as_uint(v[j][t]));  // v >= 0; NaN-propagating
        }
        am[j] = __float_as_uint(amf);

        if (flr) {
            if (c.wd_mode == WD_BF16) {
#pragma unroll
                for (int t = 0; t < 8; ++t) sum[t] = __builtin_fmaf(h.wdl, p[t], p[t]);
            } else {
#pragma unroll
                for (int t = 0; t < 8; ++t) sum[t] = p[t];
            }
#pragma unroll
            for (int t = 0; t < 8; ++t)
                sum[t] = __builtin_fmaf(
                    m[j][t],
                    __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_sqrtf(v[j][t]), h.k1l, h.k2l)), sum[t]);
            // near cancellation: the IEEE direction in the reference's order (unit_qfast)
            float dmax = 0.0f;
#pragma unroll
            for (int t = 0; t < 8; ++t) dmax = fmaxf(dmax, __builtin_fmaf(-FLR_CANCEL, fabsf(sum[t]), fabsf(p[t])));
            if (__builtin_amdgcn_ballot_w64(dmax > 0.0f) != 0) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    if (__builtin_fmaf(-FLR_CANCEL, fabsf(sum[t]), fabsf(p[t])) > 0.0f)
                        sum[t] = p[t] + decay_and_scale(h, adam_direction<false, true>(h, m[j][t], v[j][t], g[t]), p[t],
                                                        c.wd_mode);
                }
            }
        } else {
            tile_direction8<EXACT>(h, nest, m[j], v[j], g, u);
            tile_decay8(h, c.wd_mode, u, p);
#pragma unroll
            for (int t = 0; t < 8; ++t) sum[t] = p[t] + u[t];
            if constexpr (APPLY && !EXACT) {
                if (cancel_lanes8(sum, u) != 0) {
                    float ue[8];
                    tile_direction8<true>(h, nest, m[j], v[j], g, ue);
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        if (cancels(sum[t], u[t])) sum[t] = p[t] + decay_and_scale(h, ue[t], p[t], c.wd_mode);
                    }
                }
            }
        }
        if (nv > 0 && (WHOLE || !codes_only)) {
            if constexpr (!APPLY) {
                tile_store8_f32(L.updates, sp.base, eo, nv, u);
            } else if (pdt == RF_F32) {
                tile_store8_f32(L.param, sp.base, eo, nv, sum);
            } else {
                uint32_t w[4];
                if (PSR && pdt == RF_BF16) {
                    uint32_t rb[8];
                    if (c.fed && nv < 8) {  // the fed words end with the leaf
#pragma unroll
                        for (int t = 0; t < 8; ++t) rb[t] = t < nv ? gld<uint32_t>(L.param_bits, e0 + t) : 0u;
                    } else {
                        param_bits8(c, L, e0, rb);
                    }
#pragma unroll
                    for (int t = 0; t < 8; t += 2)
                        w[t / 2] = pack_hi16x2(sr_bf16_hi(sum[t], rb[t]), sr_bf16_hi(sum[t + 1], rb[t + 1]));
                } else if (pdt == RF_BF16) {
#pragma unroll
                    for (int t = 0; t < 8; t += 2) w[t / 2] = pack_bf16x2_rne(sum[t], sum[t + 1]);
                } else {
#pragma unroll
                    for (int t = 0; t < 8; t += 2) w[t / 2] = pack_f16x2_rne(sum[t], sum[t + 1]);
                }
                tile_store8_h16(L.param, sp.base, eo, nv, w);
            }
        }
    }

    // Each block's absmax in all of its lanes.  Old scales that are not
    // finite make the block slow (below) wherever it is.
    const int32_t lg = sp.lg;
    if (odd != 0) {
#pragma unroll
        for (int j = 0; j < J; ++j) av[j] = 0x7FFFFFFFu;
    }
    tile_block_max<WHOLE, J>(am, av, lg, team, red);
    float sm[J], sv[J];
    uint64_t slow = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        sm[j] = scale_from_absmax_bits(am[j]);
        sv[j] = scale_from_absmax_bits(av[j]);
        slow |= __builtin_amdgcn_ballot_w64(!(block_is_fast(am[j], sm[j]) && block_is_fast(av[j], sv[j])));
    }
    if constexpr (WHOLE) {
        if (__builtin_expect(slow != 0, 0)) return false;
    } else if (__builtin_expect(slow != 0, 0)) {
        // A block of the span with a tiny, infinite or NaN scale (in a team:
        // the workgroup's block, so that every wave is here): the span's
        // moments, still in registers, are coded by the literal search under
        // the reference's NaN-propagating absmax (adam8.py:142).  2^24 bf16
        // elements, nearest, one block in 16 of that kind, one GPU: blocks of
        // 8 116 us, of 256 70, of 4096 96; 1,139, 88 and 503 with one wave
        // recomputing the span's blocks one after the other.  The same code
        // in the WHOLE instance too cost spans without such blocks 4 %.
#pragma unroll
        for (int j = 0; j < J; ++j) {
            am[j] = av[j] = 0;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                am[j] = max(am[j], __float_as_uint(m[j][t]) & 0x7FFFFFFFu);
                av[j] = max(av[j], __float_as_uint(v[j][t]));
            }
        }
        tile_block_max<WHOLE, J>(am, av, lg, team, red);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int32_t eo = j * 512 + lane * 8;
            if (eo >= sp.len) continue;
            const float s1 = scale_from_absmax_bits(am[j]), s2 = scale_from_absmax_bits(av[j]);
            st_nt(tile_ptr<uint2>(L.mu, sp.base, 1, eo), tile_code8_literal<MSR, false>(c, L, sp.base + eo, m[j], s1));
            st_nt(tile_ptr<uint2>(L.nu, sp.base, 1, eo), tile_code8_literal<MSR, true>(c, L, sp.base + eo, v[j], s2));
            if (!team || threadIdx.x < WAVE) {
                const int64_t blk = sp.blk0 + (eo >> lg);
                store_scale(L.mu_scales, L.flags, blk, s1);
                store_scale(L.nu_scales, L.flags, blk, s2);
            }
        }
        return true;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int32_t eo = j * 512 + lane * 8;
        if (!WHOLE && j * 512 >= sp.len) continue;
        if (WHOLE || eo < sp.len) {
            const int64_t e0 = sp.base + eo;
            uint2 wm, wv;
            if constexpr (MSR) {
                if (c.packed) {
                    tile_code8_packed(c, (uint64_t)e0, m[j], v[j], sm[j], sv[j], wm, wv);
                } else {
                    wm = tile_code8_stream<false>(c, L.mu_bits, e0, m[j], sm[j]);
                    wv = tile_code8_stream<true>(c, L.nu_bits, e0, v[j], sv[j]);
                }
            } else {
                tile_code8(c.lds, m[j], v[j], sm[j], sv[j], wm, wv);
            }
            st_nt(tile_ptr<uint2>(L.mu, sp.base, 1, eo), wm);
            st_nt(tile_ptr<uint2>(L.nu, sp.base, 1, eo), wv);
            // Every lane of a block stores its (equal) scales: one store
            // instruction either way, and no branch around it.
            if (WHOLE || !team || threadIdx.x < WAVE) {
                const int64_t blk = sp.blk0 + (eo >> lg);
                store_scale(L.mu_scales, L.flags, blk, sm[j]);
                store_scale(L.nu_scales, L.flags, blk, sv[j]);
            }
        }
    }
    return true;
}

// The part of element range [lo, hi) of the leaf's code array as a span.
__device__ __forceinline__ TileSpan tile_span(const rf_adam8_leaf& L, int64_t lo, int64_t hi, int64_t blk0, int32_t lg)
{
    TileSpan sp;
    sp.base = lo;
    sp.blk0 = blk0;
    sp.len = (int32_t)max((int64_t)0, hi - lo);
    sp.rem = (int32_t)max((int64_t)0, min((int64_t)sp.len, L.size - lo));
    sp.lg = lg;
    return sp;
}

// The calling wave's part of block blk taken by the workgroup's four waves
// (KIND_QTEAM): a quarter, rounded up to whole lanes' elements.
__device__ __forceinline__ TileSpan team_span(const rf_adam8_leaf& L, int64_t blk)
{
    const int64_t bs = L.block_size;
    const int64_t quarter = (bs / 8 + WAVES_PER_WG - 1) / WAVES_PER_WG * 8;
    const int64_t lo = min(bs, (int64_t)uniform_u32(threadIdx.x / WAVE) * quarter);
    return tile_span(L, blk * bs + lo, blk * bs + min(bs, lo + quarter), blk, 10);
}

}  // namespace rf
