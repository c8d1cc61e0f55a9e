// Neighbour search over the cell tables (neighborhood_green.comp:57-86). Every
// particle meets the candidates of its search box in the reference order (z,
// then y, then x, then the particles of a cell in sorted order), several at a
// time; a wave ballot turns the accepted ones into consecutive output slots, so
// every row keeps the sequential order.
//
// Modes: COUNT writes each row's length, FILL writes the rows at the offsets
// of the scanned counts, clamped to the pair capacity the way the sequential
// schedule fills a bounded list: entries whose slot in the full list is at or
// beyond the capacity are dropped (neighbor_add.glsl:22-23). PAD does both in
// one walk: it writes every row into a fixed-stride slot of its own (stride =
// pair capacity / current particles) and counts it; when no row outgrew its
// slot and the list fits the capacity (the normal case), the rows are then
// packed into the list, and otherwise the exact COUNT-less FILL walk runs
// (the counts of PAD are the counts of COUNT). The choice is made on the
// device, so the substep needs no host synchronisation.
//
// With SPREAD the walk also carries kernel_width.comp:22-56: every entry of
// the (clamped) list spreads the particle's original kernel width to the
// neighbour (atomicMax, order-free; skipped when a plain load already shows a
// value at least as large, which is exact because the stored values only grow
// during the walk), and only the entries within the
// particle's cutoff are written, which is the list the spreading pass of the
// reference leaves behind (kernel_width.comp:54-60). The full list is then
// never materialised: COUNT counts both lists, FILL writes the short one.
#include "scene.h"

namespace apbf {

struct WalkArgs {
    float range_scale;
    GridDesc g;
    int on_target;  // spreading: kernel width from max(radius, target radius)
    uint32_t pcap;
    uint32_t stride;        // PAD, and FILL after PAD: nonzero (the slot stride is slot_stride())
    const uint32_t* gate;   // FILL after PAD: the count block (C_FALLBACK, C_ROWFIX); null otherwise
    unsigned long long* cand;  // COUNT: when set, += the candidates the walk tests (a diagnostic)
    SegmentTable seg;       // a packed batch (SEG walks): each particle's grid and cell block
};

enum WalkMode { WALK_COUNT = 0, WALK_FILL = 1, WALK_PAD = 2 };

// Entries per particle slot in the PAD layout: the pair capacity shared by the
// current particles (not by the particle capacity), so slots are as wide as
// the list allows (at most 2^26: a group's slots are indexed in 32 bits). Every
// kernel of one pair build reads the same particle count, so they agree on it.
__device__ __forceinline__ uint32_t slot_stride(uint32_t pcap, uint32_t n) {
    return min(pcap / (n ? n : 1u), 1u << 26);
}

// Inclusive scan over the 64 lanes of a wavefront (every lane active) of an
// associative, commutative op with identity 0 on unsigned values (sum, max):
// DPP row shifts inside each 16-lane row, then the row totals by readlane.
template <typename Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, Op op) {
    constexpr int ROW_SHR1 = 0x111, ROW_SHR2 = 0x112, ROW_SHR4 = 0x114, ROW_SHR8 = 0x118;
    auto shr = [](uint32_t x, auto ctrl) {  // lanes whose source leaves the row read 0
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, false);
    };
    v = op(v, shr(v, std::integral_constant<int, ROW_SHR1>{}));
    v = op(v, shr(v, std::integral_constant<int, ROW_SHR2>{}));
    v = op(v, shr(v, std::integral_constant<int, ROW_SHR4>{}));
    v = op(v, shr(v, std::integral_constant<int, ROW_SHR8>{}));
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
    const uint32_t r1 = op(r0, (uint32_t)__builtin_amdgcn_readlane((int)v, 31));
    const uint32_t r2 = op(r1, (uint32_t)__builtin_amdgcn_readlane((int)v, 47));
    const uint32_t row = (threadIdx.x & 63u) >> 4;
    const uint32_t carry = row == 0u ? 0u : (row == 1u ? r0 : (row == 2u ? r1 : r2));
    return op(v, carry);
}

// Wave-uniform copy of lane k's value (v_readlane into a scalar register).
template <typename T>
__device__ __forceinline__ T lane_value(T v, int k) {
    static_assert(sizeof(T) == 4, "32-bit values");
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}

// The walk takes a group of 64 / L consecutive particles per wavefront. The
// particles are sorted by cell, so consecutive ones search nearly the same
// cells: the wave enumerates the cells of their common search box once, in the
// reference's order (x fastest, then y, then z), as one stream of candidates,
// keeps the candidates that some particle of the group may reach in LDS, and
// tests them L at a time, each against every particle of the group
// (lane = group size * candidate + particle). Every particle meets its
// candidates in its own walk order, because the cells of its own box come in
// the same order in the common one.
//
// Exactness:
//  * Culling: the distance from a candidate to the group's bounding box is
//    formed by the same rounded operations as its distance to a particle.
//    They are monotone, so a candidate beyond the group's largest range is in
//    range of none of its particles.
//  * A candidate of the common box that lies outside the particle's own box
//    must not be accepted. An accepted candidate closer than t_inner (the
//    range less a margin above every rounding of the box's corners) lies inside
//    the own box, because grid_cell is monotone; the few beyond it have their
//    cell compared. Boxes may pass the grid's end, where cells alias, as long
//    as the common box is at most the grid wide: every cell is then visited
//    once.
//  * The kept test's fixed-point distance differs from the world-space one by
//    the rounding of the coordinates only. Below t_klo and above t_khi (the cut
//    less and plus a margin above that rounding) both agree; between them the
//    fixed-point test itself runs.
// Particles whose own box is wider than the grid (it visits cells twice), or
// whose range is negative, infinite or NaN, walk their own box alone.
//
// What bounds it: VALU issue. On a settled adaptive drop (1.1 M particles, 166
// pairs in range and 60 kept per particle) a launch with 8 lanes, the rule's there,
// tests 572 candidates per particle in 1.49 ms and 0.79 G wavefront VALU
// instructions, 88% of the issue rate; with 4 lanes 776 candidates take 1.44 ms,
// 0.79 G and 90%: about 27 per test of 64 pairs, a quarter of the total for the
// spreading's exact evaluations, a third for the candidates' look-up and
// staging. While a drop hits the pool (202 pairs in range) a launch with 8 lanes
// takes 1.94 ms and 0.87 G, 75%: the widest particle of a group makes its waves
// uneven. A wavefront per particle with look-ups, loads and conversions of its
// own took 2.61 ms and 1.59 G; 4 M particles at rest density (26 pairs each) take
// 0.93 ms against 1.69 ms with 4 lanes per particle following the box's lines.
// Also measured there, against the 4 lanes: 32 particles per wavefront 1.9 ms and 64 (one candidate
// at a time) 2.6 ms (fewer waves, and the common box's candidates grow faster
// than the shared work shrinks); a tile of candidates in the lanes and the
// particles one by one 2.3 ms (the reach of a tile culls badly along a line of
// cells); 6 and 8 waves per SIMD instead of 7 1.59 and 1.47 ms; a contiguous
// block of groups per XCD 1.86 ms (uneven regions of the scene).
constexpr uint32_t AXIS_CELLS = 32;  // cells per axis of the common box with tabulated hash bits
// A common box of more than this many times the first own box is split: a group
// across a jump of the z-curve would look up and stage what few of it reach
// (4: 1.44 ms, 3: 1.45, 6: 1.52).
constexpr float UNITE_LIMIT = 4.0f;

// Inclusive maximum over the lanes 0 .. own of a group of G <= 16 lanes.
template <uint32_t G>
__device__ __forceinline__ uint32_t group_scan_max(uint32_t v, uint32_t part) {
    auto shr = [](uint32_t x, auto ctrl) {  // lanes whose source leaves the 16-lane row read 0
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, true);
    };
    auto step = [&](uint32_t m, uint32_t from) { v = max(v, G == 16 || part >= m ? from : 0u); };
    if (G > 1) step(1, shr(v, std::integral_constant<int, 0x111>{}));
    if (G > 2) step(2, shr(v, std::integral_constant<int, 0x112>{}));
    if (G > 4) step(4, shr(v, std::integral_constant<int, 0x114>{}));
    if (G > 8) step(8, shr(v, std::integral_constant<int, 0x118>{}));
    return v;
}
// A reduction over a group of G <= 16 lanes, in every lane.
template <uint32_t G, typename T, typename Op>
__device__ __forceinline__ T group_reduce(T v, Op op) {
    auto dpp = [](T x, auto ctrl) {
        return __builtin_bit_cast(
            T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    if (G > 1) v = op(v, dpp(v, std::integral_constant<int, 0xB1>{}));   // lane ^ 1
    if (G > 2) v = op(v, dpp(v, std::integral_constant<int, 0x4E>{}));   // lane ^ 2
    if (G > 4) v = op(v, dpp(v, std::integral_constant<int, 0x141>{}));  // mirror in 8
    if (G > 8) v = op(v, dpp(v, std::integral_constant<int, 0x140>{}));  // mirror in 16
    return v;
}

template <int L, int MODE, bool SPREAD, bool SEG>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(7))) void k_walk_group(
    const int4* __restrict__ pos, const float* __restrict__ kw, const float* __restrict__ radius,
    const float* __restrict__ trad, const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
    uint32_t* __restrict__ counts, WalkArgs wa, uint32_t* __restrict__ cnt_raw, uint32_t* __restrict__ cnt_f,
    const uint32_t* __restrict__ row_raw, const uint32_t* __restrict__ row_f, uint32_t* __restrict__ col,
    uint32_t* __restrict__ ukw) {
    constexpr bool FILL = MODE == WALK_FILL;
    constexpr bool PAD = MODE == WALK_PAD;
    constexpr uint32_t WAVES = BLOCK / 64;
    constexpr bool WIDTHS = SPREAD && MODE != WALK_COUNT;
    constexpr uint32_t GROUP = 64 / L;  // particles per wavefront
    static_assert(GROUP <= 16, "a group lies in a 16-lane row");
    constexpr uint32_t EVERY = (1u << GROUP) - 1u;
    constexpr uint32_t STAGED = L == 64 ? 128 : 112;  // candidates held between tests: a multiple of L, at least 64 + L
    bool only_long_rows = false;
    if (FILL && wa.gate) {
        if (wa.gate[C_FALLBACK] == 0u) {
            if (wa.gate[C_ROWFIX] == 0u) return;
            only_long_rows = true;
        }
    }
    // candidates waiting for their tests: float(x), float(y), float(z), id; and the fixed-point x, y, z, stored width
    __shared__ float4 s_cand[WAVES][STAGED];
    __shared__ int4 s_fixed[WAVES][SPREAD ? STAGED : 1];
    // a particle's values that few tests need: its fixed-point x, y, z and own width; its exact bounds
    __shared__ int4 s_own[WAVES][GROUP];
    __shared__ float2 s_cut[WAVES][SPREAD ? GROUP : 1];
    // per axis and cell coordinate of the common box: its hash bits and its squared distance from the group's box
    __shared__ uint2 s_axis[WAVES][3][AXIS_CELLS];
    // the runs of the current 64 cells, and where they start in the current tile
    __shared__ uint32_t s_run[WAVES][64];
    __shared__ uint8_t s_head[WAVES][64];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t part = lane & (GROUP - 1u), which = lane / GROUP;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t column = (0xFFFFFFFFu / EVERY) << part;  // its lanes in either half of a ballot
    auto vadd = [](uint32_t a, uint32_t b) { return a + b; };
    const uint32_t n = counts[C_N];
    const uint32_t stride = wa.stride ? slot_stride(wa.pcap, n) : 0u;
    for (uint32_t base = (blockIdx.x * WAVES + wave) * GROUP; base < n; base += gridDim.x * WAVES * GROUP) {
        // ---- set-up of particle base + part, in all of its lanes
        const uint32_t ip = base + part;
        const bool mine = ip < n && !(only_long_rows && row_f[ip] + stride >= row_f[ip + 1]);
        bool act = mine;
        uint32_t sc = 0, lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, umax = 0, braw = 0, bf = 0;
        float t_range = 0.0f, t_inner = 0.0f, t_klo = 0.0f, t_khi = 0.0f;
        float spread_to = 0.0f;  // 1.5 okw in position units, plus a margin
        v3f pu = mk(0, 0, 0);
        bool unite = false;
        if (mine) {
            sc = SEG ? wa.seg.sid[ip] : 0u;
            const GridDesc& g = SEG ? wa.seg.grids[sc] : wa.g;
            const int4 pi = pos[ip];
            float okw = 0.0f;
            pu = vec_i(pi.x, pi.y, pi.z);
            const v3f p = pos_world(pi);
            const float kwi = kw[ip];
            const float range = kwi * wa.range_scale;
            lo[0] = grid_cell(p.x - range, g.mn[0], g.mx[0], g.res);
            lo[1] = grid_cell(p.y - range, g.mn[1], g.mx[1], g.res);
            lo[2] = grid_cell(p.z - range, g.mn[2], g.mx[2], g.res);
            hi[0] = grid_cell(p.x + range, g.mn[0], g.mx[0], g.res);
            hi[1] = grid_cell(p.y + range, g.mn[1], g.mx[1], g.res);
            hi[2] = grid_cell(p.z + range, g.mn[2], g.mx[2], g.res);
            // neighborhood_green.comp:36: in 2D the walk stays in z cell 0
            if (g.dims == 2u) lo[2] = hi[2] = 0u;
            // Bound the walk to 4 * 2^res cells per axis: wider walks only revisit
            // aliased cells, and an unbounded span (infinite range) would not end.
            const uint32_t axis = 1u << g.res;
            for (int d = 0; d < 3; ++d)
                if (hi[d] - lo[d] >= 4u * axis && hi[d] >= lo[d]) hi[d] = lo[d] + 4u * axis - 1u;
            // Distance tests compare squared distances with exact bounds (the
            // reference compares rounded square roots; sqrt_le_bound makes the two
            // agree for every input). A NaN range keeps every candidate.
            //
            // Both tests run on unscaled coordinates. The world distance is
            // p - pos_world(pj) = (float(xi) - float(xj)) * 2^-18 component-wise,
            // and the differences of integer-valued floats are 0 or at least 1 in
            // magnitude, so every rounding of the difference and of its squared
            // length commutes with the scaling by 2^-18 (no result is subnormal):
            // the squared world distance is exactly dot(u, u) * 2^-36 with
            // u = float(xi) - float(xj), and likewise for the fixed-point
            // difference. Comparing dot(u, u) with the bound times 2^36 (an exact
            // scaling; an overflow to infinity keeps the comparison's outcome, as
            // dot(u, u) * 2^-36 < 2^30) is then the same test.
            t_range = ((range != range) ? __builtin_inff() : sqrt_le_bound(range)) * 0x1p36f;
            unite = range >= 0.0f && t_range < __builtin_inff() && hi[0] - lo[0] < axis && hi[1] - lo[1] < axis &&
                    hi[2] - lo[2] < axis;
            const float far = __builtin_fabsf(p.x) + __builtin_fabsf(p.y) + __builtin_fabsf(p.z) + range;
            const float ri = range - far * 0x1p-22f;
            // alone, the common box is the own one and nothing lies outside it
            t_inner = !unite ? __builtin_inff() : (ri > 0.0f ? ri * ri * (1.0f - 0x1p-20f) * 0x1p36f : -1.0f);
            if (SPREAD) {
                const float tr = wa.on_target ? trad[ip] : 0.0f;
                okw = fmax_g(radius[ip], tr) * KERNEL_SCALE;
                const float cut = fmax_g(okw, kwi);
                s_cut[wave][part] = make_float2(sqrt_le_bound(cut) * 0x1p36f, sqrt_le_bound(okw) * 0x1p36f);
                umax = to_u32(okw * KW_RES);
                // in range and below 2^30 units apart: no difference of the fixed-point coordinates wraps
                const bool near = cut >= 0.0f && t_range < 0x1p60f;
                const float m = (far + cut) * 0x1p-20f;
                t_klo = near && cut > m ? (cut - m) * (cut - m) * (1.0f - 0x1p-20f) * 0x1p36f : -1.0f;
                t_khi = near ? (cut + m) * (cut + m) * (1.0f + 0x1p-20f) * 0x1p36f : __builtin_inff();
                spread_to = near ? (1.5f * okw + m) * 0x1p18f : __builtin_inff();
            }
            s_own[wave][part] = make_int4(pi.x, pi.y, pi.z, __builtin_bit_cast(int, okw));
            if (FILL) {
                braw = row_raw[ip];
                bf = SPREAD ? row_f[ip] : braw;
                act = braw < wa.pcap;
            }
        }
        const float own_cells = (float)(hi[0] - lo[0] + 1u) * (float)(hi[1] - lo[1] + 1u) * (float)(hi[2] - lo[2] + 1u);
        uint32_t craw = 0, cf = 0;  // this lane's accepted candidates; the row's entries so far
        uint32_t* const out = PAD ? col + (size_t)base * stride : col;
        const size_t row0 = PAD ? (size_t)(part * stride) : (size_t)bf;
        uint64_t tested = 0;
        const uint32_t unitable = (uint32_t)__ballot(unite) & EVERY;
        for (uint32_t todo = (uint32_t)__ballot(act) & EVERY; todo;) {
            // ---- the next particles that share a common box
            const int first = __builtin_ctz(todo);
            const uint32_t gsc = lane_value(sc, first);
            const GridDesc& g = SEG ? wa.seg.grids[gsc] : wa.g;
            uint32_t grp = 1u << first;
            int at = first;
            uint32_t ulo[3] = {lo[0], lo[1], lo[2]}, uhi[3] = {hi[0], hi[1], hi[2]};
            if ((unitable >> first) & 1u) {
                const bool in = ((todo >> part) & 1u) && unite && (!SEG || sc == gsc);
                for (int d = 0; d < 3; ++d) {
                    ulo[d] = ~group_scan_max<GROUP>(in ? ~lo[d] : 0u, part);
                    uhi[d] = group_scan_max<GROUP>(in ? hi[d] : 0u, part);
                }
                const uint32_t axis = 1u << g.res;
                const float cells = (float)(uhi[0] - ulo[0] + 1u) * (float)(uhi[1] - ulo[1] + 1u) *
                                    (float)(uhi[2] - ulo[2] + 1u);
                const bool fits = in && cells <= UNITE_LIMIT * lane_value(own_cells, first) &&
                                  uhi[0] - ulo[0] < axis && uhi[1] - ulo[1] < axis && uhi[2] - ulo[2] < axis;
                const uint32_t stop = todo & ~(uint32_t)__ballot(fits);
                grp |= stop ? todo & ((stop & (0u - stop)) - 1u) : todo;
                at = 31 - __builtin_clz(grp);
            }
            todo &= ~grp;
            const uint32_t lo0 = lane_value(ulo[0], at), lo1 = lane_value(ulo[1], at), lo2 = lane_value(ulo[2], at);
            const uint32_t h0 = lane_value(uhi[0], at), h1 = lane_value(uhi[1], at), h2 = lane_value(uhi[2], at);
            const uint32_t n0 = h0 >= lo0 ? h0 - lo0 + 1u : 0u, n1 = h1 >= lo1 ? h1 - lo1 + 1u : 0u,
                           n2 = h2 >= lo2 ? h2 - lo2 + 1u : 0u;
            const uint32_t cbase = SEG ? (gsc << wa.seg.shift) : 0u;
            const bool planar = g.dims == 2u;
            const bool in_group = (grp >> part) & 1u;
            // the group's bounding box and farthest range, for the candidates' culling
            constexpr float inf = __builtin_inff();
            auto group_min = [](float v) {
                v = group_reduce<GROUP>(v, [](float a, float b) { return __builtin_fminf(a, b); });
                return lane_value(v, 0);
            };
            auto group_max = [](float v) {
                v = group_reduce<GROUP>(v, [](float a, float b) { return __builtin_fmaxf(a, b); });
                return lane_value(v, 0);
            };
            const v3f gn = mk(group_min(in_group ? pu.x : inf), group_min(in_group ? pu.y : inf),
                              group_min(in_group ? pu.z : inf));
            const v3f gx = mk(group_max(in_group ? pu.x : -inf), group_max(in_group ? pu.y : -inf),
                              group_max(in_group ? pu.z : -inf));
            const float g_range = group_max(in_group ? t_range : -inf);
            const float t_mine = in_group ? t_range : -inf;  // the other lanes accept nothing
            // A cell whose box lies farther than that from the group's box holds no
            // accepted candidate. The cell boxes are widened by margins far above
            // the rounding of the hash (grid_cell) and of the distance test, and
            // the cells at the grid border and beyond (which also hold clamped and
            // aliased particles) are never culled.
            const uint32_t last_cell = (1u << g.res) - 1u;
            // A box wider than the grid visits cells twice, also for what lies past the grid's end: no culling there.
            const float thr = ((unitable >> first) & 1u) ? g_range * 1.001f + 1.0f : inf;
            auto axis_cell = [&](int d, uint32_t c, float pn, float px) -> uint2 {
                const float w = (g.mx[d] - g.mn[d]) / (float)(1u << g.res) * POS_RES;
                const float m = 1e-4f * w + 1e-6f * (__builtin_fabsf(g.mn[d]) + __builtin_fabsf(g.mx[d])) * POS_RES;
                const float a = g.mn[d] * POS_RES + (float)c * w;
                const float t = __builtin_fmaxf(__builtin_fmaxf(a - m - px, pn - (a + w + m)), 0.0f);
                const float t2 = (c == 0u || c >= last_cell) ? 0.0f : t * t;
                return make_uint2(planar && d == 2 ? 0u : zbits(c, (uint32_t)d, g.res, g.dims),
                                  __builtin_bit_cast(uint32_t, t2));
            };
            const bool table = n0 <= AXIS_CELLS && n1 <= AXIS_CELLS && n2 <= AXIS_CELLS;
            if (table) {
                const uint32_t e = lane & (AXIS_CELLS - 1u);
                if (lane < AXIS_CELLS)
                    s_axis[wave][0][e] = axis_cell(0, lo0 + e, gn.x, gx.x);
                else
                    s_axis[wave][1][e] = axis_cell(1, lo1 + e, gn.y, gx.y);
                if (lane < AXIS_CELLS) s_axis[wave][2][e] = axis_cell(2, lo2 + e, gn.z, gx.z);
                __builtin_amdgcn_wave_barrier();
            }
            uint32_t staged = 0;
            auto test_staged = [&]() {
                __builtin_amdgcn_wave_barrier();
                for (uint32_t s = 0; s < staged; s += L) {
                    const uint32_t c = s + which;
                    const float4 q = s_cand[wave][c];
                    const uint32_t j = __builtin_bit_cast(uint32_t, q.w);
                    const v3f u = pu - mk(q.x, q.y, q.z);
                    const float d2 = dot(u, u);
                    bool green = !(d2 > t_mine) && j != ip && c < staged;
                    if (!__ballot(green)) continue;
                    if (__ballot(green && d2 > t_inner)) {  // beyond the sure part of the own box: compare the cell
                        if (green && d2 > t_inner) {
                            const v3f w = mk(q.x, q.y, q.z) / POS_RES;
                            const v3f p = pu / POS_RES;
                            const float range = kw[ip] * wa.range_scale;
                            const uint32_t cm = (1u << g.res) - 1u;
                            auto outside = [&](int d, uint32_t l, float pc, float wc) {
                                const uint32_t c = l + ((grid_cell(wc, g.mn[d], g.mx[d], g.res) - l) & cm);
                                return c < grid_cell(pc - range, g.mn[d], g.mx[d], g.res) ||
                                       c > grid_cell(pc + range, g.mn[d], g.mx[d], g.res);
                            };
                            green = !(outside(0, lo0, p.x, w.x) || outside(1, lo1, p.y, w.y) ||
                                      (!planar && outside(2, lo2, p.z, w.z)));
                        }
                    }
                    if (FILL) {  // entries at or beyond the capacity are dropped
                        const uint64_t gb = __ballot(green);
                        const uint32_t ml = (uint32_t)gb & column, mh = (uint32_t)(gb >> 32) & column;
                        const uint32_t r = braw + craw + __builtin_amdgcn_mbcnt_hi(mh, __builtin_amdgcn_mbcnt_lo(ml, 0u));
                        if (r >= wa.pcap) green = false;
                        craw += (uint32_t)__popc(ml) + (uint32_t)__popc(mh);  // the row's total, in every lane
                    } else if (green) {
                        ++craw;
                    }
                    bool kept = green;
                    if (SPREAD) {
                        kept = green && d2 <= t_klo;
                        const bool open = green && d2 > t_klo && d2 <= t_khi;
                        // kernel_width.comp:41-53: the spread width is
                        // to_u32(okw * influence * 2^18) with the influence in [0, 1]:
                        // exactly umax up to a distance of okw, and at most
                        // to_u32((3 okw - 2 d) 2^18) beyond it (KW_PROPAGATION is 1/2).
                        // The neighbour's stored value starts at its own width and only
                        // grows, so an entry changes nothing where the stored value has
                        // reached umax, nor where d passes (3 okw - stored) / 2.
                        const uint32_t uj = WIDTHS ? (uint32_t)s_fixed[wave][c].w : 0u;
                        const float reach = spread_to - 0.5f * (float)uj;
                        const bool wide = WIDTHS && green && uj < umax && reach >= 0.0f && d2 <= reach * reach;
                        if (__ballot(open || wide)) {
                            uint32_t uval = 0;
                            if (open || wide) {
                                const int4 pj = s_fixed[wave][c], pi = s_own[wave][part];
                                const float2 cut = s_cut[wave][part];
                                const float okw = __builtin_bit_cast(float, pi.w);
                                const v3f v = vec_i(isub(pj.x, pi.x), isub(pj.y, pi.y), isub(pj.z, pi.z));
                                const float d2v = dot(v, v);
                                if (open) kept = d2v <= cut.x;
                                if (wide) {
                                    uval = umax;
                                    if (!(d2v <= cut.y)) {
                                        const float dfk = __builtin_sqrtf(d2v * 0x1p-36f) - okw;
                                        const float infl =
                                            fmax_g(0.0f, 1.0f - fmax_g(0.0f, dfk / (okw * KW_PROPAGATION)));
                                        uval = to_u32(okw * infl * KW_RES);
                                    }
                                }
                            }
                            if (WIDTHS) {  // one atomic per candidate
                                uval = group_reduce<GROUP>(uval, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
                                if (part == 0u && uval > uj) atomicMax(&ukw[j], uval);
                            }
                        }
                    }
                    if (MODE == WALK_COUNT) {
                        if (SPREAD && kept) ++cf;
                    } else {
                        const uint64_t kb = __ballot(kept);
                        const uint32_t ml = (uint32_t)kb & column, mh = (uint32_t)(kb >> 32) & column;
                        const uint32_t r = cf + __builtin_amdgcn_mbcnt_hi(mh, __builtin_amdgcn_mbcnt_lo(ml, 0u));
                        if (kept && (FILL || r < stride)) out[row0 + r] = j;
                        cf += (uint32_t)__popc(ml) + (uint32_t)__popc(mh);
                    }
                }
                staged = 0;
                __builtin_amdgcn_wave_barrier();
            };
            // ---- the common box's cells, 64 at a time, one per lane
            const uint64_t ncell = (uint64_t)n0 * n1 * n2;
            const float r0 = 1.0f / (float)(n0 ? n0 : 1u), r1 = 1.0f / (float)(n1 ? n1 : 1u);
            for (uint64_t c0 = 0; c0 < ncell; c0 += 64) {
                uint32_t cstart = 0, clen = 0;
                const uint64_t c = c0 + lane;
                if (c < ncell) {
                    uint32_t x, y, z;
                    if (ncell <= (1u << 20)) {
                        // (c + 1/2) / n is at least 1 / 2n from an integer, far above the roundings for c < 2^20
                        const uint32_t q = (uint32_t)(((float)(uint32_t)c + 0.5f) * r0);
                        x = (uint32_t)c - q * n0;
                        z = (uint32_t)(((float)q + 0.5f) * r1);
                        y = q - z * n1;
                    } else {
                        x = (uint32_t)(c % n0);
                        y = (uint32_t)((c / n0) % n1);
                        z = (uint32_t)(c / ((uint64_t)n0 * n1));
                    }
                    uint2 ex, ey, ez;
                    if (table) {
                        ex = s_axis[wave][0][x];
                        ey = s_axis[wave][1][y];
                        ez = s_axis[wave][2][z];
                    } else {
                        ex = axis_cell(0, lo0 + x, gn.x, gx.x);
                        ey = axis_cell(1, lo1 + y, gn.y, gx.y);
                        ez = axis_cell(2, lo2 + z, gn.z, gx.z);
                    }
                    const float cd = (__builtin_bit_cast(float, ez.y) + __builtin_bit_cast(float, ey.y)) +
                                     __builtin_bit_cast(float, ex.y);
                    if (!(cd > thr)) {
                        const uint32_t h = cbase + (ex.x | ey.x | ez.x);
                        cstart = cs[h];
                        const uint32_t cend = ce[h];
                        clen = cend > cstart ? cend - cstart : 0u;
                    }
                }
                const uint32_t incl = wave_scan(clen, vadd);
                const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
                const uint32_t off = incl - clen;  // the cell's first candidate in the stream
                // candidate = stream position + delta inside the cell; a cell whose
                // particles directly follow those of the previous non-empty cell
                // (the same delta) continues its run
                const uint32_t delta = cstart - off;
                const uint64_t nonempty = __ballot(clen > 0u);
                const uint64_t prev_mask = nonempty & below;
                const uint32_t prev = prev_mask ? 63u - (uint32_t)__clzll(prev_mask) : lane;
                const uint32_t prev_delta = (uint32_t)__shfl((int)delta, (int)prev, 64);
                const bool start = clen > 0u && (prev_mask == 0ull || prev_delta != delta);
                // the runs in order; a candidate's run is the number of starts at or before it
                const uint64_t starts = __ballot(start);
                if (start) s_run[wave][__popcll(starts & below)] = delta;
                for (uint32_t w0 = 0; w0 < total; w0 += 64u) {
                    s_head[wave][lane] = 0;
                    __builtin_amdgcn_wave_barrier();
                    if (start && off >= w0 && off - w0 < 64u) s_head[wave][off - w0] = 1;
                    __builtin_amdgcn_wave_barrier();
                    const uint64_t heads = __ballot(s_head[wave][lane] != 0);
                    const uint32_t before = (uint32_t)__popcll(__ballot(start && off < w0));
                    const bool held = w0 + lane < total;
                    const uint32_t run = before + (uint32_t)__popcll(heads & (below | (1ull << lane)));
                    const uint32_t j = held ? w0 + lane + s_run[wave][run - 1u] : base;
                    const int4 pj = pos[j];
                    const uint32_t uj = WIDTHS ? ukw[j] : 0u;
                    const v3f cu = vec_i(pj.x, pj.y, pj.z);
                    const v3f d = mk(__builtin_fmaxf(__builtin_fmaxf(cu.x - gx.x, gn.x - cu.x), 0.0f),
                                     __builtin_fmaxf(__builtin_fmaxf(cu.y - gx.y, gn.y - cu.y), 0.0f),
                                     __builtin_fmaxf(__builtin_fmaxf(cu.z - gx.z, gn.z - cu.z), 0.0f));
                    const bool take = held && !(dot(d, d) > g_range);
                    const uint64_t tb = __ballot(take);
                    if (take) {
                        const uint32_t to = staged + (uint32_t)__popcll(tb & below);
                        s_cand[wave][to] = make_float4(cu.x, cu.y, cu.z, __builtin_bit_cast(float, j));
                        if (SPREAD) s_fixed[wave][to] = make_int4(pj.x, pj.y, pj.z, (int)uj);
                    }
                    staged += (uint32_t)__popcll(tb);
                    if (MODE == WALK_COUNT) tested += (uint64_t)__popcll(tb) * (uint32_t)__popc(grp);
                    if (staged > STAGED - 64u) test_staged();
                }
            }
            test_staged();
        }
        if (!FILL) {  // the row's accepted candidates, summed over its lanes
#pragma unroll
            for (int m = (int)GROUP; m < 64; m <<= 1) craw += (uint32_t)__shfl_xor((int)craw, m, 64);
        }
        if (MODE == WALK_COUNT && SPREAD) {
#pragma unroll
            for (int m = (int)GROUP; m < 64; m <<= 1) cf += (uint32_t)__shfl_xor((int)cf, m, 64);
        }
        if (mine && which == 0u) {
            if (!FILL) {
                cnt_raw[ip] = craw;
                if (SPREAD) cnt_f[ip] = cf;
                if (PAD && cf > stride) atomicMax(&counts[C_MAXROW], cf);
            } else if (SPREAD && braw <= wa.pcap && row_raw[ip + 1] > wa.pcap) {
                // the row the capacity cuts: its kept short-list length
                counts[C_CLAMP_ROW] = ip;
                counts[C_CLAMP_KEPT] = cf;
            }
        }
        if (MODE == WALK_COUNT && wa.cand && lane == 0 && tested) atomicAdd(wa.cand, (unsigned long long)tested);
    }
    if (!FILL && blockIdx.x == 0 && threadIdx.x == 0) {
        cnt_raw[n] = 0;
        if (SPREAD) cnt_f[n] = 0;
    }
}

// After a PAD walk and the scan of its raw counts: take the exact path when a
// row outgrew its slot or the list exceeds the capacity.
__global__ void k_walk_decide(uint32_t* __restrict__ counts, uint32_t pcap) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const uint32_t stride = slot_stride(pcap, counts[C_N]);
    counts[C_FALLBACK] = counts[C_PAIRS_RAW] > pcap ? 1u : 0u;  // every row exactly (clamped list)
    counts[C_ROWFIX] = counts[C_MAXROW] > stride ? 1u : 0u;     // only rows longer than their slot
    counts[C_MAXROW_LAST] = counts[C_MAXROW];
    counts[C_MAXROW] = 0u;
}

// Packs the PAD slots into the list at the scanned offsets (16 lanes per row,
// coalesced); rows longer than their slot are left to the exact fill, and
// nothing is packed when the exact fill rewrites every row.
__global__ __launch_bounds__(BLOCK) void k_pack_rows(const uint32_t* __restrict__ counts,
                                                     const uint32_t* __restrict__ row,
                                                     const uint32_t* __restrict__ slots, uint32_t pcap,
                                                     uint32_t* __restrict__ col) {
    if (counts[C_FALLBACK]) return;
    constexpr int L = 16, B = 8;  // a lane has B loads in flight before its stores
    const uint32_t n = counts[C_N];
    const uint32_t stride = slot_stride(pcap, n);
    const int gl = threadIdx.x & (L - 1);
    for (uint32_t base = blockIdx.x * (BLOCK / L); base < n; base += gridDim.x * (BLOCK / L)) {
        const uint32_t i = base + threadIdx.x / L;
        if (i >= n) continue;
        const uint32_t b = row[i], len = row[i + 1] - b;
        if (len > stride) continue;
        const uint32_t* src = slots + (size_t)i * stride;
        for (uint32_t k0 = 0; k0 < len; k0 += (uint32_t)(B * L)) {
            uint32_t v[B];
#pragma unroll
            for (int t = 0; t < B; ++t) {
                const uint32_t k = k0 + (uint32_t)gl + (uint32_t)(t * L);
                v[t] = k < len ? src[k] : 0u;
            }
#pragma unroll
            for (int t = 0; t < B; ++t) {
                const uint32_t k = k0 + (uint32_t)gl + (uint32_t)(t * L);
                if (k < len) col[b + k] = v[t];
            }
        }
    }
}

// After a clamped spreading walk: rows after the cut row are empty, so their
// offsets all equal the end of the cut row's kept entries.
__global__ __launch_bounds__(BLOCK) void k_fix_clamped_rows(const uint32_t* __restrict__ counts, uint32_t pcap,
                                                            uint32_t* __restrict__ row_f) {
    if (counts[C_PAIRS_RAW] <= pcap) return;
    const uint32_t n = counts[C_N];
    const uint32_t p = counts[C_CLAMP_ROW];
    const uint32_t end = row_f[p] + counts[C_CLAMP_KEPT];
    for (uint32_t k = p + 1 + blockIdx.x * blockDim.x + threadIdx.x; k <= n; k += gridDim.x * blockDim.x)
        row_f[k] = end;
}

// neighborhood_brute_force.comp:31-50: particle i against every particle in
// index order, a whole wavefront per particle (64 candidates per step); the
// distance test and the capacity clamp are those of the cell walk, so the
// rows come out in the order a sequential run appends them. COUNT writes the
// row lengths, FILL the rows at the scanned offsets.
template <bool FILL>
__global__ __launch_bounds__(BLOCK) void k_brute_rows(const int4* __restrict__ pos, const float* __restrict__ kw,
                                                      const uint32_t* __restrict__ counts, float range_scale,
                                                      uint32_t pcap, uint32_t* __restrict__ cnt,
                                                      const uint32_t* __restrict__ row, uint32_t* __restrict__ col) {
    constexpr uint32_t L = 64;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t n = counts[C_N];
    const uint32_t waves = BLOCK / 64;
    for (uint32_t i = blockIdx.x * waves + threadIdx.x / 64; i < n; i += gridDim.x * waves) {
        const v3f p = pos_world(pos[i]);
        const float range = kw[i] * range_scale;
        const float t_range = (range != range) ? __builtin_inff() : sqrt_le_bound(range);
        const uint32_t b0 = FILL ? row[i] : 0u;
        uint32_t c = 0;
        bool more = !FILL || b0 < pcap;
        for (uint32_t j0 = 0; more && j0 < n; j0 += L) {
            const uint32_t j = j0 + lane;
            bool green = false;
            if (j < n && j != i) {
                const v3f d = p - pos_world(pos[j]);
                green = !(dot(d, d) > t_range);
            }
            const uint64_t bal = __ballot(green);
            if (FILL) {
                const uint32_t ridx = b0 + c + (uint32_t)__popcll(bal & below);
                if (green && ridx < pcap) col[ridx] = j;
            }
            c += (uint32_t)__popcll(bal);
            if (FILL) more = b0 + c < pcap;
        }
        if (!FILL && lane == 0) cnt[i] = c;
    }
    if (!FILL && blockIdx.x == 0 && threadIdx.x == 0) cnt[n] = 0;
}

void launch_brute(bool fill, const int4* pos, const float* kw, const uint32_t* counts, uint32_t cap,
                  float range_scale, uint32_t pcap, uint32_t* cnt, const uint32_t* row, uint32_t* col,
                  hipStream_t s) {
    uint32_t g = div_up(cap ? cap : 1, BLOCK / 64);
    g = g < 16384u ? g : 16384u;
    if (fill)
        hipLaunchKernelGGL(k_brute_rows<true>, dim3(g), dim3(BLOCK), 0, s, pos, kw, counts, range_scale, pcap, cnt,
                           row, col);
    else
        hipLaunchKernelGGL(k_brute_rows<false>, dim3(g), dim3(BLOCK), 0, s, pos, kw, counts, range_scale, pcap, cnt,
                           row, col);
}

static uint32_t walk_grid(uint32_t cap, uint32_t lanes) {
    const uint32_t groups = BLOCK / lanes;
    uint32_t g = div_up(cap ? cap : 1, groups);
    return g < 16384u ? g : 16384u;
}

void launch_walk(int mode, bool spread, const int4* pos, const float* kw, const float* radius, const float* trad,
                 int on_target, const uint32_t* cs, const uint32_t* ce, uint32_t* counts, uint32_t cap,
                 float range_scale, const GridDesc& g, uint32_t pcap, uint32_t* cnt_raw, uint32_t* cnt_f,
                 const uint32_t* row_raw, const uint32_t* row_f, uint32_t* col, uint32_t* ukw, hipStream_t s,
                 int lanes, uint32_t stride, const uint32_t* gate, const SegmentTable* seg,
                 unsigned long long* cand) {
    WalkArgs wa;
    wa.range_scale = range_scale;
    wa.g = g;
    wa.on_target = on_target;
    wa.pcap = pcap;
    wa.stride = stride;
    wa.gate = gate;
    wa.cand = cand;
    wa.seg = seg ? *seg : SegmentTable{nullptr, nullptr, nullptr, nullptr, 0u};
    const bool packed = seg && seg->sid;
    const dim3 grid(walk_grid(cap, (uint32_t)lanes)), block(BLOCK);
#define WALK(L, F, S, G)                                                                                              \
    hipLaunchKernelGGL((k_walk_group<L, F, S, G>), grid, block, 0, s, pos, kw, radius, trad, cs, ce, counts, wa,       \
                       cnt_raw, cnt_f, row_raw, row_f, col, ukw)
#define WALK_F(L, F, G)             \
    if (spread)                     \
        WALK(L, F, true, G);        \
    else                            \
        WALK(L, F, false, G)
#define WALK_G(L, G)                \
    if (mode == WALK_PAD) {         \
        WALK_F(L, WALK_PAD, G);     \
    } else if (mode == WALK_FILL) { \
        WALK_F(L, WALK_FILL, G);    \
    } else {                        \
        WALK_F(L, WALK_COUNT, G);   \
    }
#define WALK_L(L)           \
    if (packed) {           \
        WALK_G(L, true)     \
    } else {                \
        WALK_G(L, false)    \
    }
    switch (lanes) {
        case 4: WALK_L(4) break;
        case 8: WALK_L(8) break;
        case 16: WALK_L(16) break;
        default: WALK_L(64) break;
    }
#undef WALK_L
#undef WALK_G
#undef WALK_F
#undef WALK
}

void launch_walk_decide(uint32_t* counts, uint32_t pcap, hipStream_t s) {
    hipLaunchKernelGGL(k_walk_decide, dim3(1), dim3(64), 0, s, counts, pcap);
}
void launch_pack_rows(const uint32_t* counts, uint32_t cap, const uint32_t* row, const uint32_t* slots,
                      uint32_t pcap, uint32_t* col, hipStream_t s) {
    uint32_t g = div_up(cap ? cap : 1, BLOCK / 16);
    hipLaunchKernelGGL(k_pack_rows, dim3(g < 8192u ? g : 8192u), dim3(BLOCK), 0, s, counts, row, slots, pcap, col);
}

void launch_fix_clamped_rows(const uint32_t* counts, uint32_t cap, uint32_t pcap, uint32_t* row_f, hipStream_t s) {
    hipLaunchKernelGGL(k_fix_clamped_rows, dim3(stride_grid(cap + 1)), dim3(BLOCK), 0, s, counts, pcap, row_f);
}

}  // namespace apbf
