// Neighbor search of a group of 64 consecutive cell-list slots by one
// wavefront, on the matrix cores.
//
// The squared distances of 32 candidates to 32 particles are a contraction:
// with candidates and particles as offsets b, a from an anchor,
//   |a - b|^2 - r^2 = (|a|^2 - r^2) - 2 a.b + |b|^2 . 1,
// K = 4 in FP32, i.e. two v_mfma_f32_32x32x2_f32 for 1,024 pairs with the
// particle's |a|^2 - r^2 as the C operand.  The sign of a result is the hit,
// so a lane collects 32 candidates of one particle into a 32-bit mask with
// one v_alignbit each (bit o = candidate o), against about eight
// instructions and a serial append per pair in a lane-per-particle loop.
// 64 particles share the candidates' reads and conversions; exchanging the
// halves of two registers then gives every lane both mask words of its own
// particle.
// Pairs whose result lies within the FP32 error bound of the list radius are
// decided by the FP64 predicate of the host oracle, so the pair set is the
// FP64 one.
//
// Candidates are the members of the union of the particles' 27-cell
// stencils (cells outside a particle's own stencil lie beyond its list
// radius and only cost tests).  Cells are visited in ascending geometric index
// and their members in slot order: every list of every walk has this order.
// A group whose particles lie in cells far apart (a jump of the Morton
// curve, several replicas) is served in passes over windows of at most
// 5 x 5 x 5 own cells.
#pragma once

#include "cells.h"

namespace azp
{

// Own cells of one pass lie within kGroupReach of the anchor's on every axis,
// so their stencils span at most kGroupSpan cells per axis.
constexpr int kGroupReach = 2;
constexpr uint32_t kGroupSpan = 2 * kGroupReach + 3;
constexpr uint32_t kGroupCells = kGroupSpan * kGroupSpan * kGroupSpan;
// Candidates per segment of a pass (the bits of GroupLds::starts).
constexpr uint32_t kGroupSegment = 2048;

typedef float f32x16 __attribute__((ext_vector_type(16)));

// The periodic box and cell grid of one pass (wave-uniform).
struct GroupGeom
    {
    int n[3];
    double L[3], Linv[3];
    float scale[3]; // L / 2^32
    int reach[3];   // group_reach
    float slip;     // group_slip
    uint32_t cell_base;
    };

// How far a particle may lie from the middle of its pass's cells, in fixed-point
// steps, for its neighbors to stay within half a box of it: less the particle's
// and the neighbor's roundings.
inline int group_reach(double L, double r_max)
    {
    return (int)std::max(0.0, std::floor(2147483646.0 - r_max / L * 4294967296.0));
    }

// Error of r^2 near r_max^2 from the positions' fixed-point steps: a difference
// of two coordinates is off by up to L / 2^32, doubled here.
inline float group_slip(const double L[3], double r_max)
    {
    const double off = 2.0 * std::sqrt(L[0] * L[0] + L[1] * L[1] + L[2] * L[2]) / 4294967296.0;
    return (float)(off * (2.0 * r_max + off));
    }

struct GroupArgs
    {
    const double4* pos;
    const uint32_t* members;
    const uint32_t* start;     // slots of cell rank r: start[r] .. start[r + 1]
    const uint32_t* cell_rank; // storage rank of each cell; null: cells are stored by index
    const int4* cell_fixed;    // by slot: wrapped fixed-point position, type (>= ntypes: never listed)
    const double* r_listsq;
    uint32_t ntypes;
    float thr;    // largest r_list^2
    bool direct;  // no matrix tests (several list radii among more types than ONEHOT serves)
    };

// One wavefront's LDS.
struct GroupLds
    {
    uint64_t starts[kGroupSegment / 64]; // bit p: a cell's first candidate is number p of the segment
    uint32_t rows[kGroupSpan * kGroupSpan];
    uint32_t delta[kGroupCells + 1]; // slot - candidate number of each cell's members
    uint32_t first[kGroupCells + 1]; // candidate number of each cell's first member
    uint16_t seq[kGroupCells + 1];   // place of a window cell in the pass's sequence
    };

// Makes one lane's LDS writes visible to the other lanes of its wavefront.
__device__ __forceinline__ void wave_lds_fence()
    {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

__device__ __forceinline__ int lane_value(int v, int lane)
    {
    return __builtin_amdgcn_readlane(v, lane);
    }

// Exclusive sum over the wavefront (row shifts and broadcasts, no LDS).
__device__ __forceinline__ uint32_t wave_exclusive_scan(uint32_t v, uint32_t& total)
    {
    uint32_t x = v;
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false); // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false); // row_bcast:15
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false); // row_bcast:31
    total = (uint32_t)lane_value((int)x, 63);
    return x - v;
    }

// One axis of a pass's window: `len` distinct cells from s0 (periodic).
struct GroupAxis
    {
    int n, s0, len;
    __device__ GroupAxis(int n_, int anchor, int lo, int hi)
        {
        n = n_;
        const int raw = hi - lo + 3;
        const bool full = raw >= n;
        len = full ? n : raw;
        int s = anchor + lo - 1;
        s = s < 0 ? s + n : (s >= n ? s - n : s);
        s0 = full ? 0 : s;
        }
    // place of cell c in the window
    __device__ int index(int c) const
        {
        const int k = c - s0;
        return k < 0 ? k + n : k;
        }
    // q-th cell of the window in ascending cell index
    __device__ int cell(int q) const
        {
        const int wrapped = max(0, s0 + len - n);
        return q < wrapped ? q : s0 + (q - wrapped);
        }
    __device__ int step(int c, int d) const
        {
        const int x = c + d;
        return x < 0 ? x + n : (x >= n ? x - n : x);
        }
    };

// The particle a lane's column stands for.
struct GroupColumn
    {
    bool valid;
    uint32_t slot, i, cell; // cell: global cell index
    int c[3];               // cell coordinates in the grid
    int4 fixed;             // position, type
    };

// The anchor column of a pass over the columns `todo` (not 0): the middle one.
__device__ __forceinline__ int group_anchor(uint64_t todo)
    {
    const uint32_t first = (uint32_t)__builtin_ctzll(todo), last = 63u - (uint32_t)__builtin_clzll(todo);
    return __builtin_ctzll(todo >> ((first + last) / 2u) << ((first + last) / 2u));
    }

// Exchanges the upper half of p with the lower half of q: low and high
// candidates (or columns) of two values, k = 0 in lanes 0..31 and k = 1 in
// lanes 32..63, as the matrix operands take them.
__device__ __forceinline__ void swap_halves(uint32_t p, uint32_t q, uint32_t& first, uint32_t& second)
    {
    const auto r = __builtin_amdgcn_permlane32_swap(p, q, false, false);
    first = r[0];
    second = r[1];
    }
__device__ __forceinline__ void swap_halves(float p, float q, float& first, float& second)
    {
    uint32_t f, g;
    swap_halves(__float_as_uint(p), __float_as_uint(q), f, g);
    first = __uint_as_float(f);
    second = __uint_as_float(g);
    }

// Runs one pass: the columns with `todo` bits whose own cells lie in the
// window around that of the anchor column `al` (and, by `same`, in its
// system).  Returns the mask of the columns served; direct_used is set when
// it took the direct tests.  For every 64 candidates, emit(low, high, P, off,
// which) gets the column's hits among candidates P .. P + 63 and candidate
// P + off, which this lane read: its particle (MEMBERS; any for a number past
// the last candidate) or its slot (or ~0).  begin(cells, total) runs before
// the first of them.
//
// ONEHOT = 0: one list radius for every type pair (or a.direct).  Otherwise
// 2 * ONEHOT >= ntypes: K grows by one per type, the candidate's type as a
// unit vector against the particle's radii.
template<int ONEHOT, bool MEMBERS, class Begin, class Emit>
__device__ __forceinline__ uint64_t group_pass(const GroupArgs& a,
                                               const GroupGeom& G,
                                               GroupLds& s,
                                               const GroupColumn& me,
                                               uint64_t todo,
                                               int al,
                                               bool same,
                                               bool& direct_used,
                                               Begin&& begin,
                                               Emit&& emit)
    {
    const uint32_t lane = threadIdx.x & 63u, h = lane >> 5;
    int o[3], lo[3], hi[3], anchor[3];
    bool in = me.valid && same && ((todo >> lane) & 1u);
#pragma unroll
    for (int k = 0; k < 3; ++k)
        {
        anchor[k] = lane_value(me.c[k], al);
        o[k] = me.c[k] - anchor[k];
        o[k] += 2 * o[k] > G.n[k] ? -G.n[k] : (2 * o[k] < -G.n[k] ? G.n[k] : 0);
        // own cells of a pass span at most n - 2 cells: from the middle of
        // the span every one of their particles is then within L/2 - r_list
        // (grids of one or two cells take the direct tests)
        const int below = G.n[k] >= 6 || G.n[k] < 3 ? -kGroupReach : (G.n[k] == 3 ? 0 : -1);
        const int above = G.n[k] >= 7 || G.n[k] < 3 ? kGroupReach : (G.n[k] < 5 ? 0 : 1);
        in = in && o[k] >= below && o[k] <= above;
        }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        {
        lo[k] = kGroupReach;
        hi[k] = -kGroupReach;
#pragma unroll
        for (int v = -kGroupReach; v <= kGroupReach; ++v)
            if (__ballot(in && o[k] == v) != 0ull)
                {
                lo[k] = min(lo[k], v);
                hi[k] = max(hi[k], v);
                }
        }
    const uint64_t served = __ballot(in);
    // Offsets from the middle of the own cells: the difference of two is the
    // minimum image when the particle lies within L/2 - r_list of it on every
    // axis.  Otherwise the pass takes the direct tests below.
    const float sx = G.scale[0], sy = G.scale[1], sz = G.scale[2];
    auto middle = [&](int k) {
        const double f = (anchor[k] + 0.5 * (lo[k] + hi[k] + 1)) / G.n[k] - 0.5; // in box lengths
        return __builtin_amdgcn_readfirstlane((int)(uint32_t)(unsigned long long)(long long)(f * 4294967296.0));
    };
    const int fx0 = middle(0), fy0 = middle(1), fz0 = middle(2);
    const int dx0 = fixed_delta(me.fixed.x, fx0), dy0 = fixed_delta(me.fixed.y, fy0), dz0 = fixed_delta(me.fixed.z, fz0);
    const float ax = (float)dx0 * sx, ay = (float)dy0 * sy, az = (float)dz0 * sz;
    auto beyond = [](int d, int reach) { return (uint32_t)d + (uint32_t)reach > 2u * (uint32_t)reach; };
    const bool far = beyond(dx0, G.reach[0]) || beyond(dy0, G.reach[1]) || beyond(dz0, G.reach[2]) || G.n[0] < 3
                     || G.n[1] < 3 || G.n[2] < 3;
    const bool direct = a.direct || __ballot(in && far && (uint32_t)me.fixed.w < a.ntypes) != 0ull;
    direct_used = direct_used || direct;
    const GroupAxis X(G.n[0], anchor[0], lo[0], hi[0]);
    const GroupAxis Y(G.n[1], anchor[1], lo[1], hi[1]);
    const GroupAxis Z(G.n[2], anchor[2], lo[2], hi[2]);

    // the cells of the included columns' stencils, as bits of window rows
    if (lane < kGroupSpan * kGroupSpan)
        s.rows[lane] = 0u;
    wave_lds_fence();
    // once per cell: by the first of its included columns (slots of a cell are
    // consecutive)
    const uint32_t prev = (uint32_t)__shfl_up((int)me.cell, 1);
    if (in && (lane == 0u || prev != me.cell || !((served >> (lane - 1u)) & 1u)))
        {
        const uint32_t bits = (1u << X.index(X.step(me.c[0], X.n > 1 ? -1 : 0))) | (1u << X.index(me.c[0]))
                              | (1u << X.index(X.step(me.c[0], X.n > 1 ? 1 : 0)));
        for (uint32_t q = 0; q < 9u; ++q)
            {
            const int dy = (int)(q % 3u) - 1, dz = (int)(q / 3u) - 1;
            const int y = Y.index(Y.step(me.c[1], Y.n > 1 ? dy : 0));
            const int z = Z.index(Z.step(me.c[2], Z.n > 1 ? dz : 0));
            atomicOr(&s.rows[(uint32_t)z * kGroupSpan + (uint32_t)y], bits);
            }
        }
    wave_lds_fence();

    // their candidate ranges in ascending cell index: one lane per row of x,
    // the reads of a row's cells in flight together
    uint32_t st[kGroupSpan], ct[kGroupSpan], place[kGroupSpan];
    uint32_t ncell = 0, ncand = 0;
    const bool row_lane = lane < (uint32_t)(Y.len * Z.len);
    const int qz = row_lane ? (int)lane / Y.len : 0, qy = row_lane ? (int)lane % Y.len : 0;
    const int cz = Z.cell(qz), cy = Y.cell(qy);
    const uint32_t row = (uint32_t)Z.index(cz) * kGroupSpan + (uint32_t)Y.index(cy);
    const uint32_t bits = row_lane ? s.rows[row] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < kGroupSpan; ++q)
        {
        const int cx = X.cell(min((int)q, X.len - 1));
        place[q] = (uint32_t)X.index(cx);
        const uint32_t c = G.cell_base + (uint32_t)((cz * Y.n + cy) * X.n + cx);
        st[q] = a.cell_rank ? a.cell_rank[c] : c;
        }
#pragma unroll
    for (uint32_t q = 0; q < kGroupSpan; ++q)
        {
        const uint32_t r = st[q];
        st[q] = a.start[r];
        ct[q] = a.start[r + 1];
        }
#pragma unroll
    for (uint32_t q = 0; q < kGroupSpan; ++q)
        {
        ct[q] = ((int)q < X.len && ((bits >> place[q]) & 1u)) ? ct[q] - st[q] : 0u;
        ncell += ct[q] != 0u ? 1u : 0u;
        ncand += ct[q];
        }
    uint32_t cells, total;
    uint32_t k0 = wave_exclusive_scan(ncell, cells);
    uint32_t p0 = wave_exclusive_scan(ncand, total);
#pragma unroll
    for (uint32_t q = 0; q < kGroupSpan; ++q)
        if (ct[q] != 0u)
            {
            s.delta[k0] = st[q] - p0;
            s.first[k0] = p0;
            s.seq[row * kGroupSpan + place[q]] = (uint16_t)k0;
            ++k0;
            p0 += ct[q];
            }
    wave_lds_fence();
    begin(cells, total);

    // the column's own candidate number (its particle is not its neighbor)
    uint32_t self = 0xffffffffu;
    if (in)
        {
        const uint32_t own = ((uint32_t)Z.index(me.c[2]) * kGroupSpan + (uint32_t)Y.index(me.c[1])) * kGroupSpan
                             + (uint32_t)X.index(me.c[0]);
        self = me.slot - s.delta[s.seq[own]];
        }

    // |FP32 error| <= 16 2^-24 ((|a| + |b|)^2 + r^2): at most a dozen
    // roundings of partial sums no larger than that, and the rounding of the
    // offsets; |a|, |b| <= the window's diagonal.  The direct tests' own error
    // is far inside 1e-5 r^2.  The fixed-point steps' part is the larger one in
    // a box of 20,000 and more list radii.
    const float wx = (float)(X.len * G.L[0] / X.n), wy = (float)(Y.len * G.L[1] / Y.n),
                wz = (float)(Z.len * G.L[2] / Z.n);
    const float diag2 = wx * wx + wy * wy + wz * wz;
    const float band = 1e-5f * a.thr + G.slip + (direct ? 0.0f : 9.5367e-7f * (4.0f * diag2 + a.thr));

    const float asq = ax * ax + ay * ay + az * az;
    const bool listed = in && (uint32_t)me.fixed.w < a.ntypes;
    // a result is |a - b|^2 - r^2 - band: negative for every pair that may be
    // listed, and above -2 band (in the integer order of negative floats:
    // below `near_bits`) where FP32 does not decide
    // (the direct tests' differences are the pair's own: no |a|^2)
    const float c0 = !listed ? 1e30f : (direct ? -a.thr : (ONEHOT == 0 ? asq - a.thr : asq)) - band;
    const int near_bits = __float_as_int(-2.0f * band);
    // matrix operands of columns 0..31 (lanes' values of half 0) and 32..63
    float bxy[2], bzw[2], cc[2];
    swap_halves(-2.0f * ax, -2.0f * ay, bxy[0], bxy[1]);
    swap_halves(-2.0f * az, 1.0f, bzw[0], bzw[1]);
    swap_halves(c0, c0, cc[0], cc[1]);
    f32x16 C0, C1;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        {
        C0[r] = cc[0];
        C1[r] = cc[1];
        }
    [[maybe_unused]] float bt[2][ONEHOT > 0 ? ONEHOT : 1];
    if constexpr (ONEHOT > 0)
        {
#pragma unroll
        for (int t = 0; t < ONEHOT; ++t)
            {
            auto radius = [&](uint32_t tj) {
                const double rl = (listed && tj < a.ntypes) ? a.r_listsq[(uint32_t)me.fixed.w * a.ntypes + tj] : 0.0;
                return rl > 0.0 ? -(float)rl : 1e30f;
            };
            swap_halves(radius(2u * t), radius(2u * t + 1u), bt[0][t], bt[1][t]);
            }
        }

    // candidate this lane reads of each 64: rows 8 (r / 4) + 4 h + r % 4 of a
    // 32 x 32 result are registers r of lanes of half h, so half h collects
    // candidates 32 h .. 32 h + 31 of a column (the direct tests take them in
    // lane order)
    const uint32_t off = direct ? lane : 32u * ((lane >> 2) & 1u) + 16u * h + 4u * ((lane >> 3) & 3u) + (lane & 3u);
    const uint64_t upto = (2ull << off) - 1ull;

    for (uint32_t seg = 0; seg < total; seg += kGroupSegment)
        {
        for (uint32_t w = lane; w < kGroupSegment / 64; w += 64)
            s.starts[w] = 0ull;
        wave_lds_fence();
        uint32_t before = 0; // cells that start before the current 64 candidates
        for (uint32_t k = lane; k < ((cells + 63u) & ~63u); k += 64)
            {
            const uint32_t p = k < cells ? s.first[k] : 0xffffffffu;
            if (p >= seg && p - seg < kGroupSegment)
                atomicOr(reinterpret_cast<unsigned long long*>(&s.starts[(p - seg) >> 6]), 1ull << ((p - seg) & 63u));
            before += (uint32_t)__popcll(__ballot(p < seg));
            }
        wave_lds_fence();
        const uint32_t end = min(total, seg + kGroupSegment);
        uint32_t next_before = before, slot_next = 0;
        uint64_t word_next = 0;
        uint32_t member_next = 0;
        int4 cand_next;
        auto fetch = [&](uint32_t P) {
            uint64_t w = s.starts[(P - seg) >> 6];
            w = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32)
                | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w);
            const uint32_t run = next_before + (uint32_t)__popcll(w & upto) - 1u;
            const uint32_t p = P + off;
            const uint32_t at = s.delta[run] + p; // past the last candidate: not a slot
            slot_next = p < total ? at : 0xffffffffu;
            cand_next = a.cell_fixed[p < total ? at : 0u];
            if constexpr (MEMBERS)
                member_next = a.members[p < total ? at : 0u];
            word_next = w;
            next_before += (uint32_t)__popcll(w);
        };
        fetch(seg);
        for (uint32_t P = seg; P < end; P += 64)
            {
            const int4 c = cand_next;
            const uint32_t slot = slot_next, member = member_next;
            const uint64_t word = word_next;
            const uint32_t base = next_before - (uint32_t)__popcll(word);
            if (P + 64 < end)
                fetch(P + 64);
            const bool real = slot != 0xffffffffu && (uint32_t)c.w < a.ntypes;
            uint32_t low = 0, high = 0, near_low = 0, near_high = 0;
            if (!direct)
                {
                const float x = (float)fixed_delta(c.x, fx0) * sx;
                const float y = (float)fixed_delta(c.y, fy0) * sy;
                const float z = (float)fixed_delta(c.z, fz0) * sz;
                const float w = real ? x * x + y * y + z * z : 1e30f;
                float xy[2], zw[2];
                swap_halves(x, y, xy[0], xy[1]);
                swap_halves(z, w, zw[0], zw[1]);
                [[maybe_unused]] float e[ONEHOT > 0 ? ONEHOT : 1][2];
                if constexpr (ONEHOT > 0)
                    {
#pragma unroll
                    for (int t = 0; t < ONEHOT; ++t)
                        swap_halves(c.w == 2 * t ? 1.0f : 0.0f, c.w == 2 * t + 1 ? 1.0f : 0.0f, e[t][0], e[t][1]);
                    }
                uint32_t mask[2], near[2] = {0u, 0u};
#pragma unroll
                for (int g = 0; g < 2; ++g)
                    {
                    const f32x16& C = g == 0 ? C0 : C1;
                    f32x16 d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(xy[0], bxy[g], C, 0, 0, 0);
                    f32x16 d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(xy[1], bxy[g], C, 0, 0, 0);
                    d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(zw[0], bzw[g], d0, 0, 0, 0);
                    d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(zw[1], bzw[g], d1, 0, 0, 0);
                    if constexpr (ONEHOT > 0)
                        {
#pragma unroll
                        for (int t = 0; t < ONEHOT; ++t)
                            {
                            d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(e[t][0], bt[g][t], d0, 0, 0, 0);
                            d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(e[t][1], bt[g][t], d1, 0, 0, 0);
                            }
                        }
                    int least = 0;
                    uint32_t m = 0;
#pragma unroll
                    for (int r = 15; r >= 0; --r)
                        m = __builtin_amdgcn_alignbit(m, __float_as_uint(d1[r]), 31);
#pragma unroll
                    for (int r = 15; r >= 0; --r)
                        m = __builtin_amdgcn_alignbit(m, __float_as_uint(d0[r]), 31);
                    mask[g] = m;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        least = min(min(least, __float_as_int(d0[r])), __float_as_int(d1[r]));
                    if (__ballot(least < near_bits) != 0ull)
                        {
                        uint32_t sure = 0;
#pragma unroll
                        for (int r = 15; r >= 0; --r)
                            sure = __builtin_amdgcn_alignbit(sure, __float_as_uint(d1[r] + 2.0f * band), 31);
#pragma unroll
                        for (int r = 15; r >= 0; --r)
                            sure = __builtin_amdgcn_alignbit(sure, __float_as_uint(d0[r] + 2.0f * band), 31);
                        near[g] = m & ~sure;
                        }
                    }
                // both words of the lane's own column
                swap_halves(mask[0], mask[1], low, high);
                swap_halves(near[0], near[1], near_low, near_high);
                }
            else
                {
                // the candidates one after the other, each against every
                // lane's own column: 17 instructions, and 30 for a column after
                // the other against all lanes' candidates (922 particles in two
                // cells an axis: 100 us a walk, and 182)
                const uint64_t ok = __ballot(real);
                int least = 0;
                auto half = [&](int first, float extra) {
                    uint32_t m = 0;
#pragma unroll 8
                    for (int q = first + 31; q >= first; --q)
                        {
                        float shift = c0 + extra;
                        if (ONEHOT > 0 || a.direct)
                            {
                            const uint32_t tq = (uint32_t)lane_value(c.w, q);
                            const double rl = (listed && tq < a.ntypes)
                                                  ? a.r_listsq[(uint32_t)me.fixed.w * a.ntypes + tq]
                                                  : 0.0;
                            shift = rl > 0.0 ? extra - (float)rl - band : 1e30f;
                            }
                        const float x = (float)fixed_delta(lane_value(c.x, q), me.fixed.x) * sx;
                        const float y = (float)fixed_delta(lane_value(c.y, q), me.fixed.y) * sy;
                        const float z = (float)fixed_delta(lane_value(c.z, q), me.fixed.z) * sz;
                        const float d = __builtin_fmaf(x, x, __builtin_fmaf(y, y, __builtin_fmaf(z, z, shift)));
                        m = __builtin_amdgcn_alignbit(m, __float_as_uint(d), 31);
                        least = min(least, __float_as_int(d));
                        }
                    return m & (uint32_t)(ok >> first);
                };
                low = half(0, 0.0f);
                high = half(32, 0.0f);
                if (__ballot(least < near_bits) != 0ull)
                    {
                    near_low = low & ~half(0, 2.0f * band);
                    near_high = high & ~half(32, 2.0f * band);
                    }
                }
            if (__ballot((near_low | near_high) != 0u) != 0ull)
                {
                // FP32 cannot decide these: the FP64 predicate of the host oracle
                uint64_t near = listed ? (uint64_t)near_high << 32 | near_low : 0ull;
                while (near != 0ull)
                    {
                    const uint32_t q = (uint32_t)__builtin_ctzll(near);
                    near &= near - 1ull;
                    const uint32_t run = base + (uint32_t)__popcll(word & ((2ull << q) - 1ull)) - 1u;
                    const uint32_t cs = s.delta[run] + P + q;
                    const uint32_t j = a.members[cs];
                    const double4 pi = a.pos[me.i], pj = a.pos[j];
                    const double rl = a.r_listsq[(uint32_t)me.fixed.w * a.ntypes + (uint32_t)a.cell_fixed[cs].w];
                    const double ex = min_image_1d(pi.x - pj.x, G.L[0], G.Linv[0]);
                    const double ey = min_image_1d(pi.y - pj.y, G.L[1], G.Linv[1]);
                    const double ez = min_image_1d(pi.z - pj.z, G.L[2], G.Linv[2]);
                    const bool hit = rl > 0.0 && rsq3_nofma(ex, ey, ez) <= rl;
                    const uint32_t bit = 1u << (q & 31u);
                    low = q < 32u ? (hit ? low | bit : low & ~bit) : low;
                    high = q < 32u ? high : (hit ? high | bit : high & ~bit);
                    }
                }
            const uint32_t ds = self - P;
            low &= ds < 32u ? ~(1u << ds) : 0xffffffffu;
            high &= ds - 32u < 32u ? ~(1u << (ds - 32u)) : 0xffffffffu;
            emit(low, high, P, off, MEMBERS ? member : slot);
            }
        }
    return served;
    }

} // namespace azp
