// Several lanes per particle, for systems too small to fill the chip with one.
//
// The pair kernels give a particle one lane when there are enough particles:
// 256 CUs hold 262,144 lanes at four wavefronts a SIMD.  Below that the time
// is one lane's walk over its list, a serial chain that idle SIMDs don't
// shorten, so the list is dealt to 2^split lanes in batches of U entries
// (lane `sub` of a particle takes batches sub, sub + 2^split, ...), and their
// FP64 sums are added in a fixed tree at the end.  The lanes of a particle lie
// 64 >> split apart in one wavefront, so the list words that a wavefront reads
// for one batch stay consecutive.
//
// The split depends on the number of particles, the pair term and (the mixed
// pair form) the number of types, not on the list's layout, so every layout adds
// a particle's terms in the same order (up to pitches of 2^26 / 2^split: see
// launch_t).
#pragma once

#include "device_common.h"

namespace azp
{

// Up to 65,536 particles a split fills 2^18 lanes (four wavefronts a SIMD):
// Yukawa 900 particles 85 -> 12.4 us, DPD 60,000 37.5 -> 26.8, TwoPatchMorse
// 40,000 66 -> 33.  Above, a second lane has to pay for itself by the kernel's
// limits (us with one / two lanes):
//   Pair      the mixed form of one type: PerturbedLJ 90,000 31.2 / 29.4.  With
//             several types the table reads make it issue-bound: PerturbedLJ
//             90,000 48.2 / 53.8, Yukawa 67 / 72.
//   Short     Hertz, lists of about ten entries, which two lanes (mixed) or four
//             (FP64) make short enough, and the chip is full at 2^17 lanes:
//             mixed 900 particles 6.1, two 5.8, four 6.3, sixteen 7.4; 16,000
//             two 6.3, four 6.9; 130,000 9.2 / 10.2.  FP64 900 particles 9.1,
//             two 8.3, four 8.3, sixteen 12.1; 16,000 two 10.4, four 8.8.
//   PairFp64  one 512-lane workgroup a CU (LDS, registers), so the chip runs
//             rounds of 2^17 lanes, and two lanes gain where the rounds round
//             down: 160,000 PerturbedLJ 103 / 91, Yukawa 165 / 145; 195,000
//             92 / 75, 228 / 184; but PerturbedLJ of two types 90,000 62 / 71
//             and 228,000 130 / 147.
//   Dpd       70,000 45 / 38, 122,000 51 / 42.
//   Aniso     mixed 100,000 57 / 47, 131,000 59 / 50.
//   AnisoFp64 rounds of 2^16 lanes (one wavefront a SIMD at a time bound by
//             FP64 issue): 90,000 80 / 66, 100,000 81 / 85, 140,000 113 / 104,
//             180,000 115 / 122, 228,000 149 / 139.
//   Colloid   three divergent branches fill twice as many lanes: 50,000 87 with
//             2^18, 80 with 2^19; 73,000 200 -> 116.
enum class SplitTerm
    {
    Pair,
    Short,
    ShortFp64,
    PairFp64,
    Dpd,
    Aniso,
    AnisoFp64,
    Colloid,
    };
constexpr uint32_t kSplitLanes = 1u << 18;
constexpr uint32_t kSplitMax = 4;

// log2 of the lanes per particle.
inline uint32_t split_for(uint32_t N, SplitTerm term, uint32_t ntypes)
    {
    const uint32_t most = term == SplitTerm::Short ? 1u : term == SplitTerm::ShortFp64 ? 2u : kSplitMax;
    const uint32_t lanes = term == SplitTerm::Colloid ? 2 * kSplitLanes : most < kSplitMax ? kSplitLanes / 2 : kSplitLanes;
    if (N > kSplitLanes / 4 && N <= kSplitLanes)
        {
        if (term == SplitTerm::Pair && ntypes > 1)
            return 0;
        if (term == SplitTerm::PairFp64 || term == SplitTerm::AnisoFp64)
            {
            // two lanes where that takes fewer half rounds
            const uint32_t round = term == SplitTerm::PairFp64 ? kSplitLanes / 2 : kSplitLanes / 4;
            return (2 * N + round - 1) / round < 2 * ((N + round - 1) / round) ? 1u : 0u;
            }
        }
    uint32_t split = 0;
    while (split < most && ((uint64_t)N << (split + 1)) <= lanes)
        ++split;
    return split;
    }

// The workgroup-local column and the lane of that column that a lane is: a
// workgroup covers blockDim.x >> split columns, a wavefront 64 >> split.
struct SplitLane
    {
    uint32_t column;
    uint32_t sub;
    };

__device__ __forceinline__ SplitLane split_lane(uint32_t split)
    {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t shift = 6u - split;
    SplitLane s;
    s.column = ((threadIdx.x >> 6) << shift) + (lane & ((1u << shift) - 1u));
    s.sub = lane >> shift;
    return s;
    }

// The entries of one lane: entry m of its own sequence is list entry at(m).
// With a split the particle's lanes take consecutive fours.
template<bool SPLIT> struct LaneEntries
    {
    uint32_t split, first;
    __device__ __forceinline__ LaneEntries(uint32_t split_, uint32_t sub) : split(split_), first(4u * sub) { }
    __device__ __forceinline__ uint32_t at(uint32_t m) const
        {
        return SPLIT ? ((m & ~3u) << split) + first + (m & 3u) : m;
        }
    __device__ __forceinline__ uint32_t count(uint32_t nn) const
        {
        if (!SPLIT)
            return nn;
        const uint32_t rest = nn & ((4u << split) - 1u);
        return ((nn >> (2u + split)) << 2) + (rest > first ? min(rest - first, 4u) : 0u);
        }
    };

// v plus its value in the lane `across` away (32, 16, 8 or 4).  Register swaps
// and row operations: only the two lanes of a pair read each other, so the
// lanes of a column without a particle may have left.
template<int across> __device__ __forceinline__ double add_across(double v)
    {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    if constexpr (across == 32 || across == 16)
        {
        const auto swap = [](int x) {
            if constexpr (across == 32)
                return __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
            else
                return __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
        };
        const auto l = swap(lo), h = swap(hi);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
        }
    else
        {
        const auto other = [](int x) {
            if constexpr (across == 8)
                return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false); // row_ror:8
            else
                {
                const int up = __builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0x5, false);  // row_shl:4, lanes with bit 2 clear
                return __builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false);         // row_shr:4, the others
                }
        };
        return v + __hiloint2double(other(hi), other(lo));
        }
    }

// Sums over a particle's lanes, the same values in each of them.  All values
// take a stage before the next: one after the other, the exchanges' latencies
// added up to 2 us.
template<class... D> __device__ __forceinline__ void split_sum(uint32_t split, D&... v)
    {
    static_assert(kSplitMax == 4, "stages of the sum");
    if (split > 0u)
        ((v = add_across<32>(v)), ...);
    if (split > 1u)
        ((v = add_across<16>(v)), ...);
    if (split > 2u)
        ((v = add_across<8>(v)), ...);
    if (split > 3u)
        ((v = add_across<4>(v)), ...);
    }

} // namespace azp
