// Launch plans that depend on sizes only (host code), apart from the kernels so that tests can
// ask for them without a GPU.
#pragma once

#include <algorithm>

#include "common.h"

namespace gq {

// ---- gemm_q8.hip: the prefill product on int8 MFMA

struct GemmQ8Plan {
    int mt;       // 32-token tiles per workgroup
    int ks, sps;  // K splits and stages (4 quant blocks) per split
    int seg;      // stages per segment: a split's fp32 chains start anew every seg stages
};

// What bounds the rounding of a product of nb blocks: summed in fp32 chains of n blocks, whose
// sums are added one after the other, its squared error grows as n + (number of chains). `chain`
// is that figure for the order in which the fp16-pair kernel (gemm.hip) summed such a product
// when it took all of them, the yardstick of plan_gemm_q8: K steps of 2 blocks, splits while its
// tiles of 128 rows x 128 or 64 tokens leave CUs idle, and a last partial round of tiles split on
// its own (there the mean over the rows). `part_bytes` are its partials, the room that the
// workspace keeps for them. Both stay as they are when that kernel's own plan changes.
struct Fp16PairSums {
    double chain;
    size_t part_bytes;
};
inline Fp16PairSums fp16_pair_sums(int64_t N, int64_t K, int64_t M, int64_t ncu) {
    const int64_t nt = cdiv(N, 128), nb = K / QK, nk = cdiv(K, 64);
    const int64_t bm = (M > 64 && nt >= 16) || nt * cdiv(M, 128) >= ncu ? 128 : 64;
    const int64_t mtiles = cdiv(M, bm), tiles = nt * mtiles;
    auto sums = [&](int64_t want, int64_t rows) {  // `rows` weight rows in about `want` splits
        const int64_t spk = cdiv(nk, std::max<int64_t>(1, want)), ks = cdiv(nk, spk);
        return Fp16PairSums{(double)(std::min<int64_t>(2 * spk, nb) + ks),
                            ks > 1 ? (size_t)ks * M * rows * sizeof(float) : 0};
    };
    if (tiles < ncu) return sums(std::min<int64_t>({cdiv((bm == 128 ? 1 : 2) * ncu, tiles), nk / 4, 16}), N);
    if (bm == 128 && tiles > ncu && ncu % mtiles == 0) {
        const int64_t head = tiles / ncu * (ncu / mtiles), tail = (nt - head) * mtiles;
        const int64_t kt = tail > 0 && 2 * tail <= ncu ? std::min<int64_t>({ncu / tail, nk / 4, 4}) : 1;
        if (kt >= 2) {
            const double f = (double)(head * 128) / (double)N;
            const Fp16PairSums t = sums(kt, N - head * 128);
            return {f * sums(1, N).chain + (1.0 - f) * t.chain, t.part_bytes};
        }
    }
    return sums(1, N);
}

// Tiles of 32 mt tokens, ks K splits: the pair with the shortest expected launch. Measured per
// stage (Q4_0 and Q8_0 alike): a workgroup alone on its CU takes 0.56 + 0.245 mt us, two that
// share one 0.53 + 0.485 mt us together (short tiles keep more than two and stay at 0.5 us
// each), so a grid costs what its fullest CU does: 528 tiles of mt = 4 took 143 us where 512
// took 105. Smaller tiles read the weights more often, out of L2, but leave fewer rows of
// padding and fill the CUs evenly: 12288 x 4096 at 300 tokens 86 us at mt = 4, 56 at mt = 2;
// 22016 x 4096 at 333 tokens 132 and 111 (mt = 3); 16384 x 4096 at 512 stays at mt = 4. A split
// costs the reduce's launch (2 to 3 us behind the product) and its traffic (about 6 TB/s):
// 4096 x 11008 at 512 tokens 102 us in one part, 90 in three, 77 in four; 1600 x 960 at 37 tokens
// 10.9 in one, 9.9 in two. Segments cost two tiles a workgroup 5 to 7% (how many hardly
// matters), one tile 1%, or for Q8_0 its third wave per SIMD: 5120 x 960 at 333 tokens (Q4_0)
// 21.0 us as 2 tiles in two parts, 14.6 as one tile in one part and four segments.
// Where a split's one chain would pass fp16_pair_sums (in Q8_0, whose block sums, 32 products of 19
// bits and more, round there, up to 6 blocks more while that is no more than 20), workgroups of at
// most two tiles sum it in segments, cut where blocks per chain + chains are least (22016 x 4096: 12 + 11 instead
// of 129): the error is no larger than in that kernel's order, most often far smaller. The two
// kinds are timed less alike than this model says, so segments have to save a sixth where whole
// splits keep the bound too.
// Partials within part_bytes: split 0 stands in dst, the others in the workspace.
inline GemmQ8Plan plan_gemm_q8(int type, int64_t N, int64_t K, int64_t M, size_t part_bytes, int64_t ncu) {
    const int64_t nb = K / QK, ns = std::max<int64_t>(1, cdiv(nb, 4)), nt = cdiv(N, 128);
    const double slab = (double)M * (double)N * sizeof(float);
    int64_t most = 1;
    if (slab > 0) most += (int64_t)((double)part_bytes / slab);
    most = std::min<int64_t>({most, std::max<int64_t>(1, ns / 3), 16});  // at least 3 stages each
    most = cdiv(ns, cdiv(ns, most));  // the splits that many leave non-empty
    double bound = fp16_pair_sums(N, K, M, ncu).chain;
    if (type == GQ_TYPE_Q8_0) bound = std::max(bound, std::min(bound + 6.0, 20.0));
    GemmQ8Plan whole{1, 1, (int)ns, (int)ns}, cut = whole;
    double whole_us = 1e300, cut_us = 1e300;
    for (int mt = (int)std::max<int64_t>(1, std::min<int64_t>(4, cdiv(M, 32))); mt >= 1; --mt) {
        const int64_t tiles = nt * cdiv(M, 32 * mt);
        const double one = 0.56 + 0.245 * mt, two = 0.53 + 0.485 * mt;
        for (int64_t z = 1; z <= most; ++z) {
            const int64_t sps = cdiv(ns, z), ks = cdiv(ns, sps);
            if (ks != z) continue;  // the same split as a smaller z
            int64_t segs = 1, seg = sps;
            auto chain = [&] { return (double)(std::min<int64_t>(4 * seg, nb) + segs + z - 1); };
            if (mt <= 2 && chain() > bound) {
                int64_t least = seg;
                double c = chain();
                for (seg = 1; seg < sps && seg * seg <= 2 * sps; ++seg) {  // (least near sqrt(sps / 4))
                    segs = cdiv(sps, seg);
                    if (chain() <= c) c = chain(), least = seg;
                }
                seg = least, segs = cdiv(sps, least);
            }
            if (chain() > bound) continue;
            const int64_t load = cdiv(tiles * ks, ncu), pairs = load / 2;
            const bool three = mt == 1 && load > 1 && (type != GQ_TYPE_Q8_0 || segs == 1);  // registers for 3 waves a SIMD
            double us = (double)sps * (three ? 0.5 * (double)load : pairs * two + (load & 1) * one);
            if (mt > 1) us += 3.0 * (double)((load - 1) / 2);  // a further round's first loads and last stores
            if (mt == 2 && segs > 1) us *= 1.06;
            if (ks > 1) us += 2.5 + slab * 2 * (double)ks / 6e6;
            if (segs == 1 && us < whole_us) whole_us = us, whole = GemmQ8Plan{mt, (int)ks, (int)sps, (int)seg};
            if (segs > 1 && us < cut_us) cut_us = us, cut = GemmQ8Plan{mt, (int)ks, (int)sps, (int)seg};
        }
    }
    return whole_us <= 1.2 * cut_us ? whole : cut;
}

// ---- attention.hip: k_attn_pre (prompt attention)

struct AttnPrePlan {
    int nqw;  // sub-tiles of 32 queries per workgroup; its 8 waves deal the keys 8 / nqw ways
    int ks;   // key splits over workgroups
};

// NQ query vectors per kv head. Sub-tiles: 1 below 512 tiles of 32 query vectors, 2 below 1024,
// then 4, each longer over the keys but fewer workgroups. 32 / 32 heads, 128 dims, causal, us with
// 1, 2 and 4: 256 rows (256 tiles) 15.3, 17.2, 21.8; 512 rows 28.6, 22.8, 31.2; 1024 rows 64.8,
// 49.7, 50.9; 2048 rows 180, 150, 136. Between 257 and 511 tiles 2 would be faster at equal
// heads (300 rows 25.1, 19.0) and no slower at 12 / 2 (768 rows 25.4, 25.2).
// Key splits: as many as fill the CUs (one workgroup fills a CU) where each wave would otherwise
// walk 4 blocks of 32 keys or more, and keeps 2; at most `most`, the splits the caller's
// workspace holds. The merge is a launch of its own (~4 us).
inline AttnPrePlan plan_attn_pre(int64_t NQ, int64_t Hkv, int64_t n_kv, int64_t most) {
    const int64_t t32 = cdiv(NQ, 32) * Hkv;
    const int nqw = t32 >= 1024 ? 4 : t32 >= 512 ? 2 : 1;
    const int64_t wgs = cdiv(NQ, 32 * nqw) * Hkv, per_wave = cdiv(n_kv, 32) / (8 / nqw);
    if (per_wave < 4) return {nqw, 1};
    return {nqw, (int)std::max<int64_t>(1, std::min<int64_t>({256 / wgs, per_wave / 2, most, 8}))};
}

}  // namespace gq
