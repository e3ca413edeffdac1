// tfgfa_plan.h - which forward kernel runs a problem: host code only, shared by the launch
// (tfgfa_fwd.hip) and the binding, so the rule can be tested without a GPU.
#ifndef TFGFA_PLAN_H
#define TFGFA_PLAN_H

#include <algorithm>

namespace tfgfa {

// A grid that leaves CUs idle, or fills them once, takes as long as its longest wave's chain of
// half-steps (one per 32 keys, ~0.4 us each whatever runs beside them); splitting the keys over
// several waves shortens the chain, at the price of a merge and, where fewer than 4 waves share a K/V
// tile, of more traffic from the L2.
//   kWhole    fwd_kernel, 4 row waves, one group: the most work per byte, three workgroups a CU
//   kHalves   fwd_split_kernel: one 32-row block, 4 waves
//   kGroups2  4 row waves x 2 key groups (128 rows, 8 waves): one workgroup a CU
//   kPairs    2 row waves x 2 key groups (64 rows, 4 waves): two a CU, one past 64 head dims
//   kGroups4  2 row waves x 4 key groups (64 rows, 8 waves): one a CU, head dims up to 64
// The lines below are where the measured times cross on 256 CUs.  They rest on every plan timed over
// 21600 problems (up to 640 128-row blocks, chains of 1 to 128 halves, causal with N_q = N_k, 2 N_k
// and 4 N_k, unmasked, and drawn sizes, head dims 32 to 128, both types): what they choose takes 1.0043
// of the best plan's time in the mean, and at most 1.03 of the time of kHalves up to one block per CU
// and kWhole past it but for 13 problems (1.08 the most).
// Some of the rows (bf16, us, graph replays; "blocks": 128-row query blocks, h: halves of the longest
// chain; * the choice):
//   D = 64, N x N causal         blocks  h   kWhole kHalves kGroups2 kPairs kGroups4
//     H32 N128                      32    4     5.4    4.1*     5.8     4.8     5.2
//     H14 N1152                    126   36    15.7   10.3     13.6    10.6     9.8*
//     H25 N704 (550 row blocks)    150   22    10.7    8.5*    10.1     8.8     9.3
//     H18 N1152                    162   36    15.8   11.0     13.6    10.9*   11.1
//     H192 N128                    192    4     5.6*   6.5      6.1     5.9     8.7
//     H46 N448                     184   14     8.3    7.8      8.3     7.4*    9.4
//     H21 N1152                    189   36    16.2   14.4     14.0    11.7*   13.4
//     H12 N2048                    192   64    24.6   18.5     20.7    16.5    15.6*
//     H30 N960                     240   30    13.4   13.4     12.3    10.6*   13.0
//     H30 N1152                    270   36    16.3   16.8     14.0    11.8*   17.3
//     H20 N2048                    320   64    25.4   26.7     21.0    18.4*   24.6
//     H24 N2048                    384   64    26.0   30.1     21.4*   23.2    26.7
//   D = 64, unmasked (16 heads) or causal with N_q well past N_k (marked c): every chain is as long
//     768 x 64                      96    2     4.5*   5.0      5.5     5.0     5.4
//     1024 x 960                   128   30    13.5   12.4*    12.8    10.1     9.7
//     1024 x 1152                  128   36    15.5   13.3     13.7    10.7    10.6*
//     1280 x 352                   160   11     7.8*  10.1      8.3     8.2    12.0
//     1536 x 704                   192   22    11.1   15.0     11.1*   11.4    14.3
//     1792 x 1152                  224   36    15.6   23.2     14.1*   14.6    18.3
//     2048 x 448                   256   14     8.8*  13.9      9.3     9.6    12.5
//     2048 x 1312                  256   41    17.6   26.4     16.1*   17.0    20.8
//     2176 x 1152                  272   36    21.3*  28.6     26.2    21.7    26.3
//     H37 896 x 448 c              259   14     9.3*  13.9     11.3    11.7    16.0
//     H12 4096 x 2048 c            384   64    28.6*  41.5     34.3    30.6    34.0
//   D = 128, N x N causal
//     H18 N448                      72   14    12.0    9.5*    12.2    11.3
//     H20 N704 (440 row blocks)    120   22    15.7   14.5     15.2    13.6*
//     H12 N1312                    132   41    24.8   22.5     22.4    18.7*
//     H80 N256                     160    8    10.3*  13.2     11.4    13.7
//     H29 N704                     174   22    17.7   23.4     16.3*   18.5
//     H21 N1152                    189   36    24.9   32.8     22.5    22.5*
//     H30 N1152                    270   36    25.5   43.0     22.8*   30.3
//     H39 N832                     273   26    20.7*  39.3     21.4    26.1
//     H32 N2048                    512   64    47.0  107.5     43.4*   62.8
//   D = 128, unmasked (16 heads; 8 where marked)
//     512 x 448                     64   14    11.8    9.8*    13.0    10.9
//     768 x 192                     96    6     8.2*   9.8     10.1     8.5
//     1024 x 704                   128   22    15.9   22.5     16.1    13.6*
//     H8 2176 x 448                136   14    11.9*  24.3     13.1    19.8
//     1536 x 1152                  192   36    22.5   44.3     21.3*   31.5
//     2176 x 2048                  272   64    49.1* 112.6     64.1    71.7
// The choice depends on the sizes only, never on strides or outputs, so every instance of one
// problem takes the same arithmetic.
enum class Plan { kWhole, kHalves, kGroups2, kPairs, kGroups4 };

inline Plan choose_plan(long long heads, int cu_count, int Nq, int Nk, int D, bool causal) {
  auto pieces = [](long long n, int size) { return (n + size - 1) / size; };
  const long long cu = cu_count;
  const long long h = pieces(causal ? std::min(Nq, Nk) : Nk, 32);
  const long long blocks = heads * pieces(Nq, 128);
  const long long pair_blocks = heads * pieces(Nq, 64);  // kPairs' and kGroups4's grid
  const long long row_blocks = heads * pieces(Nq, 32);   // kHalves' grid
  // Causal chains have every length up to h, until N_q passes N_k: then more and more have h.  Where
  // most are shorter, a second round's short ones run beside the first's long ones.
  const bool triangle = causal && 4LL * Nq <= 5LL * Nk;
  const bool wedge = causal && 5LL * Nq <= 8LL * Nk;
  const bool half = causal && Nq <= 2LL * Nk;
  if (blocks > 2 * cu) return Plan::kWhole;
  if (D <= 64) {
    // One or two halves: four waves have nothing to share, unless the grid is too small to matter.
    if (h <= 2 && 4 * blocks > cu && !(triangle && 2 * blocks <= cu) && !(causal && row_blocks <= cu))
      return Plan::kWhole;
    // One round of kHalves is two workgroups a CU; a triangle's second one fits beside it.
    if (h <= 32 && (row_blocks <= 2 * cu || (triangle && h >= 14 && 15 * row_blocks <= 32 * cu) ||
                    (triangle && h >= 20 && 5 * row_blocks <= 12 * cu)))
      return Plan::kHalves;
    if (pair_blocks <= cu) return Plan::kGroups4;  // one round
    if (blocks <= cu) {
      if ((causal && h >= 57 && 5 * blocks <= (triangle ? 4 : 3) * cu) ||
          (triangle && h >= 33 && 8 * blocks <= 5 * cu))
        return Plan::kGroups4;
      if (triangle) return h >= 7 ? Plan::kPairs : Plan::kWhole;
      if (half) return h >= (6 * blocks <= 5 * cu ? 8 : 15) ? Plan::kPairs : Plan::kWhole;
      if (h <= 14) return causal && h >= 8 && 5 * pair_blocks <= 6 * cu ? Plan::kPairs : Plan::kWhole;
      return causal && 5 * blocks <= 4 * cu ? Plan::kPairs : Plan::kGroups2;
    }
    if (wedge && 4 * blocks <= 5 * cu && h >= (6 * blocks <= 7 * cu ? 24 : 28)) return Plan::kPairs;
    return (triangle && h >= 56) || (half && h >= 36 && 8 * blocks <= 9 * cu) ? Plan::kGroups2 : Plan::kWhole;
  }
  // One round of kHalves, and of kPairs, is one workgroup a CU.
  if (row_blocks <= cu || (half && h >= 10 && 4 * row_blocks <= 5 * cu) ||
      (triangle && h >= 11 && 5 * row_blocks <= 7 * cu) || (triangle && h >= 18 && 2 * row_blocks <= 3 * cu))
    return Plan::kHalves;
  if (2 * blocks <= cu) return h >= 8 ? Plan::kPairs : Plan::kWhole;
  if ((pair_blocks <= cu && h >= 9) || (half && h >= (triangle ? 20 : 22) && 8 * pair_blocks <= 9 * cu))
    return Plan::kPairs;
  if (blocks <= cu) {
    if (!triangle) return h >= 20 ? Plan::kGroups2 : Plan::kWhole;
    return h <= 12 ? Plan::kWhole : h >= 28 && 4 * blocks <= 3 * cu ? Plan::kPairs : Plan::kGroups2;
  }
  return (triangle && h >= (4 * blocks <= 5 * cu ? 32 : 56)) || (half && h >= 64 && 8 * blocks <= 9 * cu)
             ? Plan::kGroups2
             : Plan::kWhole;
}

}  // namespace tfgfa

#endif  // TFGFA_PLAN_H
