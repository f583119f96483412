// Host plan of the Nl > 1 crossing (crossing_plan.cpp); no device code.
#pragma once
#include <cstdint>
#include <vector>

namespace tups {

// Plan of the Nl > 1 crossing over the nonzero elements of M (crossing_plan.cpp).
// For each target pair p the kept rows (l1, l2, Q) are packed into blocks of
// kPlanRows that need few inner indices j = l3 + Nl l4 + Nl^2 R; kPlanBlocks
// blocks (kPlanSlots for each of four waves) form a group, one workgroup per
// column tile.  Groups of pair 0 come first, then those of pair 1.
constexpr int kPlanRows = 16, kPlanSlots = 2, kPlanBlocks = 4 * kPlanSlots;
constexpr int kPlanChunk = 104;  // inner indices staged at once: 52 KB of LDS, three workgroups per CU; a byte counts them
struct PaePlanHost {
  int groups[2] = {0, 0};
  int chunks = 1;             // the most staging chunks of a (group, routine)
  int chunk_len = 0;          // the longest staging chunk
  long long steps = 0;        // MFMA k-steps (16 rows x 4 inner indices) of all blocks
  std::vector<int> ubeg;      // [(group 2 + routine) (chunks + 1) + c]: first entry of staging chunk c in ulist
  std::vector<int> ulist;     // inner indices to stage
  std::vector<int> seg;       // [((group 2 + routine) chunks + c) kPlanBlocks + slot] 2 + {0, 1}: k-steps begin, end
  std::vector<int> kidx;      // [step]: LDS rows of its four inner indices within their chunk, a byte each
  std::vector<int> kj;        // [4 step + k]: the inner index, -1 for padding
  std::vector<int> step_blk;  // [step]: (group kPlanBlocks + slot) 2 + routine
  std::vector<int> brow;      // [(group kPlanBlocks + slot) kPlanRows + r]: row l1 + Nl l2 + Nl^2 m, -1 for none
  std::vector<int> used;      // [i]: inner index with a nonzero element in some routine
  std::vector<int> used_by;   // [i]: bit 2 p + routine set when that routine needs used[i]
};
// support: [k = 2 p + routine][l1 + Nl l2][j], nonzero where M_k has a nonzero element for some Q
void build_pae_plan(const std::vector<uint8_t>& support, const std::vector<int>& rows, int nl, int nibz, int kk,
                    PaePlanHost& out);

}  // namespace tups
