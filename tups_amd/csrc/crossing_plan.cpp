// Host plan of the Nl > 1 crossing over the nonzero elements of M.
//
// A crossing term sums over j = (l3, l4, R), but M(l1, l2, l3, l4, Q, R) vanishes
// for most of them whatever Q is: the shell R has to be one that the bonds of l1
// and l3 (and of l2 and l4) reach together.  At Nl = 5 a row (l1, l2) has 3 to 26
// of its 100 inner indices, at Nl = 9 1 to 54 of 486.  So the rows (l1, l2, Q) of
// one or of a few (l1, l2) form a block of 16 with the union of their indices as
// its inner dimension, in MFMA k-steps of four, instead of all rows in order with
// every index.
#include "crossing_plan.h"

#include <algorithm>
#include <numeric>

namespace tups {

namespace {

struct Block {
  std::vector<int> rows;
  std::vector<uint8_t> need[2];  // per routine: inner index needed
};

// Blocks of one target pair.  A class (l1, l2) fills whole blocks first; what is
// left of it goes on into the open block as far as it fits (split), or only when
// it fits entirely.  Splitting fills every block, at the price of wider unions.
std::vector<Block> pack_rows(const std::vector<std::vector<int>>& cls, const uint8_t* sup0, const uint8_t* sup1,
                             int nl, int kk, bool split) {
  std::vector<Block> out;
  int open = -1;
  auto add = [&](int b, int l, const int* r, size_t n) {
    Block& x = out[b];
    x.rows.insert(x.rows.end(), r, r + n);
    for (int k = 0; k < 2; ++k) {
      const uint8_t* s = (k ? sup1 : sup0) + (size_t)l * kk;
      for (int j = 0; j < kk; ++j) x.need[k][j] |= s[j];
    }
  };
  auto fresh = [&]() {
    Block b;
    b.need[0].assign(kk, 0);
    b.need[1].assign(kk, 0);
    out.push_back(std::move(b));
    return (int)out.size() - 1;
  };
  // l1 slowest: the blocks of a group then share most of their (l3, R)
  for (int l1 = 0; l1 < nl; ++l1)
    for (int l2 = 0; l2 < nl; ++l2) {
      const int l = l1 + nl * l2;
      const std::vector<int>& r = cls[l];
      size_t at = 0;
      while (r.size() - at >= (size_t)kPlanRows) {
        add(fresh(), l, r.data() + at, kPlanRows);
        at += kPlanRows;
      }
      while (at < r.size()) {
        const size_t left = r.size() - at;
        size_t room = open >= 0 ? kPlanRows - out[open].rows.size() : 0;
        if (room == 0 || (!split && room < left)) {
          open = fresh();
          room = kPlanRows;
        }
        const size_t n = std::min(left, room);
        add(open, l, r.data() + at, n);
        at += n;
      }
    }
  return out;
}

long long steps_of(const Block& b) {
  long long n = 0;
  for (int k = 0; k < 2; ++k) n += (std::accumulate(b.need[k].begin(), b.need[k].end(), 0) + 3) / 4;
  return n;
}

}  // namespace

void build_pae_plan(const std::vector<uint8_t>& support, const std::vector<int>& rows, int nl, int nibz, int kk,
                    PaePlanHost& out) {
  out = PaePlanHost();
  const int nl2 = nl * nl;
  std::vector<std::vector<int>> cls(nl2);
  if (rows.empty())
    for (int r = 0; r < nl2 * nibz; ++r) cls[r % nl2].push_back(r);
  else
    for (int r : rows) cls[r % nl2].push_back(r);
  struct Group {
    std::vector<Block> slot;       // kPlanBlocks, empty ones without rows
    std::vector<int> u[2];         // staged inner indices per routine
    int nchunk[2] = {0, 0}, len[2] = {0, 0};
  };
  std::vector<Group> groups;
  for (int p = 0; p < 2; ++p) {
    const uint8_t* s0 = support.data() + (size_t)(2 * p) * nl2 * kk;
    const uint8_t* s1 = s0 + (size_t)nl2 * kk;
    std::vector<Block> best;
    long long cost = -1;
    for (int split = 0; split < 2; ++split) {
      std::vector<Block> b = pack_rows(cls, s0, s1, nl, kk, split != 0);
      long long n = 0;
      for (const Block& x : b) n += steps_of(x);
      if (cost < 0 || n < cost) {
        cost = n;
        best = std::move(b);
      }
    }
    const int nb = (int)best.size();
    const int ng = (nb + kPlanBlocks - 1) / kPlanBlocks;
    out.groups[p] = ng;
    for (int g = 0; g < ng; ++g) {
      const int b0 = (int)((long long)nb * g / ng), b1 = (int)((long long)nb * (g + 1) / ng);
      Group gr;
      gr.slot.resize(kPlanBlocks);
      // the blocks over the four waves: longest first to the least loaded wave with room
      std::vector<int> order(b1 - b0);
      std::iota(order.begin(), order.end(), b0);
      std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return steps_of(best[x]) > steps_of(best[y]); });
      long long load[4] = {0, 0, 0, 0};
      int cnt[4] = {0, 0, 0, 0};
      for (int b : order) {
        int w = -1;
        for (int i = 0; i < 4; ++i)
          if (cnt[i] < kPlanSlots && (w < 0 || load[i] < load[w])) w = i;
        load[w] += steps_of(best[b]);
        gr.slot[w * kPlanSlots + cnt[w]++] = best[b];
      }
      for (int k = 0; k < 2; ++k) {
        for (int j = 0; j < kk; ++j)
          if (std::any_of(gr.slot.begin(), gr.slot.end(),
                          [&](const Block& b) { return !b.rows.empty() && b.need[k][j]; }))
            gr.u[k].push_back(j);
        gr.nchunk[k] = ((int)gr.u[k].size() + kPlanChunk - 1) / kPlanChunk;
        gr.len[k] = gr.nchunk[k] ? ((int)gr.u[k].size() + gr.nchunk[k] - 1) / gr.nchunk[k] : 0;
        out.chunks = std::max(out.chunks, gr.nchunk[k]);
        out.chunk_len = std::max(out.chunk_len, gr.len[k]);
      }
      groups.push_back(std::move(gr));
    }
  }
  const int nc = out.chunks;
  std::vector<int> mask(kk, 0);
  out.ubeg.resize(groups.size() * 2 * (nc + 1));
  out.seg.resize(groups.size() * 2 * nc * kPlanBlocks * 2);
  out.brow.assign(groups.size() * kPlanBlocks * kPlanRows, -1);
  for (size_t g = 0; g < groups.size(); ++g) {
    const Group& gr = groups[g];
    const int p = (int)g >= out.groups[0] ? 1 : 0;
    for (int sl = 0; sl < kPlanBlocks; ++sl)
      std::copy(gr.slot[sl].rows.begin(), gr.slot[sl].rows.end(),
                out.brow.begin() + (g * kPlanBlocks + sl) * kPlanRows);
    for (int k = 0; k < 2; ++k) {
      const int first = (int)out.ulist.size();
      out.ulist.insert(out.ulist.end(), gr.u[k].begin(), gr.u[k].end());
      for (int j : gr.u[k]) mask[j] |= 1 << (2 * p + k);
      const int total = (int)gr.u[k].size();
      for (int c = 0; c <= nc; ++c) out.ubeg[(g * 2 + k) * (nc + 1) + c] = first + std::min(total, c * gr.len[k]);
      for (int c = 0; c < nc; ++c)
        for (int sl = 0; sl < kPlanBlocks; ++sl) {
          const Block& b = gr.slot[sl];
          int* seg = &out.seg[(((g * 2 + k) * nc + c) * kPlanBlocks + sl) * 2];
          seg[0] = (int)out.step_blk.size();
          int n = 0, last = 0;
          const int u0 = std::min(total, c * gr.len[k]), u1 = std::min(total, (c + 1) * gr.len[k]);
          for (int u = u0; u < u1; ++u) {
            if (b.rows.empty() || !b.need[k][gr.u[k][u]]) continue;
            if (n % 4 == 0) {
              out.step_blk.push_back((int)(g * kPlanBlocks + sl) * 2 + k);
              out.kidx.push_back(0);
            }
            last = u - u0;
            out.kidx.back() |= last << (8 * (n % 4));
            out.kj.push_back(gr.u[k][u]);
            ++n;
          }
          // the last step repeats a staged row against zeros
          for (; n % 4; ++n) {
            out.kidx.back() |= last << (8 * (n % 4));
            out.kj.push_back(-1);
          }
          seg[1] = (int)out.step_blk.size();
        }
    }
  }
  out.steps = (long long)out.step_blk.size();
  for (int j = 0; j < kk; ++j)
    if (mask[j]) {
      out.used.push_back(j);
      out.used_by.push_back(mask[j]);
    }
}

}  // namespace tups
