// Half-length transforms on the host: over every planned length and grids
// from its shortest to its longest, the rule's inequalities hold, the buffers
// a half-length request puts into its workspace do not overlap, and the pass B
// and image items of a launch name every (row block, share) and every (cell,
// part) once.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "ldm_plan.h"

int main() {
  int fails = 0, halves = 0, wholes = 0, shared = 0, whole_shared = 0;
#define CHECK(c, ...) \
  if (!(c)) { std::fprintf(stderr, "check failed: %s: ", #c); std::fprintf(stderr, __VA_ARGS__); std::fprintf(stderr, "\n"); ++fails; }
  radis_ldm_db db;
  db.n = 1000;
  for (int64_t nv = 300; nv < 1100000; nv = nv * 41 / 40 + 7)
    for (int m_cap : {1, 2, 9, 16, 30, 61, 144, 400})
      for (double wg : {0.0, 0.01, 5.0})
        for (int tile : {0, 16, 1024}) {
          Req R;
          R.r.tile_w = tile;
          R.r.Tgas = 1000.0;
          R.nv = nv;
          R.delta_w = 0.002;
          R.wg_hi = wg;
          R.i1 = 1000;
          R.m_cap = m_cap;
          if (plan_fft(nv, 0, R.plan)) continue;
          choose_split_b(&R, 1, 256);
          size_t total = 0;
          if (layout_request(R, total)) continue;
          CHECK(check_layout(R, total) == 0, "nv %lld: %s", (long long)nv, g_err);
          CHECK(R.tL == (int64_t)R.tn1 * R.tn2, "split");
          if (!R.half) {
            ++wholes;
            CHECK(R.tL == R.plan.L && R.n_cell == 0 && R.n_share <= 4, "whole length");
            if (R.n_share > 2) {  // their buffers behind Y, every (row block, share) once
              ++whole_shared;
              const size_t y1 = R.off_y + (size_t)((m_cap + 1) / 2) * R.plan.L * 8;
              CHECK(R.off_share >= y1 && R.off_share + (size_t)R.n_share * R.tL * 8 <= R.off_rows, "whole-length shares");
              std::set<int> once;
              const LdmItemPlan P = item_plan(db, R);
              const int b0 = plan_items(P) - P.n_rowB - P.n_colC;
              for (int i = b0; i < b0 + P.n_rowB; ++i) once.insert(plan_item(P, i).w);
              for (int w : once) CHECK((w >> 4) < (R.tn1 >> R.bX[1]) && (w & 15) < R.n_share, "row block and share");
              CHECK((int)once.size() == P.n_rowB, "every row block and share once");
            }
            continue;
          }
          ++halves;
          shared += R.n_share > 2;
          const int64_t V = nv + 1, gap = R.tL - nv;
          CHECK(R.plan.fc && R.plan.wrap_k > 0 && R.fill_groups == 1 && R.tL * 2 == R.plan.L && R.tL >= V, "half of a compiled split");
          CHECK(gap >= (int64_t)IMG_TILES_PER_GAP * R.tile_w && gap >= IMG_SIGMAS_PER_GAP * wg * std::sqrt(10.0) / (2.3548 * R.delta_w),
                "gap %lld", (long long)gap);
          CHECK(5 * (int64_t)R.cell_tiles * R.tile_w <= 2 * gap && R.n_cell <= IMG_MAX_CELLS && R.n_cell >= 1 &&
                    (int64_t)R.n_cell * R.cell_tiles >= R.n_tiles && (int64_t)(R.n_cell - 1) * R.cell_tiles < R.n_tiles, "cells");
          const size_t pcap = (m_cap + 1) / 2, share = (size_t)R.tL * 8;
          const size_t y0 = R.off_y, y1 = y0 + pcap * share, img1 = R.off_img + (size_t)R.n_cell * IMG_NODES * 8,
                       mom1 = R.off_mom + (size_t)R.n_tiles * std::max(1, m_cap / 2 < LDM_MAX_AX ? m_cap / 2 : LDM_MAX_AX) * 16,
                       end = y0 + pcap * (size_t)R.plan.L * 8;
          CHECK(R.off_ldm + pcap * 2 * R.stride * 4 <= R.off_b && R.off_b + 2 * share <= y0, "LDM, B, Y");
          CHECK(y1 <= R.off_img && img1 <= R.off_mom && mom1 <= end, "Y, correction, moments");
          CHECK(R.off_share == R.off_b ? R.n_share <= 2 : (mom1 <= R.off_share && R.off_share + R.n_share * share <= end), "shares");
          CHECK(R.off_free >= mom1 && (R.off_share == R.off_b || R.off_free >= R.off_share + R.n_share * share) && R.off_free <= end + 255,
                "unused part");
          const LdmItemPlan P = item_plan(db, R);
          std::set<std::pair<int, int>> seen;
          const int b0 = plan_items(P) - P.n_rowB - P.n_colC, rb = R.tn1 >> R.bX[1];
          CHECK(P.n_rowB == rb * R.n_share, "pass B items");
          for (int i = b0; i < b0 + P.n_rowB; ++i) {
            const int4 t = plan_item(P, i);
            const int k = t.y * R.split_b + t.z;
            CHECK(k / R.n_share < rb && t.w == (k / R.n_share << 4 | k % R.n_share), "row block");
            seen.insert({k / R.n_share, k % R.n_share});
          }
          CHECK((int)seen.size() == P.n_rowB, "every row block and share once");
          seen.clear();
          for (int i = 0; i < P.n_img; ++i) {
            const int4 t = plan_item(P, plan_items(P) + i);
            CHECK(t.y < R.n_cell && t.z * IMG_TARGETS < R.n_cell * IMG_NODES, "image item");
            seen.insert({t.y, t.z});
          }
          CHECK((int)seen.size() == P.n_img && P.n_img == R.n_cell * ((R.n_cell * IMG_NODES + IMG_TARGETS - 1) / IMG_TARGETS),
                "every cell and part once");
        }
  // the shares' pairs: [P s inv >> 16, P (s + 1) inv >> 16), the last up to P
  for (unsigned n = 1; n <= 8; ++n)
    for (unsigned P = 0; P <= 128 * 128 / 2; ++P) {
      const unsigned inv = 65536u / n;
      unsigned at = 0;
      for (unsigned s = 0; s < n; ++s) {
        const unsigned e = s + 1 == n ? P : (unsigned)(P * (s + 1)) * inv >> 16;
        if (e < at || e - at > P / n + 2) { CHECK(false, "share %u of %u, %u pairs", s, n, P); break; }
        at = e;
      }
    }
  CHECK(halves > 1000 && wholes > 1000 && shared > 100 && whole_shared > 100, "%d half-length, %d whole, %d with more than two shares", halves, wholes, shared);
  std::printf("%d half-length plans (%d with more than two shares), %d whole, %d failed checks\n", halves, shared, wholes, fails);
  return fails ? 1 : 0;
}
