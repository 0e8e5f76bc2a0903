// Edges of the host planning, one section per argument:
//   wide_tile   an explicit fill tile too wide for two LDM rows is refused by
//               the planning itself, alone and beside requests that plan
//   shares_in_y pass B's partial spectra in Y: no share's overlaps what another
//               reads or writes
//   axis_groups width candidate blocks per workgroup from the whole launch's
//   half_cost   half-length transforms where they cost the launch less
//   image_room  pass B's shares beside many image items
//   no_allocation  planning a lone request allocates nothing
//   scratch     the no-allocation entry point's array holds what it held with
//               the plain splits' tables
//   bytes       the admission figure: at most one transform's buffers and a
//               second partial spectrum, and no less than what batches of such
//               requests lay out
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "ldm_plan.h"

long g_news = 0;  // allocations through operator new
void* operator new(size_t n) {
  ++g_news;
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

int g_fail = 0;
#define CHECK(c, ...)                                  \
  do {                                                 \
    if (!(c)) {                                        \
      std::fprintf(stderr, "check failed: %s: ", #c);  \
      std::fprintf(stderr, __VA_ARGS__);               \
      std::fprintf(stderr, "\n");                      \
      ++g_fail;                                        \
    }                                                  \
  } while (0)

// A request of nv points and m_cap LDM rows (widths of a 0.002 cm-1 grid).
Req request(int64_t nv, int m_cap, int tile_w = 0, int flags = 0) {
  Req R;
  R.r.tile_w = tile_w;
  R.r.Tgas = 1000.0;
  R.r.flags = flags;
  R.nv = nv;
  R.delta_w = 0.002;
  R.wg_hi = 0.01;
  R.i1 = 1000;
  R.m_cap = R.m_need = m_cap;
  CHECK(plan_fft(nv, 0, R.plan) == 0, "%s", g_err);
  return R;
}

void wide_tile() {
  for (int64_t nv : {9000, 20001, 150001, 500001})
    for (int w : {2048, 4096})
      for (int m_cap : {1, 2, 3, 16, 144})
        for (int beside : {0, 1, 2}) {  // alone, before and after a request that plans
          Req reqs[2] = {request(nv, m_cap, w), request(20001, 16)};
          if (beside == 2) std::swap(reqs[0], reqs[1]);
          const int n = beside ? 2 : 1;
          const bool fits = fill_tile_bytes(m_cap, w) <= (size_t)FILL_LDS_MAX || 2 * fill_tile_bytes(1, w) <= (size_t)FILL_LDS_TARGET;
          const int rc = choose_split_b(reqs, n, 256);
          CHECK(rc == (fits ? 0 : RADIS_LDM_ERANGE), "nv %lld, W %d, %d rows: %d", (long long)nv, w, m_cap, rc);
          size_t total = 0;
          CHECK((layout_request(reqs[beside == 2], total) == 0) == fits, "W %d, %d rows", w, m_cap);
        }
}

// Partial spectra in Y: every share of every number of pairs up to the planned
// one writes a pair of its own that no other share reads (share_pairs, and
// k_finalize for share_at).
void shares_in_y() {
  int split = 0;
  for (int64_t nv : {4000, 9000, 20001, 50001, 150001})
    for (int m_cap = 1; m_cap <= 144; ++m_cap) {
      Req R = request(nv, m_cap, 0, RADIS_LDM_MIN_RMS);
      CHECK(choose_split_b(&R, 1, 256, true) == 0, "%s", g_err);
      size_t total = 0;
      CHECK(layout_request(R, total) == 0 && check_layout(R, total) == 0, "%s", g_err);
      CHECK(!R.half && R.share_in_y == (R.n_share > 1), "whole length");
      if (R.n_share == 1) continue;
      ++split;
      const int pcap = (m_cap + 1) / 2, n = R.n_share;
      const unsigned inv = 65536u / n;
      for (int P = 0; P <= pcap; ++P) {
        auto lo = [&](int s) { return s == n ? P : (int)((unsigned)(P * s) * inv >> 16); };
        std::vector<int> reader(pcap, -1), writer(pcap, -1);
        for (int s = 0; s < n; ++s)
          for (int p = lo(s); p < lo(s + 1); ++p) reader[p] = s;
        for (int p = 0; p < P; ++p) CHECK(reader[p] >= 0, "pair %d of %d unread", p, P);
        for (int s = 0; s < n; ++s) {
          const int at = lo(s + 1) > lo(s) ? lo(s) : P + s;
          CHECK(at < pcap && writer[at] < 0 && (reader[at] < 0 || reader[at] == s), "share %d of %d, %d of %d pairs: at %d", s, n, P, pcap, at);
          if (at < pcap) writer[at] = s;
        }
      }
    }
  CHECK(split > 300, "%d split", split);
}

// Axis items: a block each where a launch has few, in groups of up to
// LDM_SKY_GROUP where it has many, whatever number of requests they belong to.
void axis_groups() {
  for (int64_t n : {300000, 5000000, 100000000})
    for (int count : {1, 4, 32, 256}) {
      radis_ldm_db db;
      db.n = n;
      db.has_sky = true;
      std::vector<Req> reqs;
      int64_t blocks = 0;
      for (int i = 0; i < count; ++i) {
        Req R = request(20001, 16);
        R.i0 = 1 + n / 40 * (i % 13);
        R.i1 = n - 1 - n / 50 * (i % 17);
        blocks += R.i1 / LDM_SKY_BLOCK - (R.i0 + LDM_SKY_BLOCK - 1) / LDM_SKY_BLOCK;
        reqs.push_back(R);
      }
      CHECK(choose_split_b(reqs.data(), count, 256, true) == 0, "%s", g_err);
      int64_t items = 0;
      size_t total = 0;
      for (Req& R : reqs) {
        CHECK(layout_request(R, total) == 0, "%s", g_err);
        const LdmItemPlan P = item_plan(db, R);
        CHECK(P.n_g <= LDM_SKY_WGS && (int64_t)P.n_g * P.G >= P.fb1 - P.g0 && (int64_t)(P.n_g - 1) * P.G < P.fb1 - P.g0, "groups cover the window");
        items += P.n_g;
      }
      // (each request's last group may be short)
      CHECK(items <= LDM_SKY_WGS + blocks / LDM_SKY_GROUP + count, "%d windows of %lld lines: %lld items for %lld blocks", count,
            (long long)n, (long long)items, (long long)blocks);
      if (blocks <= LDM_SKY_WGS) CHECK(items == blocks, "a block each: %lld of %lld", (long long)items, (long long)blocks);
    }
}

// Which launches run at half length: measured ones (times on both sides are at
// half_loss_ns).
void half_cost() {
  const struct { int count; int64_t nv; int m_cap; int64_t lines; bool half; } cases[] = {
      {200, 12000, 18, 48000, true},    {200, 15541, 18, 62000, false}, {64, 15541, 38, 62000, false},
      {64, 17000, 38, 68000, true},     {64, 46900, 18, 190000, false}, {16, 63800, 18, 250000, false},
      {4, 63800, 12, 250000, false},    {16, 40001, 38, 160000, true},  {64, 120417, 18, 480000, true},
      {1, 200001, 12, 5000, true},      {1, 500001, 27, 5000000, true}, {1, 19500, 84, 78000, true},
      {1, 600001, 144, 100000000, true}, {1, 600001, 345, 50000000, true}, {1, 600001, 345, 200000000, false}};
  for (const auto& c : cases) {
    std::vector<Req> reqs(c.count, request(c.nv, c.m_cap));
    for (Req& R : reqs) R.i1 = c.lines;
    CHECK(choose_split_b(reqs.data(), c.count, 256, true) == 0, "%s", g_err);
    for (const Req& R : reqs) CHECK(R.half == c.half, "%d x %lld points, %d rows", c.count, (long long)c.nv, c.m_cap);
  }
  // many windows of random sizes mix both lengths, a few keep one
  for (int count : {32, 256}) {
    std::vector<Req> reqs;
    int halves = 0, can = 0;
    for (int i = 0; i < count; ++i) {
      reqs.push_back(request(14000 + 86000 * (int64_t)(i * 37 % 256) / 256, 14 + i % 8));
      Req R = reqs.back();
      R.may_half = true;
      CHECK(plan_exec(R) == 0, "%s", g_err);
      can += R.half;
    }
    CHECK(choose_split_b(reqs.data(), count, 256, true) == 0, "%s", g_err);
    for (const Req& R : reqs) {
      halves += R.half;
      if (count == 256) CHECK(!R.half || R.half_loss <= 0, "a request that costs more than it saves");
    }
    CHECK(count == 32 ? halves == can : halves > count / 3 && halves < can, "%d of %d half, %d can", halves, count, can);
  }
}

// Pass B's shares beside many image items: the rows' pairs are still split.
void image_room() {
  for (int m_cap : {38, 84}) {
    std::vector<Req> reqs(4, request(46900, m_cap));
    for (Req& R : reqs) R.i1 = 190000;
    CHECK(choose_split_b(reqs.data(), 4, 256, true) == 0, "%s", g_err);
    for (const Req& R : reqs) CHECK(R.n_share >= 2, "%d rows, half %d: %d shares, %d image items", m_cap, (int)R.half, R.n_share, R.half ? image_items(R.n_cell) : 0);
  }
}

// What the no-allocation entry point plans with, plan to scratch layout.
void no_allocation() {
  radis_ldm_db db;
  db.n = 5000000;
  db.has_sky = true;
  for (int64_t nv : {4000, 20001, 150001, 600001})
    for (int m_cap : {1, 18, 144, 700})
      for (int flags : {0, RADIS_LDM_MIN_RMS, RADIS_LDM_GENERIC_FFT}) {
        const long before = g_news;
        Req R;
        R.r.Tgas = 1000.0;
        R.r.flags = flags;
        R.nv = nv;
        R.delta_w = 0.002;
        R.wg_hi = 0.01;
        R.i0 = 1;
        R.i1 = db.n;
        R.m_cap = R.m_need = m_cap;
        int64_t b = 0;
        size_t work = 0;
        NoallocLayout S;
        int rc = plan_fft(nv, 0, R.plan, 0, !(flags & RADIS_LDM_GENERIC_FFT), false);
        if (!rc) rc = choose_split_b(&R, 1, 256);
        if (!rc) rc = layout_request(R, work);
        const LdmItemPlan P = item_plan(db, R);
        if (!rc) noalloc_layout(R, P, plan_items(P) + P.n_img, work, S);
        if (!rc) rc = request_bytes(R, 256, b);
        CHECK(rc == 0, "%s", g_err);
        CHECK(g_news == before, "nv %lld, %d rows: %ld allocations", (long long)nv, m_cap, g_news - before);
      }
}

// LDM, Y, a partial spectrum (two where pass B is split over two shares: four
// pairs or more, and twice the row blocks fit four workgroups per CU), rows,
// axis partials, correction table, fill items at the full tile width, tables.
int64_t figure(const Req& R, int n_cu) {
  size_t t = 0;
  auto put = [&](size_t n) { t = align_up(t + n, 256); };
  const size_t pcap = (R.m_cap + 1) / 2, L = R.plan.L;
  put(pcap * 2 * align_up(R.nv + 1, 64) * 4);
  put(pcap * L * 8);
  put(L * 8);
  if (R.plan.fc && pcap >= 4 && 2 * (R.plan.n1 / fc_rows_b(R.plan.n2)) <= 4 * n_cu) put(L * 8);
  put((size_t)R.m_cap * 16);
  put((size_t)((R.i1 - R.i0 + LDM_AX_CHUNK - 1) / LDM_AX_CHUNK + 2) * 32);
  put((size_t)(R.plan.wrap_k ? std::max(1, std::min(R.m_cap / 2, LDM_MAX_AX)) : 0) * R.plan.wrap_k * 4);
  int w = R.r.tile_w ? R.r.tile_w : choose_tile(R.m_cap), groups = 1;
  if (fill_tile_bytes(R.m_cap, w) > (size_t)FILL_LDS_MAX) {
    if (!R.r.tile_w) w = FILL_GROUP_TILE_W;
    const int rows = (int)((size_t)FILL_LDS_TARGET / fill_tile_bytes(1, w)) & ~1;
    groups = (R.m_cap + rows - 1) / rows;
  }
  return (int64_t)t + (R.nv + w) / w * groups * 16 + (int64_t)(R.plan.n1 + R.plan.n2 + 1024 + (L >> LDM_TW_LO_BITS) + 1) * 8 + 64 * 1024;
}

void bytes() {
  int halves = 0, wholes = 0;
  for (int64_t nv = 2000; nv < 1000000; nv = nv * 21 / 20 + 7)
    for (int m_cap : {1, 4, 9, 16, 18, 30, 61, 144, 700})
      for (int flags : {0, RADIS_LDM_MIN_RMS})
        for (int tile : {0, 32}) {
          Req R = request(nv, m_cap, tile, flags);
          int64_t b = 0;
          CHECK(request_bytes(R, 256, b) == 0, "%s", g_err);
          CHECK(b <= figure(R, 256), "nv %lld, %d rows: %lld B, %lld for two shares", (long long)nv, m_cap, (long long)b,
                (long long)figure(R, 256));
          (R.half ? halves : wholes)++;
          // alone, with others of its kind, and with others of other sizes
          for (int n : {1, 2, 5, 9})
            for (int mixed : {0, 1}) {
              std::vector<Req> reqs;
              int64_t sum = 0;
              for (int i = 0; i < n; ++i) {
                Req Q = mixed && i ? request(nv * (1 + i) / 3 + 1500, 4 + 7 * i, 0, i % 2 ? RADIS_LDM_MIN_RMS : 0) : request(nv, m_cap, tile, flags);
                int64_t q = 0;
                CHECK(request_bytes(Q, 256, q) == 0, "%s", g_err);
                sum += q;
                reqs.push_back(mixed && i ? request(nv * (1 + i) / 3 + 1500, 4 + 7 * i, 0, i % 2 ? RADIS_LDM_MIN_RMS : 0) : request(nv, m_cap, tile, flags));
              }
              CHECK(choose_split_b(reqs.data(), n, 256, true) == 0, "%s", g_err);
              size_t total = 0;
              int64_t tw = LDM_WRAP_LC * 8;
              for (Req& Q : reqs) {
                CHECK(layout_request(Q, total) == 0, "%s", g_err);
                tw += ((int64_t)Q.tn1 + Q.tn2) * 8 + (int64_t)twl_bytes(Q) + 3 * 256;
              }
              CHECK((int64_t)total + tw <= sum, "nv %lld, %d rows, %d requests: %lld B of %lld", (long long)nv, m_cap, n,
                    (long long)total + tw, (long long)sum);
            }
        }
  CHECK(halves > 100 && wholes > 100, "%d half, %d whole", halves, wholes);
}

// Bytes of scratch with the tables of the plain splits: full-width fill tiles and
// column blocks, one pass B share (two where it is split), width candidates in
// groups of eight blocks or more, axes without tile ranges.
size_t plain_scratch(const radis_ldm_db& db, const Req& R, const LdmItemPlan& P) {
  size_t t = 0;
  auto put = [&](size_t n) { t = align_up(t + n, 256); };
  const size_t pcap = (R.m_cap + 1) / 2, L = R.plan.L;
  put(1024);
  put(sizeof(LdmAxes) - sizeof(LdmAxes::pair) - 2 * sizeof(LdmAxes::tlo));
  put(sizeof(LdmResult));
  const int64_t blocks = P.n_g ? P.fb1 - P.g0 : 0, G = std::max<int64_t>(8, (blocks + 599) / 600);
  size_t items = P.n_lo + (blocks + G - 1) / G + P.n_hi + (R.wrap_rows + 1) / 2 + (size_t)R.wide_tiles * R.fill_groups;
  const bool two = R.plan.fc && pcap >= 4 && 2 * (R.plan.n1 / fc_rows_b(R.plan.n2)) <= 1024;
  if (R.plan.fc)
    items += pcap * (R.plan.n2 / fc_cols_a(R.plan.n1)) + (two ? 2 : 1) * (R.plan.n1 / fc_rows_b(R.plan.n2)) + R.plan.n2 / fc_cols_c(R.plan.n1);
  else
    items += pcap * P.n_colA + P.n_rowB + P.n_colC;
  put(items * 16);
  put(R.plan.n1 * 8);
  put(R.plan.n2 * 8);
  put((size_t)(((L + 1023) >> LDM_TW_LO_BITS) + 1024) * 8);
  put(LDM_WRAP_LC * 8);
  size_t work = 0;
  auto buf = [&](size_t n) { work = align_up(work + n, 256); };
  buf(pcap * 2 * align_up(R.nv + 1, 64) * 4);
  buf(pcap * L * 8);
  buf(L * 8);
  if (two) buf(L * 8);
  buf((size_t)R.m_cap * 16);
  buf((size_t)((R.i1 - R.i0 + LDM_AX_CHUNK - 1) / LDM_AX_CHUNK + 2) * 32);
  buf((size_t)R.wrap_rows * R.plan.wrap_k * 4);
  put(work);
  return t;
}

void scratch() {
  int at_limit = 0;
  auto check = [&](int64_t n, int64_t nv, int m_cap, int tile, int flags) {
    radis_ldm_db db;
    db.n = n;
    db.has_sky = n >= LDM_SKY_BLOCK;
    Req R = request(nv, m_cap, tile, flags);
    R.i0 = 1;
    R.i1 = n;
    if (flags & (RADIS_LDM_GENERIC_FFT | RADIS_LDM_PERIOD_L))
      CHECK(plan_fft(nv, 0, R.plan, 0, !(flags & RADIS_LDM_GENERIC_FFT), (flags & RADIS_LDM_PERIOD_L) != 0) == 0, "%s", g_err);
    CHECK(choose_split_b(&R, 1, 256) == 0, "%s", g_err);
    size_t work = 0;
    CHECK(layout_request(R, work) == 0 && check_layout(R, work) == 0, "%s", g_err);
    const LdmItemPlan P = item_plan(db, R);
    NoallocLayout S;
    noalloc_layout(R, P, plan_items(P) + P.n_img, work, S);
    const size_t before = plain_scratch(db, R, P), limit = (size_t)RADIS_LDM_NOALLOC_BYTES;
    // what fits with the plain splits fits the array
    if (before <= limit) CHECK(S.bytes <= limit + SCRATCH_TABLES, "%lld lines, nv %lld, %d rows: %zu, plain %zu", (long long)n, (long long)nv, m_cap, S.bytes, before);
    if (before > limit / 2) CHECK(S.bytes <= before + SCRATCH_TABLES, "%lld lines, nv %lld, %d rows: %zu, plain %zu", (long long)n, (long long)nv, m_cap, S.bytes, before);
    at_limit += before > limit / 2 && before < 2 * limit;
    // and the tables and the workspace do not overlap
    CHECK(S.work + work <= S.bytes && S.twc + (size_t)LDM_WRAP_LC * 8 <= S.work && S.twl < S.twc &&
              (S.items < S.tw1 || (S.items >= S.work + R.off_free && S.items + 16 * (size_t)(plan_items(P) + P.n_img) <= S.work + work)), "scratch layout");
  };
  check(2000000, 521910, 40, 32, RADIS_LDM_PERIOD_L);  // within 2 KB of the limit
  for (int64_t n : {1000, 300000, 4100000, 100000000})
    for (int64_t nv = 3000; nv < 5000000; nv = nv * 11 / 10 + 1)
      for (int m_cap = 1; m_cap < 9000; m_cap = m_cap * 5 / 4 + 1)
        for (int flags : {0, RADIS_LDM_MIN_RMS, RADIS_LDM_GENERIC_FFT, RADIS_LDM_PERIOD_L})
          if ((size_t)((m_cap + 1) / 2) * nv * 24 < (2u << 30)) check(n, nv, m_cap, 0, flags);
  CHECK(at_limit > 100, "%d near the limit", at_limit);
}

}  // namespace

int main(int argc, char** argv) {
  const struct { const char* name; void (*run)(); } sections[] = {{"wide_tile", wide_tile}, {"axis_groups", axis_groups}, {"half_cost", half_cost}, {"image_room", image_room}, {"no_allocation", no_allocation}, {"bytes", bytes}, {"scratch", scratch}, {"shares_in_y", shares_in_y}};
  for (const auto& s : sections)
    if (argc == 2 && !std::strcmp(argv[1], s.name)) {
      s.run();
      std::printf("%s: %d failed checks\n", s.name, g_fail);
      return g_fail ? 1 : 0;
    }
  std::fprintf(stderr, "no such section\n");
  return 2;
}
