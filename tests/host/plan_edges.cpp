// Edges of the host planning, one section per argument:
//   wide_tile   an explicit fill tile too wide for two LDM rows is refused by
//               the planning itself, alone and beside requests that plan
#include <cstdio>
#include <cstring>

#include "ldm_plan.h"

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

}  // namespace

int main(int argc, char** argv) {
  const struct { const char* name; void (*run)(); } sections[] = {{"wide_tile", wide_tile}};
  for (const auto& s : sections)
    if (argc == 2 && !std::strcmp(argv[1], s.name)) {
      s.run();
      std::printf("%s: %d failed checks\n", s.name, g_fail);
      return g_fail ? 1 : 0;
    }
  std::fprintf(stderr, "no such section\n");
  return 2;
}
