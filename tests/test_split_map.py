"""Split counts per row tile (SplitMap in csrc/attn_params.h), compiled for the host: every (row tile, split) is one unit of a
KV head, found again from its number, the longest share keeps the asked-for length, and the shortest length is found without
trying each.  And the other rules of the same header: split and slice counts, the order of units, how rows are merged."""
import re
import subprocess

from diffgemma_amd import attention as A, build, capi

PROGRAM = r"""
#include "attn_params.h"
#include <algorithm>
#include <cstdio>
#include <vector>
int main() {
  using namespace dg;
  for (uint32_t n = 1; n <= 70; n += n < 6 ? 1 : 13)
    for (uint32_t len = 1; len <= 20; ++len)
      for (uint32_t base = 0; base <= 40; base += 8)
        for (uint32_t per = 0; per <= 3; ++per) {
          auto tiles = [&](uint32_t mt) { return base + 1 + mt * per / 2; };
          SplitMap m;
          const uint32_t most = (tiles(n - 1) + len - 1) / len;
          if (make_split_map(n, len, tiles, &m) != (most <= kMapSplits)) return std::printf("n %u len %u most %u\n", n, len, most), 1;
          if (most > kMapSplits) continue;
          if (m.n != most) return std::printf("n %u len %u: %u splits\n", n, len, m.n), 1;
          std::vector<uint32_t> seen(n, 0);
          uint32_t units = 0;
          for (uint32_t mt = 0; mt < n; ++mt) {
            if (map_splits(m, mt) != (tiles(mt) + len - 1) / len) return std::printf("mt %u: %u splits\n", mt, map_splits(m, mt)), 1;
            units += map_splits(m, mt);
          }
          if (units != m.units) return std::printf("units %u %u\n", units, m.units), 1;
          for (uint32_t u = 0; u < m.units; ++u) {
            const uint32_t s = map_split_of(m, u), mt = m.first[s] + u - m.cum[s];
            if (mt >= n || s >= map_splits(m, mt) || (seen[mt] & (1u << s))) return std::printf("unit %u: mt %u split %u\n", u, mt, s), 1;
            seen[mt] |= 1u << s;
          }
        }
  // the shortest length: what trying every one finds, looked at a bounded number of times, once where no row tile can do with less
  for (uint32_t n = 1; n <= 64; n += 9)
    for (uint32_t base = 0; base <= 1100; base += base < 40 ? 8 : 353)
      for (uint32_t per = 0; per <= 3; ++per)
        for (uint32_t budget = n; budget <= 128; budget += 37)
          for (uint32_t len = 1; len <= 60; len += 1 + len / 2)
            for (uint32_t limit = 0; limit <= 520; limit += 1 + limit / 2) {
              uint32_t calls = 0;
              auto tiles = [&](uint32_t mt) { return ++calls, base + 1 + mt * per / 2; };
              SplitMap want, got;
              bool found = false;
              for (uint32_t l = len; l <= limit && !found; ++l) found = make_split_map(n, l, tiles, &want) && want.units <= budget;
              calls = 0;
              if (shortest_split_map(n, len, limit, budget, tiles, &got) != found) return std::printf("n %u base %u len %u limit %u budget %u\n", n, base, len, limit, budget), 1;
              if (calls > 1u + 12u * n || (per == 0 && limit && n * ((base + limit) / limit) > budget && calls > 1u))
                return std::printf("n %u base %u len %u limit %u budget %u: %u calls\n", n, base, len, limit, budget, calls), 1;
              if (!found) continue;
              bool same = got.n == want.n && got.units == want.units;
              for (uint32_t i = 0; i < kMapSplits; ++i) same = same && got.first[i] == want.first[i] && got.cum[i] == want.cum[i];
              if (!same) return std::printf("n %u base %u len %u limit %u budget %u: another map\n", n, base, len, limit, budget), 1;
            }
  std::puts("ok");
  return 0;
}
"""


ROUNDS = r"""
#include "attn_params.h"
#include <cstdio>
int main() {
  using namespace dg;
  double all = 0, seen = 0;
  for (uint32_t cus : {256u, 80u})
    for (uint32_t base = 1; base <= 700; base += base < 70 ? 1 : 37)
      for (uint32_t tiles = 1; tiles <= 5400; tiles += 1 + tiles / 7)
        for (uint32_t least : {1u, 6u, 14u, 16u})
          for (uint32_t most : {least, std::max(least, std::min(tiles / 4, 64u)), std::max(least, std::min(tiles / 2, 128u))})
            for (uint32_t start : {3u, 4u}) {
              uint32_t want = least, looked = 0;
              uint64_t want_cost = UINT64_MAX;
              for (uint32_t s = least; s <= most; ++s) {
                const uint64_t cost = ((uint64_t)base * s + cus - 1) / cus * ((tiles + s - 1) / s + start);
                if (cost < want_cost) want_cost = cost, want = s;
              }
              const uint32_t got = splits_in_rounds(base, tiles, least, most, cus, start, &looked);
              if (got != want)
                return std::printf("base %u tiles %u least %u most %u cus %u: %u, not %u\n", base, tiles, least, most, cus, got, want), 1;
              all += most - least + 1, seen += looked;
            }
  if (seen * 6 > all) return std::printf("%.0f counts looked at of %.0f\n", seen, all), 1;
  // a canvas of many rows: as many workgroups as 32 bits hold
  if (splits_in_rounds(1u << 24, 1000, 6, 64, 256, 3) != 6) return 1;
  std::puts("ok");
  return 0;
}
"""


BY_ROWS = r"""
#include "attn_params.h"
#include <cstdio>
int main() {
  using namespace dg;
  FastDiv by[kMapSplits];
  for (uint32_t i = 0; i < kMapSplits; ++i) by[i] = make_fast_div(i + 1);
  for (uint32_t n = 1; n <= 70; n += n < 6 ? 1 : 13)
    for (uint32_t len = 1; len <= 20; ++len)
      for (uint32_t base = 0; base <= 40; base += 8)
        for (uint32_t per = 0; per <= 3; ++per) {
          SplitMap m;
          if (!make_split_map(n, len, [&](uint32_t mt) { return base + 1 + mt * per / 2; }, &m)) continue;
          uint32_t u = 0;
          for (uint32_t mt = 0; mt < n; ++mt)
            for (uint32_t s = 0; s < map_splits(m, mt); ++s, ++u) {
              const MapUnit got = map_unit_by_rows(m, by, u);
              if (got.mt != mt || got.split != s || got.splits != map_splits(m, mt)) return std::printf("n %u len %u unit %u\n", n, len, u), 1;
            }
          if (u != m.units) return std::printf("units %u %u\n", u, m.units), 1;
        }
  // both sides of each line: 20 or 10 key tiles to a row tile, and where many row tiles see more than a few thousand keys
  if (!rows_before_splits(2, 4, 80) || rows_before_splits(2, 4, 81) || !rows_before_splits(2, 5, 50) || rows_before_splits(2, 5, 51)) return 2;
  if (!rows_before_splits(2, 16, 104) || rows_before_splits(2, 16, 105) || !rows_before_splits(8, 1, 20) || rows_before_splits(1, 1, 11)) return 3;
  std::puts("ok");
  return 0;
}
"""


def test_units_by_row_tile(tmp_path):
    """A split map's workgroups in the order by row tile, then split: every unit once, and the lines of the rule that takes it."""
    run_program(tmp_path, BY_ROWS)


BY_ROWS_CALLS = r"""
#include "attn_params.h"
#include <cstdio>
using namespace dg;
int main() {
  struct Call { uint32_t hkv, n_mtiles, n_splits, key_tiles, map_n; bool by_rows; uint32_t from_hbm, hd; };
  const Call calls[] = {
%s  };
  for (const Call& c : calls) {
    AttnParams p = {};
    p.hkv = c.hkv, p.n_mtiles = c.n_mtiles, p.n_splits = c.n_splits, p.tile_first = 3, p.tile_end = 3 + c.key_tiles;
    p.touch_ahead = c.from_hbm;
    SplitMap map = {};
    map.n = c.map_n;
    if (units_by_row_tile(p, map, c.hd) != c.by_rows)
      return std::printf("%%u KV heads, %%u row tiles, %%u splits, %%u key tiles\\n", c.hkv, c.n_mtiles, c.n_splits, c.key_tiles), 1;
  }
  // merged in runs: the same, or KV heads in eights, from head_dim 256 on
  AttnParams p = {};
  p.hkv = 8, p.n_mtiles = 1, p.rows_total = 74, p.rows_pad = 128, p.n_splits = 3, p.part_half = 1, p.tile_end = 9;
  for (uint32_t hd = 32; hd <= 512; hd *= 2)
    for (uint32_t shared = 0; shared < 2; ++shared) {
      const MergePlan m = plan_merge(p, SplitMap{}, hd, false, shared != 0);
      if (!m.at_once || m.rows.run != (hd >= 256 ? 19u : 0u) || m.rows.span != (hd >= 256 ? 76u : 74u)) return std::printf("head_dim %%u\n", hd), 1;
      if (plan_merge(p, SplitMap{}, hd, true, shared != 0).at_once) return 1;
    }
  p.hkv = 2, p.n_mtiles = 4, p.rows_total = 392, p.rows_pad = 512;
  for (uint32_t shared = 0; shared < 2; ++shared) {
    const MergePlan m = plan_merge(p, SplitMap{}, 512, false, shared != 0);
    if (!m.at_once || m.rows.run != (shared ? 0u : 32u) || m.rows.span != (shared ? 392u : 512u)) return 1;
  }
  std::puts("ok");
  return 0;
}
"""


def test_calls_whose_units_go_by_row_tile(tmp_path):
    """(KV heads, row tiles of a KV head, splits, key tiles, a map's splits): with fewer than eight row tiles only where every XCD has an equal
    run out of one of them; from eight on by the number of key tiles, fewer where the rows come from HBM; not
    with KV heads in eights, nor below head_dim 256."""
    calls = [((2, 2, 14, 14, 0), True), ((2, 3, 7, 14, 0), False), ((2, 2, 3, 3, 0), False), ((2, 2, 9, 17, 0), False), ((2, 1, 4, 4, 0), True),
             ((2, 3, 8, 14, 0), False), ((2, 2, 4, 14, 4), False), ((1, 4, 12, 12, 0), True), ((1, 7, 8, 12, 0), False), ((1, 8, 5, 12, 0), True),
             ((2, 4, 7, 14, 0), True), ((2, 5, 7, 14, 0), True), ((2, 16, 6, 33, 0), True), ((2, 16, 8, 105, 0), False), ((2, 44, 4, 44, 4), True)]
    cold = [((2, 16, 8, 96, 0), True), ((2, 16, 8, 97, 0), False), ((2, 16, 8, 102, 0), False), ((2, 8, 12, 83, 0), True), ((2, 64, 2, 126, 2), True),
            ((2, 4, 7, 14, 0), True), ((2, 4, 14, 78, 0), True), ((2, 4, 14, 79, 0), False)]
    calls += [((2, 16, 8, 104, 0), True), ((2, 4, 14, 80, 0), True), ((8, 1, 6, 12, 0), False), ((16, 2, 6, 12, 0), False), ((12, 2, 6, 12, 0), True)]
    rows = "".join("    {%d, %d, %d, %d, %d, %s, %d, %d},\n" % (*c, str(yes and hd >= 256).lower(), hbm, hd)
                   for hd in (32, 128, 256, 512) for hbm, forms in ((0, calls), (1, cold)) for c, yes in forms)
    run_program(tmp_path, BY_ROWS_CALLS % rows)


PATHS = r"""
#include "dg_attn_api.hip"
#include <cstdio>
#include <string>
int main() {
  const struct { unsigned char desc[sizeof(dg_attn_desc)]; const char* path; } calls[] = {
%s  };
  for (const auto& c : calls) {
    dg_attn_desc d;
    std::memcpy(&d, c.desc, sizeof(d));
    Plan pl;
    if (make_plan(&d, 256, &pl) != DG_OK) return 1;
    dg::AttnParams p = {};
    p.hkv = d.n_kv_heads, p.n_mtiles = pl.n_mtiles, p.n_splits = pl.n_splits, p.rows_total = pl.rows_total, p.rows_pad = pl.rows_pad;
    p.tile_first = pl.tile_first, p.tile_end = pl.tile_end, p.part_half = pl.part_half;
    const dg::MergePlan m = dg::plan_merge(p, pl.map, d.head_dim, false, pl.wsplit);
    const std::string path = std::string(pl.wsplit ? "shared" : dg::units_by_row_tile(p, pl.map, d.head_dim) ? "by row tile" : "by split") +
                             (pl.map.n ? ", map" : !m.at_once ? ", streamed" : m.rows.run ? ", in runs" : ", in turn") + (pl.part_half ? ", f16" : ", f32");
    if (path != c.path) return std::printf("%%u rows behind %%u: %%s, not %%s\n", d.canvas, d.kv_len, path.c_str(), c.path), 1;
  }
  std::puts("ok");
  return 0;
}
"""


def test_paths_of_the_order_tests(tmp_path):
    """The order of the units, the merge and the partial rows' type that the GPU tests' calls are named for are those they get."""
    from test_gpu_split_plan import MAP_FORMS, ORDER_FLAGS, ORDER_FORMS, map_workload, order_workload
    calls = [(order_workload(*f[:6]).desc(flags=ORDER_FLAGS), f[6]) for f in ORDER_FORMS]
    calls += [(map_workload(*f[:5]).desc(), f[5] + ", map, f16") for f in MAP_FORMS]
    rows = "".join('    {{%s}, "%s"},\n' % (",".join(map(str, bytes(d))), path) for d, path in calls)
    run_program(tmp_path, PATHS % rows, "-I", str(build.CSRC.parent.parent / "include"),
                "-L", str(build.LIB_PATH.parent), "-l:" + build.LIB_NAME, "-Wl,-rpath," + str(build.LIB_PATH.parent))


MERGE_RUNS = r"""
#include "attn_params.h"
#include <cstdio>
#include <vector>
using namespace dg;
int main() {
  const uint32_t heads[] = {1, 2, 3, 4, 5, 8, 12, 16}, rows[] = {1, 8, 74, 127, 128, 129, 333, 392, 512, 576, 768, 1600, 2048, 4095};
  for (uint32_t hkv : heads)
    for (uint32_t rt : rows)
      for (uint32_t S = 2; S <= kMergeFewSplits; ++S) {
        const uint32_t mt = (rt + kBlockM - 1) / kBlockM, T = hkv * mt, per = (T * S + 7) / 8;
        // which XCD writes split s of row tile t of a KV head: whole heads in either order, else by row tile, then split
        auto wrote = [&](uint32_t h, uint32_t t, uint32_t s) { return ((h * mt + t) * S + s) / per; };
        const MergeRuns r = merge_runs(hkv, rt, mt, S);
        std::vector<uint32_t> seen(hkv * rt, 0);
        const FastDiv by = make_fast_div(r.span);
        uint64_t own = 0;
        for (uint32_t b = 0; b < 8 * r.run; ++b)
          for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t n = merge_row(b, w, r.run), h = fast_div(n, by), row = n - h * r.span;
            if (h >= hkv || row >= rt) continue;
            ++seen[h * rt + row];
            uint32_t here = 0;
            for (uint32_t s = 0; s < S; ++s) here += wrote(h, row / kBlockM, s) == b % 8 ? 1 : 0;
            own += here;
            const bool whole = hkv % 8 == 0 || (T % 8 == 0 && T * S % 8 == 0);
            if (whole && here != S) return std::printf("%u heads, %u rows, %u splits: row %u of head %u\n", hkv, rt, S, row, h), 1;
          }
        for (uint32_t n : seen)
          if (n != 1) return std::printf("%u heads, %u rows, %u splits: a row %u times\n", hkv, rt, S, n), 2;
        // row tiles cut by the end of a run: half of what is merged was written there at the least
        if (T >= 8 && own * 2 < (uint64_t)hkv * rt * S) return std::printf("%u heads, %u rows, %u splits: %g\n", hkv, rt, S, (double)own / (hkv * rt * S)), 3;
        // in turn: every row once
        std::fill(seen.begin(), seen.end(), 0u);
        for (uint32_t b = 0; b < (hkv * rt + 3) / 4; ++b)
          for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t n = merge_row(b, w, 0), h = fast_div(n, make_fast_div(rt));
            if (h < hkv) ++seen[n];
          }
        for (uint32_t n : seen)
          if (n != 1) return 4;
      }
  std::puts("ok");
  return 0;
}
"""


def test_rows_are_merged_where_they_were_written(tmp_path):
    """The merge's runs of rows, one for each XCD, against the split kernel's runs of units: every row once, on the XCD that wrote its
    partial rows where no row tile is cut by the end of a run, and on one that wrote most of them otherwise."""
    run_program(tmp_path, MERGE_RUNS)


def test_keys_an_xcd_reads_before_the_merge(tmp_path):
    """KV heads of an XCD, rounded up, times their keys, and an eighth of the partial rows, against 6 MiB."""
    mib = 1 << 20
    wrong = " || ".join(f"dg::merge_on_xcd({hkv}, {head}, {part}) != {str(yes).lower()}" for hkv, head, part, yes in (
        (1, 6 * mib, 0, True), (2, 5 * mib, 8 * mib, True), (2, 5 * mib, 8 * mib + 8, False), (8, 6 * mib, 0, True), (8, 6 * mib + 1, 0, False),
        (12, 3 * mib, 0, True), (12, 3 * mib + 1, 0, False), (16, 3 * mib, 0, True), (17, 2 * mib, 0, True), (17, 3 * mib, 0, False)))
    run_program(tmp_path, '#include "attn_params.h"\n#include <cstdio>\nint main() { if (%s) return 1; std::puts("ok"); return 0; }\n' % wrong)


def test_units_of_a_split_map(tmp_path):
    run_program(tmp_path, PROGRAM)


def test_splits_in_rounds_of_the_chip(tmp_path):
    """What working out the cost of every count finds, by looking at a sixth of them."""
    run_program(tmp_path, ROUNDS)


def test_slices_of_the_gather(tmp_path):
    """The slices that test_gather_slices names are those its calls get."""
    from test_gpu_topk_parity import GATHER_SLICES
    wrong = " || ".join(f"dg::topk_gather_slices({rows} * 16) != {n}" for rows, n in GATHER_SLICES)
    run_program(tmp_path, '#include "attn_params.h"\n#include <cstdio>\nint main() { if (%s) return 1; std::puts("ok"); return 0; }\n' % wrong)
    assert {n for _, n in GATHER_SLICES} == {1, 2, 4}


def run_program(tmp_path, program, *more):
    src, exe = tmp_path / "map.hip", tmp_path / "map"
    src.write_text(program)
    res = subprocess.run([build.hipcc_path(), *build.HIP_FLAGS, "-I", str(build.CSRC), str(src), *more, "-o", str(exe)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout


def test_where_a_split_map_is_planned():
    """Causal rows behind a short prefix, 16-bit partial rows; not behind a long one, not with a window, fp32 partial rows, an
    explicit count or equal rows.  The scratch covers the entry points that read the prefix on the device, too."""
    half = capi.DG_ATTN_F_F16_PARTIALS
    desc = lambda rows, kv, cr, **kw: A.make_desc(rows, 16, 2, 512, kv, causal_rows=cr, **{"flags": half, **kw})
    assert capi.resolved_splits(desc(1024, 0, 1024)) == 3 and capi.resolved_splits(desc(700, 700, 700)) == 4
    assert capi.resolved_splits(desc(1024, 0, 1024, kv_dtype=capi.DG_F16, flags=0)) == 3
    for d in (desc(1024, 0, 1024, flags=0), desc(1024, 20000, 1024), desc(1024, 0, 0), desc(1024, 0, 1024, n_splits=2)):
        assert capi.resolved_splits(d) == 2
    row_tiles = 2 * 64 * 128
    assert capi.workspace_bytes(desc(1024, 0, 1024)) >= 2 * row_tiles * (512 * 2 + 8)      # two equal splits


def test_shares_no_shorter_than_partial_rows_pay_for():
    """(rows, prefix) of causal rows -> the largest split count of a row tile: a share is as long as where the partial rows of all row
    tiles cost what shorter shares save, so that row tiles up to that length stay one share and their rows fp32 until the output."""
    half = capi.DG_ATTN_F_F16_PARTIALS
    for kw in ({"flags": half}, {"kv_dtype": capi.DG_F16, "flags": 0}):
        splits = lambda rows, kv: capi.resolved_splits(A.make_desc(rows, 16, 2, 512, kv, causal_rows=rows, **kw))
        assert [splits(*c) for c in ((1024, 0), (901, 0), (700, 0), (800, 100), (512, 0), (600, 200), (350, 300))] == [3, 3, 3, 3, 3, 3, 4]


def test_every_merge_instance_can_be_reached():
    """The merge that asks for all rows at once: one instance per split count up to 8 and every second to 16, with a map only up to
    the splits a map gives, fp32 rows up to 8."""
    names = subprocess.run(["nm", "-C", str(build.LIB_PATH)], stdout=subprocess.PIPE, text=True, check=True).stdout
    built = set(re.findall(r"attn_merge_few_kernel<(\d+)u, (true|false), (\d+)u>", names))
    few = [str(n) for n in range(2, 9)]
    want = {(n, "false", "0") for n in few + ["10", "12", "14", "16"]} | {(n, "true", "0") for n in few}
    assert built == want | {(n, "false", c) for n in few for c in "12"}


def test_split_counts_that_keep_the_merge_short():
    """(rows, keys) of 16 heads over 2 -> splits: to 16 with at most a merge workgroup per compute unit, a share of up to three tiles
    more, or 8 in all, taken for it; past that to 8 where a share gets one tile longer."""
    splits = lambda rows, keys: capi.resolved_splits(A.make_desc(rows, 16, 2, 512, keys - rows, flags=capi.DG_ATTN_F_F16_PARTIALS))
    assert [splits(64, 1264), splits(32, 3700), splits(32, 4064), splits(48, 4500)] == [14, 15, 16, 29]
    assert [splits(72, 1000), splits(80, 841), splits(96, 1264), splits(96, 1700), splits(72, 1500)] == [8, 7, 8, 11, 12]


def test_shares_of_a_short_range():
    """(rows, prefix, heads, KV heads) of a sliding layer -> workgroups to a row tile: by what their tiles, a second launch and their
    partial rows cost; one where that is no gain, and past 112 rows of 16 heads."""
    shares = lambda rows, kv, hq=16, hkv=8: capi.resolved_splits(A.make_desc(rows, hq, hkv, 256, kv, window=1024))
    assert [shares(rows, 4000) for rows in (16, 48, 64, 80, 96, 112, 128, 256)] == [5, 5, 3, 3, 3, 3, 1, 1]
    assert [shares(112, 781), shares(96, 861), shares(64, 829), shares(32, 200)] == [1, 4, 4, 1]
    assert [shares(100, 800, 16, 2), shares(32, 800, 48, 8), shares(112, 4000, 8, 1)] == [4, 1, 3]
