"""Which cache rows a key tile's loads touch: the arithmetic every tile loader shares (tile_rows, tile_is_edge in
csrc/attn_params.h), compiled for the host.  A row before the first key the workgroup sees, or past the last key, may lie
outside the caller's allocation (a holder of a key range passes a shifted base) and must not be read."""
import subprocess

from diffgemma_amd import build

PROGRAM = r"""
#include "attn_params.h"
#include <algorithm>
#include <cstdio>
#include <vector>
int main() {
  using namespace dg;
  const uint32_t span = 3 * kBlockN + 2;
  // the keys a kernel is told of: those of the cache, or up to the key tile in which a range [begin, end) ends
  for (uint32_t keys = 1; keys <= span; ++keys)
    for (uint32_t end = 0; end <= keys; ++end)
      for (uint32_t begin = 0; begin <= end; ++begin) {
        const uint32_t first = begin / kBlockN, last = std::max(first, (end + kBlockN - 1) / kBlockN), told = keys_of_range(first, last, keys);
        if (told > keys || (end > begin && (told < end || told > (end + kBlockN - 1) / kBlockN * kBlockN)) || (end == keys && told != keys))
          return std::printf("[%u, %u) of %u: %u keys\n", begin, end, keys, told), 1;
      }
  for (uint32_t t_all = 1; t_all <= span; ++t_all)
    for (uint32_t lo = 0; lo <= t_all + kBlockN; ++lo)
      for (uint32_t t0 = 0; t0 < t_all; t0 += kBlockN) {
        const TileRows r = tile_rows(t0, lo, t_all);
        const uint32_t see = lo < t_all ? lo : t_all - 1u;      // (rows that see nothing: any row that exists)
        bool clamped = false;
        for (uint32_t i = 0; i < (uint32_t)kBlockN; ++i) {
          const uint32_t row = t0 + (i < r.first ? r.first : i > r.last ? r.last : i);
          clamped |= row != t0 + i;
          // inside the keys that exist, and not before the first visible one unless the whole tile is
          if (row >= t_all || (row < see && see < t0 + kBlockN)) return std::printf("t_all %u lo %u t0 %u row %u\n", t_all, lo, t0, row), 1;
          if (t0 + i >= lo && t0 + i < t_all && row != t0 + i) return std::printf("moved a visible row %u\n", t0 + i), 1;
        }
        // loads for tiles behind t0, the last one: nothing behind the last key, and nothing before the first visible one where t0 is
        // the first tile too
        const uint32_t pos = past_end_pos(t0, lo, t_all, 0u);
        const TileRows past = tile_rows(pos, 0u, t_all);
        if (pos + past.last >= t_all || pos < t0 || (see < t0 + kBlockN && pos + past.first < see) || past_end_pos(t0, lo, t_all, 63u) != t0)
          return std::printf("t_all %u lo %u t0 %u: past the end at %u\n", t_all, lo, t0, pos), 1;
        // touches of a row tile whose last tile is t0 and whose first one, with `lo` in it, is anywhere before: from the fourth on
        for (uint32_t tb = lo / kBlockN; tb <= t0 / kBlockN; ++tb)
          for (uint32_t tile = tb + 3u; tile < tb + 8u; ++tile) {
            const uint32_t at = std::min(tile * kBlockN, pos);
            for (uint32_t i = 0; i < (uint32_t)kBlockN; ++i) {
              const uint32_t row = at + std::min(i, t_all - 1u - at);
              if (row >= t_all || row < see || (tile * kBlockN <= t0 && row != std::min(tile * kBlockN + i, t_all - 1u)))
                return std::printf("t_all %u lo %u t0 %u: touches row %u\n", t_all, lo, t0, row), 1;
            }
          }
        if (clamped && !tile_is_edge(t0, lo, t_all)) return std::printf("t_all %u lo %u t0 %u: no edge tile\n", t_all, lo, t0), 1;
      }
  // touches of the one-launch kernel: every key of the range, and no other
  for (uint32_t per = 8; per <= 64; per *= 2)
    for (uint32_t pos0 = 0; pos0 <= 33; pos0 += 11)
      for (uint32_t n = 1; n <= 130; ++n) {
        std::vector<bool> seen(n);
        for (uint32_t u = 0; u < (n + per - 1) / per; ++u)
          for (uint32_t i = 0; i < per; ++i) {
            const uint32_t pos = touched_pos(pos0, pos0 + n, per, u, i);
            if (pos < pos0 || pos >= pos0 + n) return std::printf("%u to a touch, [%u, %u): touches row %u\n", per, pos0, pos0 + n, pos), 1;
            seen[pos - pos0] = true;
          }
        if (std::count(seen.begin(), seen.end(), true) != n) return std::printf("%u to a touch, %u keys: not all\n", per, n), 1;
      }
  std::puts("ok");
  return 0;
}
"""


def test_no_row_outside_the_visible_keys_is_read(tmp_path):
    src, exe = tmp_path / "rows.hip", tmp_path / "rows"
    src.write_text(PROGRAM)
    res = subprocess.run([build.hipcc_path(), *build.HIP_FLAGS, "-I", str(build.CSRC), str(src), "-o", str(exe)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout


def test_k_and_v_tiles_of_the_one_launch_kernel_share_the_rule():
    """The one-launch kernel once clamped V's first tile and not K's."""
    text = (build.CSRC / "attn_wsplit.hip").read_text()
    assert text.count("tile_is_edge(") == 1 and text.count("tile_rows(tile * kBlockN, lo_min, p.t_all)") == 1
    assert text.count("is_edge(tile)") == 2        # where K's loads go out and where V's do


def test_kernels_are_told_of_the_keys_of_a_range_alone():
    """Behind a range of one tile that begins inside it the split kernel once loaded up to 31 rows past the range: its loads ended
    with the last key of the cache."""
    api, text = (build.CSRC / "dg_attn_api.hip").read_text(), (build.CSRC / "attn_mfma.hip").read_text()
    assert api.count("p.t_all = dg::keys_of_range(pl.tile_first, pl.tile_end, pl.t_all);") == api.count("  p.t_all = ") == 1
    assert "t_last = past_end_pos((te - 1u) * kBlockN, lo_min, p.t_all, p.ring_mask)" in text
    assert text.count("min(t0, t_last), 0u, p.t_all, p.ring_mask") == text.count("min(t0, t_last)") == 2


def test_touches_of_the_split_kernel_begin_with_the_first_visible_key():
    """They once began with the tile: up to 31 rows before a share of one tile that begins inside it."""
    text = (build.CSRC / "attn_mfma.hip").read_text()
    assert text.count("lds_dma_touch(") == 1 and text.count("tp = min(tile * kBlockN, t_last);") == 1
    assert text.count("row = min(li >> 3, p.t_all - 1u - tp);") == 1


def test_touches_of_the_one_launch_kernel_stay_in_its_range():
    """They once ended with the last key, up to 63 rows behind the keys of a workgroup's range."""
    text = (build.CSRC / "attn_wsplit.hip").read_text()
    assert text.count("lds_dma_touch(") == 1 and text.count("touched_pos(pos0, pos1, RPT,") == 1
    assert "pos1 = min(mt_end * kBlockN, p.t_all)" in text
