// CPU check of the pair passes in 128 x 128 tiles: for every job size and
// pair, the tiles of batch_desc.h cover exactly the 64 x 64 tasks of the same
// pass, once each, and the plan builder's segments for them
// (fapi::build_fw_batch) count those tiles, job by job, in launches of pair
// passes only.  Prints "ok" and exits 0 when everything holds.
#include <stdio.h>

#include <map>
#include <utility>
#include <vector>

#include "batch_desc.h"

typedef std::map<std::pair<int, int>, int> Tiles;

static bool maps_agree() {
  for (int nb = 3; nb <= 41; nb++)
    for (int r = 0; r + 1 < nb; r += 2) {
      Tiles small, big;
      int I, J;
      for (int i = 0; i < (nb - 2) * (nb - 2); i++) {
        fapk::pair_tile(r, nb, i, &I, &J);
        small[{I, J}]++;
      }
      for (int i = 0; i < fapk::pair128_count(nb); i++) {
        fapk::pair128_tile(r, nb, i, &I, &J);
        for (int q = 0; q < 4; q++) {
          const int a = 2 * I + (q >> 1), b = 2 * J + (q & 1);
          if (a < nb && b < nb) big[{a, b}]++;
        }
      }
      if (small != big) {
        printf("nb %d pair %d: %zu tasks, %zu covered\n", nb, r, small.size(), big.size());
        return false;
      }
    }
  return true;
}

static bool segments_agree(const std::vector<int32_t> &n, bool expect) {
  std::vector<int32_t *> mats(n.size(), nullptr);
  std::vector<int64_t> ld(n.begin(), n.end());
  fapi::FwBatchDesc d;
  fapi::build_fw_batch((int32_t)n.size(), mats.data(), n.data(), ld.data(), &d);
  const int launches = (int)d.launch_tasks.size();
  bool any = false;
  for (int p = 0; p < launches; p++) {
    if (d.pair128_off[p] < 0) continue;
    any = true;
    int at = 0;
    for (int q = d.seg_off[p], k = d.pair128_off[p]; q < d.seg_off[p + 1]; q++, k++) {
      const fapk::BatchSeg &a = d.segs[q], &b = d.segs[k];
      const int count = fapk::pair128_count(d.jobs[a.job].nb);
      if ((a.kind_r & 7) != fapk::TASK_REST2 || a.job != b.job || a.kind_r != b.kind_r ||
          b.first != at || b.count != count)
        return false;
      at += count;
    }
    if (at != d.pair128_tasks[p]) return false;
  }
  d.drop_pair128();
  for (int p = 0; p < launches; p++)
    if (d.pair128_off[p] >= 0) return false;
  return any == expect && (int)d.segs.size() == d.seg_off.back();
}

int main() {
  if (!maps_agree()) return 1;
  std::vector<int32_t> uneven;
  for (int i = 0; i < 200; i++) uneven.push_back(64 + (i * 977) % 1985);
  if (!segments_agree(uneven, true) || !segments_agree(std::vector<int32_t>(64, 512), true) ||
      !segments_agree(std::vector<int32_t>(8, 512), false) ||   // too few tiles
      !segments_agree(std::vector<int32_t>(500, 192), false) || // half-empty last blocks
      !segments_agree({64, 128}, false))
    return 1;
  printf("ok\n");
  return 0;
}
