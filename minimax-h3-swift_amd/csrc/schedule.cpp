// The attention kernel's persistent schedule, built on the host from a plan's
// row lengths. Pure C++, no device code, so CPU tests can compile it:
// h3hip_plan_create uploads plan_schedule's lists (over half rows where those end
// earlier) and h3hip_plan_schedule gives them back; h3hip_schedule exposes the
// lists over whole rows.
#include <algorithm>
#include <cstdint>
#include <numeric>
#include <queue>
#include <utility>
#include <vector>

#include "plan.h"

namespace h3hip {

// The attention kernel's schedule: which (head, q-tile) work units each of
// its persistent workgroups runs, and in what order.
//
// Workgroups are handed to the 8 XCDs round-robin (workgroup b runs on XCD
// b % 8), and each XCD has its own L2. So each XCD gets its own list, laid
// out for L2 reuse: long rows (the dense prefix rows, ~8x the median) first,
// grouped by head so that units streaming the same head's K/V run side by
// side, then a contiguous (head, q-tile) range so neighbouring q-tiles of one
// head, which share most of their key tiles under local masks, are resident
// together. The XCD lists are balanced by cost (tiles + a fixed per-unit
// overhead). Each list is then dealt to the XCD's workgroups in list order,
// every unit to the workgroup that the cost model frees first -- the order in
// which the hardware's own dispatch would hand them out -- so the units an
// XCD runs at one time stay neighbours in its list.
// Cost of a unit in tile times beyond its tiles (merge, store, first loads),
// measured on MI355X (band rules: 1.8 us per tile, the rest per unit).
constexpr int kUnitOverhead = 2;

// Deals a list to `count` workgroups in list order, every unit to the one that
// is free first (the lowest index of several), and appends each unit's
// workgroup to wg. Costs are whole numbers of at most max_cost, so all free
// times lie in a window of max_cost + 1 ticks from the earliest: a ring of
// buckets, one bit per workgroup, finds the next one in a step or two. For the
// 10,000 units of 250 x 250 tiles x 40 heads on 256 workgroups build_schedule
// takes 140 us so and 396 us with a priority queue and a vector per workgroup
// (one core of the build host). The queue stays for more than 64 workgroups
// per XCD, which do not fit in a bucket's word.
static void deal(const std::vector<int32_t>& list, const std::vector<int32_t>& len, int count,
                 std::vector<int32_t>& wg) {
  if (count > 64) {
    std::priority_queue<std::pair<int64_t, int>, std::vector<std::pair<int64_t, int>>,
                        std::greater<std::pair<int64_t, int>>>
        free_at;
    for (int c = 0; c < count; c++) free_at.push({0, c});
    for (int32_t u : list) {
      const auto [t, c] = free_at.top();
      free_at.pop();
      wg.push_back(c);
      free_at.push({t + len[u & 0xffff] + kUnitOverhead, c});
    }
    return;
  }
  int32_t max_cost = 1;
  for (int32_t u : list) max_cost = std::max(max_cost, len[u & 0xffff] + kUnitOverhead);
  const int32_t window = max_cost + 1;
  std::vector<uint64_t> free_at(window, 0);
  free_at[0] = count == 64 ? ~0ull : (1ull << count) - 1;
  int32_t now = 0;
  for (int32_t u : list) {
    while (free_at[now] == 0) now = now + 1 == window ? 0 : now + 1;
    const uint64_t c = free_at[now] & (0 - free_at[now]);
    free_at[now] ^= c;
    int32_t then = now + len[u & 0xffff] + kUnitOverhead;
    if (then >= window) then -= window;
    free_at[then] |= c;
    wg.push_back(__builtin_ctzll(c));
  }
}

// Every (head, row) unit exactly once: a dropped unit would leave its output rows
// unwritten, a duplicated one would race with itself.
static int check_units(int32_t heads, int32_t rows, const std::vector<int32_t>& work) {
  std::vector<uint8_t> seen((size_t)heads * rows, 0);
  bool ok = work.size() == (size_t)heads * rows;
  for (size_t i = 0; ok && i < work.size(); i++) {
    const int32_t h = work[i] >> 16, r = work[i] & 0xffff;
    ok = h >= 0 && h < heads && r < rows && !seen[(size_t)h * rows + r];
    if (ok) seen[(size_t)h * rows + r] = 1;
  }
  if (!ok) {
    set_error("internal: the attention schedule does not list each of the %lld units once",
              (long long)heads * rows);
    return H3HIP_EHIP;
  }
  return H3HIP_OK;
}

int build_schedule(const std::vector<int32_t>& row_ptr, int32_t heads, int32_t groups,
                   std::vector<int32_t>& work_ptr, std::vector<int32_t>& work) {
  const int32_t nq = (int32_t)row_ptr.size() - 1;
  const int kXcd = 8;
  std::vector<int32_t> len(nq);
  for (int32_t i = 0; i < nq; i++) len[i] = row_ptr[i + 1] - row_ptr[i];
  std::vector<int32_t> sorted_len(len);
  std::sort(sorted_len.begin(), sorted_len.end());
  const int32_t median = nq ? sorted_len[nq / 2] : 0;
  const int32_t long_at = std::max<int32_t>(4 * median, median + 16);

  std::vector<std::vector<int32_t>> lists(kXcd);
  std::vector<double> cost(kXcd, 0.0);
  auto enc = [](int32_t h, int32_t qt) { return (h << 16) | qt; };

  // Long rows, one group per head, groups placed greedily on the least-loaded XCD.
  std::vector<int32_t> long_rows;
  for (int32_t i = 0; i < nq; i++)
    if (len[i] >= long_at) long_rows.push_back(i);
  std::stable_sort(long_rows.begin(), long_rows.end(),
                   [&](int32_t a, int32_t b) { return len[a] > len[b]; });
  double long_cost = 0;
  for (int32_t i : long_rows) long_cost += len[i] + kUnitOverhead;
  for (int32_t h = 0; h < heads && !long_rows.empty(); h++) {
    const int x = (int)(std::min_element(cost.begin(), cost.end()) - cost.begin());
    for (int32_t i : long_rows) lists[x].push_back(enc(h, i));
    cost[x] += long_cost;
  }

  // Regular rows: one contiguous (head, q-tile) sequence split into ranges that
  // top every XCD up to the same total.
  std::vector<int32_t> rows;   // regular rows, the same for every head
  double reg_cost = 0;
  for (int32_t i = 0; i < nq; i++)
    if (len[i] < long_at) {
      rows.push_back(i);
      reg_cost += len[i] + kUnitOverhead;
    }
  const size_t n_regular = rows.size() * heads;
  double total = reg_cost * heads;
  for (double c : cost) total += c;
  const double target = total / kXcd;
  size_t pos = 0, row = 0;
  int32_t head = 0;
  // Fill the least-loaded XCDs first so ranges stay contiguous per XCD.
  std::vector<int> order(kXcd);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost[a] < cost[b]; });
  for (int oi = 0; oi < kXcd; oi++) {
    const int x = order[oi];
    lists[x].reserve(lists[x].size() + n_regular / kXcd * 2);
    for (; pos < n_regular && (oi == kXcd - 1 || cost[x] < target); pos++) {
      const int32_t qt = rows[row];
      lists[x].push_back(enc(head, qt));
      cost[x] += len[qt] + kUnitOverhead;
      if (++row == rows.size()) row = 0, head++;
    }
  }
  // Each XCD's list onto its groups / 8 workgroups (workgroup c*8 + x is the
  // c-th of XCD x): every unit's workgroup in list order, then a counting sort.
  const int per_xcd = groups / kXcd;
  std::vector<int32_t> wg;
  wg.reserve((size_t)heads * nq);
  work_ptr.assign(groups + 1, 0);
  for (int x = 0; x < kXcd; x++) {
    const size_t first = wg.size();
    deal(lists[x], len, per_xcd, wg);
    for (size_t i = first; i < wg.size(); i++) {
      wg[i] = wg[i] * kXcd + x;
      work_ptr[wg[i] + 1]++;
    }
  }
  for (int b = 0; b < groups; b++) work_ptr[b + 1] += work_ptr[b];
  work.assign(wg.size(), 0);
  std::vector<int32_t> next(work_ptr.begin(), work_ptr.end() - 1);
  size_t at = 0;
  for (int x = 0; x < kXcd; x++)
    for (int32_t u : lists[x]) work[next[wg[at++]]++] = u;
  return check_units(heads, nq, work);
}

// One unit per workgroup at most (heads x rows <= groups), a contiguous range per
// XCD, so that the units of a head share its L2.
static int spread_units(int32_t heads, int32_t rows, int32_t groups,
                        std::vector<int32_t>& work_ptr, std::vector<int32_t>& work) {
  const int64_t units = (int64_t)heads * rows;
  std::vector<int32_t> at(groups, -1);
  for (int x = 0; x < 8; x++) {
    const int32_t first = (int32_t)(units * x / 8), last = (int32_t)(units * (x + 1) / 8);
    for (int32_t i = first; i < last; i++) at[(i - first) * 8 + x] = (i / rows) << 16 | i % rows;
  }
  work.clear();
  work_ptr.assign(groups + 1, 0);
  for (int32_t b = 0; b < groups; b++) {
    if (at[b] >= 0) work.push_back(at[b]);
    work_ptr[b + 1] = (int32_t)work.size();
  }
  return check_units(heads, rows, work);
}

// Cost of a unit beyond its tiles and of a tile, in whole units' tiles, for the
// comparison below: a rule on the cautious side, not the cost of a half unit, which
// depends on how busy the chip is. Alone on its CU a half unit takes 0.73-0.82 of a
// whole one's time (dense rows of 3, 8, 16 and 42 tiles on MI355X: 7.8, 11.4, 17.4
// and 38.9 us against 10.2, 15.4, 23.6 and 51.8, launch included); where all CUs
// work, two take 1.13-1.28 of one (the constants say 1.7). Of 327 plans timed both
// ways (equal, local, axial and drawn rows, 8 to 1,536 units) it picks the faster
// units, or units within 0.5% of them, for 304. For 22 it stays with whole units
// where half ones are up to 15% faster; one runs half units that are 3% slower.
constexpr double kFullUnit = 2.0, kHalfUnit = 1.7, kHalfTile = 0.85;
// Whole units per workgroup up to which half units are looked at. Past it a
// launch is bound by the chip's throughput, where half units take 1.13-1.28 times
// the whole ones' time.
constexpr int kHalfUnitsUpTo = 6;

// The time the cost model gives the longest workgroup of these lists.
static double longest_workgroup(const std::vector<int32_t>& row_ptr,
                                const std::vector<int32_t>& work_ptr,
                                const std::vector<int32_t>& work, double unit, double tile) {
  double worst = 0;
  for (size_t b = 0; b + 1 < work_ptr.size(); b++) {
    double t = 0;
    for (int32_t i = work_ptr[b]; i < work_ptr[b + 1]; i++) {
      const int32_t row = work[i] & 0xffff;
      t += unit + tile * (row_ptr[row + 1] - row_ptr[row]);
    }
    worst = std::max(worst, t);
  }
  return worst;
}

// Whole units, or half units (64 queries, bsattn_half.hip) where their longest
// workgroup ends earlier: few units (917 tokens x 8 heads: 15.9 -> 11.8 us), or few
// long rows among short ones (31,885 tokens x 2 heads of the local rule, whose 5
// prefix rows see all 250 tiles: 295 -> 236 us).
int plan_schedule(const std::vector<int32_t>& row_ptr, int32_t heads, int32_t groups,
                  bool& half_units, std::vector<int32_t>& work_ptr, std::vector<int32_t>& work) {
  half_units = false;
  int rc = build_schedule(row_ptr, heads, groups, work_ptr, work);
  if (rc != H3HIP_OK) return rc;
  const int32_t n = (int32_t)row_ptr.size() - 1;
  if ((int64_t)heads * n > kHalfUnitsUpTo * (int64_t)groups) return H3HIP_OK;
  std::vector<int32_t> half_rows(2 * (size_t)n + 1, 0), half_ptr, half_work;
  for (size_t r = 0; r + 1 < half_rows.size(); r++)
    half_rows[r + 1] = half_rows[r] + row_ptr[r / 2 + 1] - row_ptr[r / 2];
  // build_schedule balances the XCDs by cost and gives some workgroups two units
  // where each could have one (4,096 tokens x 4 heads of a band: 15.4 us, spread
  // 11.1, full units 14.1).
  rc = 2 * (int64_t)heads * n <= groups
           ? spread_units(heads, 2 * n, groups, half_ptr, half_work)
           : build_schedule(half_rows, heads, groups, half_ptr, half_work);
  if (rc != H3HIP_OK) return rc;
  if (longest_workgroup(half_rows, half_ptr, half_work, kHalfUnit, kHalfTile) <
      longest_workgroup(row_ptr, work_ptr, work, kFullUnit, 1.0)) {
    half_units = true;
    work_ptr = std::move(half_ptr);
    work = std::move(half_work);
  }
  return H3HIP_OK;
}

}  // namespace h3hip

extern "C" int h3hip_schedule(const int32_t* row_ptr, int32_t n_tiles, int32_t heads,
                              int32_t groups, int32_t* work_ptr, int32_t* work) {
  using h3hip::set_error;
  if (!row_ptr || !work_ptr || !work) {
    set_error("NULL argument");
    return H3HIP_EINVAL;
  }
  if (n_tiles <= 0 || n_tiles > 32767 || heads <= 0 || heads >= 32768 || groups <= 0 ||
      groups % 8 != 0) {
    set_error("bad shape: n_tiles %d heads %d groups %d (groups a positive multiple of 8)",
              n_tiles, heads, groups);
    return H3HIP_EINVAL;
  }
  std::vector<int32_t> rp(row_ptr, row_ptr + n_tiles + 1);
  if (rp[0] != 0) {
    set_error("row_ptr[0] must be 0");
    return H3HIP_EINVAL;
  }
  for (int32_t i = 0; i < n_tiles; i++)
    if (rp[i + 1] < rp[i] || rp[i + 1] - rp[i] > n_tiles) {
      set_error("row_ptr is not a CSR row pointer over %d columns at row %d", n_tiles, i);
      return H3HIP_EINVAL;
    }
  std::vector<int32_t> wp, w;
  const int rc = h3hip::build_schedule(rp, heads, groups, wp, w);
  if (rc != H3HIP_OK) return rc;
  std::copy(wp.begin(), wp.end(), work_ptr);
  std::copy(w.begin(), w.end(), work);
  return H3HIP_OK;
}
