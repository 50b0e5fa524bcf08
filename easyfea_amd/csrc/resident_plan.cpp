// Host side of a resident solve's plan: the bisection of the nodes into blocks
// and the blocks' neighbour tables, on host arrays.
//
// A plan is built once per pattern, inside the first solve on it.  On the device
// with torch's sorts the tables took 3 to 4 ms, but the first use of those
// operations in a process loads their code objects (130 to 600 ms), and numpy's
// bisection of a million nodes took 380 ms.  Here parts and blocks are
// independent tasks, which a few threads take in turn.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <limits>
#include <thread>
#include <vector>

#include "efea_common.h"
#include "resident.h"

namespace efea {

constexpr int WORKERS = 8;          // threads at most, the bisection's 2^3 among them
constexpr int64_t ALONE = 1 << 16;  // nodes or neighbours below which one thread is as fast

// f(task) for every task, by up to `workers` threads, the caller among
// them (fewer where threads cannot be had).  f does not throw.
template <typename F>
static void for_tasks(int tasks, int workers, const F& f) {
  std::atomic<int> next{0};
  auto take = [&] {
    for (int i; (i = next.fetch_add(1)) < tasks;) f(i);
  };
  std::vector<std::thread> ts;
  try {
    for (int w = 1; w < workers; ++w) ts.emplace_back(take);
  } catch (const std::exception&) {
  }
  take();
  for (auto& t : ts) t.join();
}

struct AxisNode {
  double x;
  int id;
  bool operator<(const AxisNode& o) const { return x < o.x || (x == o.x && id < o.id); }
};

// Nodes [lo, hi) of `order` into k parts numbered from p0; s: scratch as long as
// order; levels: how often the halves may still go to two threads.
static void bisect(const double* coord, AxisNode* s, int* order, int* part_ptr, int64_t lo, int64_t hi, int k,
                   int p0, int levels) {
  if (k == 1) {
    std::sort(order + lo, order + hi);
    part_ptr[p0] = (int)lo;
    return;
  }
  double mn[3], mx[3];
  for (int d = 0; d < 3; ++d) {
    mn[d] = std::numeric_limits<double>::infinity();
    mx[d] = -mn[d];
  }
  for (int64_t i = lo; i < hi; ++i)
    for (int d = 0; d < 3; ++d) {
      const double c = coord[3 * (int64_t)order[i] + d];
      mn[d] = c < mn[d] ? c : mn[d];
      mx[d] = c > mx[d] ? c : mx[d];
    }
  int axis = 0;
  for (int d = 1; d < 3; ++d)
    if (mx[d] - mn[d] > mx[axis] - mn[axis]) axis = d;
  const int64_t mid = lo + (hi - lo) * (k / 2) / k;
  if (mid > lo && mid < hi) {
    for (int64_t i = lo; i < hi; ++i) {
      const double c = coord[3 * (int64_t)order[i] + axis];
      s[i] = {std::isnan(c) ? std::numeric_limits<double>::infinity() : c, order[i]};
    }
    std::nth_element(s + lo, s + mid, s + hi);
    for (int64_t i = lo; i < hi; ++i) order[i] = s[i].id;
  }
  for_tasks(2, levels > 0 && hi - lo > ALONE ? 2 : 1, [&](int half) {
    if (half == 0)
      bisect(coord, s, order, part_ptr, lo, mid, k / 2, p0, levels - 1);
    else
      bisect(coord, s, order, part_ptr, mid, hi, k - k / 2, p0 + k / 2, levels - 1);
  });
}

int resident_bisect(int Nn, const double* coord, int parts, int* order, int* part_ptr) {
  try {
    std::vector<AxisNode> s(Nn);
    for (int i = 0; i < Nn; ++i) order[i] = i;
    bisect(coord, s.data(), order, part_ptr, 0, Nn, parts, 0, 3);
    part_ptr[parts] = Nn;
  } catch (const std::exception& e) {
    set_error("resident_bisect: %s", e.what());
    return EFEA_ERR_SIZE;
  }
  return EFEA_OK;
}

int resident_neighbours(int Nn, const int* node_ptr, const int* node_cols, int lanes, int slots, int passes, int nblk,
                        const int* rows, unsigned short* lidx, int* halo_ptr, int* halo_ex, int halo_room, int* pub,
                        int* pub_ptr, int* pub_pos, int* self, int* nex, int* max_halo) {
  constexpr int RT = 512, RNW = RT / 64;
  const int per = 64 / lanes, nloc = per * RNW * passes, kept = lanes == 1 ? slots - 1 : slots;
  const int npos = nblk * nloc;
  std::atomic<int> bad{0};
  try {
    std::vector<int> pos(Nn, -1);
    for (int p = 0; p < npos; ++p) {
      if (rows[p] < -1 || rows[p] >= Nn) bad = 1;
      else if (rows[p] >= 0) pos[rows[p]] = p;
    }
    for (int n = 0; n < Nn; ++n)
      if (pos[n] < 0 || node_ptr[n + 1] < node_ptr[n]) bad = 1;
    for (int k = node_ptr[0]; !bad && k < node_ptr[Nn]; ++k)
      if (node_cols[k] < 0 || node_cols[k] >= Nn) bad = 1;
    if (bad) {
      set_error("resident_neighbours: rows or columns out of range, or a node without a position");
      return EFEA_ERR_ARG;
    }
    std::vector<std::vector<int>> halo(nblk);  // positions, ascending
    std::vector<std::atomic<unsigned char>> read(npos);
    for (auto& r : read) r.store(0, std::memory_order_relaxed);
    for_tasks(nblk, node_ptr[Nn] > 4 * ALONE ? WORKERS : 1, [&](int b) {
      std::vector<int>& h = halo[b];
      const int b0 = b * nloc;
      try {
        for (int p = 0; p < nloc; ++p) {
          const int n = rows[b0 + p];
          for (int k = n >= 0 ? node_ptr[n] : 0; n >= 0 && k < node_ptr[n + 1]; ++k) {
            const int q = pos[node_cols[k]];
            if (q / nloc != b) h.push_back(q);
          }
        }
      } catch (const std::exception&) {
        bad = 2;
        return;
      }
      std::sort(h.begin(), h.end());
      h.erase(std::unique(h.begin(), h.end()), h.end());
      for (int q : h) read[q].store(1, std::memory_order_relaxed);
      unsigned short* out = lidx + (int64_t)b * passes * kept * RT;
      std::fill(out, out + (int64_t)passes * kept * RT, (unsigned short)0);
      for (int p = 0; p < nloc; ++p) {
        const int n = rows[b0 + p], chunk = p / per;
        self[b0 + p] = 0;
        if (n < 0) continue;
        const int k0 = node_ptr[n], cnt = node_ptr[n + 1] - k0;
        int s = cnt;  // scalar rows: the node itself comes first, without an entry
        if (lanes == 1) {
          for (int k = 0; k < cnt; ++k)
            if (node_cols[k0 + k] == n) s = k;
          if (s < cnt) self[b0 + p] = s;
        }
        for (int k = 0; k < cnt; ++k) {
          if (k == s) continue;
          const int num = k < s && s < cnt ? k + 1 : k, slot = num / lanes - (slots - kept);
          if (slot < 0 || slot >= kept) {
            bad = 3;
            continue;
          }
          const int q = pos[node_cols[k0 + k]];
          const int local =
              q / nloc == b ? q - b0 : nloc + (int)(std::lower_bound(h.begin(), h.end(), q) - h.begin());
          const int thread = chunk % RNW * 64 + p % per * lanes + num % lanes;
          out[((int64_t)(chunk / RNW) * kept + slot) * RT + thread] = (unsigned short)local;
        }
      }
    });
    if (bad) {
      set_error(bad == 2 ? "resident_neighbours: out of memory" : "resident_neighbours: a row longer than its slots");
      return bad == 2 ? EFEA_ERR_SIZE : EFEA_ERR_ARG;
    }
    int e = 0;
    for (int b = 0; b < nblk; ++b) {
      pub_ptr[b] = e;
      for (int p = 0; p < nloc; ++p) {
        const int q = b * nloc + p;
        pub[q] = -1;
        if (!read[q].load(std::memory_order_relaxed)) continue;
        pub_pos[e] = p;
        pub[q] = e++;
      }
    }
    pub_ptr[nblk] = *nex = e;
    int64_t total = 0;
    size_t most = 0;
    for (const auto& h : halo) {
      total += (int64_t)h.size();
      most = std::max(most, h.size());
    }
    if (total > halo_room) {
      set_error("resident_neighbours: room for %d halo entries, %lld needed", halo_room, (long long)total);
      return EFEA_ERR_SIZE;
    }
    int at = 0;
    for (int b = 0; b < nblk; ++b) {
      halo_ptr[b] = at;
      for (int q : halo[b]) halo_ex[at++] = pub[q];
    }
    halo_ptr[nblk] = at;
    *max_halo = (int)most;
  } catch (const std::exception& ex) {
    set_error("resident_neighbours: %s", ex.what());
    return EFEA_ERR_SIZE;
  }
  return EFEA_OK;
}

}  // namespace efea
