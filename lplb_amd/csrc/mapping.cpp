// Expert placement: EPLB packing and replication, and the planner's layout of physical experts, on the host, in C++ alone:
// it is part of liblplb_hip.so and, for hosts without a GPU or ROCm, the whole of liblplb_host.so.
//
// It runs once per re-shuffle, on a few hundred numbers, between two batches: what it costs is the host time
// of the call.  update_redundancy_mapping at 256 experts on 32 ranks, history on the GPU: 755 us as numpy loops
// (one interpreted argmin per expert and pass) and three copies to the GPU, 42 us here, of which the arithmetic
// is 12 and the two synchronising copies most of the rest (20.9 us with 64 experts per node and 29
// with 256, which place.hip places on the GPU).  Behaviour follows the reference's embedded EPLB (lplb/eplb.py:6-190) and its
// use in the planner (lplb/planner.py:115-182); weights are 32-bit floats throughout, items of equal weight
// are taken in index order and a tie between packs goes to the lowest (the reference sorts unstably).
#include "error.h"

#include <algorithm>
#include <cmath>
#include <exception>
#include <numeric>
#include <vector>

namespace lplb {

// Heaviest first, equal ones in index order, NaN last.
template <typename T> static void order_by_weight(const T *weight, int n, std::vector<int> &order) {
  order.resize(n);
  std::iota(order.begin(), order.end(), 0);
  const auto earlier = [weight](int a, int b) {
    const T x = weight[a], y = weight[b];
    return x > y || (std::isnan(y) && !std::isnan(x));
  };
  if (n > 16) {
    std::stable_sort(order.begin(), order.end(), earlier);
    return;
  }
  for (int i = 1; i < n; ++i) {   // (the library's sort allocates)
    const int item = order[i];
    int k = i;
    for (; k > 0 && earlier(item, order[k - 1]); --k)
      order[k] = order[k - 1];
    order[k] = item;
  }
}

// n items into n_packs packs of n / n_packs each, heaviest first, each into the lightest pack with room left.
static void pack_balanced(const float *weight, int n, int n_packs, int64_t *pack_of, int64_t *rank_in_pack) {
  const int room = n / n_packs;
  if (room == 1) {
    for (int i = 0; i < n; ++i) {
      pack_of[i] = i;
      rank_in_pack[i] = 0;
    }
    return;
  }
  // The packs with room, in the order of their numbers.  Only those: among loads of infinity a search over all packs would
  // come upon a full one.
  std::vector<float> load(n_packs, 0.0f);
  std::vector<int> open(n_packs), fill(n_packs, 0), order;
  std::iota(open.begin(), open.end(), 0);
  order_by_weight(weight, n, order);
  int n_open = n_packs;
  for (const int item : order) {
    int best = 0;
    for (int k = 1; k < n_open; ++k)
      if (load[k] < load[best] || (std::isnan(load[k]) && !std::isnan(load[best])))
        best = k;
    pack_of[item] = open[best];
    rank_in_pack[item] = fill[best]++;
    load[best] += weight[item];
    if (fill[best] == room) {
      --n_open;
      for (int k = best; k < n_open; ++k) {
        load[k] = load[k + 1];
        open[k] = open[k + 1];
        fill[k] = fill[k + 1];
      }
    }
  }
}

// n_phy - n_log replicas, each of the expert whose load per copy is largest then.
static void replicate(const float *weight, int n_log, int n_phy, int64_t *phy2log, int64_t *rank, int64_t *logcnt) {
  for (int i = 0; i < n_log; ++i) {
    phy2log[i] = i;
    rank[i] = 0;
    logcnt[i] = 1;
  }
  for (int slot = n_log; slot < n_phy; ++slot) {
    int best = 0;
    float heaviest = weight[0] / (float)logcnt[0];
    for (int i = 1; i < n_log && !std::isnan(heaviest); ++i) {
      const float w = weight[i] / (float)logcnt[i];
      if (w > heaviest || std::isnan(w)) {
        best = i;
        heaviest = w;
      }
    }
    phy2log[slot] = best;
    rank[slot] = logcnt[best]++;
  }
}

// Sum of n floats in eight interleaved partial sums, halved recursively beyond 128: the order in which a
// numpy sum adds them up.  Groups of equal content then weigh the same whoever adds them up.
static float sum_pairwise(const float *v, int n) {
  if (n < 8) {
    float s = 0.0f;
    for (int i = 0; i < n; ++i)
      s += v[i];
    return s;
  }
  if (n > 128) {
    const int half = n / 2 / 8 * 8;
    return sum_pairwise(v, half) + sum_pairwise(v + half, n - half);
  }
  float r[8];
  for (int k = 0; k < 8; ++k)
    r[k] = v[k];
  int i = 8;
  for (; i + 8 <= n; i += 8)
    for (int k = 0; k < 8; ++k)
      r[k] += v[i + k];
  float s = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
  for (; i < n; ++i)
    s += v[i];
  return s;
}

// One layer: whole groups onto nodes, replicas inside each node, physical experts onto the node's GPUs.
static void rebalance_layer(const float *weight, int n_log, int n_phy, int n_groups, int n_nodes, int n_gpus,
                            int64_t *phy2log, int64_t *phyrank, int64_t *logcnt) {
  const int group_size = n_log / n_groups, groups_per_node = n_groups / n_nodes;
  const int log_per_node = n_log / n_nodes, phy_per_node = n_phy / n_nodes, phy_per_gpu = n_phy / n_gpus;
  std::vector<float> group_weight(n_groups), node_weight(n_log), phy_weight(phy_per_node);
  std::vector<int64_t> g_pack(n_groups), g_rank(n_groups), log_of(n_log);   // log_of: node-ordered -> logical
  for (int g = 0; g < n_groups; ++g)
    group_weight[g] = sum_pairwise(weight + (int64_t)g * group_size, group_size);
  pack_balanced(group_weight.data(), n_groups, n_nodes, g_pack.data(), g_rank.data());
  for (int g = 0; g < n_groups; ++g)
    for (int k = 0; k < group_size; ++k) {
      const int64_t at = (g_pack[g] * groups_per_node + g_rank[g]) * group_size + k;
      log_of[at] = (int64_t)g * group_size + k;
      node_weight[at] = weight[log_of[at]];
    }
  std::vector<int64_t> phy2node(phy_per_node), rank(phy_per_node), count(log_per_node), pack(phy_per_node), place(phy_per_node);
  for (int node = 0; node < n_nodes; ++node) {
    const float *w = node_weight.data() + (int64_t)node * log_per_node;
    const int64_t *to_log = log_of.data() + (int64_t)node * log_per_node;
    replicate(w, log_per_node, phy_per_node, phy2node.data(), rank.data(), count.data());
    for (int i = 0; i < phy_per_node; ++i)
      phy_weight[i] = w[phy2node[i]] / (float)count[phy2node[i]];
    pack_balanced(phy_weight.data(), phy_per_node, n_gpus / n_nodes, pack.data(), place.data());
    for (int i = 0; i < phy_per_node; ++i) {
      const int64_t at = (int64_t)node * phy_per_node + pack[i] * phy_per_gpu + place[i];
      phy2log[at] = to_log[phy2node[i]];
      phyrank[at] = rank[i];
    }
    for (int i = 0; i < log_per_node; ++i)
      logcnt[to_log[i]] = count[i];
  }
}

// No exception crosses the C boundary.
template <typename F> static int without_exceptions(F &&f) {
  try {
    return f();
  } catch (const std::exception &e) {
    return fail(LPLB_EINVAL, "expert placement: %s", e.what());
  }
}

static int check_rebalance(int n_log, int n_phy, int n_groups, int n_nodes, int n_gpus) {
  LPLB_REQUIRE(n_log > 0 && n_groups > 0 && n_nodes > 0 && n_gpus > 0, LPLB_EINVAL, "rebalance_experts: sizes must be positive");
  LPLB_REQUIRE(n_log % n_groups == 0 && n_groups % n_nodes == 0 && n_gpus % n_nodes == 0 && n_phy % n_gpus == 0 && n_phy >= n_log,
               LPLB_EINVAL, "rebalance_experts: %d experts in %d groups, %d physical ones, do not divide over %d nodes with %d GPUs",
               n_log, n_groups, n_phy, n_nodes, n_gpus);
  return LPLB_OK;
}

} // namespace lplb

extern "C" int lplb_balanced_packing(const float *weight, int n_layers, int n_items, int n_packs, int64_t *pack_index,
                                     int64_t *rank_in_pack) {
  using namespace lplb;
  LPLB_REQUIRE(n_layers >= 0 && n_items > 0 && n_packs > 0 && n_items % n_packs == 0, LPLB_EINVAL,
               "balanced_packing: %d items do not divide over %d packs", n_items, n_packs);
  LPLB_REQUIRE(weight && pack_index && rank_in_pack, LPLB_EINVAL, "balanced_packing: null pointer");
  return without_exceptions([&] {
    for (int64_t x = 0; x < n_layers; ++x)
      pack_balanced(weight + x * n_items, n_items, n_packs, pack_index + x * n_items, rank_in_pack + x * n_items);
    return LPLB_OK;
  });
}

extern "C" int lplb_replicate_experts(const float *weight, int n_rows, int n_log, int n_phy, int64_t *phy2log, int64_t *rank,
                                      int64_t *logcnt) {
  using namespace lplb;
  LPLB_REQUIRE(n_rows >= 0 && n_log > 0 && n_phy >= n_log, LPLB_EINVAL, "replicate_experts: %d physical, %d logical experts", n_phy, n_log);
  LPLB_REQUIRE(weight && phy2log && rank && logcnt, LPLB_EINVAL, "replicate_experts: null pointer");
  for (int64_t x = 0; x < n_rows; ++x)
    replicate(weight + x * n_log, n_log, n_phy, phy2log + x * n_phy, rank + x * n_phy, logcnt + x * n_log);
  return LPLB_OK;
}

extern "C" int lplb_rebalance_experts(const float *weight, int n_layers, int n_log, int n_phy, int n_groups, int n_nodes,
                                      int n_gpus, int64_t *phy2log, int64_t *phyrank, int64_t *logcnt) {
  using namespace lplb;
  const int rc = check_rebalance(n_log, n_phy, n_groups, n_nodes, n_gpus);
  if (rc != LPLB_OK)
    return rc;
  LPLB_REQUIRE(n_layers >= 0 && weight && phy2log && phyrank && logcnt, LPLB_EINVAL, "rebalance_experts: null pointer");
  return without_exceptions([&] {
    for (int64_t x = 0; x < n_layers; ++x)
      rebalance_layer(weight + x * n_log, n_log, n_phy, n_groups, n_nodes, n_gpus, phy2log + x * n_phy, phyrank + x * n_phy,
                      logcnt + x * n_log);
    return LPLB_OK;
  });
}

namespace lplb {

static int build_mapping(const float *weight, const double *history, const int32_t *r2o, int group_size,
                         int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes, int32_t *phy2log,
                         int32_t *log2phy, int32_t *logcnt) {
  const int G = group_size, D = dup_per_rank;
  LPLB_REQUIRE(r2o && phy2log && log2phy && logcnt && (weight == nullptr) == (history == nullptr), LPLB_EINVAL,
               "build_mapping: null pointer");
  LPLB_REQUIRE(G > 0 && D > 0 && ep_size > 0 && n_nodes > 0 && n_logical > 0 && ep_size % G == 0 && n_logical % ep_size == 0, LPLB_EINVAL,
               "build_mapping: %d logical experts on %d ranks in groups of %d", n_logical, ep_size, G);
  const int n_group = ep_size / G, L = n_logical / ep_size, P = n_physical / ep_size, C = (P - L) / D, CD = C * D;
  LPLB_REQUIRE(P >= L && CD <= L && (int64_t)ep_size * (L + CD) == n_physical, LPLB_EINVAL,
               "build_mapping: %d physical experts do not lay out %d logical ones on %d ranks with %d slots for replicas",
               n_physical, n_logical, ep_size, D);
  // the experts of every rank, those that get a replica first
  std::vector<int64_t> ranks(n_logical);
  if (!weight) {
    std::iota(ranks.begin(), ranks.end(), 0);
  } else {
    const bool by_node = n_group % n_nodes == 0;
    const int rc = check_rebalance(n_logical, n_logical, by_node ? n_group : 1, by_node ? n_nodes : 1, ep_size);
    if (rc != LPLB_OK)
      return rc;
    std::vector<int64_t> unused_rank(n_logical), unused_count(n_logical);
    rebalance_layer(weight, n_logical, n_logical, by_node ? n_group : 1, by_node ? n_nodes : 1, ep_size, ranks.data(),
                    unused_rank.data(), unused_count.data());
    std::vector<double> load(L);
    std::vector<int> order;
    std::vector<int64_t> sorted(L);
    for (int rank = 0; rank < ep_size; ++rank) {
      int64_t *mine = ranks.data() + (int64_t)rank * L;
      for (int k = 0; k < L; ++k)
        load[k] = history[mine[k]];
      order_by_weight(load.data(), L, order);
      for (int k = 0; k < L; ++k)
        sorted[k] = mine[order[k]];
      std::copy(sorted.begin(), sorted.end(), mine);
    }
  }
  for (int g = 0; g < n_group; ++g)
    for (int i = 0; i < G; ++i) {
      int32_t *row = phy2log + (int64_t)(g * G + i) * P;
      const int64_t *mine = ranks.data() + (int64_t)(g * G + i) * L;
      for (int k = 0; k < L; ++k)
        row[k] = (int32_t)mine[k];
      for (int d = 0; d < D; ++d) {
        int from = r2o[i * D + d];
        LPLB_REQUIRE(from >= -G && from < G, LPLB_EINVAL, "build_mapping: r2o[%d][%d] = %d is no rank of a group of %d", i, d, from, G);
        from = from < 0 ? from + G : from;
        for (int c = 0; c < C; ++c)   // replica (c, d) of rank i <- original (c, d) of rank r2o[i, d]
          row[L + c * D + d] = (int32_t)ranks[(int64_t)(g * G + from) * L + c * D + d];
      }
    }
  // originals before replicas: physical experts by (place on the rank, rank)
  int most = 0;
  std::fill(logcnt, logcnt + n_logical, 0);
  std::fill(log2phy, log2phy + 2 * (int64_t)n_logical, -1);
  for (int place = 0; place < P; ++place)
    for (int rank = 0; rank < ep_size; ++rank) {
      const int phy = rank * P + place, e = phy2log[phy];
      if (logcnt[e] < 2)
        log2phy[2 * (int64_t)e + logcnt[e]] = phy;
      most = std::max(most, ++logcnt[e]);
    }
  LPLB_REQUIRE(most == 2, LPLB_EINVAL, "every logical expert may have at most one replica (got %d copies)", most);
  return LPLB_OK;
}

} // namespace lplb

extern "C" int lplb_build_mapping(const float *weight, const double *history, const int32_t *r2o, int group_size,
                                  int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes, int32_t *phy2log,
                                  int32_t *log2phy, int32_t *logcnt) {
  return lplb::without_exceptions([&] {
    return lplb::build_mapping(weight, history, r2o, group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, phy2log, log2phy,
                               logcnt);
  });
}
