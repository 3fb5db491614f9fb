// The planner's layout of physical experts from a load history that is on the GPU, as one workgroup
// (lplb_place_experts).  Same result as lplb_build_mapping on the host (mapping.cpp), bit for bit: experts are spread over the
// ranks by greedy packing, heaviest first, each into the lightest pack with room (lplb/eplb.py:6-46), each rank's experts
// are sorted heaviest first and the first of them get the replicas (lplb/planner.py:127-182).
//
// On the host the arithmetic takes 11 us, but the history has to come over (a copy the host waits for) and the tables have to go
// back (another).  Here nothing crosses: one launch, and the host waits once, because the tables are there for every stream
// when the call returns.  update_redundancy_mapping of 256 experts on 32 ranks of 4 nodes, history on the GPU: 43.6 -> 27.0 us,
// of which the kernel is 8.7.  What bounds that is the packing, a serial chain of one step per expert of a node (64 here), 68 ns
// each: least load by DPP, its lane from a ballot; the nodes are packed side by side, a wave each.  The sorts rank every item by
// counting those ahead of it.
#include "map_kernel.h"

namespace lplb {

// A core of the host takes 30 ns for a step of the packing.  Per call, host / here: 64 experts of a node 43.6 / 27.0 us, 128 42.1 / 32.0
// (8 ranks) and 43.5 / 33.1 (16), 256 45.0 / 44.2 and, into 32 packs, 45.6 / 45.5: from there on the host is as fast.
constexpr int kPlaceMaxPerNode = 128;
constexpr int kPlaceMaxExperts = 1024, kPlaceMaxPacks = 64, kPlaceMaxEdges = 2 * kWave;

// Floats in an order that unsigned comparison understands; -0 is 0.
__device__ inline uint32_t ascending(float v) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v + 0.0f);
  return b >> 31 ? ~b : b | 0x80000000u;
}
// Heaviest first, NaN last.
__device__ inline uint32_t heaviest_first(float v) { return v != v ? 0xffffffffu : ~ascending(v); }
__device__ inline bool heavier(double x, double y) { return x > y || (y != y && x == x); }

struct PlaceArgs {
  const void *history;
  const int32_t *r2o;
  int32_t *phy2log, *log2phy, *logcnt;
  int G, D, L, P, ep_size, n_logical, per_node, n_nodes, packs;
  uint32_t magic_G, magic_D, magic_L, magic_P, magic_per_node;   // fast_div_magic
};

template <int CTRL> __device__ inline uint32_t min_dpp(uint32_t v) {
  return min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffffu, (int)v, CTRL, 0xF, 0xF, false));
}
// One node's experts, in `order`, into its packs: lane = pack, PACKS lanes at least (8, 16, 32 or 64).  SIMPLE: no weight is
// negative or not a number, so a load's bits are in its order.  packed[pack * room + place] = expert.
// A step is: least key by DPP, the first lane that has it from a ballot; what that lane's load and key will be is worked out
// beside.  (A load that is not a number is taken first, of equal ones the first; a full pack never.)
template <int PACKS, bool SIMPLE>
__device__ inline void pack_node(const int32_t *order, const float *weight, int n, int packs, int room, int32_t *packed, int lane) {
  constexpr uint32_t kFull = 0xffffffffu;
  auto key_of = [](float v) {
    return SIMPLE ? __builtin_bit_cast(uint32_t, v) : v != v ? 0u : ascending(v);
  };
  const unsigned long long mask = packs == kWave ? ~0ull : (1ull << packs) - 1;
  float load = 0.0f;
  int fill = 0;
  uint32_t key = lane < packs ? key_of(0.0f) : kFull;
  for (int s0 = 0; s0 < n; s0 += kWave) {
    const int item = s0 + lane < n ? order[s0 + lane] : 0;
    const int weight_bits = __builtin_bit_cast(int, weight[item]);
    const int end = min(kWave, n - s0);
    int place = 0;   // lane = item: where it goes
    auto step = [&](int s) {
      const float sum = load + __builtin_bit_cast(float, __builtin_amdgcn_readlane(weight_bits, s));
      const uint32_t next = fill + 1 >= room ? kFull : key_of(sum);
      uint32_t least = min_dpp<0xB1>(key);   // quad_perm [1,0,3,2]
      least = min_dpp<0x4E>(least);          // quad_perm [2,3,0,1]
      least = min_dpp<0x141>(least);         // row_half_mirror
      if constexpr (PACKS > 8)
        least = min_dpp<0x128>(least);       // row_ror:8
      if constexpr (PACKS > 16) {
        auto of_row = [in_row = (int)least](int at) { return (uint32_t)__builtin_amdgcn_readlane(in_row, at); };
        least = min(of_row(0), of_row(16));
        if constexpr (PACKS > 32)
          least = min(least, min(of_row(32), of_row(48)));
      }
      const int best = __builtin_ctzll(__ballot(key == least) & mask);
      const int at = best * room + __builtin_amdgcn_readlane(fill, best);
      const bool chosen = lane == best;
      place = lane == s ? at : place;
      key = chosen ? next : key;
      load = chosen ? sum : load;
      fill += chosen ? 1 : 0;
    };
    int s = 0;
    for (; s + 4 <= end; s += 4)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        step(s + k);
    for (; s < end; ++s)
      step(s);
    if (lane < end)
      packed[place] = item;
  }
}
template <bool SIMPLE>
__device__ inline void pack_node_of(const int32_t *order, const float *weight, int n, int packs, int room, int32_t *packed, int lane) {
  if (packs <= 8)
    pack_node<8, SIMPLE>(order, weight, n, packs, room, packed, lane);
  else if (packs <= 16)
    pack_node<16, SIMPLE>(order, weight, n, packs, room, packed, lane);
  else if (packs <= 32)
    pack_node<32, SIMPLE>(order, weight, n, packs, room, packed, lane);
  else
    pack_node<64, SIMPLE>(order, weight, n, packs, room, packed, lane);
}

template <typename T> __global__ __launch_bounds__(kPlaceMaxExperts) void place_experts(PlaceArgs a) {
  __shared__ uint32_t key[kPlaceMaxExperts];
  __shared__ float weight[kPlaceMaxExperts];
  __shared__ double load_of[kPlaceMaxExperts];
  __shared__ int32_t order[kPlaceMaxExperts], packed[kPlaceMaxExperts], sorted[kPlaceMaxExperts], replica[kPlaceMaxExperts];
  __shared__ int32_t from_rank[kPlaceMaxEdges];
  __shared__ int not_simple;
  fetch_arguments_now(a.history, a.n_logical, a.magic_P);
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n = a.n_logical, per_node = a.per_node, room = a.L;
  if (tid == 0)
    not_simple = 0;
  __syncthreads();
  for (int i = tid; i < a.G * a.D; i += nt) {
    const int from = a.r2o[i];
    from_rank[i] = min(max(from < 0 ? from + a.G : from, 0), a.G - 1);   // (checked on the host)
  }
  for (int i = tid; i < n; i += nt) {
    const T v = static_cast<const T *>(a.history)[i];
    const float w = (float)v;
    weight[i] = w;
    load_of[i] = (double)v;
    key[i] = heaviest_first(w);
    replica[i] = -1;
    if (!(w >= 0.0f))
      not_simple = 1;
  }
  __syncthreads();
  if (room > 1) {
    // ---- each node's experts, heaviest first, equal ones in index order: four threads count what is ahead of an expert ----
    for (int i = tid / 4; i < n; i += nt / 4) {
      const int first = (int)fast_div((uint32_t)i, a.magic_per_node) * per_node;
      const uint32_t mine = key[i];
      int ahead = 0;
#pragma unroll 4
      for (int j = first + tid % 4; j < first + per_node; j += 4) {
        const uint32_t other = key[j];
        ahead += other < mine || (other == mine && j < i);
      }
      ahead += __builtin_amdgcn_update_dpp(0, ahead, 0xB1, 0xF, 0xF, true);
      ahead += __builtin_amdgcn_update_dpp(0, ahead, 0x4E, 0xF, 0xF, true);
      if (tid % 4 == 0)
        order[first + ahead] = i;
    }
    __syncthreads();
    // ---- packing, one wave per node ----
    for (int node = wave_s; node < a.n_nodes; node += nt / kWave) {
      const int first = node * per_node;
      if (not_simple)
        pack_node_of<false>(order + first, weight, per_node, a.packs, room, packed + first, lane);
      else
        pack_node_of<true>(order + first, weight, per_node, a.packs, room, packed + first, lane);
    }
  } else {
    for (int i = tid; i < n; i += nt)
      packed[i] = i;
  }
  __syncthreads();
  // ---- each rank's experts, heaviest first, equal ones in the order they were packed ----
  for (int i = tid; i < n; i += nt) {
    const int first = (int)fast_div((uint32_t)i, a.magic_L) * room, item = packed[i];
    const double mine = load_of[item];
    int ahead = 0;
#pragma unroll 4
    for (int k = first; k < first + room; ++k) {
      const double other = load_of[packed[k]];
      ahead += heavier(other, mine) || (k < i && !heavier(mine, other));
    }
    sorted[first + ahead] = item;
  }
  __syncthreads();
  // ---- physical experts: a rank's originals, then the replicas of its neighbours' first ones ----
  for (int phy = tid; phy < a.ep_size * a.P; phy += nt) {
    const int rank = (int)fast_div((uint32_t)phy, a.magic_P), place = phy - rank * a.P;
    int e;
    if (place < a.L) {
      e = sorted[rank * a.L + place];
      a.log2phy[2 * e] = phy;
    } else {
      const int slot = place - a.L, d = slot - (int)fast_div((uint32_t)slot, a.magic_D) * a.D;
      const int group = (int)fast_div((uint32_t)rank, a.magic_G) * a.G;
      e = sorted[(group + from_rank[(rank - group) * a.D + d]) * a.L + slot];
      replica[e] = phy;
    }
    a.phy2log[phy] = e;
  }
  __syncthreads();
  for (int e = tid; e < n; e += nt) {
    a.log2phy[2 * e + 1] = replica[e];
    a.logcnt[e] = replica[e] < 0 ? 1 : 2;
  }
}

static bool is_a_deployment(int G, int D, int ep_size, int n_logical, int n_physical, int n_nodes) {
  if (G <= 0 || D <= 0 || ep_size <= 0 || n_nodes <= 0 || n_logical <= 0 || ep_size % G != 0 || n_logical % ep_size != 0)
    return false;
  const int L = n_logical / ep_size, P = n_physical / ep_size, C = (P - L) / D;
  return P > L && C > 0 && C * D <= L && (int64_t)ep_size * (L + C * D) == n_physical;
}
// Groups go onto nodes only where every node takes one, so that no group has to be weighed; else all ranks are one node.
static int packed_nodes(int G, int ep_size, int n_nodes) { return ep_size / G % n_nodes == 0 ? n_nodes : 1; }
static bool is_placed_here(int G, int D, int ep_size, int n_logical, int n_physical, int n_nodes) {
  const int n_group = ep_size / G, nodes = packed_nodes(G, ep_size, n_nodes);
  return (nodes == 1 ? n_group % n_nodes != 0 || n_group == 1 : n_group == nodes) && ep_size % nodes == 0 &&
         n_logical <= kPlaceMaxExperts && (n_logical / nodes <= kPlaceMaxPerNode || n_logical == ep_size) &&
         ep_size / nodes <= kPlaceMaxPacks && G * D <= kPlaceMaxEdges && n_physical < 65536;
}

} // namespace lplb

extern "C" int lplb_place_experts_covers(int group_size, int dup_per_rank, int ep_size, int n_logical, int n_physical,
                                         int n_nodes) {
  using namespace lplb;
  return is_a_deployment(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes) &&
         is_placed_here(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes);
}

extern "C" int lplb_place_experts(const void *history, int history_type, const int32_t *r2o, int group_size,
                                  int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes,
                                  int32_t *phy2log, int32_t *log2phy, int32_t *logcnt, lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(history && r2o && phy2log && log2phy && logcnt, LPLB_EINVAL, "place_experts: null pointer");
  LPLB_REQUIRE(is_a_deployment(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes), LPLB_EINVAL,
               "place_experts: %d logical and %d physical experts on %d ranks in groups of %d with %d slots for replicas",
               n_logical, n_physical, ep_size, group_size, dup_per_rank);
  LPLB_REQUIRE(is_placed_here(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes), LPLB_EUNSUPPORTED,
               "place_experts: %d groups on %d nodes, %d experts on %d ranks are placed on the host only",
               ep_size / group_size, n_nodes, n_logical, ep_size);
  const int G = group_size, D = dup_per_rank, L = n_logical / ep_size, P = n_physical / ep_size;
  const int nodes = packed_nodes(G, ep_size, n_nodes);
  const auto magic = [](int d) { return fast_div_magic((uint32_t)d); };
  const PlaceArgs a{history, r2o, phy2log, log2phy, logcnt, G, D, L, P, ep_size, n_logical, n_logical / nodes, nodes, ep_size / nodes,
                    magic(G), magic(D), magic(L), magic(P), magic(n_logical / nodes)};
  const dim3 block(kPlaceMaxExperts);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  switch (history_type) {
  case LPLB_INT32: launch(place_experts<int32_t>, dim3(1), block, 0, s, a); break;
  case LPLB_INT64: launch(place_experts<int64_t>, dim3(1), block, 0, s, a); break;
  case LPLB_FLOAT32: launch(place_experts<float>, dim3(1), block, 0, s, a); break;
  case LPLB_FLOAT64: launch(place_experts<double>, dim3(1), block, 0, s, a); break;
  default: return fail(LPLB_EINVAL, "place_experts: unknown history_type %d", history_type);
  }
  LPLB_HIP_TRY(hipGetLastError());
  LPLB_HIP_TRY(hipStreamSynchronize(s));
  return LPLB_OK;
}
