// The planner's layout of physical experts from a load history that is on the GPU, as one workgroup
// (lplb_place_experts).  Same result as lplb_build_mapping on the host (mapping.cpp), bit for bit: experts are spread over the
// ranks by greedy packing, heaviest first, each into the lightest pack with room (lplb/eplb.py:6-46), each rank's experts
// are sorted heaviest first and the first of them get the replicas (lplb/planner.py:127-182).
//
// On the host the arithmetic takes 11 us, but the history has to come over (a copy the host waits for) and the tables have to go
// back (another).  Here nothing crosses: one launch, and the host waits once, because the tables are there for every stream
// when the call returns.  update_redundancy_mapping of 256 experts on 32 ranks of 4 nodes, history on the GPU: 46.1 us by the host,
// 20.9 here, of which the kernel is 5.3 (8.7 with the lightest pack searched for in every step) and an empty kernel's launch and wait 11.1; 24.2
// where the caller made the tables' views behind the wait instead of ahead of it.  What bounds it is
// the packing, a serial chain of one step per expert of a node, 30 ns each (pack_node); the nodes are packed side by side, a wave
// each.  With 256 experts on one node the kernel takes 13.2 us: 7.7 of packing, 2 of ranking every item by counting those ahead of it.
#include "map_kernel.h"

namespace lplb {

// lplb_place_experts has always refused more than this; lplb_place_on_large_nodes does not.
constexpr int kPlaceMaxPerNode = 128;
// The ranking's work is the square of a node's experts, and the host's arithmetic is a small part of a call there.  Per call, host /
// here (views behind the wait), into 8 packs: 256 experts of a node 45.5 / 32.4 us, 384 47.7 / 39.3, 512 49.7 / 47.3, 640 51.9 / 55.9; into 32 packs 256 46.6 / 35.3,
// 512 50.5 / 52.7.  (What the caller waits for, one call and a synchronisation: 8 packs, 256 54.1 / 35.4, 512 58.4 / 50.0.)  With weights that
// are negative or not numbers, which loads are not, a step takes longer: 384 of a node, views ahead of the wait, 48.4 / 51.3, waited for 57.5 / 54.0;
// without, 48.8 / 35.6 and 57.4 / 38.2.
constexpr int kPlaceMaxPerLargeNode = 384;
constexpr int kPlaceMaxExperts = 1024, kPlaceMaxPacks = 64, kPlaceMaxEdges = 2 * kWave;
// Where a node's experts are laid side by side in fours (a node has two at least where there is something to pack), and four more.
__host__ __device__ constexpr int padded_to_four(int n) { return (n + 3) / 4 * 4; }
constexpr int kPlaceMaxNodeWords = kPlaceMaxExperts / 2 * padded_to_four(2) + 4;

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
  uint32_t magic_G, magic_D, magic_L, magic_per_node;   // fast_div_magic
};

// One node's experts, heaviest first, into its packs, each into the lightest pack with room.  The packs lie sorted over the lanes,
// lightest first and by number among equals, so that a step is: lane 0's load with the next weight, and every lane takes what the
// insertion of that leaves at its place, which is its own key, the next lane's or the new one: max(mine, min(next lane's, new)).
// A key is the load, as bits in the order of numbers, above the pack's number and what is in it (so that a key gets greater also by a
// weight of zero); a pack without room goes to the end.  No search, no ballot and, up to 16 packs, nothing wave-uniform in the
// chain: 30 ns a step, 68 with the least load searched for by DPP and a ballot among packs that stay where they are.
// SIMPLE: no weight is negative or not a number.  Loads are their own bits then and only grow, and a key is a double whose order as a
// number is that of its bits (one instruction a comparison).  ROW: at most 16 packs.
// packed[pack * room + place] = expert; order, weight: the node's experts and their weights, heaviest first; places: room for n and up to
// three more, 16-byte aligned as weight is.
typedef float f32x4_in_lds __attribute__((ext_vector_type(4)));
typedef uint32_t pack_key __attribute__((ext_vector_type(2)));   // number and fill, load
constexpr int kLanesInRow = 16;
constexpr uint32_t kFullPack[2] = {0xffffffffu, 0x7fe00000u};   // by SIMPLE; above every load's
template <bool SIMPLE> __device__ inline uint32_t load_bits(float v) {
  return SIMPLE ? __builtin_bit_cast(uint32_t, v) : v != v ? 0u : ascending(v);   // (a load that is not a number is taken first)
}
template <bool SIMPLE> __device__ inline float load_of_bits(uint32_t b) {
  return __builtin_bit_cast(float, SIMPLE ? b : b >> 31 ? b ^ 0x80000000u : ~b);
}
template <bool ROW, bool SIMPLE>
__device__ inline void pack_node(const int32_t *order, const float *weight, int32_t *places, int n, int packs, int room, int32_t *packed,
                                 int lane) {
  constexpr uint32_t kFull = kFullPack[SIMPLE];
  constexpr int kNextLane = ROW ? 0x101 /* row_shl:1 */ : 0x130 /* wave_shl:1 */;
  if (!ROW || lane < kLanesInRow) {
    pack_key key{(uint32_t)lane << 16, lane < packs ? load_bits<SIMPLE>(0.0f) : kFull};
    pack_key next{0xffffffffu, kFull};   // of the next lane; the last has none, where this stays
    f32x4_in_lds w = *reinterpret_cast<const f32x4_in_lds *>(weight);
    for (int s = 0; s < n; s += 4) {
      const f32x4_in_lds next_w = *reinterpret_cast<const f32x4_in_lds *>(weight + s + 4);   // (past the last: not used)
      i32x4 at;
#pragma unroll
      for (int k = 0; k < 4; ++k) {   // (steps past the last find every pack full and leave that so)
        pack_key first;
        if constexpr (ROW) {
          first.x = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key.x, 0x150 /* row_newbcast:0 */, 0xF, 0xF, true);
          first.y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key.y, 0x150, 0xF, 0xF, true);
        } else {
          first.x = (uint32_t)__builtin_amdgcn_readfirstlane((int)key.x);
          first.y = (uint32_t)__builtin_amdgcn_readfirstlane((int)key.y);
        }
        next.x = (uint32_t)__builtin_amdgcn_update_dpp((int)next.x, (int)key.x, kNextLane, 0xF, 0xF, false);
        next.y = (uint32_t)__builtin_amdgcn_update_dpp((int)next.y, (int)key.y, kNextLane, 0xF, 0xF, false);
        const float sum = load_of_bits<SIMPLE>(first.y) + w[k];
        pack_key mine{first.x + 1, load_bits<SIMPLE>(sum)};
        mine.y = (mine.x & 0xffffu) == (uint32_t)room ? kFull : mine.y;
        at[k] = (int)mine.x;
        if constexpr (SIMPLE) {
          // (written out: the compiler makes a NaN quiet first, which is none here; two wait states before a DPP operand)
          double lesser;
          asm("v_min_f64 %1, %2, %3\n\tv_max_f64 %0, %0, %1\n\ts_nop 1"
              : "+v"(key), "=&v"(lesser) : "v"(next), "v"(mine));
        } else {
          const uint64_t n64 = __builtin_bit_cast(uint64_t, next), m64 = __builtin_bit_cast(uint64_t, mine);
          const uint64_t own = lane == 0 ? 0 : __builtin_bit_cast(uint64_t, key);   // (a load may get less)
          key = __builtin_bit_cast(pack_key, max(own, min(n64, m64)));
        }
      }
      *reinterpret_cast<i32x4 *>(places + s) = at;   // (the same from every lane)
      w = next_w;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int s = lane; s < n; s += kWave) {
    const int at = places[s];
    packed[(at >> 16) * room + (at & 0xffff) - 1] = order[s];
  }
}

template <typename T> __global__ __launch_bounds__(kPlaceMaxExperts) void place_experts(PlaceArgs a) {
  __shared__ uint64_t key[kPlaceMaxExperts];   // in the order of packing: weight, then index
  __shared__ float weight[kPlaceMaxExperts];
  __shared__ double load_of[kPlaceMaxExperts];
  __shared__ int32_t order[kPlaceMaxExperts], packed[kPlaceMaxExperts], resorted[kPlaceMaxExperts];
  __shared__ __attribute__((aligned(16))) float node_weight[kPlaceMaxNodeWords];   // by node (padded), heaviest first
  __shared__ __attribute__((aligned(16))) int32_t node_places[kPlaceMaxNodeWords];
  __shared__ int32_t host_of[kPlaceMaxEdges];   // by rank and slot of a group: the rank that hosts the copy
  __shared__ int not_simple, out_of_order, repeated;
  fetch_arguments_now(a.history, a.n_logical, a.magic_per_node);
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n = a.n_logical, per_node = a.per_node, padded = padded_to_four(per_node), room = a.L;
  if (tid == 0)
    not_simple = out_of_order = repeated = 0;
  __syncthreads();
  auto source_of = [&](int i) {   // by rank and slot of a group: the rank whose expert is copied there
    const int from = a.r2o[i];
    return min(max(from < 0 ? from + a.G : from, 0), a.G - 1);
  };
  static_assert(kPlaceMaxEdges <= kPlaceMaxExperts, "an edge per thread");
  const int edge = nt - 1 - tid, my_host = (int)fast_div((uint32_t)edge, a.magic_D);   // (the last waves', which seldom have a node to pack)
  const int my_edge = edge < a.G * a.D ? source_of(edge) * a.D + edge - my_host * a.D : -1;
  if (my_edge >= 0)
    host_of[my_edge] = my_host;
  for (int i = tid; i < n; i += nt) {
    const T v = static_cast<const T *>(a.history)[i];
    const float w = (float)v;
    weight[i] = w;
    load_of[i] = (double)v;
    key[i] = (uint64_t)heaviest_first(w) << 32 | (uint32_t)i;
    if (!(w >= 0.0f))
      not_simple = 1;
  }
  __syncthreads();
  if (room > 1) {
    // ---- each node's experts, heaviest first, equal ones in index order: four threads count what is ahead of an expert (a comparison
    //      of 64 bits and an addition each) ----
    for (int i = tid / 4; i < n; i += nt / 4) {
      const int node = (int)fast_div((uint32_t)i, a.magic_per_node), first = node * per_node;
      const uint64_t mine = key[i];
      int ahead = 0;
#pragma unroll 8
      for (int j = tid % 4; j < per_node; j += 4)
        ahead += key[first + j] < mine;
      ahead += __builtin_amdgcn_update_dpp(0, ahead, 0xB1, 0xF, 0xF, true);
      ahead += __builtin_amdgcn_update_dpp(0, ahead, 0x4E, 0xF, 0xF, true);
      if (tid % 4 == 0) {
        order[first + ahead] = i;
        node_weight[node * padded + ahead] = weight[i];
      }
    }
    __syncthreads();
    // ---- packing, one wave per node ----
    for (int node = wave_s; node < a.n_nodes; node += nt / kWave) {
      auto pack = [&](auto in_row, auto simple) {
        pack_node<decltype(in_row)::value, decltype(simple)::value>(order + node * per_node, node_weight + node * padded, node_places + node * padded,
                                                                    per_node, a.packs, room, packed + node * per_node, lane);
      };
      if (a.packs <= kLanesInRow)
        not_simple ? pack(std::true_type{}, std::false_type{}) : pack(std::true_type{}, std::true_type{});
      else
        not_simple ? pack(std::false_type{}, std::false_type{}) : pack(std::false_type{}, std::true_type{});
    }
  } else {
    for (int i = tid; i < n; i += nt)
      packed[i] = i;
  }
  // (where a column repeats a rank, that rank's entry has another host for all of its hosts but one; entries of ranks left out were never written)
  if (my_edge >= 0 && host_of[my_edge] != my_host)
    repeated = 1;
  __syncthreads();
  // ---- each rank's experts, heaviest first, equal ones in the order they were packed.  They were packed heaviest first: what is
  //      out of order is what only the packing, which rounds loads to 32 bits, took for equal ----
  const int32_t *sorted = packed;
  if (room > 1) {
    for (int i = tid; i < n - 1; i += nt)
      if ((int)fast_div((uint32_t)i + 1, a.magic_L) * room != i + 1 && heavier(load_of[packed[i + 1]], load_of[packed[i]]))
        out_of_order = 1;
    __syncthreads();
    if (out_of_order) {
      for (int i = tid; i < n; i += nt) {
        const int first = (int)fast_div((uint32_t)i, a.magic_L) * room, item = packed[i];
        const double mine = load_of[item];
        int ahead = 0;
#pragma unroll 4
        for (int k = first; k < first + room; ++k) {
          const double other = load_of[packed[k]];
          ahead += heavier(other, mine) || (k < i && !heavier(mine, other));
        }
        resorted[first + ahead] = item;
      }
      __syncthreads();
      sorted = resorted;
    }
  }
  // ---- physical experts: a rank's originals; of its first ones a copy on the rank that hosts the slot.  The values of r2o are the caller's:
  //      with a rank repeated in a column its hosts are looked for one by one (none, or several, of which log2phy has the last), as host_of
  //      says nothing about the ranks left out ----
  for (int i = tid; i < n; i += nt) {
    const int rank = (int)fast_div((uint32_t)i, a.magic_L), place = i - rank * a.L, e = sorted[i], phy = rank * a.P + place;
    int replica = -1;
    if (place < a.P - a.L) {
      const int d = place - (int)fast_div((uint32_t)place, a.magic_D) * a.D;
      const int group = (int)fast_div((uint32_t)rank, a.magic_G) * a.G;
      if (!repeated) {
        replica = (group + host_of[(rank - group) * a.D + d]) * a.P + a.L + place;
        a.phy2log[replica] = e;
      } else {
        for (int host = 0; host < a.G; ++host)
          if (source_of(host * a.D + d) == rank - group) {
            replica = (group + host) * a.P + a.L + place;
            a.phy2log[replica] = e;
          }
      }
    }
    a.phy2log[phy] = e;
    a.log2phy[2 * e] = phy;
    a.log2phy[2 * e + 1] = replica;
    a.logcnt[e] = replica < 0 ? 1 : 2;
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
static bool is_placed_here(int G, int D, int ep_size, int n_logical, int n_physical, int n_nodes, int most_per_node) {
  const int n_group = ep_size / G, nodes = packed_nodes(G, ep_size, n_nodes);
  return (nodes == 1 ? n_group % n_nodes != 0 || n_group == 1 : n_group == nodes) && ep_size % nodes == 0 &&
         n_logical <= kPlaceMaxExperts && (n_logical / nodes <= most_per_node || n_logical == ep_size) &&
         ep_size / nodes <= kPlaceMaxPacks && G * D <= kPlaceMaxEdges && n_physical < 65536;
}

static bool covers(int G, int D, int ep_size, int n_logical, int n_physical, int n_nodes, int most_per_node) {
  return is_a_deployment(G, D, ep_size, n_logical, n_physical, n_nodes) &&
         is_placed_here(G, D, ep_size, n_logical, n_physical, n_nodes, most_per_node);
}

static int place(const void *history, int history_type, const int32_t *r2o, int G, int D, int ep_size, int n_logical, int n_physical,
                 int n_nodes, int most_per_node, int32_t *phy2log, int32_t *log2phy, int32_t *logcnt, hipStream_t s) {
  LPLB_REQUIRE(history && r2o && phy2log && log2phy && logcnt, LPLB_EINVAL, "place_experts: null pointer");
  LPLB_REQUIRE(is_a_deployment(G, D, ep_size, n_logical, n_physical, n_nodes), LPLB_EINVAL,
               "place_experts: %d logical and %d physical experts on %d ranks in groups of %d with %d slots for replicas",
               n_logical, n_physical, ep_size, G, D);
  LPLB_REQUIRE(is_placed_here(G, D, ep_size, n_logical, n_physical, n_nodes, most_per_node), LPLB_EUNSUPPORTED,
               "place_experts: %d groups on %d nodes, %d experts on %d ranks are placed on the host only",
               ep_size / G, n_nodes, n_logical, ep_size);
  const int L = n_logical / ep_size, P = n_physical / ep_size, nodes = packed_nodes(G, ep_size, n_nodes);
  const auto magic = [](int d) { return fast_div_magic((uint32_t)d); };
  const PlaceArgs a{history, r2o, phy2log, log2phy, logcnt, G, D, L, P, ep_size, n_logical, n_logical / nodes, nodes, ep_size / nodes,
                    magic(G), magic(D), magic(L), magic(n_logical / nodes)};
  const dim3 block(kPlaceMaxExperts);
  switch (history_type) {
  case LPLB_INT32: launch(place_experts<int32_t>, dim3(1), block, 0, s, a); break;
  case LPLB_INT64: launch(place_experts<int64_t>, dim3(1), block, 0, s, a); break;
  case LPLB_FLOAT32: launch(place_experts<float>, dim3(1), block, 0, s, a); break;
  case LPLB_FLOAT64: launch(place_experts<double>, dim3(1), block, 0, s, a); break;
  default: return fail(LPLB_EINVAL, "place_experts: unknown history_type %d", history_type);
  }
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}
static int wait_for(hipStream_t s) {
  LPLB_HIP_TRY(hipStreamSynchronize(s));
  return LPLB_OK;
}

} // namespace lplb

extern "C" int lplb_place_experts_covers(int group_size, int dup_per_rank, int ep_size, int n_logical, int n_physical,
                                         int n_nodes) {
  return lplb::covers(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, lplb::kPlaceMaxPerNode);
}
extern "C" int lplb_place_on_large_nodes_covers(int group_size, int dup_per_rank, int ep_size, int n_logical, int n_physical,
                                                int n_nodes) {
  return lplb::covers(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, lplb::kPlaceMaxPerLargeNode);
}

extern "C" int lplb_place_experts(const void *history, int history_type, const int32_t *r2o, int group_size,
                                  int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes,
                                  int32_t *phy2log, int32_t *log2phy, int32_t *logcnt, lplb_stream_t stream) {
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = lplb::place(history, history_type, r2o, group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, lplb::kPlaceMaxPerNode,
                             phy2log, log2phy, logcnt, s);
  return rc == LPLB_OK ? lplb::wait_for(s) : rc;
}
extern "C" int lplb_place_on_large_nodes(const void *history, int history_type, const int32_t *r2o, int group_size,
                                         int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes,
                                         int32_t *phy2log, int32_t *log2phy, int32_t *logcnt, lplb_stream_t stream) {
  const int rc = lplb_place_on_large_nodes_begin(history, history_type, r2o, group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes,
                                                 phy2log, log2phy, logcnt, stream);
  return rc == LPLB_OK ? lplb_place_wait(stream) : rc;
}
extern "C" int lplb_place_on_large_nodes_begin(const void *history, int history_type, const int32_t *r2o, int group_size,
                                               int dup_per_rank, int ep_size, int n_logical, int n_physical, int n_nodes,
                                               int32_t *phy2log, int32_t *log2phy, int32_t *logcnt, lplb_stream_t stream) {
  return lplb::place(history, history_type, r2o, group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, lplb::kPlaceMaxPerLargeNode,
                     phy2log, log2phy, logcnt, static_cast<hipStream_t>(stream));
}
extern "C" int lplb_place_wait(lplb_stream_t stream) { return lplb::wait_for(static_cast<hipStream_t>(stream)); }
