// libnpc.so: the `npc` operator library for PyTorch-ROCm.
//
// Registers the hot-path operators under the names and C++ signatures the
// reference binds with TORCH_LIBRARY(npc, m) in src/pybind.cc:18-48, so that
// torch.ops.npc.<name>(...) keeps working.  Every operator is a thin host
// wrapper: it checks its tensors, allocates outputs with torch, and calls the
// C ABI of libapt_hip.so (include/apt_amd.h) on the current HIP stream.
// Operators whose reference implementation exchanges data with other GPUs
// over NCCL are registered too, and raise.
#include <ATen/hip/HIPEvent.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>
#include <torch/torch.h>

#include <array>
#include <deque>
#include <memory>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/apt_amd.h"

namespace npc {

using torch::Tensor;
using IdType = int64_t;  // reference src/utils.h:14

namespace {

struct State {  // counterpart of NPCState, reference src/state.h:32-63
  int64_t rank = 0, local_rank = 0, world_size = 1, node_size = 1;
  // graph (reference GraphStorage, state.h:18-23)
  bool has_graph = false;
  Tensor indptr, indices, cached_indptr, cached_indices, adj_pos_map;
  apt_graph graph{};
  // features (reference FeatStorage, state.h:10-16)
  bool has_feat = false;
  Tensor local_feats, cache_feats, feat_pos_map, cpu_feat_pos_map;
  bool identity_map = false;
  apt_feat_store feat{};
  // bucketing
  Tensor shuffle_min_vids, remote_worker_map;
  int64_t shuffle_id_offset = 0, num_remote_workers = 0;
  // sampling
  uint64_t rng_seed = 7777777;  // reference src/cuda/npc_kernel.cu:292
  int64_t sample_calls = 0;
  // How load_subtensor reports requested nodes that have no row here (the reference reads out of bounds):
  //   0 not at all (rows are zero-filled), 1 deferred (default): the miss counter travels to pinned host memory
  //   behind the gather and is looked at by the next operator call or by check_errors(), so no call waits for
  //   the GPU; 2 immediate: the call waits for its own counter and raises itself.
  int miss_check = 1;
  bool strict = true;   // feat_shuffle's pack checks permutations it did not produce itself
  struct PendingCheck {
    Tensor dev, host;
    std::shared_ptr<at::cuda::CUDAEvent> done;
  };
  std::deque<PendingCheck> pending_checks;
  // permutations handed out by shuffle_seeds / cluster_and_permute (kept alive, with their versions): bijections
  // by construction, which feat_shuffle's pack need not check
  std::deque<std::pair<Tensor, uint32_t>> own_permutations;
  // relabel_csc on a registered graph: a rank table of its own, a workspace that grows with the largest call, and
  // the unique list the last call returned (kept alive so that its address cannot be reused) with its version
  Tensor ranked_table, ranked_ws, ranked_counts, ranked_last;
  uint32_t ranked_last_version = 0;
  bool ranked_enabled = true;
  // A sampling operator call that has placed the bids of the relabel_csc call the reference's sampler makes
  // next (apt_sample_neighbors_bidding): its seeds and sampled ids (kept alive, with their versions) and the slot
  // states that call will take over.  A relabel_csc with other tensors finds abandoned bids in the table and
  // starts a fresh batch.
  struct RankedPending {
    bool valid = false, continued = false;
    Tensor seeds, neighbors, states;
    uint32_t seeds_version = 0, neighbors_version = 0;
  } ranked_pending;
  // pinned host words that the relabel operators read their counts into (a copy to pageable memory is staged)
  Tensor pinned_counts;
  // fused multi-hop driver: rank table of the registered graph, workspace of the last plan
  Tensor rank_table, mb_workspace;
  int64_t mb_batch = -1;
  std::vector<int64_t> mb_fanouts;
  // sample_blocks' output buffers (upper-bound sized).  Ring 0 (the default) = fresh tensors on every call,
  // as the reference's operators return them; set_block_buffer_ring(n) hands out n registry-owned sets in
  // turn instead: what call k returned is then overwritten by call k + n
  struct BlockBuffers {
    Tensor nodes, sizes, format_ws;
    std::vector<Tensor> nb, rl, ct, row, col, csc;
    bool formats = false;
  };
  std::vector<BlockBuffers> mb_ring;
  int64_t mb_ring_size = 0, mb_ring_pos = 0;
};

State& S() {
  // the C library found at run time must be the one this file's header describes
  static const bool abi_ok = [] {
    TORCH_CHECK(apt_abi_version() == APT_ABI_VERSION, "npc: libapt_hip.so has ABI version ", apt_abi_version(),
                ", libnpc.so was built against ", APT_ABI_VERSION);
    return true;
  }();
  (void)abi_ok;
  static State s;
  return s;
}

void check(int status) {
  TORCH_CHECK(status == APT_OK, "npc: ", apt_last_error(), " (status ", status, ")");
}

void* stream() { return static_cast<void*>(c10::hip::getCurrentHIPStream().stream()); }

c10::Device device() {
  TORCH_CHECK(torch::cuda::is_available(), "npc: no GPU; the operators have no CPU implementation");
  return c10::Device(c10::kCUDA, c10::hip::current_device());
}

Tensor ids_on_device(const Tensor& t, const char* name) {
  TORCH_CHECK(t.scalar_type() == torch::kInt64, "npc: ", name, " must be int64");
  TORCH_CHECK(t.dim() == 1, "npc: ", name, " must be 1-D");
  return t.to(device()).contiguous();
}

const int64_t* i64(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr<int64_t>() : nullptr; }

torch::TensorOptions i64_opts() { return torch::TensorOptions().dtype(torch::kInt64).device(device()); }

int64_t* pinned_counts() {
  auto& s = S();
  if (!s.pinned_counts.defined())
    s.pinned_counts = torch::zeros({4}, torch::TensorOptions().dtype(torch::kInt64).pinned_memory(true));
  return s.pinned_counts.data_ptr<int64_t>();
}

// A few device counts on the host, through pinned memory of the calling thread (operators of a backward pass run on
// autograd's threads).  Waits for the current stream.
const int64_t* read_counts(const Tensor& dev) {
  static thread_local Tensor host;
  if (!host.defined()) host = torch::zeros({8}, torch::TensorOptions().dtype(torch::kInt64).pinned_memory(true));
  host.narrow(0, 0, dev.numel()).copy_(dev, /*non_blocking=*/true);
  c10::hip::getCurrentHIPStream().synchronize();
  return host.data_ptr<int64_t>();
}

}  // namespace

// ---------------------------------------------------------------- registries
void SetTopology(IdType rank, IdType world_size, IdType node_size) {
  TORCH_CHECK(world_size >= 1 && world_size <= APT_MAX_BUCKETS && rank >= 0 && rank < world_size &&
                  node_size >= 1,
              "npc: bad topology");
  S().rank = rank;
  S().world_size = world_size;
  S().node_size = node_size;
  S().local_rank = rank % node_size;
}

void SetRngSeed(IdType seed) {
  S().rng_seed = static_cast<uint64_t>(seed);
  S().sample_calls = 0;
}

// Looks at the miss counters of earlier load_subtensor calls that have arrived (wait: all of them) and raises for
// the first that is not zero.
void PollChecks(bool wait) {
  auto& q = S().pending_checks;
  while (!q.empty()) {
    auto& p = q.front();
    if (wait) p.done->synchronize();
    else if (!p.done->query()) break;
    const int64_t m = p.host.data_ptr<int64_t>()[0];
    q.pop_front();
    TORCH_CHECK_INDEX(m == 0, "npc: load_subtensor (an earlier call): ", m,
                      " requested node(s) have no feature row on this GPU; their rows were zero-filled");
  }
}

void CheckErrors() { PollChecks(true); }

void SetStrict(bool strict) {
  S().strict = strict;
  S().miss_check = strict ? 1 : 0;
}

void SetMissCheck(std::string mode) {
  TORCH_CHECK(mode == "off" || mode == "deferred" || mode == "immediate",
              "npc: set_miss_check: 'off', 'deferred' or 'immediate'");
  PollChecks(true);
  S().miss_check = mode == "off" ? 0 : mode == "deferred" ? 1 : 2;
}

// relabel_csc goes through the registered graph's rank table where it can (default) or always through the
// hash table (false).
static void drop_pending_bids();
void SetRankedRelabel(bool enabled) {
  S().ranked_enabled = enabled;
  S().ranked_last = Tensor();
  drop_pending_bids();
}

// How many registry-owned sets of output buffers sample_blocks hands out in turn.  0 (the default) = fresh
// tensors on every call.  With n > 0 a call costs less (no allocation), but what call k returned is
// overwritten by call k + n whatever stream or consumer still holds it.
IdType BlockBufferRing() { return S().mb_ring_size; }

void SetBlockBufferRing(IdType sets) {
  TORCH_CHECK(sets >= 0 && sets <= 64, "npc: set_block_buffer_ring: 0..64 sets");
  S().mb_ring_size = sets;
  S().mb_ring.clear();
  S().mb_ring_pos = 0;
}

// reference src/cache_feats.cc:14-61
void CacheFeatsShared(IdType num_total_nodes, Tensor localnode_feats, Tensor cached_feats,
                      Tensor cached_idx, Tensor localnode_idx, IdType feat_dim_offset) {
  auto& s = S();
  TORCH_CHECK(localnode_feats.dim() == 2, "npc: localnode_feats must be [num_local, feat_dim]");
  TORCH_CHECK(localnode_feats.element_size() == 2 || localnode_feats.element_size() == 4,
              "npc: features must have 2- or 4-byte elements");
  const int64_t n_local = localnode_feats.size(0), feat_dim = localnode_feats.size(1);
  const int64_t n_cached = cached_feats.dim() == 2 ? cached_feats.size(0) : 0;
  auto local_idx = ids_on_device(localnode_idx, "localnode_idx");
  auto cache_idx = ids_on_device(cached_idx, "cached_idx");
  TORCH_CHECK(local_idx.numel() == n_local, "npc: localnode_idx must name every local row");
  TORCH_CHECK(cache_idx.numel() == n_cached, "npc: cached_idx must name every cached row");
  if (n_local)
    TORCH_CHECK(local_idx.min().item<int64_t>() >= 0 && local_idx.max().item<int64_t>() < num_total_nodes,
                "npc: localnode_idx out of range");
  if (n_cached)
    TORCH_CHECK(cache_idx.min().item<int64_t>() >= 0 && cache_idx.max().item<int64_t>() < num_total_nodes,
                "npc: cached_idx out of range");
  const int64_t rank_dim = n_cached ? cached_feats.size(1) : feat_dim - feat_dim_offset;
  TORCH_CHECK(feat_dim_offset >= 0 && feat_dim_offset + rank_dim <= feat_dim,
              "npc: feat_dim_offset + cached width exceeds the local feature width");
  s.local_feats = localnode_feats.to(device()).contiguous();
  auto pos = torch::full({num_total_nodes}, -1, i64_opts());  // FEAT_NOT_EXIST, src/utils.h:20
  pos.index_put_({local_idx}, -torch::arange(n_local, i64_opts()) - 2);  // ENCODE_ID, src/utils.h:17
  s.cpu_feat_pos_map = pos.cpu();  // without cache entries, src/cache_feats.cc:52
  s.cache_feats = Tensor();
  if (n_cached) {
    TORCH_CHECK(cached_feats.scalar_type() == localnode_feats.scalar_type(),
                "npc: cached_feats dtype differs from localnode_feats");
    s.cache_feats = cached_feats.to(device()).contiguous();
    pos.index_put_({cache_idx}, torch::arange(n_cached, i64_opts()));  // the cache wins, :53-55
  }
  s.feat_pos_map = pos;
  s.identity_map = n_cached == 0 && n_local == num_total_nodes &&
                   torch::equal(local_idx, torch::arange(n_local, i64_opts()));
  s.feat.local_table = s.local_feats.data_ptr();
  s.feat.num_local_rows = n_local;
  s.feat.local_dim = feat_dim;
  s.feat.cache_table = n_cached ? s.cache_feats.data_ptr() : nullptr;
  s.feat.num_cache_rows = n_cached;
  s.feat.pos_map = s.identity_map ? nullptr : pos.data_ptr<int64_t>();
  s.feat.num_total_nodes = num_total_nodes;
  s.feat.col_offset = feat_dim_offset;
  s.feat.out_dim = rank_dim;
  s.feat.elem_size = static_cast<int>(localnode_feats.element_size());
  s.has_feat = true;
}

// reference src/cache_graphs.cc:12-49
void MixCacheGraphs(IdType num_cached_nodes, Tensor cached_node_idx, Tensor cached_indptr,
                    Tensor cached_indices, Tensor global_indptr, Tensor global_indices) {
  auto& s = S();
  TORCH_CHECK(num_cached_nodes == cached_node_idx.numel(),
              "npc: num_cached_nodes != cached_node_idx.numel()");  // reference CHECK :19
  s.indptr = ids_on_device(global_indptr, "global_indptr");
  s.indices = ids_on_device(global_indices, "global_indices");
  const int64_t total = s.indptr.numel() - 1;
  TORCH_CHECK(total >= 0, "npc: global_indptr is empty");
  s.graph = apt_graph{};
  s.graph.indptr = s.indptr.data_ptr<int64_t>();
  s.graph.indices = i64(s.indices);
  s.graph.row_begin = 0;
  s.graph.num_rows = total;
  s.graph.num_total_nodes = total;
  s.rank_table = Tensor();
  s.ranked_table = Tensor();
  s.ranked_ws = Tensor();
  s.ranked_last = Tensor();
  s.ranked_pending = {};
  s.adj_pos_map = Tensor();
  if (num_cached_nodes > 0) {
    auto idx = ids_on_device(cached_node_idx, "cached_node_idx");
    s.cached_indptr = ids_on_device(cached_indptr, "cached_indptr");
    s.cached_indices = ids_on_device(cached_indices, "cached_indices");
    TORCH_CHECK(s.cached_indptr.numel() == num_cached_nodes + 1,
                "npc: cached_indptr must have num_cached_nodes + 1 entries");
    TORCH_CHECK(idx.min().item<int64_t>() >= 0 && idx.max().item<int64_t>() < total,
                "npc: cached_node_idx out of range");
    s.adj_pos_map = -torch::arange(total, i64_opts()) - 2;  // ENCODE_ID(v), :37-40
    s.adj_pos_map.index_put_({idx}, torch::arange(num_cached_nodes, i64_opts()));
    s.graph.cached_indptr = s.cached_indptr.data_ptr<int64_t>();
    s.graph.cached_indices = i64(s.cached_indices);
    s.graph.num_cached_rows = num_cached_nodes;
    s.graph.adj_pos_map = s.adj_pos_map.data_ptr<int64_t>();
  }
  s.has_graph = true;
}

// A contiguous-range partition: nodes outside [row_begin, row_begin + rows)
// have no adjacency.  No counterpart in the reference.
void RegisterGraphPartition(Tensor indptr, Tensor indices, IdType row_begin, IdType num_total_nodes) {
  auto& s = S();
  s.indptr = ids_on_device(indptr, "indptr");
  s.indices = ids_on_device(indices, "indices");
  TORCH_CHECK(s.indptr.numel() >= 1, "npc: indptr is empty");
  s.adj_pos_map = Tensor();
  s.graph = apt_graph{};
  s.graph.indptr = s.indptr.data_ptr<int64_t>();
  s.graph.indices = i64(s.indices);
  s.graph.row_begin = row_begin;
  s.graph.num_rows = s.indptr.numel() - 1;
  s.graph.num_total_nodes = num_total_nodes;
  s.rank_table = Tensor();
  s.ranked_table = Tensor();
  s.ranked_ws = Tensor();
  s.ranked_last = Tensor();
  s.ranked_pending = {};
  s.has_graph = true;
}

// reference src/core.cc:102-108
void RegisterMinVids(Tensor shuffle_min_vids, IdType shuffle_id_offset) {
  S().shuffle_min_vids = ids_on_device(shuffle_min_vids, "shuffle_min_vids");
  S().shuffle_id_offset = shuffle_id_offset;
}

// reference src/core.cc:110-125 (state only)
void RegisterMultiMachinesScheme(Tensor remote_worker_map, Tensor remote_worker_id) {
  S().remote_worker_map = ids_on_device(remote_worker_map, "remote_worker_map");
  S().num_remote_workers = remote_worker_id.numel();
}

// ---------------------------------------------------------------- hot path
static bool same_tensor(const Tensor& kept, uint32_t version, const Tensor& t) {
  return kept.defined() && kept.data_ptr() == t.data_ptr() && kept.numel() == t.numel() && version == t._version();
}

// Forgets bids that a sampling call placed for a relabel_csc call that did not come.  Those of a call that
// continued a batch have also set per-slot flags in the workspace, which only that relabel_csc would have
// consumed: the workspace is cleared.  (The bids themselves are harmless: the next call on the table starts a new
// batch.)
static void drop_pending_bids() {
  auto& s = S();
  if (s.ranked_pending.valid && s.ranked_pending.continued && s.ranked_ws.defined())
    check(apt_minibatch_workspace_init(s.ranked_ws.data_ptr(), static_cast<size_t>(s.ranked_ws.numel()), stream()));
  if (s.ranked_pending.valid && s.ranked_counts.defined()) s.ranked_counts.zero_();   // seeds it counted as outside
  s.ranked_pending = {};
}

// The rank table of the registered graph for relabel_csc (a table of its own) and a workspace for `items` items.
static bool ranked_resources(int64_t items) {
  auto& s = S();
  auto u8 = torch::TensorOptions().dtype(torch::kUInt8).device(device());
  if (!s.ranked_table.defined()) {
    const size_t bytes = apt_rank_table_bytes(s.graph.num_total_nodes);
    if (bytes == 0) return false;
    s.ranked_table = torch::empty({static_cast<int64_t>(bytes)}, u8);
    check(apt_rank_table_init(s.ranked_table.data_ptr(), bytes, stream()));
    s.ranked_counts = torch::zeros({2}, i64_opts());
    s.ranked_last = Tensor();
    s.ranked_pending = {};
  }
  const size_t need = apt_relabel_ranked_workspace_bytes(items);
  if (need == 0) return false;
  if (!s.ranked_ws.defined() || static_cast<size_t>(s.ranked_ws.numel()) < need) {
    // (a new workspace starts with clean flags; bids placed under the old one are abandoned)
    s.ranked_ws = torch::empty({static_cast<int64_t>(std::max<size_t>(need, 256) * 2)}, u8);
    check(apt_minibatch_workspace_init(s.ranked_ws.data_ptr(), static_cast<size_t>(s.ranked_ws.numel()), stream()));
    s.ranked_last = Tensor();
    s.ranked_pending = {};
  }
  return true;
}

// One hop of sampling.  Where the relabel_csc call that the reference's sampler makes next
// (python/npc/sampler.py:187-203) will go through the rank table, its bids are placed here, by the sampling kernel
// itself, and that call only ranks the owners.
static void sample_hop(const Tensor& f, IdType fanout, bool replace, uint64_t rng_seed, int hop, Tensor& out,
                       int64_t* counts) {
  auto& s = S();
  const int64_t n = f.numel(), items = n + n * fanout;
  if (s.ranked_enabled && fanout <= 64 && items > 8192 && items <= apt_relabel_ranked_max_items() &&
      s.graph.num_total_nodes > 0 && ranked_resources(items)) {
    // the batch continues if these seeds are the unique list the last relabel_csc returned and nothing has bid since
    const bool continued = !s.ranked_pending.valid && same_tensor(s.ranked_last, s.ranked_last_version, f);
    s.ranked_last = Tensor();
    drop_pending_bids();
    auto states = torch::empty({n * fanout}, i64_opts());
    check(apt_sample_neighbors_bidding(&s.graph, i64(f), n, nullptr, static_cast<int>(fanout), replace, rng_seed, hop,
                                       out.data_ptr<int64_t>(), counts, nullptr, continued ? 1 : 0,
                                       s.ranked_table.data_ptr(), s.graph.num_total_nodes, states.data_ptr<int64_t>(),
                                       s.ranked_counts.data_ptr<int64_t>() + 1, s.ranked_ws.data_ptr(),
                                       static_cast<size_t>(s.ranked_ws.numel()), stream()));
    auto& p = s.ranked_pending;
    p.valid = true;
    p.continued = continued;
    p.seeds = f;
    p.neighbors = out;
    p.states = states;
    p.seeds_version = f._version();
    p.neighbors_version = out._version();
    return;
  }
  check(apt_sample_neighbors(&s.graph, i64(f), n, nullptr, static_cast<int>(fanout), replace, rng_seed, hop,
                             out.data_ptr<int64_t>(), counts, nullptr, stream()));
}

std::tuple<Tensor, Tensor> SampleNeighbors(Tensor seeds, IdType fanout, bool replace, IdType rng_seed,
                                           IdType hop) {
  auto& s = S();
  TORCH_CHECK(s.has_graph, "npc: no graph registered (mix_cache_graphs)");
  TORCH_CHECK(fanout > 0, "npc: fanout must be > 0");
  auto f = ids_on_device(seeds, "seeds");
  auto out = torch::empty({f.numel() * fanout}, i64_opts());
  auto cnt = torch::empty({f.numel()}, i64_opts());
  sample_hop(f, fanout, replace, static_cast<uint64_t>(rng_seed), static_cast<int>(hop), out, cnt.data_ptr<int64_t>());
  return {out, cnt};
}

// The whole multi-hop loop of MixedPSNeighborSampler.sample, DP branch (reference
// python/npc/sampler.py:187-203,358-364: sample -> relabel -> frontier = unique, per
// hop) as one operator: every kernel of the batch is enqueued by one C call, the
// sizes stay on the device, and the host waits once, to cut the outputs to size.
// hop_fanouts: from the seeds outward.  Returns
//   [sizes (CPU int64[H + 2]: frontier rows entering each hop, input nodes, edges),
//    input_nodes, then per hop h: neighbors_h, relabeled_h, counts_h]
// with neighbors / relabeled in the fixed-stride layout [rows_h * fanout_h], -1 = no edge.
// The rank table and workspace live in the registry and are reused: calls must be
// ordered on one stream.
// with_formats: each hop's block is also emitted as COO + CSC before that one wait;
// appended per hop: coo_row_h, coo_col_h, csc_indptr_h (sizes then carries the hops'
// edge counts after its H + 2 entries).
std::vector<Tensor> SampleBlocks(Tensor seeds, std::vector<int64_t> hop_fanouts, bool replace, IdType rng_seed,
                                 bool with_formats) {
  auto& s = S();
  TORCH_CHECK(s.has_graph, "npc: no graph registered (mix_cache_graphs)");
  const int H = static_cast<int>(hop_fanouts.size());
  TORCH_CHECK(H >= 1 && H <= APT_MAX_HOPS, "npc: sample_blocks: 1..", APT_MAX_HOPS, " hops");
  auto sd = ids_on_device(seeds, "seeds");
  const int64_t B = sd.numel();
  TORCH_CHECK(B > 0, "npc: sample_blocks: no seeds");
  std::vector<int> fan(H);
  for (int h = 0; h < H; ++h) {
    TORCH_CHECK(hop_fanouts[h] > 0 && hop_fanouts[h] <= (1 << 20), "npc: sample_blocks: bad fanout");
    fan[h] = static_cast<int>(hop_fanouts[h]);
  }
  auto u8 = torch::TensorOptions().dtype(torch::kUInt8).device(device());
  if (!s.rank_table.defined()) {
    const size_t bytes = apt_rank_table_bytes(s.graph.num_total_nodes);
    TORCH_CHECK(bytes > 0, "npc: sample_blocks: graph too large for the rank table");
    s.rank_table = torch::empty({static_cast<int64_t>(bytes)}, u8);
    check(apt_rank_table_init(s.rank_table.data_ptr(), bytes, stream()));
  }
  if (s.mb_batch != B || s.mb_fanouts != hop_fanouts || !s.mb_workspace.defined()) {
    const size_t need = apt_minibatch_workspace_bytes(B, fan.data(), H);
    TORCH_CHECK(need > 0, "npc: sample_blocks: unsupported batch / fanouts");
    s.mb_workspace = torch::empty({static_cast<int64_t>(need)}, u8);
    check(apt_minibatch_workspace_init(s.mb_workspace.data_ptr(), need, stream()));
    s.mb_batch = B;
    s.mb_fanouts = hop_fanouts;
  }
  std::vector<int64_t> cap(H + 1);
  for (int h = 0; h <= H; ++h) {
    cap[h] = apt_minibatch_capacity(B, fan.data(), H, h);
    TORCH_CHECK(cap[h] > 0, "npc: sample_blocks: unsupported batch / fanouts");
  }
  // Output buffers at their upper bounds: a set of the ring (reused, see State::mb_ring) or fresh ones.
  State::BlockBuffers fresh;
  State::BlockBuffers* bufp = &fresh;
  if (s.mb_ring_size > 0) {
    if (static_cast<int64_t>(s.mb_ring.size()) != s.mb_ring_size) s.mb_ring.assign(s.mb_ring_size, State::BlockBuffers());
    bufp = &s.mb_ring[s.mb_ring_pos];
    s.mb_ring_pos = (s.mb_ring_pos + 1) % s.mb_ring_size;
  }
  State::BlockBuffers& b = *bufp;
  const bool fits = b.nodes.defined() && b.nodes.numel() == cap[H] && static_cast<int>(b.nb.size()) == H &&
                    b.sizes.numel() == H + 2 + (with_formats ? H : 0) && (!with_formats || b.formats) &&
                    [&] {
                      for (int h = 0; h < H; ++h)
                        if (b.nb[h].numel() != cap[h] * fan[h] || b.ct[h].numel() != cap[h]) return false;
                      return true;
                    }();
  if (!fits) {
    b = State::BlockBuffers();
    b.nodes = torch::empty({cap[H]}, i64_opts());
    b.sizes = torch::empty({H + 2 + (with_formats ? H : 0)}, i64_opts());
    b.nb.resize(H); b.rl.resize(H); b.ct.resize(H);
    for (int h = 0; h < H; ++h) {
      b.nb[h] = torch::empty({cap[h] * fan[h]}, i64_opts());
      b.rl[h] = torch::empty({cap[h] * fan[h]}, i64_opts());
      b.ct[h] = torch::empty({cap[h]}, i64_opts());
    }
    if (with_formats) {
      size_t need = 256;
      for (int h = 0; h < H; ++h) {
        const size_t bytes = apt_block_workspace_bytes(cap[h], fan[h], cap[h + 1], 0);
        TORCH_CHECK(bytes > 0, "npc: sample_blocks: block sizes out of range");
        need = std::max(need, bytes);
      }
      b.format_ws = torch::empty({static_cast<int64_t>(need)}, u8);   // the hops run one after the other
      b.row.resize(H); b.col.resize(H); b.csc.resize(H);
      for (int h = 0; h < H; ++h) {
        b.row[h] = torch::empty({cap[h] * fan[h]}, i64_opts());
        b.col[h] = torch::empty({cap[h] * fan[h]}, i64_opts());
        b.csc[h] = torch::empty({cap[h] + 1}, i64_opts());
      }
      b.formats = true;
    }
  }
  b.sizes.zero_();
  Tensor &nodes = b.nodes, &sizes = b.sizes;
  std::vector<Tensor>&nb = b.nb, &rl = b.rl, &ct = b.ct, &row = b.row, &col = b.col, &csc = b.csc;
  std::vector<int64_t*> nbp(H), rlp(H), ctp(H);
  for (int h = 0; h < H; ++h) {
    nbp[h] = nb[h].data_ptr<int64_t>();
    rlp[h] = rl[h].data_ptr<int64_t>();
    ctp[h] = ct[h].data_ptr<int64_t>();
  }
  const int rc = apt_minibatch_sample(&s.graph, i64(sd), B, fan.data(), H, replace ? 1 : 0,
                                      static_cast<uint64_t>(rng_seed), nullptr, s.rank_table.data_ptr(),
                                      s.graph.num_total_nodes, nodes.data_ptr<int64_t>(), nbp.data(), rlp.data(),
                                      ctp.data(), sizes.data_ptr<int64_t>(), s.mb_workspace.data_ptr(),
                                      static_cast<size_t>(s.mb_workspace.numel()), stream());
  if (rc != APT_OK) s.mb_workspace = Tensor();  // re-initialised by the next call
  check(rc);
  if (with_formats) {
    int64_t* dev_sizes = sizes.data_ptr<int64_t>();
    for (int h = 0; h < H; ++h)
      check(apt_block_formats(rlp[h], cap[h], dev_sizes + h, fan[h], cap[h + 1], row[h].data_ptr<int64_t>(),
                              col[h].data_ptr<int64_t>(), csc[h].data_ptr<int64_t>(), dev_sizes + H + 2 + h, nullptr,
                              nullptr, nullptr, b.format_ws.data_ptr(), static_cast<size_t>(b.format_ws.numel()),
                              stream()));
  }
  auto host = sizes.cpu();  // the one wait of the batch
  const int64_t* hs = host.data_ptr<int64_t>();
  std::vector<Tensor> out{host, nodes.narrow(0, 0, hs[H])};
  for (int h = 0; h < H; ++h) {
    out.push_back(nb[h].narrow(0, 0, hs[h] * fan[h]));
    out.push_back(rl[h].narrow(0, 0, hs[h] * fan[h]));
    out.push_back(ct[h].narrow(0, 0, hs[h]));
  }
  if (with_formats)
    for (int h = 0; h < H; ++h) {
      out.push_back(row[h].narrow(0, 0, hs[H + 2 + h]));
      out.push_back(col[h].narrow(0, 0, hs[H + 2 + h]));
      out.push_back(csc[h].narrow(0, 0, hs[h] + 1));
    }
  return out;
}

// COO / CSC / CSR of a fixed-stride block (what DGL derives from (row, col) in the
// reference, python/npc/sampler.py:59-69).  Returns [coo_row, coo_col, csc_indptr]
// (+ [csr_indptr, csr_indices, csr_eids] with want_csr), cut to the edge count.
std::vector<Tensor> BlockFormats(Tensor relabeled, IdType num_dst, IdType fanout, IdType num_src, bool want_csr) {
  auto rl = ids_on_device(relabeled, "relabeled");
  TORCH_CHECK(num_dst >= 0 && fanout > 0 && num_src >= 0, "npc: block_formats: bad shape");
  TORCH_CHECK(rl.numel() >= num_dst * fanout, "npc: block_formats: relabeled shorter than num_dst * fanout");
  const int64_t slots = num_dst * fanout;
  const size_t need = apt_block_workspace_bytes(num_dst, static_cast<int>(fanout), num_src, want_csr);
  TORCH_CHECK(need > 0 || slots == 0, "npc: block_formats: sizes out of range");
  auto ws = torch::empty({static_cast<int64_t>(std::max<size_t>(need, 256))},
                         torch::TensorOptions().dtype(torch::kUInt8).device(device()));
  auto row = torch::empty({slots}, i64_opts()), col = torch::empty({slots}, i64_opts());
  auto csc = torch::empty({num_dst + 1}, i64_opts()), edges = torch::zeros({1}, i64_opts());
  Tensor csr, ci, ce;
  if (want_csr) {
    csr = torch::empty({num_src + 1}, i64_opts());
    ci = torch::empty({slots}, i64_opts());
    ce = torch::empty({slots}, i64_opts());
  }
  check(apt_block_formats(i64(rl), num_dst, nullptr, static_cast<int>(fanout), num_src, row.data_ptr<int64_t>(),
                          col.data_ptr<int64_t>(), csc.data_ptr<int64_t>(), edges.data_ptr<int64_t>(),
                          want_csr ? csr.data_ptr<int64_t>() : nullptr, want_csr ? ci.data_ptr<int64_t>() : nullptr,
                          want_csr ? ce.data_ptr<int64_t>() : nullptr, ws.data_ptr(),
                          static_cast<size_t>(ws.numel()), stream()));
  const int64_t e = edges.item<int64_t>();
  std::vector<Tensor> out{row.narrow(0, 0, e), col.narrow(0, 0, e), csc};
  if (want_csr) {
    out.push_back(csr);
    out.push_back(ci.narrow(0, 0, e));
    out.push_back(ce.narrow(0, 0, e));
  }
  return out;
}

// reference src/sampling.cc:13-17
std::vector<Tensor> LocalSamplingNeibhorsOneLayer(Tensor seeds, IdType fanout) {
  auto& s = S();
  TORCH_CHECK(s.has_graph, "npc: no graph registered (mix_cache_graphs)");
  TORCH_CHECK(fanout > 0, "npc: fanout must be > 0");
  auto f = ids_on_device(seeds, "seeds");
  auto out = torch::empty({f.numel() * fanout}, i64_opts());
  sample_hop(f, fanout, true, s.rng_seed, static_cast<int>(s.sample_calls), out, nullptr);
  s.sample_calls += 1;
  return {f, out};
}

// relabel_csc through the rank table of the registered graph (apt_relabel_ranked).  The reference's sampler calls
// relabel_csc once per hop with seeds = the unique list of the hop before (python/npc/sampler.py:187-203): such a
// call continues the batch, its seeds are already in the table.  -> false when an id does not fit the table (the
// caller then takes the hash table).
static bool RelabelRanked(const Tensor& sd, const Tensor& nb, Tensor& unique, Tensor& relabeled) {
  auto& s = S();
  const int64_t items = sd.numel() + nb.numel();
  const int64_t len = s.graph.num_total_nodes;
  if (!ranked_resources(items)) return false;
  // bids placed by the sampling call for exactly these tensors?  Bids placed for others are abandoned: the table's
  // batch cannot be continued then.
  auto& p = s.ranked_pending;
  const bool marked = p.valid && nb.numel() > 0 && same_tensor(p.neighbors, p.neighbors_version, nb) &&
                      same_tensor(p.seeds, p.seeds_version, sd);
  const bool continued = marked ? p.continued
                                : !p.valid && same_tensor(s.ranked_last, s.ranked_last_version, sd);
  s.ranked_last = Tensor();
  unique = torch::empty({items}, i64_opts());
  relabeled = marked ? p.states : torch::empty({nb.numel()}, i64_opts());
  if (marked) s.ranked_pending = {};
  else drop_pending_bids();
  int64_t* host = pinned_counts();
  host[0] = host[1] = -1;
  // ranked_counts[1] counts ids beyond the graph; it is zero unless the previous call found some
  check(apt_relabel_ranked(i64(sd), sd.numel(), nullptr, i64(nb), nb.numel(), 0, (continued ? 1 : 0) | (marked ? 2 : 0),
                           s.ranked_table.data_ptr(), len,
                           unique.data_ptr<int64_t>(), nb.numel() ? relabeled.data_ptr<int64_t>() : nullptr,
                           s.ranked_counts.data_ptr<int64_t>(), s.ranked_counts.data_ptr<int64_t>() + 1, host,
                           s.ranked_ws.data_ptr(),
                           static_cast<size_t>(s.ranked_ws.numel()), stream()));
  if (host[1] != 0) {  // ids beyond the graph: not a valid relabel, and the table's batch is not continued
    s.ranked_counts.zero_();
    relabeled = Tensor();
    return false;
  }
  unique = unique.narrow(0, 0, host[0]);
  s.ranked_last = unique;
  s.ranked_last_version = unique._version();
  return true;
}

// reference src/relabel.cc:9-15
std::vector<Tensor> RelabelCSC(Tensor seeds, Tensor neighbors) {
  auto& s = S();
  auto sd = ids_on_device(seeds, "seeds");
  auto nb = ids_on_device(neighbors, "neighbors");
  const int64_t items = sd.numel() + nb.numel();
  // Small inputs: one workgroup with its table in LDS (inside apt_relabel).  Larger ones: the rank table of the
  // registered graph, if there is one and the ids fit it; else the hash table in device memory.
  if (s.has_graph && s.ranked_enabled && items > 8192 && items <= apt_relabel_ranked_max_items() &&
      s.graph.num_total_nodes > 0) {
    Tensor unique, relabeled;
    if (RelabelRanked(sd, nb, unique, relabeled)) return {unique, relabeled};
  }
  s.ranked_last = Tensor();
  if (s.ranked_pending.valid) {   // a sampling call has counted ids beyond the graph, or its bids are not used
    drop_pending_bids();
    if (s.ranked_counts.defined()) s.ranked_counts.zero_();
  }
  const size_t need = apt_relabel_workspace_bytes(items);
  TORCH_CHECK(need > 0, "npc: relabel_csc: ", items, " items exceed the supported maximum");
  auto ws = torch::empty({static_cast<int64_t>(need)}, torch::TensorOptions().dtype(torch::kUInt8).device(device()));
  auto unique = torch::empty({items}, i64_opts());
  auto relabeled = torch::empty({nb.numel()}, i64_opts());
  auto count = torch::empty({1}, i64_opts());
  int64_t* host_count = pinned_counts();
  *host_count = -1;
  check(apt_relabel(i64(sd), sd.numel(), nullptr, i64(nb), nb.numel(), 0, unique.data_ptr<int64_t>(),
                    relabeled.data_ptr<int64_t>(), count.data_ptr<int64_t>(), host_count,
                    ws.data_ptr(), need, stream()));
  return {unique.narrow(0, 0, *host_count), relabeled};
}

// reference src/load_subtensor.cc:19-40
Tensor LoadSubtensor(Tensor node_id) {
  auto& s = S();
  TORCH_CHECK(s.has_feat, "npc: no features registered (cache_feats_shared)");
  PollChecks(false);
  auto idx = ids_on_device(node_id, "node_id");
  auto out = torch::empty({idx.numel(), s.feat.out_dim}, s.local_feats.options());
  Tensor miss;
  if (s.miss_check != 0) miss = torch::zeros({1}, i64_opts());
  check(apt_gather_rows(&s.feat, i64(idx), idx.numel(), nullptr, out.data_ptr(),
                        s.miss_check != 0 ? miss.data_ptr<int64_t>() : nullptr, stream()));
  if (s.miss_check == 2) {
    const int64_t m = miss.item<int64_t>();
    TORCH_CHECK_INDEX(m == 0, "npc: load_subtensor: ", m,
                      " requested node(s) have no feature row on this GPU");
  } else if (s.miss_check == 1) {
    // the counter follows the gather to pinned host memory; nobody waits for it here
    State::PendingCheck p;
    p.dev = miss;
    p.host = torch::empty({1}, torch::TensorOptions().dtype(torch::kInt64).pinned_memory(true));
    p.host.copy_(miss, /*non_blocking=*/true);
    p.done = std::make_shared<at::cuda::CUDAEvent>();
    p.done->record();
    s.pending_checks.push_back(std::move(p));
    if (s.pending_checks.size() > 64) {   // a caller that never lets one arrive: wait for the oldest
      s.pending_checks.front().done->synchronize();
      PollChecks(false);
    }
  }
  return out;
}

// reference src/load_subtensor.cc:10-17: two index_selects, the result on the host
// as there.  The local table lives in HBM here, so the rows come from the GPU; the
// ids are checked on the host first (the map copy is a host tensor), where the
// reference's host index_select would raise: an id outside the map or without a
// local row never reaches a kernel.
Tensor CPULoadSubtensor(Tensor node_id) {
  auto& s = S();
  TORCH_CHECK(s.has_feat, "npc: no features registered (cache_feats_shared)");
  TORCH_CHECK(node_id.scalar_type() == torch::kInt64, "npc: node_id must be int64");
  auto ids = node_id.cpu().contiguous().view({-1});
  const int64_t total = s.cpu_feat_pos_map.numel();
  const int64_t* idp = ids.data_ptr<int64_t>();
  const int64_t* map = s.cpu_feat_pos_map.data_ptr<int64_t>();
  auto pos = torch::empty({ids.numel()}, torch::TensorOptions().dtype(torch::kInt64));
  int64_t* pp = pos.data_ptr<int64_t>();
  const int64_t n_local = s.local_feats.size(0);
  for (int64_t i = 0; i < ids.numel(); ++i) {
    const int64_t v = idp[i];
    TORCH_CHECK_INDEX(v >= 0 && v < total, "npc: cpu_load_subtensor: node id ", v, " at position ", i,
                      " is outside [0, ", total, ")");
    const int64_t row = -map[v] - 2;  // ENCODE_ID, src/utils.h:17
    TORCH_CHECK_INDEX(row >= 0 && row < n_local, "npc: cpu_load_subtensor: node ", v, " at position ", i,
                      " has no local feature row");
    pp[i] = row;
  }
  return s.local_feats.index_select(0, pos.to(s.local_feats.device())).cpu();
}

std::tuple<Tensor, Tensor, Tensor, Tensor> ClusterAndPermuteLocal(Tensor seeds) {
  auto& s = S();
  TORCH_CHECK(s.shuffle_min_vids.defined(), "npc: register_min_vids has not been called");
  TORCH_CHECK(s.shuffle_min_vids.numel() >= s.world_size + 1, "npc: min_vids shorter than world_size + 1");
  auto ids = ids_on_device(seeds, "seeds");
  const int W = static_cast<int>(s.world_size);
  const int node_beg = static_cast<int>(s.rank - (s.rank % s.node_size));  // src/sampling.cc:168-169
  auto size = torch::empty({W}, i64_opts()), offset = torch::empty({W}, i64_opts());
  auto sorted = torch::empty({ids.numel()}, i64_opts()), perm = torch::empty({ids.numel()}, i64_opts());
  const size_t need = apt_bucket_workspace_bytes(ids.numel(), W);
  TORCH_CHECK(need > 0, "npc: bucketing: unsupported size");
  auto ws = torch::empty({static_cast<int64_t>(need)}, torch::TensorOptions().dtype(torch::kUInt8).device(device()));
  check(apt_cluster_permute(i64(ids), ids.numel(), nullptr, s.shuffle_min_vids.data_ptr<int64_t>(), W,
                            s.shuffle_id_offset, static_cast<int>(s.rank), node_beg,
                            node_beg + static_cast<int>(s.node_size), size.data_ptr<int64_t>(),
                            offset.data_ptr<int64_t>(), sorted.data_ptr<int64_t>(),
                            perm.data_ptr<int64_t>(), ws.data_ptr(), need, stream()));
  auto& own = s.own_permutations;
  own.emplace_back(perm, perm._version());
  if (own.size() > 8) own.pop_front();
  return {size, offset, sorted, perm};
}

// reference src/sampling.cc:19-50: virtual nodes of SP mode (local arithmetic, no exchange)
static Tensor MapToVir(const char* who, IdType fanout, const Tensor* dst, IdType num_dst, Tensor src) {
  auto& s = S();
  TORCH_CHECK(s.shuffle_min_vids.defined(), "npc: ", who, ": register_min_vids has not been called");
  TORCH_CHECK(s.shuffle_min_vids.numel() >= s.world_size + 1, "npc: min_vids shorter than world_size + 1");
  TORCH_CHECK(fanout > 0, "npc: ", who, ": fanout must be > 0");
  auto sv = ids_on_device(src, "src");
  Tensor dv;
  if (dst != nullptr) {
    dv = ids_on_device(*dst, "dst");
    num_dst = dv.numel();
  }
  const int node_beg = static_cast<int>(s.rank - (s.rank % s.node_size));
  auto out = torch::empty({(dst != nullptr ? num_dst : 0) + sv.numel()}, i64_opts());
  check(apt_map_to_vir(dst != nullptr ? i64(dv) : nullptr, num_dst, i64(sv), sv.numel(), static_cast<int>(fanout),
                       s.shuffle_min_vids.data_ptr<int64_t>(), static_cast<int>(s.world_size),
                       s.shuffle_id_offset, static_cast<int>(s.rank), node_beg,
                       node_beg + static_cast<int>(s.node_size), out.data_ptr<int64_t>(), stream()));
  return out;
}
Tensor SrcDsttoVir(IdType fanout, Tensor dst, Tensor src) { return MapToVir("srcdst_to_vir", fanout, &dst, 0, src); }
Tensor SrcToVir(IdType fanout, IdType num_dst, Tensor src) {
  TORCH_CHECK(num_dst >= 0, "npc: src_to_vir: num_dst must be >= 0");
  return MapToVir("src_to_vir", fanout, nullptr, num_dst, src);
}

// reference src/sampling.cc:159-193; with one GPU both all-to-alls are identity copies
std::tuple<Tensor, Tensor, Tensor, Tensor> ShuffleSeeds(Tensor seeds) {
  TORCH_CHECK(S().world_size == 1,
              "npc: shuffle_seeds exchanges ids between GPUs; only world_size 1 is available "
              "(cluster_and_permute gives the local half)");
  auto r = ClusterAndPermuteLocal(seeds);
  auto off = std::get<1>(r).cpu();
  return {std::get<2>(r), std::get<3>(r), off.clone(), off};
}

// reference src/load_subtensor.cc:83-86
std::tuple<Tensor, Tensor, Tensor> ClusterReqs(Tensor node_id) {
  auto& s = S();
  TORCH_CHECK(s.has_feat && s.remote_worker_map.defined() && s.shuffle_min_vids.defined(),
              "npc: cluster_reqs needs cache_feats_shared, register_min_vids and "
              "register_multi_machines_scheme");
  TORCH_CHECK(s.shuffle_min_vids.numel() >= s.world_size + 1 && s.remote_worker_map.numel() >= s.world_size,
              "npc: min_vids / remote_worker_map shorter than world_size");
  auto ids = ids_on_device(node_id, "node_id");
  const int R = static_cast<int>(s.num_remote_workers);
  auto size = torch::empty({R}, i64_opts());
  auto sorted = torch::empty({ids.numel()}, i64_opts()), perm = torch::empty({ids.numel()}, i64_opts());
  const size_t need = apt_bucket_workspace_bytes(ids.numel(), R);
  TORCH_CHECK(need > 0, "npc: bucketing: unsupported size");
  auto ws = torch::empty({static_cast<int64_t>(need)}, torch::TensorOptions().dtype(torch::kUInt8).device(device()));
  check(apt_cluster_reqs(i64(ids), ids.numel(), nullptr, s.feat_pos_map.data_ptr<int64_t>(),
                         s.feat_pos_map.numel(), s.remote_worker_map.data_ptr<int64_t>(),
                         s.shuffle_min_vids.data_ptr<int64_t>(), static_cast<int>(s.world_size), R,
                         size.data_ptr<int64_t>(), nullptr, sorted.data_ptr<int64_t>(),
                         perm.data_ptr<int64_t>(), ws.data_ptr(), need, stream()));
  return {size, sorted, perm};
}

// reference src/feat_shuffle.cc:9-30 with one GPU
Tensor FeatShuffle(Tensor inputs, Tensor send_offset, Tensor recv_offset, Tensor permutation,
                   IdType feat_dim, IdType fwd_flag) {
  TORCH_CHECK(S().world_size == 1,
              "npc: feat_shuffle exchanges rows between GPUs; only world_size 1 is available");
  TORCH_CHECK(inputs.is_cuda() && (inputs.element_size() == 2 || inputs.element_size() == 4),
              "npc: feat_shuffle needs a GPU tensor with 2- or 4-byte elements");
  auto x = inputs.reshape({-1, feat_dim}).contiguous();
  auto perm = ids_on_device(permutation, "permutation");
  const int64_t n_out = recv_offset.index({-1}).item<int64_t>();
  if (fwd_flag) {
    TORCH_CHECK(x.size(0) == n_out, "npc: with one GPU the received row count equals the sent one");
    auto out = torch::empty({perm.numel(), feat_dim}, x.options());
    check(apt_permute_rows(x.data_ptr(), x.size(0), i64(perm), perm.numel(), feat_dim,
                           static_cast<int>(x.element_size()), out.data_ptr(), stream()));
    return out;
  }
  TORCH_CHECK(perm.numel() == x.size(0), "npc: permutation must name every input row");
  // rows that no permutation entry names (none when it is a bijection, as ShuffleSeeds makes it) are flagged by
  // the scatter and zeroed afterwards: cheaper than zero-filling the whole output first
  auto out = torch::empty({n_out, feat_dim}, x.options());
  auto ws = torch::empty({static_cast<int64_t>(apt_scatter_workspace_bytes(n_out))},
                         torch::TensorOptions().dtype(torch::kUInt8).device(device()));
  check(apt_scatter_rows(x.data_ptr(), i64(perm), perm.numel(), feat_dim, static_cast<int>(x.element_size()),
                         out.data_ptr(), n_out, ws.data_ptr(), static_cast<size_t>(ws.numel()), stream()));
  bool own = false;   // a permutation this library produced is a bijection onto [0, n): nothing to check
  for (const auto& p : S().own_permutations)
    own |= p.first.data_ptr() == perm.data_ptr() && p.first.numel() == perm.numel() && p.second == perm._version() &&
           perm.numel() == n_out;
  if (S().strict && !own) {
    // The reference's pack is index_select_backward (src/feat_shuffle.cc:14-16): rows named more than once
    // add up.  The scatter keeps one of them, which is the same thing only for a permutation without
    // repeats (what ShuffleSeeds produces).  The flags tell: as many rows named as entries <=> no repeats and
    // nothing out of range; otherwise the sum is formed the reference's way.
    const int64_t named = ws.narrow(0, 0, n_out).sum().item<int64_t>();
    if (named != perm.numel()) {
      TORCH_CHECK_INDEX(perm.numel() == 0 || (perm.min().item<int64_t>() >= 0 && perm.max().item<int64_t>() < n_out),
                        "npc: feat_shuffle: permutation entry outside [0, ", n_out, ")");
      out = torch::zeros({n_out, feat_dim}, x.options()).index_add_(0, perm, x);
    }
  }
  return out;
}

// ---------------------------------------------------------------- aggregation
namespace {

Tensor feat2d(const Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 &&
                  (t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kBFloat16),
              "npc: ", name, " must be a 2-D fp32 or bf16 GPU tensor");
  return t.contiguous();
}

// out_num = output_offset[-1] is read on the host, as in the reference (src/spmm.cc:13).
Tensor spmm(int mode, Tensor coo_row, Tensor coo_col, Tensor input, const Tensor* edata, Tensor coo_offset,
            const Tensor* input_offset, Tensor output_offset) {
  auto row = ids_on_device(coo_row, "coo_row"), col = ids_on_device(coo_col, "coo_col");
  auto x = feat2d(input, "input");
  auto coo = ids_on_device(coo_offset, "coo_offset");
  auto oo = ids_on_device(output_offset, "output_offset");
  TORCH_CHECK(coo.numel() >= 2 && oo.numel() >= coo.numel() - 1 && row.numel() == col.numel(),
              "npc: spmm: bad offsets or edge lists");
  const int nseg = static_cast<int>(coo.numel() - 1);
  Tensor io, ed;
  if (input_offset) io = ids_on_device(*input_offset, "input_offset");
  if (edata) {
    ed = feat2d(*edata, "edata");
    TORCH_CHECK(ed.scalar_type() == x.scalar_type() && ed.size(0) == row.numel() && ed.size(1) == x.size(1),
                "npc: spmm: edata must be [E, dim] of the input dtype");
  }
  if (mode == 1) TORCH_CHECK(x.size(0) == row.numel(), "npc: spmm_copy_e_sum needs one input row per edge");
  TORCH_CHECK(!input_offset || io.numel() >= nseg, "npc: spmm: input_offset is shorter than the segments");
  const int64_t E = row.numel();
  // The edge-parallel sum: atomics where a row's edges are not together.
  const auto by_edge = [&](int64_t out_num) {
    auto out = torch::zeros({out_num, x.size(1)}, x.options().dtype(torch::kFloat32));
    auto flag = torch::empty({1}, torch::TensorOptions().dtype(torch::kInt32).device(device()));
    check(apt_coo_is_grouped(i64(col), E, flag.data_ptr<int>(), stream()));
    check(apt_spmm_sum(mode, i64(row), i64(col), E, x.data_ptr(), x.size(0), edata ? ed.data_ptr() : nullptr, x.size(1),
                       static_cast<int>(x.element_size()), i64(coo), input_offset ? i64(io) : nullptr, i64(oo), nseg,
                       out.data_ptr<float>(), out_num, flag.data_ptr<int>(), stream()));
    return out.to(x.scalar_type());
  };
  // Ordering the edges costs some 30 us of launches, as much as about 2 M atomic additions: few edges or short rows are
  // added up as they come.  Edges in any order, by edge / ordered: 16 k of 64 features, 65 k of 16 (2^20 additions) 57 / 77,
  // 54 / 77 us; 260 k of 4 94 / 83; 16 k of 256, 65 k of 64, 260 k of 16 (2^22) 91 / 77, 93 / 76, 95 / 81; 1 M of 64 887 / 169.
  // Edges grouped by output row need no order: 46 / 45 us up to 2^22, 92 / 90 for 1 M of 64.
  if (E * x.size(1) <= int64_t{1} << 21) return by_edge(oo.index({-1}).item<int64_t>());
  // every edge's rows, whether the edges come grouped by output row (a block's COO does), the number of output rows, and
  // whether some may have very many edges: the last three are read back in one copy
  auto keys = torch::empty({2, E}, i64_opts());
  auto probe = torch::empty({3}, i64_opts());
  check(apt_coo_prepare(i64(row), i64(col), E, i64(coo), input_offset ? i64(io) : nullptr, i64(oo), nseg,
                        i64(oo) + oo.numel() - 1, keys.data_ptr<int64_t>(), keys.data_ptr<int64_t>() + E,
                        probe.data_ptr<int64_t>(), stream()));
  const int64_t* host = read_counts(probe);
  const int grouped = host[0] != 0, has_long = host[2] != 0;
  const int64_t out_num = host[1];
  const size_t need = apt_coo_sum_workspace_bytes(E, out_num, grouped, has_long, x.size(1));
  if (need > 0) {
    auto ws = torch::empty({static_cast<int64_t>(need)}, x.options().dtype(torch::kUInt8));
    auto out = torch::empty({out_num, x.size(1)}, x.options());
    check(apt_coo_sum(mode, i64(keys), E ? i64(keys) + E : nullptr, E, grouped, has_long, x.data_ptr(), x.size(0),
                      edata ? ed.data_ptr() : nullptr, x.size(1), static_cast<int>(x.element_size()), out.data_ptr(),
                      out_num, ws.data_ptr(), need, stream()));
    return out;
  }
  return by_edge(out_num);   // more edges or rows than the ordering takes
}

Tensor sddmm(int op, Tensor coo_row, Tensor coo_col, Tensor lhs, Tensor rhs, Tensor coo_offset,
             Tensor lhs_offset, Tensor rhs_offset) {
  auto row = ids_on_device(coo_row, "coo_row"), col = ids_on_device(coo_col, "coo_col");
  auto l = feat2d(lhs, "lhs"), r = feat2d(rhs, "rhs");
  TORCH_CHECK(l.scalar_type() == r.scalar_type() && l.size(1) == r.size(1) && row.numel() == col.numel(),
              "npc: sddmm: lhs/rhs mismatch");
  auto coo = ids_on_device(coo_offset, "coo_offset");
  auto lo = ids_on_device(lhs_offset, "lhs_offset"), ro = ids_on_device(rhs_offset, "rhs_offset");
  TORCH_CHECK(coo.numel() >= 2 && lo.numel() >= coo.numel() - 1 && ro.numel() >= coo.numel() - 1,
              "npc: sddmm: bad offsets");
  auto out = torch::empty({row.numel(), l.size(1)}, l.options());
  check(apt_coo_combine(op, i64(row), i64(col), row.numel(), l.data_ptr(), l.size(0), r.data_ptr(), r.size(0),
                  l.size(1), static_cast<int>(l.element_size()), i64(coo), i64(lo), i64(ro),
                  static_cast<int>(coo.numel() - 1), out.data_ptr(), stream()));
  return out;
}

}  // namespace

// reference src/spmm.cc:9-42
Tensor CopyUSum(Tensor coo_row, Tensor coo_col, Tensor input, Tensor coo_offset, Tensor input_offset,
                Tensor output_offset) {
  return spmm(0, coo_row, coo_col, input, nullptr, coo_offset, &input_offset, output_offset);
}
Tensor CopyESum(Tensor coo_row, Tensor coo_col, Tensor input, Tensor coo_offset, Tensor output_offset) {
  return spmm(1, coo_row, coo_col, input, nullptr, coo_offset, nullptr, output_offset);
}
Tensor UMulESum(Tensor coo_row, Tensor coo_col, Tensor input, Tensor edata, Tensor coo_offset,
                Tensor input_offset, Tensor output_offset) {
  return spmm(2, coo_row, coo_col, input, &edata, coo_offset, &input_offset, output_offset);
}
// reference src/sddmm.cc:9-31
Tensor UAddV(Tensor coo_row, Tensor coo_col, Tensor lhs, Tensor rhs, Tensor coo_offset, Tensor lhs_offset,
             Tensor rhs_offset) {
  return sddmm(0, coo_row, coo_col, lhs, rhs, coo_offset, lhs_offset, rhs_offset);
}
Tensor UMulV(Tensor coo_row, Tensor coo_col, Tensor lhs, Tensor rhs, Tensor coo_offset, Tensor lhs_offset,
             Tensor rhs_offset) {
  return sddmm(1, coo_row, coo_col, lhs, rhs, coo_offset, lhs_offset, rhs_offset);
}

// ---------------------------------------------------------------- dense layers over a block's rows
namespace {

// A product whose weight's gradient is wanted, dw = dy^T x, and its bias's, the column sums of dy; dy counts where `relu`
// is positive if that is given.  Without x the sums alone.
struct WeightGrad {
  Tensor dy, x;
  bool want_bias = false;
  Tensor relu;
  Tensor dw{}, db{};
};
// Gradients of one or two products, of one type, in one launch (apt_linear_wgrads).
template <size_t N>
void weight_grads(std::array<WeightGrad, N>& all, size_t count = N) {
  apt_wgrad_product products[N] = {};
  int es = 0;
  bool empty = false;
  for (size_t i = 0; i < count; ++i) {
    WeightGrad& g = all[i];
    g.dy = g.dy.contiguous();
    if (g.x.defined()) g.x = g.x.contiguous();
    if (g.relu.defined()) g.relu = g.relu.contiguous();
    es = static_cast<int>(g.dy.element_size());
    products[i].m = g.dy.size(0);
    products[i].n = g.dy.size(1);
    products[i].k = g.x.defined() ? g.x.size(1) : 0;
    empty |= g.x.defined() && products[i].k == 0;
  }
  const size_t need = empty ? 0 : apt_linear_wgrads_workspace_bytes(products, static_cast<int>(count), es);
  if (need == 0) {   // a weight beyond the kernel's sizes, or without elements
    for (size_t i = 0; i < count; ++i) {
      WeightGrad& g = all[i];
      const Tensor dy = g.relu.defined() ? at::threshold_backward(g.dy, g.relu, 0) : g.dy;
      if (g.x.defined()) g.dw = dy.t().mm(g.x);
      if (g.want_bias) g.db = dy.sum(0);
    }
    return;
  }
  auto ws = torch::empty({static_cast<int64_t>(need)}, all[0].dy.options().dtype(torch::kUInt8));
  for (size_t i = 0; i < count; ++i) {
    WeightGrad& g = all[i];
    apt_wgrad_product& q = products[i];
    if (g.x.defined()) g.dw = torch::empty({q.n, q.k}, g.dy.options());
    if (g.want_bias) g.db = torch::empty({q.n}, g.dy.options());
    q.dy = g.dy.data_ptr();
    q.out = g.relu.defined() ? g.relu.data_ptr() : nullptr;
    q.x = g.x.defined() ? g.x.data_ptr() : nullptr;
    q.dw = g.dw.defined() ? g.dw.data_ptr() : nullptr;
    q.db = g.db.defined() ? g.db.data_ptr() : nullptr;
  }
  check(apt_linear_wgrads(products, static_cast<int>(count), es, ws.data_ptr(), need, stream()));
}
std::tuple<Tensor, Tensor> linear_wgrad(const Tensor& dy, const Tensor& x, bool want_bias) {
  std::array<WeightGrad, 1> g{WeightGrad{dy, x, want_bias}};
  weight_grads(g);
  return {g[0].dw, g[0].db};
}

// Whether apt_rows_product takes a weight [n, k]: contiguous along a side.
bool product_takes(const Tensor& w) {
  const int64_t n = w.size(0), k = w.size(1), sn = w.stride(0), sk = w.stride(1);
  return (sk == 1 && sn >= k && (n + 256) * sn <= (1 << 30)) || (sn == 1 && sk >= n && (k + 32) * sk <= (1 << 30));
}

// Whether apt_rows_product is the faster for such sizes.  It reads the rows once for every column tile whose weights fit
// LDS, and costs the host a third of a library product (6 us of 21): it wins where the rows are what counts, where a second
// product and its sum are spared, and where both are short.  GPU us, library / here, 20 k | 54 k | 124 k | 460 k rows:
//   100 -> 256 10/8 16/16 67/25 169/99     128 -> 64 5/5 7/8 27/12 59/32       128 -> 256 7/10 12/16 43/23 113/100
//   128 -> 512 10/16 21/21 46/36 188/169   188 -> 256 12/11 19/21 78/33 215/101   256 -> 128 7/10 12/15 24/23 105/80
//   256 -> 256 9/15 16/25 30/37 151/110    512 -> 128 9/15 18/21 34/34 160/118    512 -> 256 12/19 22/32 44/55 227/178
//   1000 -> 64 16/16 28/27 74/51           1024 -> 128 12/24 23/42 57/76          1024 -> 1024 46/92 101/217 235/471
//   333 -> 333 25/29 66/59 111/121         100 + 100 -> 256 23/13 35/23 142/40 403/113
//   256 + 256 -> 256, 0.15 of the rows in the second: 15/18 24/26 43/41 193/125
bool product_pays(int64_t m, int64_t n, int64_t k, int64_t k2) {
  const int64_t steps = (k + 31) / 32 + (k2 + 31) / 32;
  const bool once = n <= 64 || (n <= 128 && steps <= 16);   // one column tile, if any fits
  if (steps <= 4 || (k2 > 0 && steps <= 16) || (k % 32 != 0 && k % 2 == 0 && steps <= 8)) return true;
  if (m * n <= (k % 2 == 0 ? 1300000000 : 650000000) / k) return true;
  return m >= 100000 && (once || (m >= 300000 && k % 32 == 0 && k <= 512 && n <= 256));
}

// x w^T (+ x2 w2^T on the first rows) (+ b) with w [n, k] of any strides; `onto`: added to (and returned).  fp32 rows
// take apt_rows_gemm, bf16 rows apt_rows_product or the library's product.
Tensor dense(const Tensor& x_in, const Tensor& w, const Tensor& x2_in = Tensor(), const Tensor& w2 = Tensor(),
             const Tensor& b = Tensor(), Tensor onto = Tensor(), bool relu = false) {
  const int64_t m = x_in.size(0), k = x_in.size(1), n = w.size(0);
  const bool pair = x2_in.defined();
  const int64_t m2 = pair ? x2_in.size(0) : 0, k2 = pair ? x2_in.size(1) : 0;
  TORCH_CHECK(w.size(1) == k && (!pair || (w2.size(0) == n && w2.size(1) == k2 && m2 <= m)) && (!b.defined() || b.numel() == n),
              "npc: a layer's rows have ", k, " columns, its weight is ", n, " x ", w.size(1), " (or the bias does not fit)");
  const size_t need = x_in.scalar_type() == torch::kFloat32 ? apt_rows_gemm_workspace_bytes(n, k, k2) : 0;
  if (need > 0) {
    auto x = x_in.contiguous();
    Tensor x2 = pair ? x2_in.contiguous() : Tensor(), bias = b.defined() ? b.contiguous() : Tensor();
    const bool accumulate = onto.defined();
    auto y = accumulate ? onto : torch::empty({m, n}, x.options());
    auto ws = torch::empty({static_cast<int64_t>(need)}, x.options().dtype(torch::kUInt8));
    check(apt_rows_gemm(x.data_ptr<float>(), k, w.data_ptr<float>(), w.stride(0), w.stride(1),
                        pair ? x2.data_ptr<float>() : nullptr, k2, pair ? w2.data_ptr<float>() : nullptr,
                        pair ? w2.stride(0) : 0, pair ? w2.stride(1) : 0, m, m2, n,
                        bias.defined() ? bias.data_ptr<float>() : nullptr, accumulate, relu, y.data_ptr<float>(), ws.data_ptr(),
                        need, stream()));
    return y;
  }
  if (x_in.scalar_type() == torch::kBFloat16 && apt_rows_product_fits(m, n, k, k2) && product_pays(m, n, k, k2) && product_takes(w) &&
      (!pair || product_takes(w2)) && (!b.defined() || b.scalar_type() == torch::kBFloat16)) {
    auto x = x_in.contiguous();
    Tensor x2 = pair ? x2_in.contiguous() : Tensor(), bias = b.defined() ? b.contiguous() : Tensor();
    const bool accumulate = onto.defined();
    auto y = accumulate ? onto : torch::empty({m, n}, x.options());
    check(apt_rows_product(x.data_ptr(), k, w.data_ptr(), w.stride(0), w.stride(1), pair ? x2.data_ptr() : nullptr, k2,
                           pair ? w2.data_ptr() : nullptr, pair ? w2.stride(0) : 0, pair ? w2.stride(1) : 0, m, m2, n,
                           bias.defined() ? bias.data_ptr() : nullptr, accumulate, relu, y.data_ptr(), stream()));
    return y;
  }
  Tensor y;
  if (onto.defined()) {   // (in one rounding)
    y = onto.addmm_(x_in, w.t());
    if (b.defined()) y.add_(b);
  } else {
    y = at::linear(x_in, w, b.defined() ? std::optional<Tensor>(b) : std::nullopt);
  }
  if (pair) y.narrow(0, 0, m2).addmm_(x2_in, w2.t());
  return relu ? y.relu_() : y;
}

// Whether a call is part of a training step.  Its fp32 products are the library's (`exact` below): they give the bits of nn.Linear, and a
// ReLU whose input changes sign with the last bit (one or two of 10^7) moves a weight's gradient by up to 6e-5.
template <typename... Tensors>
bool trains(const Tensors&... t) {
  return torch::GradMode::is_enabled() && (t.requires_grad() || ...);
}
bool exact(bool train, const Tensor& x) { return train && x.scalar_type() == torch::kFloat32; }
Tensor product(bool library, const Tensor& x, const Tensor& w, const Tensor& b = Tensor()) {
  return library ? at::linear(x, w, b.defined() ? std::optional<Tensor>(b) : std::nullopt)
               : dense(x, w, Tensor(), Tensor(), b);
}

// What a gradient needs is kept until then; the rest stays free to be changed in place.
Tensor kept_if(bool needed, const Tensor& t) { return needed ? t : Tensor(); }
// Slots and CSR of a block that was made in inference mode: autograd keeps no such tensor, but a copy of it.
Tensor keepable(bool train, const Tensor& t) { return train && t.is_inference() ? t.clone() : t; }
std::optional<Tensor> keepable(bool train, const std::optional<Tensor>& t) {
  return t.has_value() ? std::optional<Tensor>(keepable(train, *t)) : t;
}

// y = x w^T + b (or x w with `kn`: w is [k, n]).
struct BlockLinearFn : public torch::autograd::Function<BlockLinearFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w,
                        const std::optional<Tensor>& b, bool kn, bool train) {
    ctx->save_for_backward({kept_if(w.requires_grad(), x), kept_if(x.requires_grad(), w)});
    ctx->saved_data["kn"] = kn;
    ctx->saved_data["bias"] = b.has_value() && b->requires_grad();
    if (exact(train, x) && kn) return at::mm(x, w);
    return product(exact(train, x), x, kn ? w.t() : w, b.value_or(Tensor()));
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1], &dy = grads[0];
    const bool kn = ctx->saved_data["kn"].toBool(), bias = ctx->saved_data["bias"].toBool();
    Tensor dx, dw, db;
    if (torch::GradMode::is_enabled()) {   // a graph of the gradients is wanted: operations that carry one
      if (ctx->needs_input_grad(0)) dx = kn ? dy.mm(w.t()) : dy.mm(w);
      if (ctx->needs_input_grad(1)) dw = kn ? x.t().mm(dy) : dy.t().mm(x);
      if (bias) db = dy.sum(0);
    } else {
      if (ctx->needs_input_grad(0)) dx = dense(dy, kn ? w : w.t());
      if (ctx->needs_input_grad(1)) std::tie(dw, db) = kn ? linear_wgrad(x, dy, false) : linear_wgrad(dy, x, bias);
      else if (bias) db = dy.sum(0);
    }
    return {dx, dw, db, Tensor(), Tensor()};
  }
};

}  // namespace

Tensor BlockLinear(const Tensor& x, const Tensor& w, const std::optional<Tensor>& b, bool kn) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == w.scalar_type() &&
                  (x.scalar_type() == torch::kFloat32 || x.scalar_type() == torch::kBFloat16),
              "npc: block_linear needs 2-D fp32 or bf16 GPU tensors of one dtype");
  TORCH_CHECK(!kn || !b.has_value(), "npc: block_linear: a [k, n] weight takes no bias");
  return BlockLinearFn::apply(x, w, b, kn, trains(x, w) || (b.has_value() && trains(*b)));
}

// ---------------------------------------------------------------- aggregation over a block, with its gradient
namespace {

void check_block(const char* who, const Tensor& relabeled, int64_t num_dst, int64_t fanout) {
  TORCH_CHECK_TYPE(relabeled.is_cuda() && relabeled.scalar_type() == torch::kInt64 && relabeled.is_contiguous(), "npc: ", who,
                   ": the block's slots must be a contiguous int64 tensor on the GPU");
  TORCH_CHECK(num_dst >= 0 && fanout > 0 && relabeled.numel() >= num_dst * fanout, "npc: ", who,
              ": the block has fewer than num_dst * fanout slots");
}

// The edges of every source of a block: slots (4-byte, apt_block_transpose), or, for a block too large for that, the
// destinations of its CSR (8-byte), with the table of the sources that have very many and `scratch` bytes beside it.
// Enqueued on the current stream; nothing is read back.
struct SourceOrder {
  Tensor memory, csr_indptr, csr_index;
  const void* indptr = nullptr;
  const void* index = nullptr;
  void* table = nullptr;        // NULL: no source can have so many
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  int bytes = 4;
  int64_t edges = 0;            // what index holds
};
size_t aligned(size_t x) { return (x + 255) / 256 * 256; }

// of a CSR
SourceOrder source_order_csr(const Tensor& csr_indptr, const Tensor& csr_index, int64_t num_src, size_t scratch) {
  SourceOrder o;
  o.csr_indptr = csr_indptr;
  o.csr_index = csr_index;
  o.indptr = csr_indptr.data_ptr();
  o.index = csr_index.numel() > 0 ? csr_index.data_ptr() : nullptr;
  o.bytes = 8;
  o.edges = csr_index.numel();
  if (const size_t need = apt_long_rows_bytes(o.edges)) {
    o.memory = torch::empty({static_cast<int64_t>(aligned(need) + scratch)}, csr_indptr.options().dtype(torch::kUInt8));
    o.table = o.memory.data_ptr();
    o.scratch = static_cast<char*>(o.table) + aligned(need);
    o.scratch_bytes = scratch;
    check(apt_find_long_rows(o.indptr, 8, num_src, o.edges, o.table, stream()));
  }
  return o;
}

SourceOrder source_order(const Tensor& relabeled, int64_t num_dst, int64_t fanout, int64_t num_src, size_t scratch) {
  const int64_t slots = std::max<int64_t>(num_dst * fanout, 1);
  const int f = static_cast<int>(fanout);
  const auto u8 = relabeled.options().dtype(torch::kUInt8);
  if (const size_t need = apt_block_transpose_workspace_bytes(num_dst, f, num_src)) {
    SourceOrder o;
    o.edges = num_dst * fanout;
    const size_t offsets = aligned(4 * (static_cast<size_t>(num_src) + 1)), entries = aligned(4 * static_cast<size_t>(slots)),
                 table = aligned(apt_long_rows_bytes(o.edges));
    o.scratch_bytes = std::max(need, scratch);   // first the transpose's, then the caller's
    o.memory = torch::empty({static_cast<int64_t>(offsets + entries + table + o.scratch_bytes)}, u8);
    char* at = static_cast<char*>(o.memory.data_ptr());
    o.indptr = at;
    o.index = at + offsets;
    o.table = table > 0 ? at + offsets + entries : nullptr;
    o.scratch = at + offsets + entries + table;
    check(apt_block_transpose(i64(relabeled), num_dst, f, num_src, reinterpret_cast<uint32_t*>(at),
                              reinterpret_cast<uint32_t*>(at + offsets), o.table, o.scratch, need, stream()));
    return o;
  }
  const size_t need = apt_block_workspace_bytes(num_dst, f, num_src, 1);
  TORCH_CHECK(need > 0, "npc: block of ", num_dst, " x ", fanout, " slots and ", num_src, " sources is out of range");
  auto ws = torch::empty({static_cast<int64_t>(need)}, u8);
  auto coo = torch::empty({2, slots}, relabeled.options()), csc = torch::empty({num_dst + 1}, relabeled.options());
  auto edges = torch::empty({1}, relabeled.options()), eids = torch::empty({slots}, relabeled.options());
  auto indptr = torch::empty({num_src + 1}, relabeled.options()), index = torch::empty({slots}, relabeled.options());
  check(apt_block_formats(i64(relabeled), num_dst, nullptr, f, num_src, coo.data_ptr<int64_t>(),
                          coo.data_ptr<int64_t>() + slots, csc.data_ptr<int64_t>(), edges.data_ptr<int64_t>(),
                          indptr.data_ptr<int64_t>(), index.data_ptr<int64_t>(), eids.data_ptr<int64_t>(), ws.data_ptr(), need,
                          stream()));
  return source_order_csr(indptr, index, num_src, scratch);
}

// The gradient of the block sum / mean towards its input, from the block's CSR if it has one.
Tensor aggregate_backward(const Tensor& dz_in, const Tensor& relabeled, int64_t num_dst, int64_t fanout, int64_t num_src,
                          const Tensor& dst_scale, const Tensor& csr_indptr, const Tensor& csr_indices, float scale = 1.f) {
  auto dz = dz_in.contiguous();
  auto dx = torch::empty({num_src, dz.size(1)}, dz.options());
  const bool csr = csr_indptr.defined() && csr_indptr.numel() == num_src + 1;
  const size_t scratch =
      apt_block_aggregate_backward_workspace_bytes(csr ? csr_indices.numel() : num_dst * fanout, dz.size(1));
  const SourceOrder o = csr ? source_order_csr(csr_indptr, csr_indices, num_src, scratch)
                            : source_order(relabeled, num_dst, fanout, num_src, scratch);
  check(apt_block_aggregate_backward(o.indptr, o.index, o.bytes, static_cast<int>(fanout), num_src, o.edges, o.table,
                                     dst_scale.defined() ? dst_scale.data_ptr<float>() : nullptr, scale, dz.data_ptr(), num_dst,
                                     dz.size(1), static_cast<int>(dz.element_size()), dx.data_ptr(), o.scratch, o.scratch_bytes,
                                     stream()));
  return dx;
}

// -> (sum or mean, 1 / degree per destination when `mean`)
std::tuple<Tensor, Tensor> aggregate_forward(const Tensor& relabeled, int64_t num_dst, int64_t fanout, const Tensor& x,
                                             bool mean, float scale = 1.f, const Tensor& bias = Tensor(), bool relu = false,
                                             const Tensor& base = Tensor()) {
  auto out = torch::empty({num_dst, x.size(1)}, x.options());
  Tensor inv;
  if (mean) inv = torch::empty({num_dst}, x.options().dtype(torch::kFloat32));
  check(apt_block_aggregate(i64(relabeled), num_dst, static_cast<int>(fanout), x.data_ptr(), x.size(0), x.size(1),
                            static_cast<int>(x.element_size()), mean, scale, bias.defined() ? bias.data_ptr() : nullptr,
                            base.defined() ? base.data_ptr() : nullptr, relu, out.data_ptr(),
                            mean ? inv.data_ptr<float>() : nullptr, stream()));
  return {out, inv};
}

std::optional<Tensor> maybe(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// The same inside a backward pass whose own graph may be wanted (create_graph).
Tensor aggregate_gradient(const Tensor& dz, const Tensor& relabeled, int64_t num_dst, int64_t fanout, int64_t num_src,
                          const Tensor& dst_scale, const Tensor& csr_indptr, const Tensor& csr_indices, double scale = 1.0);

struct BlockAggregateFn : public torch::autograd::Function<BlockAggregateFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& relabeled, int64_t num_dst,
                        int64_t fanout, bool mean, const std::optional<Tensor>& csr_indptr,
                        const std::optional<Tensor>& csr_indices) {
    auto r = aggregate_forward(relabeled, num_dst, fanout, x, mean);
    ctx->save_for_backward({relabeled, std::get<1>(r), csr_indptr.value_or(Tensor()), csr_indices.value_or(Tensor())});
    ctx->saved_data["num_dst"] = num_dst;
    ctx->saved_data["fanout"] = fanout;
    ctx->saved_data["num_src"] = x.size(0);
    return std::get<0>(r);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Tensor dx;
    if (ctx->needs_input_grad(0))
      dx = aggregate_gradient(grads[0], saved[0], ctx->saved_data["num_dst"].toInt(), ctx->saved_data["fanout"].toInt(),
                              ctx->saved_data["num_src"].toInt(), saved[1], saved[2], saved[3]);
    return {dx, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// That gradient is linear in dz, and its own gradient is the sum (or mean) again.
struct AggregateGradientFn : public torch::autograd::Function<AggregateGradientFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& dz, const Tensor& relabeled, int64_t num_dst,
                        int64_t fanout, int64_t num_src, const std::optional<Tensor>& dst_scale,
                        const std::optional<Tensor>& csr_indptr, const std::optional<Tensor>& csr_indices, double scale) {
    ctx->save_for_backward({relabeled, csr_indptr.value_or(Tensor()), csr_indices.value_or(Tensor())});
    ctx->saved_data["num_dst"] = num_dst;
    ctx->saved_data["fanout"] = fanout;
    ctx->saved_data["mean"] = dst_scale.has_value();
    ctx->saved_data["scale"] = scale;
    return aggregate_backward(dz, relabeled, num_dst, fanout, num_src, dst_scale.value_or(Tensor()), csr_indptr.value_or(Tensor()),
                              csr_indices.value_or(Tensor()), static_cast<float>(scale));
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Tensor ddz = BlockAggregateFn::apply(grads[0].contiguous(), saved[0], ctx->saved_data["num_dst"].toInt(),
                                         ctx->saved_data["fanout"].toInt(), ctx->saved_data["mean"].toBool(), maybe(saved[1]),
                                         maybe(saved[2]));
    const double scale = ctx->saved_data["scale"].toDouble();
    if (scale != 1.0) ddz = ddz * scale;
    return {ddz, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor aggregate_gradient(const Tensor& dz, const Tensor& relabeled, int64_t num_dst, int64_t fanout, int64_t num_src,
                          const Tensor& dst_scale, const Tensor& csr_indptr, const Tensor& csr_indices, double scale) {
  if (torch::GradMode::is_enabled())
    return AggregateGradientFn::apply(dz, relabeled, num_dst, fanout, num_src, maybe(dst_scale), maybe(csr_indptr),
                                      maybe(csr_indices), scale);
  return aggregate_backward(dz, relabeled, num_dst, fanout, num_src, dst_scale, csr_indptr, csr_indices,
                            static_cast<float>(scale));
}

}  // namespace

Tensor BlockAggregate(const Tensor& relabeled, int64_t num_dst, int64_t fanout, const Tensor& x, bool mean,
                      const std::optional<Tensor>& csr_indptr, const std::optional<Tensor>& csr_indices) {
  check_block("block_aggregate", relabeled, num_dst, fanout);
  TORCH_CHECK_TYPE(x.is_cuda() && x.dim() == 2 &&
                       (x.scalar_type() == torch::kFloat32 || x.scalar_type() == torch::kBFloat16),
                   "npc: block_aggregate: input must be a 2-D fp32 or bf16 GPU tensor");
  const bool train = trains(x);
  return BlockAggregateFn::apply(x.contiguous(), keepable(train, relabeled), num_dst, fanout, mean, keepable(train, csr_indptr),
                                 keepable(train, csr_indices));
}

// ---------------------------------------------------------------- GraphSAGE layer
namespace {

// The gradient towards what a layer's ReLU was applied to (`out`: its result; undefined: no ReLU).
Tensor before_relu(const Tensor& grad, const Tensor& out) {
  return (out.defined() ? at::threshold_backward(grad, out, 0) : grad).contiguous();
}

// x[:num_dst] w_self^T + bias + mean over the block of x, times w_neigh^T; the product comes before the mean where it
// makes the rows shorter.  As one function the two products and their gradients are added up in the kernels that form
// them: no pass over the result to add them, no zero-filled gradient of the destinations' rows.
struct SageLayerFn : public torch::autograd::Function<SageLayerFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w_neigh, const Tensor& w_self,
                        const std::optional<Tensor>& bias, const Tensor& relabeled, int64_t num_dst, int64_t fanout,
                        const std::optional<Tensor>& csr_indptr, const std::optional<Tensor>& csr_indices, bool relu,
                        bool train) {
    const Tensor b = bias.value_or(Tensor()), self = x.narrow(0, 0, num_dst);
    const bool first = x.size(1) > w_self.size(0);
    Tensor mean, inv, out;
    const bool apart = train;   // the products by the library
    if (first) {
      const Tensor base = product(apart, self, w_self, b);
      std::tie(out, inv) = aggregate_forward(relabeled, num_dst, fanout, product(apart, x, w_neigh), true, 1.f, Tensor(), relu,
                                             base);
    } else {
      std::tie(mean, inv) = aggregate_forward(relabeled, num_dst, fanout, x, true);
      if (apart) {
        out = product(true, self, w_self, b);
        const Tensor neigh = product(true, mean, w_neigh);
        check(apt_add_rows(out.data_ptr(), neigh.data_ptr(), out.numel(), static_cast<int>(out.element_size()), relu, stream()));
      } else {
        out = dense(self, w_self, mean, w_neigh, b, Tensor(), relu);
      }
    }
    ctx->save_for_backward({kept_if(w_neigh.requires_grad() || w_self.requires_grad(), x), kept_if(x.requires_grad(), w_neigh),
                            kept_if(x.requires_grad(), w_self), relabeled, inv, kept_if(w_neigh.requires_grad(), mean),
                            csr_indptr.value_or(Tensor()), csr_indices.value_or(Tensor()), relu ? out : Tensor()});
    ctx->saved_data["bias"] = bias.has_value() && bias->requires_grad();
    ctx->saved_data["first"] = first;
    ctx->saved_data["num_src"] = x.size(0);
    ctx->saved_data["num_dst"] = num_dst;
    ctx->saved_data["fanout"] = fanout;
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w_neigh = saved[1], &w_self = saved[2], &relabeled = saved[3], &inv = saved[4];
    const bool bias = ctx->saved_data["bias"].toBool(), first = ctx->saved_data["first"].toBool();
    const int64_t num_dst = ctx->saved_data["num_dst"].toInt(), fanout = ctx->saved_data["fanout"].toInt();
    const int64_t num_src = ctx->saved_data["num_src"].toInt();
    const auto spread = [&](const Tensor& d) {
      return aggregate_gradient(d, relabeled, num_dst, fanout, num_src, inv, saved[6], saved[7]);
    };
    const Tensor self = x.defined() ? x.narrow(0, 0, num_dst) : x;
    const bool want_x = ctx->needs_input_grad(0), want_n = ctx->needs_input_grad(1), want_s = ctx->needs_input_grad(2);
    // where the weights' gradients alone read the gradient, the ReLU's mask is applied as they do
    const bool masked = saved[8].defined() && !want_x && !(first && want_n) && !torch::GradMode::is_enabled();
    const Tensor dz = masked ? grads[0] : before_relu(grads[0], saved[8]);
    Tensor dpre, dx, dwn, dws, db;
    if (first && (want_x || want_n)) dpre = spread(dz);
    if (torch::GradMode::is_enabled()) {   // a graph of the gradients is wanted: operations that carry one
      if (want_x)
        dx = (first ? dpre.mm(w_neigh) : spread(dz.mm(w_neigh))) +
             at::constant_pad_nd(dz.mm(w_self), {0, 0, 0, num_src - num_dst});
      if (want_n)
        dwn = first ? dpre.t().mm(x)
                    : dz.t().mm(BlockAggregateFn::apply(x, relabeled, num_dst, fanout, true, std::nullopt, std::nullopt));
      if (want_s) dws = dz.t().mm(self);
      if (bias) db = dz.sum(0);
    } else {
      const Tensor relu = masked ? saved[8] : Tensor();
      std::array<WeightGrad, 2> g;
      size_t count = 0;
      if (want_s || bias) g[count++] = WeightGrad{dz, want_s ? self : Tensor(), bias, relu};
      if (want_n) g[count++] = first ? WeightGrad{dpre, x} : WeightGrad{dz, saved[5], false, relu};
      if (count > 0) weight_grads(g, count);
      if (want_s) dws = g[0].dw;
      if (bias) db = g[0].db;
      if (want_n) dwn = g[count - 1].dw;
      if (want_x)
        dx = first ? dense(dpre, w_neigh.t(), dz, w_self.t()) : [&] {
          Tensor d = spread(dense(dz, w_neigh.t()));
          dense(dz, w_self.t(), Tensor(), Tensor(), Tensor(), d.narrow(0, 0, num_dst));
          return d;
        }();
    }
    return {dx, dwn, dws, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

}  // namespace

Tensor SageLayer(const Tensor& relabeled, int64_t num_dst, int64_t fanout, const Tensor& x, const Tensor& w_neigh,
                 const Tensor& w_self, const std::optional<Tensor>& bias, const std::optional<Tensor>& csr_indptr,
                 const std::optional<Tensor>& csr_indices, bool relu) {
  check_block("sage_layer", relabeled, num_dst, fanout);
  const auto t = x.scalar_type();
  TORCH_CHECK_TYPE(x.is_cuda() && x.dim() == 2 && (t == torch::kFloat32 || t == torch::kBFloat16),
                   "npc: sage_layer: input must be a 2-D fp32 or bf16 GPU tensor");
  const auto fits = [&](const Tensor& w) {
    return w.is_cuda() && w.dim() == 2 && w.scalar_type() == t && w.size(1) == x.size(1) && w.size(0) == w_self.size(0);
  };
  TORCH_CHECK(fits(w_neigh) && fits(w_self) && x.size(1) > 0 && w_self.size(0) > 0 && num_dst <= x.size(0) &&
                  (!bias.has_value() || (bias->is_cuda() && bias->scalar_type() == t && bias->dim() == 1 &&
                                         bias->size(0) == w_self.size(0))),
              "npc: sage_layer: weights, bias and input do not fit each other");
  const bool train = trains(x, w_neigh, w_self) || (bias.has_value() && trains(*bias));
  return SageLayerFn::apply(x.contiguous(), w_neigh, w_self, bias, keepable(train, relabeled), num_dst, fanout,
                            keepable(train, csr_indptr), keepable(train, csr_indices), relu, train);
}

// ---------------------------------------------------------------- GCN layer
namespace {

// right * (sum over the block of (left * x) w) + bias, w [in, out]: the factors of the normalisation, of the rows before
// and after.  Without gradients both are one factor of the sum (a training step keeps the bits of separate operations,
// see `trains`); in the gradients they are one.  Factor, bias and ReLU are applied where the sum is stored.
struct GcnLayerFn : public torch::autograd::Function<GcnLayerFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w,
                        const std::optional<Tensor>& bias, const Tensor& relabeled, int64_t num_dst, int64_t fanout,
                        double left, double right, const std::optional<Tensor>& csr_indptr,
                        const std::optional<Tensor>& csr_indices, bool relu, bool train) {
    const Tensor b = bias.has_value() ? bias->contiguous() : Tensor();
    const bool as_mm = exact(train, x);
    const Tensor h = as_mm ? at::mm(left == 1.0 ? x : at::mul(x, left), w) : dense(x, w.t());
    const double scale = left * right;
    const Tensor out = std::get<0>(aggregate_forward(relabeled, num_dst, fanout, h, false,
                                                     static_cast<float>(as_mm ? right : scale), b, relu));
    ctx->save_for_backward({kept_if(w.requires_grad(), x), kept_if(x.requires_grad(), w), relabeled,
                            csr_indptr.value_or(Tensor()), csr_indices.value_or(Tensor()), relu ? out : Tensor()});
    ctx->saved_data["bias"] = bias.has_value() && bias->requires_grad();
    ctx->saved_data["num_src"] = x.size(0);
    ctx->saved_data["num_dst"] = num_dst;
    ctx->saved_data["fanout"] = fanout;
    ctx->saved_data["scale"] = scale;
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1];
    const Tensor dz = before_relu(grads[0], saved[5]);
    Tensor dh, dx, dw, db;
    if (ctx->needs_input_grad(0) || ctx->needs_input_grad(1))
      dh = aggregate_gradient(dz, saved[2], ctx->saved_data["num_dst"].toInt(), ctx->saved_data["fanout"].toInt(),
                              ctx->saved_data["num_src"].toInt(), Tensor(), saved[3], saved[4],
                              ctx->saved_data["scale"].toDouble());
    const bool bias = ctx->saved_data["bias"].toBool();
    if (torch::GradMode::is_enabled()) {   // a graph of the gradients is wanted: operations that carry one
      if (ctx->needs_input_grad(0)) dx = dh.mm(w.t());
      if (ctx->needs_input_grad(1)) dw = x.t().mm(dh);
      if (bias) db = dz.sum(0);
    } else {
      if (ctx->needs_input_grad(0)) dx = dense(dh, w);
      std::array<WeightGrad, 2> g;
      size_t count = 0;
      if (bias) g[count++] = WeightGrad{dz, Tensor(), true};
      if (ctx->needs_input_grad(1)) g[count++] = WeightGrad{x, dh};
      if (count > 0) weight_grads(g, count);
      if (bias) db = g[0].db;
      if (ctx->needs_input_grad(1)) dw = g[count - 1].dw;
    }
    return {dx, dw, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

}  // namespace

Tensor GcnLayer(const Tensor& relabeled, int64_t num_dst, int64_t fanout, const Tensor& x, const Tensor& w,
                const std::optional<Tensor>& bias, double left, double right, const std::optional<Tensor>& csr_indptr,
                const std::optional<Tensor>& csr_indices, bool relu) {
  check_block("gcn_layer", relabeled, num_dst, fanout);
  const auto t = x.scalar_type();
  TORCH_CHECK_TYPE(x.is_cuda() && x.dim() == 2 && (t == torch::kFloat32 || t == torch::kBFloat16),
                   "npc: gcn_layer: input must be a 2-D fp32 or bf16 GPU tensor");
  TORCH_CHECK(w.is_cuda() && w.dim() == 2 && w.scalar_type() == t && w.size(0) == x.size(1) && w.numel() > 0 &&
                  (!bias.has_value() || (bias->is_cuda() && bias->scalar_type() == t && bias->dim() == 1 &&
                                         bias->size(0) == w.size(1))),
              "npc: gcn_layer: weight, bias and input do not fit each other");
  const bool train = trains(x, w) || (bias.has_value() && trains(*bias));
  return GcnLayerFn::apply(x.contiguous(), w, bias, keepable(train, relabeled), num_dst, fanout, left, right,
                           keepable(train, csr_indptr), keepable(train, csr_indices), relu, train);
}

// ---------------------------------------------------------------- GAT layer, from the dense product to the bias
namespace {

// The layer's gradients as operations that carry a graph (create_graph): it is stated again in torch, with the slots as an
// index, and differentiated.  v: ft, attn_l, attn_r and the bias, or undefined.
torch::autograd::variable_list gat_gradients_with_graph(const std::vector<Tensor>& v, const Tensor& relabeled, int64_t num_dst,
                                                        int64_t fanout, double slope, const Tensor& d_out) {
  std::vector<Tensor> in, wanted;   // aliases: a tensor that is given twice has a gradient in each place
  for (const Tensor& t : v) {
    in.push_back(t.defined() ? t.view_as(t) : t);
    if (t.defined() && t.requires_grad()) wanted.push_back(in.back());
  }
  const int64_t n = v[0].size(0), heads = v[0].size(1), dim = v[0].size(2);
  const Tensor ids = relabeled.narrow(0, 0, num_dst * fanout).view({num_dst, fanout});
  const Tensor missing = (ids < 0).logical_or(ids >= n).unsqueeze(-1);
  const Tensor at = ids.clamp(0, std::max<int64_t>(n - 1, 0)).view(-1);
  const Tensor ft = in[0].to(torch::kFloat32);
  const Tensor el = (ft * in[1].view({heads, dim})).sum(-1), er = (ft.narrow(0, 0, num_dst) * in[2].view({heads, dim})).sum(-1);
  const Tensor e = at::leaky_relu(el.index_select(0, at).view({num_dst, fanout, heads}) + er.unsqueeze(1), slope);
  const Tensor a = at::softmax(e.masked_fill(missing, -1e30), 1).masked_fill(missing, 0);
  Tensor out = (a.unsqueeze(-1) * ft.index_select(0, at).view({num_dst, fanout, heads, dim})).sum(1).to(v[0].scalar_type());
  if (in[3].defined()) out = out + in[3].view({heads, dim});
  auto grads = torch::autograd::grad({out}, wanted, {d_out}, /*retain_graph=*/true, /*create_graph=*/true, /*allow_unused=*/true);
  torch::autograd::variable_list result(v.size());
  size_t next = 0;
  for (size_t i = 0; i < v.size(); ++i)
    if (v[i].defined() && v[i].requires_grad()) result[i] = grads[next++];
  return result;
}

struct GatLayerFn : public torch::autograd::Function<GatLayerFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& ft, const Tensor& attn_l, const Tensor& attn_r,
                        const std::optional<Tensor>& bias, const Tensor& relabeled, int64_t num_dst, int64_t fanout,
                        double slope, bool want_grad, const std::optional<Tensor>& csr_indptr,
                        const std::optional<Tensor>& csr_indices, const std::optional<Tensor>& csr_eids,
                        const std::optional<Tensor>& csc_indptr, bool relu, bool wide) {
    const int64_t n = ft.size(0), heads = ft.size(1), dim = ft.size(2);
    const auto f32 = ft.options().dtype(torch::kFloat32);
    auto scores = torch::empty({(n + num_dst) * heads}, f32);   // el, then er
    float* el = scores.data_ptr<float>();
    float* er = el + n * heads;
    auto out = torch::empty({num_dst, heads, dim}, wide ? f32 : ft.options());
    Tensor attn;
    if (want_grad) attn = torch::empty({num_dst * fanout, heads}, f32);
    Tensor b = bias.has_value() ? bias->to(out.scalar_type()).contiguous() : Tensor();
    if (!want_grad && out.scalar_type() == torch::kFloat32) {
      check(apt_gat_layer_infer(i64(relabeled), num_dst, static_cast<int>(fanout), ft.data_ptr(), n, static_cast<int>(heads), dim,
                                static_cast<int>(ft.element_size()), attn_l.data_ptr(), attn_r.data_ptr(),
                                static_cast<int>(attn_l.element_size()), b.defined() ? b.data_ptr<float>() : nullptr, relu,
                                static_cast<float>(slope), el, out.data_ptr<float>(), stream()));
      return out;
    }
    check(apt_gat_layer(i64(relabeled), num_dst, static_cast<int>(fanout), ft.data_ptr(), n, static_cast<int>(heads), dim,
                        static_cast<int>(ft.element_size()), attn_l.data_ptr(), attn_r.data_ptr(),
                        static_cast<int>(attn_l.element_size()), b.defined() ? b.data_ptr() : nullptr, relu,
                        static_cast<float>(slope), wide, el, er, out.data_ptr(), want_grad ? attn.data_ptr<float>() : nullptr,
                        stream()));
    if (want_grad) {
      const bool csr = csr_indptr.has_value() && csr_indices.has_value() && csr_eids.has_value() && csc_indptr.has_value() &&
                       csr_indptr->numel() == n + 1;
      ctx->save_for_backward({ft, attn_l, attn_r, relabeled, scores, attn, csr ? *csr_indptr : Tensor(),
                              csr ? *csr_indices : Tensor(), csr ? *csr_eids : Tensor(), csr ? *csc_indptr : Tensor(),
                              relu ? out : Tensor(), bias.value_or(Tensor())});
      ctx->saved_data["num_dst"] = num_dst;
      ctx->saved_data["fanout"] = fanout;
      ctx->saved_data["slope"] = slope;
      ctx->saved_data["bias"] = bias.has_value();
    }
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &ft = saved[0], &attn_l = saved[1], &attn_r = saved[2], &relabeled = saved[3], &scores = saved[4],
                 &attn = saved[5];
    const int64_t num_dst = ctx->saved_data["num_dst"].toInt(), fanout = ctx->saved_data["fanout"].toInt();
    const int64_t n = ft.size(0), heads = ft.size(1), dim = ft.size(2);
    const bool bias = ctx->saved_data["bias"].toBool();
    const Tensor d_out = before_relu(grads[0], saved[10]);
    if (torch::GradMode::is_enabled()) {
      auto out = gat_gradients_with_graph({ft, attn_l, attn_r, saved[11]}, relabeled, num_dst, fanout,
                                          ctx->saved_data["slope"].toDouble(), d_out);
      out.resize(15);
      return out;
    }
    SourceOrder o;
    Tensor eids, csc;
    int64_t edges = 0;
    if (saved[6].defined()) {
      eids = saved[8];
      csc = saved[9];
      o = source_order_csr(saved[6], saved[7], n, 0);
    } else if (apt_block_transpose_workspace_bytes(num_dst, static_cast<int>(fanout), n) > 0) {
      o = source_order(relabeled, num_dst, fanout, n, 0);
    } else {
      auto f = BlockFormats(relabeled, num_dst, fanout, n, true);
      csc = f[2];
      eids = f[5];
      o = source_order_csr(f[3], f[4], n, 0);
    }
    if (o.bytes == 8) edges = o.edges;
    auto d_ft = torch::empty_like(ft), d_al = torch::empty_like(attn_l), d_ar = torch::empty_like(attn_r);
    Tensor d_bias;
    if (bias) d_bias = torch::empty({heads, dim}, ft.options());
    const size_t need = apt_gat_layer_backward_workspace_bytes(num_dst, static_cast<int>(fanout), n, static_cast<int>(heads),
                                                               dim, edges);
    auto ws = torch::empty({static_cast<int64_t>(need)}, ft.options().dtype(torch::kUInt8));
    const float* el = scores.data_ptr<float>();
    check(apt_gat_layer_backward(i64(relabeled), num_dst, static_cast<int>(fanout), ft.data_ptr(), n,
                                 static_cast<int>(heads), dim, static_cast<int>(ft.element_size()), attn_l.data_ptr(),
                                 attn_r.data_ptr(), static_cast<int>(attn_l.element_size()),
                                 static_cast<float>(ctx->saved_data["slope"].toDouble()), el, el + n * heads,
                                 attn.data_ptr<float>(), d_out.data_ptr(), o.indptr, o.index, o.bytes,
                                 o.bytes == 8 ? i64(eids) : nullptr, o.bytes == 8 ? i64(csc) : nullptr, edges,
                                 o.table, d_ft.data_ptr(), d_al.data_ptr(), d_ar.data_ptr(), bias ? d_bias.data_ptr() : nullptr,
                                 ws.data_ptr(), need, stream()));
    torch::autograd::variable_list out(15);
    out[0] = d_ft;
    out[1] = d_al;
    out[2] = d_ar;
    if (bias) out[3] = d_bias;
    return out;
  }
};

}  // namespace

// ft [num_src, heads, dim] -> [num_dst, heads, dim] (apt_gat_layer), with its gradients.  attn_l, attn_r [heads, dim]
// fp32 or bf16, bias [heads, dim] (or any shape of that many elements) of ft's type.  fp32_result: of bf16 rows too, and
// nothing rounded on the way to it, if no gradient is wanted.
Tensor GatLayer(const Tensor& relabeled, int64_t num_dst, int64_t fanout, const Tensor& ft, const Tensor& attn_l,
                const Tensor& attn_r, const std::optional<Tensor>& bias, double slope,
                const std::optional<Tensor>& csr_indptr, const std::optional<Tensor>& csr_indices,
                const std::optional<Tensor>& csr_eids, const std::optional<Tensor>& csc_indptr, bool relu, bool fp32_result) {
  check_block("gat_layer", relabeled, num_dst, fanout);
  const auto good = [](const Tensor& t) {
    return t.is_cuda() && (t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kBFloat16);
  };
  TORCH_CHECK_TYPE(good(ft) && ft.dim() == 3, "npc: gat_layer: ft must be a [num_src, heads, dim] fp32 or bf16 GPU tensor");
  TORCH_CHECK_TYPE(good(attn_l) && attn_r.scalar_type() == attn_l.scalar_type() && attn_r.is_cuda(),
                   "npc: gat_layer: attn_l and attn_r must be fp32 or bf16 GPU tensors of one type");
  TORCH_CHECK(attn_l.numel() == ft.size(1) * ft.size(2) && attn_r.numel() == attn_l.numel() && num_dst <= ft.size(0),
              "npc: gat_layer: attn_l / attn_r must be [heads, dim], num_dst at most num_src");
  std::optional<Tensor> b = bias;
  if (b.has_value()) {
    TORCH_CHECK(b->is_cuda() && b->scalar_type() == ft.scalar_type() && b->numel() == ft.size(1) * ft.size(2),
                "npc: gat_layer: bias must have heads * dim elements of ft's type");
    b = b->reshape({ft.size(1), ft.size(2)});
  }
  const bool want_grad = torch::GradMode::is_enabled() && (ft.requires_grad() || attn_l.requires_grad() || attn_r.requires_grad() ||
                                                          (b.has_value() && b->requires_grad()));
  return GatLayerFn::apply(ft.contiguous(), attn_l.contiguous(), attn_r.contiguous(), b, keepable(want_grad, relabeled), num_dst, fanout,
                           slope, want_grad, keepable(want_grad, csr_indptr), keepable(want_grad, csr_indices),
                           keepable(want_grad, csr_eids), keepable(want_grad, csc_indptr), relu,
                           fp32_result && !want_grad && ft.scalar_type() == torch::kBFloat16);
}

// ---------------------------------------------------------------- peers only
#define NPC_NEEDS_PEERS(name)                                                              \
  TORCH_CHECK(false, "npc." name " talks to other GPUs over NCCL in the reference; this " \
                     "library builds one GPU's share only")

Tensor NCCLGetUniqueId() { NPC_NEEDS_PEERS("nccl_get_unique_id"); }
void Initialize(IdType, IdType, IdType, Tensor, IdType) { NPC_NEEDS_PEERS("init"); }
void AlltoAll(Tensor, Tensor, Tensor, Tensor, IdType, IdType) { NPC_NEEDS_PEERS("alltoall"); }
Tensor CrossMachineLoadSubtensor(Tensor) { NPC_NEEDS_PEERS("crossmachine_load_subtensor"); }
std::vector<Tensor> NPSampleAndShuffle(Tensor, IdType) { NPC_NEEDS_PEERS("np_sample_and_shuffle"); }
std::vector<Tensor> SPSampleAndShuffle(IdType, Tensor, Tensor, Tensor, IdType) {
  NPC_NEEDS_PEERS("sp_sample_and_shuffle");
}
std::vector<Tensor> SPSampleShuffleSrc(Tensor) { NPC_NEEDS_PEERS("sp_sample_shuffle_src"); }
std::vector<Tensor> MPSampleShuffle(Tensor, Tensor, Tensor) { NPC_NEEDS_PEERS("mp_sample_shuffle"); }
Tensor SPFeatShuffle(Tensor, Tensor, Tensor, IdType, IdType, IdType) { NPC_NEEDS_PEERS("sp_feat_shuffle"); }
Tensor MPFeatShuffleFwd(Tensor, Tensor, Tensor, IdType) { NPC_NEEDS_PEERS("mp_feat_shuffle_fwd"); }
Tensor MPFeatShuffleBwd(Tensor, Tensor, Tensor, IdType) { NPC_NEEDS_PEERS("mp_feat_shuffle_bwd"); }

TORCH_LIBRARY(npc, m) {
  // same names and order as the reference's src/pybind.cc:18-48
  m.def("nccl_get_unique_id", &NCCLGetUniqueId)
      .def("init", &Initialize)
      .def("alltoall", &AlltoAll)
      .def("cache_feats_shared", &CacheFeatsShared)
      .def("mix_cache_graphs", &MixCacheGraphs)
      .def("register_min_vids", &RegisterMinVids)
      .def("register_multi_machines_scheme", &RegisterMultiMachinesScheme)
      .def("cpu_load_subtensor", &CPULoadSubtensor)
      .def("load_subtensor", &LoadSubtensor)
      .def("crossmachine_load_subtensor", &CrossMachineLoadSubtensor)
      .def("cluster_reqs", &ClusterReqs)
      .def("local_sample_one_layer", &LocalSamplingNeibhorsOneLayer)
      .def("srcdst_to_vir", &SrcDsttoVir)
      .def("src_to_vir", &SrcToVir)
      .def("np_sample_and_shuffle", &NPSampleAndShuffle)
      .def("sp_sample_and_shuffle", &SPSampleAndShuffle)
      .def("sp_sample_shuffle_src", &SPSampleShuffleSrc)
      .def("mp_sample_shuffle", &MPSampleShuffle)
      .def("feat_shuffle", &FeatShuffle)
      .def("sp_feat_shuffle", &SPFeatShuffle)
      .def("mp_feat_shuffle_fwd", &MPFeatShuffleFwd)
      .def("mp_feat_shuffle_bwd", &MPFeatShuffleBwd)
      .def("shuffle_seeds", &ShuffleSeeds)
      .def("relabel_csc", &RelabelCSC)
      .def("spmm_copy_u_sum", &CopyUSum)
      .def("spmm_copy_e_sum", &CopyESum)
      .def("spmm_u_mul_e_sum", &UMulESum)
      .def("sddmm_u_add_v", &UAddV)
      .def("sddmm_u_mul_v", &UMulV)
      // additions (no counterpart in the reference)
      .def("sample_neighbors", &SampleNeighbors)
      .def("sample_blocks", &SampleBlocks)
      .def("block_formats", &BlockFormats)
      .def("block_linear", &BlockLinear)
      .def("block_aggregate", &BlockAggregate)
      .def("sage_layer(Tensor relabeled, int num_dst, int fanout, Tensor x, Tensor w_neigh, Tensor w_self, Tensor? bias, "
           "Tensor? csr_indptr, Tensor? csr_indices, bool relu=False) -> Tensor", &SageLayer)
      .def("gcn_layer(Tensor relabeled, int num_dst, int fanout, Tensor x, Tensor w, Tensor? bias, float left, float right, "
           "Tensor? csr_indptr, Tensor? csr_indices, bool relu=False) -> Tensor", &GcnLayer)
      .def("gat_layer(Tensor relabeled, int num_dst, int fanout, Tensor ft, Tensor attn_l, Tensor attn_r, Tensor? bias, "
           "float slope, Tensor? csr_indptr, Tensor? csr_indices, Tensor? csr_eids, Tensor? csc_indptr, bool relu=False, "
           "bool fp32_result=False) -> Tensor", &GatLayer)
      .def("cluster_and_permute", &ClusterAndPermuteLocal)
      .def("register_graph_partition", &RegisterGraphPartition)
      .def("set_topology", &SetTopology)
      .def("set_rng_seed", &SetRngSeed)
      .def("set_strict", &SetStrict)
      .def("set_miss_check", &SetMissCheck)
      .def("check_errors", &CheckErrors)
      .def("set_ranked_relabel", &SetRankedRelabel)
      .def("set_block_buffer_ring", &SetBlockBufferRing)
      .def("block_buffer_ring", &BlockBufferRing);
}

}  // namespace npc
