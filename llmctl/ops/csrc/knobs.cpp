// Native side of llmctl.config.knobs: kernel-selection knobs the HIP launchers consult
// (flash-attention split / priority / wave count, dK/dV schedule, decode splits, decode skinny
// GEMM version).  Python pushes the resolved PerfKnobs here once (llmctl.config.knobs.apply);
// a launcher reads knob("name", default) -- no environment lookups on the hot path.
#include <hip/hip_runtime_api.h>
#include <torch/library.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace llmctl {
namespace {
std::mutex& mu() {
  static std::mutex m;
  return m;
}
std::map<std::string, int64_t>& table() {
  static std::map<std::string, int64_t> t;
  return t;
}
}  // namespace

int64_t knob(const char* name, int64_t dflt) {
  std::lock_guard<std::mutex> lk(mu());
  auto it = table().find(name);
  return it == table().end() ? dflt : it->second;
}

void set_knob(const std::string& name, int64_t value) {
  std::lock_guard<std::mutex> lk(mu());
  table()[name] = value;
}

void clear_knobs() {
  std::lock_guard<std::mutex> lk(mu());
  table().clear();
}

// Memset nodes of a recorded graph (a hipGraph_t as an integer): library calls record them too, and on this part they have given wrong results on
// replays after the first, so a caller that finds any runs its calls eagerly.
int64_t graph_memsets(int64_t graph) {
  const hipGraph_t g = reinterpret_cast<hipGraph_t>(static_cast<uintptr_t>(graph));
  size_t n = 0;
  TORCH_CHECK(g != nullptr && hipGraphGetNodes(g, nullptr, &n) == hipSuccess, "llmctl: graph_memsets: not a recorded graph");
  std::vector<hipGraphNode_t> nodes(n);
  TORCH_CHECK(n == 0 || hipGraphGetNodes(g, nodes.data(), &n) == hipSuccess, "llmctl: graph_memsets: nodes");
  int64_t found = 0;
  for (hipGraphNode_t node : nodes) {
    hipGraphNodeType type;
    TORCH_CHECK(hipGraphNodeGetType(node, &type) == hipSuccess, "llmctl: graph_memsets: node type");
    found += type == hipGraphNodeTypeMemset;
  }
  return found;
}
}  // namespace llmctl
