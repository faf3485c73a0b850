#include "hetero_graph.h"

#include <algorithm>
#include <numeric>

#include "range.h"

#include "hip_ops.h"

namespace gs {

void HeteroGraph::LoadFromHomo(
    const std::vector<std::string>& node_types,
    const std::vector<std::tuple<std::string, std::string, std::string>>& edge_types,
    const std::vector<c10::intrusive_ptr<Graph>>& edge_relations) {
  TORCH_CHECK(edge_types.size() == edge_relations.size(),
              "one relation graph per edge type is required");
  node_type_id_.clear();
  edge_type_id_.clear();
  relations_ = edge_relations;
  metapath_cache_.clear();
  for (size_t i = 0; i < node_types.size(); ++i) node_type_id_[node_types[i]] = static_cast<int64_t>(i);
  tables_.clear();
  for (size_t i = 0; i < edge_types.size(); ++i) {
    edge_type_id_[std::get<1>(edge_types[i])] = static_cast<int64_t>(i);
    auto csc = edge_relations[i]->GetCSC();
    TORCH_CHECK(csc != nullptr, "relation ", std::get<1>(edge_types[i]), " has no CSC format");
    TORCH_CHECK(csc->indptr.is_cuda() && csc->indices.is_cuda(),
                "Not implemented warning: relation graphs must live on the GPU");
    const int idb = csc->indices.scalar_type() == torch::kInt32 ? 4 : 8;
    if (i == 0) id_bytes_ = idb;
    TORCH_CHECK(idb == id_bytes_, "relation graphs differ in id dtype");
    tables_.push_back({reinterpret_cast<int64_t>(csc->indptr.data_ptr()),
                       reinterpret_cast<int64_t>(csc->indices.data_ptr()), csc->indptr.numel() - 1});
    device_ = csc->indptr.device();
  }
  std::vector<int64_t> all(tables_.size());
  std::iota(all.begin(), all.end(), 0);
  all_ = Path();
  if (!all.empty()) all_ = Upload({}, all);
}

HeteroGraph::Path HeteroGraph::Upload(std::vector<int64_t> values, const std::vector<int64_t>& relations) const {
  const int64_t length = static_cast<int64_t>(values.size()), R = static_cast<int64_t>(relations.size());
  Path path;
  for (int k = 0; k < 3; ++k)
    for (int64_t r : relations) values.push_back(tables_[r][k]);
  for (int64_t r : relations) path.num_nodes += tables_[r][2];
  auto all = torch::tensor(values, torch::dtype(torch::kInt64)).to(device_);
  path.steps = all.narrow(0, 0, length);
  path.indptr = all.narrow(0, length, R);
  path.indices = all.narrow(0, length + R, R);
  path.sizes = all.narrow(0, length + 2 * R, R);
  return path;
}

c10::intrusive_ptr<Graph> HeteroGraph::GetHomoGraph(const std::string& edge_type) const {
  auto it = edge_type_id_.find(edge_type);
  TORCH_CHECK(it != edge_type_id_.end(), "unknown edge type ", edge_type);
  return relations_[it->second];
}

torch::Tensor HeteroGraph::MetapathRandomWalkFused(torch::Tensor seeds,
                                                   const std::vector<std::string>& metapath) {
  Range range("gs::MetapathRandomWalk");
  auto cached = metapath_cache_.find(metapath);
  if (cached == metapath_cache_.end()) {
    // the relations that the path takes, in the order in which it meets them (their offsets are what a
    // walk may pack, and another large relation is none of its business)
    std::vector<int64_t> used, steps;
    for (const auto& name : metapath) {
      auto it = edge_type_id_.find(name);
      TORCH_CHECK(it != edge_type_id_.end(), "unknown edge type ", name, " in metapath");
      auto at = std::find(used.begin(), used.end(), it->second);
      steps.push_back(at - used.begin());
      if (at == used.end()) used.push_back(it->second);
    }
    Path path;
    if (used.size() == tables_.size()) {  // (all: their tables are there, and only the steps go up)
      for (int64_t& step : steps) step = used[step];
      path = all_;
      path.steps = torch::tensor(steps, torch::dtype(torch::kInt64)).to(device_);
    } else {
      path = Upload(std::move(steps), used);
    }
    cached = metapath_cache_.emplace(metapath, path).first;
  }
  const Path& path = cached->second;
  return hip::MetapathWalk(seeds, path.steps, path.indptr, path.indices, path.sizes, path.num_nodes, id_bytes_)
      .reshape({seeds.numel(), -1});
}

}  // namespace gs
