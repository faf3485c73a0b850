// gs::HeteroGraph -- a set of relation graphs keyed by edge type, with the
// fused metapath random walk (API of the reference's src/hetero_graph.h:36-66).
#pragma once

#include <torch/custom_class.h>
#include <torch/script.h>

#include <array>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "graph.h"

namespace gs {

class HeteroGraph : public torch::CustomClassHolder {
 public:
  HeteroGraph() {}

  // edge_types[i] = (source node type, edge type, destination node type); the
  // middle string is the key a metapath refers to; edge_relations[i] holds the
  // CSC of relation i.
  void LoadFromHomo(
      const std::vector<std::string>& node_types,
      const std::vector<std::tuple<std::string, std::string, std::string>>& edge_types,
      const std::vector<c10::intrusive_ptr<Graph>>& edge_relations);

  c10::intrusive_ptr<Graph> GetHomoGraph(const std::string& edge_type) const;

  // One walker per seed, step t follows relation metapath[t].  Returns the flat
  // [len(metapath)+1][n] trace with shape [n, len(metapath)+1].
  torch::Tensor MetapathRandomWalkFused(torch::Tensor seeds,
                                        const std::vector<std::string>& metapath);

 private:
  std::map<std::string, int64_t> node_type_id_, edge_type_id_;
  std::vector<c10::intrusive_ptr<Graph>> relations_;
  // of every relation: the addresses of its indptr and its indices, and its columns
  std::vector<std::array<int64_t, 3>> tables_;
  torch::Device device_ = torch::kCPU;
  int id_bytes_ = 8;
  // A metapath on the GPU, with the tables of the relations that it takes
  struct Path {
    torch::Tensor steps, indptr, indices, sizes;
    int64_t num_nodes = 0;  // of its relations together
  };
  // (in one copy: the steps, then three columns of the relations' tables)
  Path Upload(std::vector<int64_t> steps, const std::vector<int64_t>& relations) const;
  // Every relation's tables, uploaded when the graph is loaded (no steps): a path that takes all of them
  // goes up alone.  With the tables in the path's copy, a new graph's first walk, 13 k walkers of four steps, took
  // 78-88 us for 57, a third of it the first small copy after the load.
  Path all_;
  // metapaths already uploaded (the reference re-uploads on every call, src/hetero_graph.cc:66-69)
  std::map<std::vector<std::string>, Path> metapath_cache_;
};

}  // namespace gs
