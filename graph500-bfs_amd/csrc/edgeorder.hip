// edgeorder.hip -- when a graph's edges are ordered for the validator, and when
// the order goes again (order_edges makes it, validate.hip uses it; host code).
//
// The order is a copy of the edges that only saves time, so it is made for a
// graph's second pass over its edges, once, is done without where there is no
// room for it, and is given up, for good, to an allocation that would fail.
#include <algorithm>
#include <new>

#include "internal.hpp"

namespace g500 {

namespace {

// Graphs that hold an order.  Never destroyed: handles may be released by
// destructors that run after those of this file.
struct Holders {
  std::mutex mu;
  std::vector<g500_graph*> graphs;
};
Holders& holders() {
  static Holders* h = new Holders;
  return *h;
}

}  // namespace

std::shared_ptr<const OrderedEdges> held_order(g500_graph* g) {
  std::lock_guard<std::mutex> lock(g->order_mu);
  return g->ordered;
}

std::shared_ptr<const OrderedEdges> order_for_pass(g500_graph* g, hipStream_t s) {
  {
    std::lock_guard<std::mutex> lock(g->order_mu);
    if (g->edge_passes++ == 0 || g->order_tried) return g->ordered;
    g->order_tried = true;
  }
  std::shared_ptr<const OrderedEdges> order;
  try {
    order = order_edges(g, s);
  } catch (const Error& e) {
    if (e.code != G500_ERR_NOMEM) throw;
  } catch (const std::bad_alloc&) {
  }
  if (order) {
    Holders& h = holders();
    std::lock_guard<std::mutex> lock(h.mu);
    h.graphs.push_back(g);
    std::lock_guard<std::mutex> glock(g->order_mu);
    g->ordered = order;
  }
  return order;
}

void forget_ordered_edges(g500_graph* g) {
  Holders& h = holders();
  std::lock_guard<std::mutex> lock(h.mu);
  h.graphs.erase(std::remove(h.graphs.begin(), h.graphs.end(), g), h.graphs.end());
}

void drop_ordered_edges(int device) {
  std::vector<std::shared_ptr<const OrderedEdges>> dropped;  // released without the locks
  Holders& h = holders();
  std::lock_guard<std::mutex> lock(h.mu);
  for (size_t i = 0; i < h.graphs.size();) {
    g500_graph* g = h.graphs[i];
    std::lock_guard<std::mutex> glock(g->order_mu);
    // a validation that uses it holds a reference, and can only get one here
    if (g->device != device || g->ordered.use_count() != 1) {
      ++i;
      continue;
    }
    dropped.push_back(std::move(g->ordered));
    h.graphs.erase(h.graphs.begin() + (ptrdiff_t)i);
  }
}

}  // namespace g500
