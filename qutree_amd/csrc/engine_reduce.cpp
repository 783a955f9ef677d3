// Which matrices a compressed sweep forms.
//
// Apply (and the gradient's mean fields) use most h-matrices and holes only
// inside coefficient-weighted sums: at a node the terms that lie wholly below
// a child enter as ONE matrix sum_l c_l h_l, and a factor x_i inside the node
// meets the outside only as ONE mean field sum_j c_ij hole_j.  Such a sum is
// itself a contraction at the node: with h_l = <A| h_l(c0) x h_l(c1) |A> it is
//     sum_l c_l h_l = sum_g <A| F_g x G_g |A>,
// where the terms that agree in one factor are merged into a group whose
// other factor is a sum again, one level further down (h-matrices) or up
// (holes).  For pair couplings over l modes below a node that is l / 2 + 2
// groups in place of l (l + 1) / 2 matrices and their combination; for the
// mean field of one mode two groups in place of a hole per outside mode.
//
// The choice is made per node and kind, from what is asked of it: a matrix
// wanted by itself is formed by itself; the sums whose matrices are wanted by
// nothing else are formed as such when that takes fewer contractions.  Sums of
// matrices that exist anyway are combined (combine_kernel).
//
// Order on the device: the single h-matrices bottom-up beside the density
// tree; one combination launch for the sums of them; then layer by layer,
// top-down, the holes and mean fields, and beside them, bottom-up, the summed
// h-matrices (which no hole reads); the combinations of holes; Apply.
//
// Per-term matrices that no sum needs are not formed in a sweep;
// qtg_engine_get_matrix forms them when it is asked for one (term_engine).
#include <algorithm>
#include <map>

#include "engine.hpp"

namespace qtg {

namespace {
// terms with equal matrix merged, ordered by matrix
std::vector<std::pair<int64_t, cd>> merged(const std::vector<std::pair<int64_t, cd>>& t) {
  std::map<int64_t, cd> m;
  for (auto& x : t) m[x.first] += x.second;
  return std::vector<std::pair<int64_t, cd>>(m.begin(), m.end());
}
}  // namespace

// The greedy merge of aggregate(), without forming anything: summands that
// agree on every slot but `fs` (largest group first) with their weighted
// list of matrices on that slot.
std::vector<Engine::Group> Engine::merge_groups(const std::vector<Summand>& tl, int S) const {
  std::vector<Group> out;
  std::vector<char> alive(tl.size(), 1);
  size_t nalive = tl.size();
  while (nalive > 1) {
    int best_s = -1;
    std::vector<int> best;
    for (int sl = 0; sl < S; ++sl) {
      std::map<std::vector<int64_t>, std::vector<int>> gm;
      for (size_t t = 0; t < tl.size(); ++t) {
        if (!alive[t]) continue;
        std::vector<int64_t> k = tl[t].ids;
        k.erase(k.begin() + sl);
        gm[k].push_back((int)t);
      }
      for (auto& kv : gm)
        if (kv.second.size() > std::max<size_t>(1, best.size())) {
          best = kv.second;
          best_s = sl;
        }
    }
    if (best_s < 0) break;
    Group g;
    g.ids = tl[best[0]].ids;
    g.fs = best_s;
    std::vector<std::pair<int64_t, cd>> terms;
    for (int t : best) {
      terms.push_back({tl[t].ids[best_s], tl[t].coef});
      alive[t] = 0;
      --nalive;
    }
    g.terms = merged(terms);
    if (g.terms.size() == 1) {  // one matrix after all
      g.ids[best_s] = g.terms[0].first;
      g.coef = g.terms[0].second;
      g.fs = -1;
      g.terms.clear();
    }
    out.push_back(g);
  }
  for (size_t t = 0; t < tl.size(); ++t)
    if (alive[t]) {
      Group g;
      g.ids = tl[t].ids;
      g.coef = tl[t].coef;
      out.push_back(g);
    }
  return out;
}

int Engine::matrix_sum(const SlotRef& slot, int d, const std::vector<std::pair<int64_t, cd>>& terms, int64_t& off) {
  auto key = std::make_tuple(slot.node, (int)slot.kind, std::vector<std::pair<int64_t, std::pair<double, double>>>());
  for (auto& t : terms) std::get<2>(key).push_back({t.first, {t.second.real(), t.second.imag()}});
  auto f = sumKey_.find(key);
  if (f != sumKey_.end()) return f->second;
  MatSum s;
  s.slot = slot;
  s.d = d;
  s.terms = terms;
  s.out = off;
  off += (int64_t)d * d;
  for (auto& t : terms)
    if (t.first >= 0 && highSlots_.count(t.first)) highSlots_.insert(s.out);
  sums_.push_back(s);
  sumOf_[s.out] = (int)sums_.size() - 1;
  return sumKey_[key] = (int)sums_.size() - 1;
}

std::vector<Engine::Summand> Engine::take_groups(const std::vector<Group>& groups, const std::vector<SlotRef>& slots,
                                                 const std::vector<int>& sdim, int64_t& off) {
  std::vector<Summand> out;
  for (const Group& g : groups) {
    Summand s;
    s.coef = g.coef;
    s.ids = g.ids;
    if (g.fs >= 0) {
      s.ids[g.fs] = sums_[matrix_sum(slots[g.fs], sdim[g.fs], g.terms, off)].out;
      s.coef = cd(1.0, 0.0);
    }
    out.push_back(s);
  }
  return out;
}

std::vector<Engine::SlotRef> Engine::node_slots(const HNode& v, std::vector<int>& sdim) const {
  std::vector<SlotRef> s;
  sdim.clear();
  if (v.bottom) {
    s.push_back({v.addr, SlotRef::LEAF});
    sdim.push_back(v.dims[0]);
  } else {
    for (int c : v.children) {
      s.push_back({c, SlotRef::H});
      sdim.push_back(tree_.nodes[c].n);
    }
  }
  if (!v.top()) {
    s.push_back({v.addr, SlotRef::HOLE});
    sdim.push_back(v.n);
  }
  return s;
}

void Engine::want(const SlotRef& slot, int64_t id, bool early, bool hard) {
  if (id < 0 || slot.kind == SlotRef::LEAF) return;
  auto f = sumOf_.find(id);
  if (f == sumOf_.end()) {
    (slot.kind == SlotRef::H ? hWant_ : qWant_)[slot.node].single.insert(id);
    return;
  }
  MatSum& s = sums_[f->second];
  s.early |= early;
  s.hard |= hard;
  (slot.kind == SlotRef::H ? hWant_ : qWant_)[slot.node].sums.insert(f->second);
}

// Chooses, for every node, the single matrices and the summed ones that the
// wanted Apply and gradient summands need: hWant_ and qWant_ (by which plan()
// keeps items of h_items_), fused_ (summed contractions) and the combinations
// h_combA_ (sums of h-matrices) and h_comb1_ (sums of holes).
void Engine::reduce_plan(const std::vector<std::vector<std::pair<int64_t, int>>>& hent,
                         const std::vector<std::vector<std::pair<int64_t, int>>>& qent, int64_t& off) {
  const int NN = (int)tree_.nodes.size();
  std::vector<std::map<int64_t, int>> hrep(NN), qrep(NN);
  for (int a = 0; a < NN; ++a) {
    for (auto& e : hent[a]) hrep[a][e.first] = e.second;
    for (auto& e : qent[a]) qrep[a][e.first] = e.second;
  }
  auto leafmat = [&](int l, int mode) -> int64_t {
    for (auto& lm : sop_.terms[l].leafmats)
      if (lm.first == mode) return leafOff_[lm.second];
    return -1;
  };
  // what Apply and the gradient ask for
  std::vector<int> sdim;
  for (auto& v : tree_.nodes) {
    const auto slots = node_slots(v, sdim);
    for (auto& s : summ_[v.addr])
      for (size_t i = 0; i < slots.size(); ++i) want(slots[i], s.ids[i], false, false);
    if (v.top() || gsumm_.empty()) continue;
    const HNode& p = tree_.nodes[v.parent];
    const auto ps = node_slots(p, sdim);
    for (auto& s : gsumm_[v.addr])
      for (size_t i = 0; i < ps.size(); ++i) want(ps[i], s.ids[i], false, false);
  }
  fused_.clear();
  std::vector<int> byDepth(NN);
  for (int a = 0; a < NN; ++a) byDepth[a] = a;
  std::stable_sort(byDepth.begin(), byDepth.end(),
                   [&](int a, int b) { return tree_.nodes[a].depth < tree_.nodes[b].depth; });
  // ---- holes, deepest first: a node's children have said what they need of it
  for (int i = NN - 1; i >= 0; --i) {
    const HNode& v = tree_.nodes[byDepth[i]];
    if (v.top()) continue;
    const HNode& p = tree_.nodes[v.parent];
    Want& w = qWant_[v.addr];
    std::vector<SlotRef> slots;
    std::vector<int> dims;
    for (int c : p.children)
      if (c != v.addr) {
        slots.push_back({c, SlotRef::H});
        dims.push_back(tree_.nodes[c].n);
      }
    if (!p.top()) {
      slots.push_back({p.addr, SlotRef::HOLE});
      dims.push_back(p.n);
    }
    // the summand of one hole matrix at the parent
    auto factors = [&](int64_t atom) {
      const int l = qrep[v.addr].at(atom);
      Summand t;
      for (int c : p.children)
        if (c != v.addr) t.ids.push_back(l >= 0 && active_[l][c] ? hslot_[l][c] : -1);
      if (!p.top()) t.ids.push_back(l >= 0 ? holeslot_[l][p.addr] : rhoslot_[p.addr]);
      return t;
    };
    std::set<int64_t> have = w.single;
    have.insert(rhoslot_[v.addr]);
    std::set<int64_t> extra;
    std::vector<std::vector<Group>> gs;
    std::vector<int> cand;
    size_t ngroups = 0;
    bool hard = false;
    for (int si : w.sums) {
      const MatSum& s = sums_[si];
      hard |= s.hard;
      std::vector<Summand> tl;
      for (auto& t : s.terms) {
        Summand x = factors(t.first);
        x.coef = t.second;
        tl.push_back(x);
        if (!have.count(t.first)) extra.insert(t.first);
      }
      gs.push_back(merge_groups(tl, (int)slots.size()));
      cand.push_back(si);
      ngroups += gs.back().size();
    }
    if (!cand.empty() && (hard || ngroups <= extra.size())) {
      for (size_t k = 0; k < cand.size(); ++k) {
        sums_[cand[k]].fused = true;
        Fused f;
        f.node = p.addr;
        f.k = v.childIdx;
        f.out = sums_[cand[k]].out;
        f.level = v.depth;
        f.slots = slots;
        f.groups = take_groups(gs[k], slots, dims, off);
        for (auto& g : f.groups)
          for (size_t q = 0; q < slots.size(); ++q) want(slots[q], g.ids[q], true, true);
        fused_.push_back(f);
      }
    } else {
      w.single.insert(extra.begin(), extra.end());
    }
    for (int64_t a : w.single) {
      const Summand t = factors(a);
      for (size_t q = 0; q < slots.size(); ++q) want(slots[q], t.ids[q], true, true);
    }
  }
  // ---- h-matrices, top-down
  for (int i = 0; i < NN; ++i) {
    const HNode& c = tree_.nodes[byDepth[i]];
    if (c.top()) continue;
    Want& w = hWant_[c.addr];
    std::vector<int> dims;
    std::vector<SlotRef> slots = node_slots(c, dims);
    slots.pop_back();  // the node's own hole: not a factor of its h-matrices
    auto factors = [&](int64_t atom) {
      const int l = hrep[c.addr].at(atom);
      Summand t;
      if (c.bottom) t.ids.push_back(leafmat(l, c.leaf.mode));
      else
        for (int ch : c.children) t.ids.push_back(active_[l][ch] ? hslot_[l][ch] : -1);
      return t;
    };
    // sums that a hole reads come from single matrices
    for (int si : w.sums)
      if (sums_[si].early || c.bottom)
        for (auto& t : sums_[si].terms)
          if (t.first >= 0) w.single.insert(t.first);
    std::set<int64_t> extra;
    std::vector<std::vector<Group>> gs;
    std::vector<int> cand;
    size_t ngroups = 0;
    for (int si : w.sums) {
      const MatSum& s = sums_[si];
      std::set<int64_t> need;
      bool ident = false;
      for (auto& t : s.terms) {
        ident |= t.first < 0;
        if (t.first >= 0 && !w.single.count(t.first)) need.insert(t.first);
      }
      if (ident) w.single.insert(need.begin(), need.end());  // a sum with the identity is combined
      if (ident || need.empty()) continue;
      extra.insert(need.begin(), need.end());
      std::vector<Summand> tl;
      for (auto& t : s.terms) {
        Summand x = factors(t.first);
        x.coef = t.second;
        tl.push_back(x);
      }
      gs.push_back(merge_groups(tl, (int)slots.size()));
      cand.push_back(si);
      ngroups += gs.back().size();
    }
    if (!cand.empty() && ngroups <= extra.size()) {
      for (size_t k = 0; k < cand.size(); ++k) {
        sums_[cand[k]].fused = true;
        Fused f;
        f.node = c.addr;
        f.k = c.order() - 1;
        f.out = sums_[cand[k]].out;
        f.slots = slots;
        f.groups = take_groups(gs[k], slots, dims, off);
        f.d = sums_[cand[k]].d;
        for (auto& g : f.groups)
          for (size_t q = 0; q < slots.size(); ++q) want(slots[q], g.ids[q], false, false);
        fused_.push_back(f);
      }
    } else {
      w.single.insert(extra.begin(), extra.end());
    }
    for (int64_t a : w.single) {
      const Summand t = factors(a);
      for (size_t q = 0; q < slots.size(); ++q) want(slots[q], t.ids[q], true, false);
    }
  }
  // ---- levels of the summed h-matrices: one above the summed ones they
  // read.  The groups that read none (the couplings across the node's own
  // children, most of the work) are formed for all nodes in the first layer
  // and added to the short rest, so the chain from layer to layer is two
  // groups long.
  std::map<int64_t, int> lev;
  std::vector<Fused> parts;
  for (int i = NN - 1; i >= 0; --i)
    for (auto& f : fused_) {
      if (f.node != byDepth[i] || f.level > 0) continue;
      f.level = 1;
      std::vector<Summand> first, chain;
      for (auto& g : f.groups) {
        int l = 0;
        for (size_t q = 0; q < f.slots.size(); ++q) {
          auto x = lev.find(g.ids[q]);
          if (x != lev.end()) l = std::max(l, x->second);
        }
        f.level = std::max(f.level, l + 1);
        (l > 0 ? chain : first).push_back(g);
      }
      if (!chain.empty() && !first.empty()) {
        Fused part = f;
        part.level = 1;
        part.groups = first;
        part.out = off;
        off += (int64_t)f.d * f.d;
        if (highSlots_.count(f.out)) highSlots_.insert(part.out);
        f.groups = chain;
        f.add = part.out;
        parts.push_back(part);
      }
      lev[f.out] = f.level;
    }
  fused_.insert(fused_.end(), parts.begin(), parts.end());
  // ---- combinations of the sums that are not formed as such; sums of leaf
  // operators are constants
  h_combA_.clear();
  h_combtA_.clear();
  leafSums_.clear();
  for (const MatSum& s : sums_) {
    if (s.fused) continue;
    if (s.slot.kind == SlotRef::LEAF) {
      std::vector<cd> m((size_t)s.d * s.d, 0.0);
      for (auto& t : s.terms) {
        if (t.first < 0) {
          for (int k = 0; k < s.d; ++k) m[k + (size_t)k * s.d] += t.second;
          continue;
        }
        const size_t li = std::find(leafOff_.begin(), leafOff_.end(), t.first) - leafOff_.begin();
        for (size_t e = 0; e < m.size(); ++e) m[e] += t.second * sop_.leafMatrices[li][e];
      }
      leafSums_.push_back({s.out, m});
      continue;
    }
    const bool h = s.slot.kind == SlotRef::H;
    std::vector<CombOut>& co = h ? h_combA_ : h_comb1_;
    std::vector<CombTerm>& ct = h ? h_combtA_ : h_combt1_;
    CombOut o{};
    o.out = s.out;
    o.n = s.d;
    o.t0 = (int32_t)ct.size();
    for (auto& t : s.terms) ct.push_back({t.second.real(), t.second.imag(), t.first});
    o.t1 = (int32_t)ct.size();
    co.push_back(o);
  }
}

}  // namespace qtg
