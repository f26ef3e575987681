// gfx950 memory passes, what the target compiler may assume about pointers: distinct arrays, read-only parameters.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

// ================================================================ pointers that change places while the kernel runs
// `for t: src = a; dst = b; if (t & 1) { src = b; dst = a; } <step>` on arrays in memory: within a step nothing is stored to
// what `src` names, and the device compiler takes that for all steps: it reads an element that all threads read, or a single
// thread behind a test, by a scalar load.  The scalar cache does not see vector stores, and the element is that of an earlier
// step.  (`s[i, 5]` in a step that also reduces the row, 2 rows of 2051 floats; `s[i, 4 j % 2051]` for j = 2049, which only
// thread 0 of 512 has.)  The pointers get an offset of zero from a vector register, with which no address is the same for
// all threads as far as the compiler knows.  Arrays in LDS and loops on the host are not concerned.
Stmts Pass::swapped_pointers(const Stmts& ss0) {
  auto in_memory = [](const Type& t) { return is_alias_type(t) && t.mem != Mem::LDS; };
  std::function<Stmts(const Stmts&, bool, bool)> walk = [&](const Stmts& ss, bool in_loop, bool loop_body) {
    std::set<Name> here, inside;       // pointers declared by these statements, and anywhere in them
    std::map<Name, size_t> last;       // the last of these statements that sets a pointer
    for (size_t i = 0; in_loop && i < ss.size(); ++i) {
      if (ss[i]->k == Stmt::Def) here.insert(ss[i]->id);
      visit_stmts({ss[i]}, [&](const S& c) { if (c->k == Stmt::Def) inside.insert(c->id); });
      if (ss[i]->k == Stmt::For || ss[i]->k == Stmt::While) continue;
      visit_stmts({ss[i]}, [&](const S& c) {
        if (c->k == Stmt::Assign && c->dst->k == Expr::Var && in_memory(c->dst->ty)) last[c->dst->name] = i;
        if (c->k == Stmt::Def && c->expr && c->expr->k == Expr::IfExpr && in_memory(c->ty)) last[c->id] = i;
      });
    }
    Stmts out;
    for (size_t i = 0; i < ss.size(); ++i) {
      const S& s = ss[i];
      const bool loop = s->k == Stmt::While || (s->k == Stmt::For && s->map.k == GpuMap::None && !s->unroll);
      auto r = clone(s);
      r->body = walk(s->body, in_loop || loop, loop);
      r->els = walk(s->els, in_loop, false);
      out.push_back(r);
      for (auto& l : last)
        if (l.second == i && (here.count(l.first) || (loop_body && !inside.count(l.first)))) out.push_back(mk_rawstmt(l.first.str() + " += parpy_vector_zero();"));
    }
    return out;
  };
  return walk(ss0, false, false);
}

// ================================================================ no-alias scopes for array aliases
// `src = a; dst = b; if (c) { src = b; dst = a; } <rest>`: in <rest> the two aliases always name
// different arrays, but the target compiler only sees two selected pointers that may be equal, so
// it keeps every load from `src` behind the preceding store to `dst`.  When every combination of
// the selections gives pairwise different arrays, and <rest> reaches those arrays through the
// aliases only, <rest> is put into a scope whose parameters are the aliases, declared not to
// alias each other.  Loads of the (independent) iterations that a thread runs of a parallel loop
// can then be shared and merged: the four states of a thread that have the same predecessors load
// them once, and own-state loads and stores become 128-bit LDS accesses.
bool Pass::is_alias_type(const Type& t) { return t.k == Type::Pointer || (t.k == Type::Tensor && !t.shape.empty()); }

bool Pass::alias_target(const E& e, const AliasCfg& cfg, Name* out) {
  if (!e || e->k != Expr::Var) return false;
  auto it = cfg.find(e->name);
  *out = it == cfg.end() ? e->name : it->second;
  return true;
}

// statements that only (re)point aliases: applies them to every configuration, false if anything else is found
bool Pass::apply_alias_stmt(const S& st, std::vector<AliasCfg>& cfgs, std::vector<Name>& order) {
  if ((st->k == Stmt::Def && is_alias_type(st->ty)) ||
      (st->k == Stmt::Assign && st->dst->k == Expr::Var && is_alias_type(st->dst->ty))) {
    Name a = st->k == Stmt::Def ? st->id : st->dst->name;
    for (auto& c : cfgs) {
      Name t;
      if (!alias_target(st->expr, c, &t)) return false;
      c[a] = t;
    }
    if (std::find(order.begin(), order.end(), a) == order.end()) order.push_back(a);
    return true;
  }
  if (st->k == Stmt::If && !(st->body.empty() && st->els.empty())) {
    std::vector<AliasCfg> then_c = cfgs, else_c = cfgs;
    for (auto& c : st->body) if (!apply_alias_stmt(c, then_c, order)) return false;
    for (auto& c : st->els) if (!apply_alias_stmt(c, else_c, order)) return false;
    cfgs = then_c;
    cfgs.insert(cfgs.end(), else_c.begin(), else_c.end());
    return cfgs.size() <= 16;
  }
  return false;
}

// With `wrap` the rest of the block goes into a scope whose pointer parameters carry the promise; without it the
// kernel only records which local pointers never coincide (the printer's access packing asks).
Stmts Pass::noalias_scopes(const Stmts& ss, bool wrap) {
  Stmts cur;
  for (auto& s : ss) {
    auto r = clone(s);
    r->body = noalias_scopes(s->body, wrap);
    r->els = noalias_scopes(s->els, wrap);
    cur.push_back(r);
  }
  // the first run of alias-only statements of this block
  size_t a = 0;
  while (a < cur.size() && !(cur[a]->k == Stmt::Def && is_alias_type(cur[a]->ty))) ++a;
  if (a == cur.size()) return cur;
  std::vector<AliasCfg> cfgs(1);
  std::vector<Name> order;
  size_t b = a;
  while (b < cur.size()) {
    std::vector<AliasCfg> trial = cfgs;
    std::vector<Name> otrial = order;
    if (!apply_alias_stmt(cur[b], trial, otrial)) break;
    cfgs = trial;
    order = otrial;
    ++b;
  }
  if (order.size() < 2 || b == cur.size()) return cur;
  std::set<Name> targets;
  for (auto& c : cfgs) {
    std::set<Name> seen;
    for (auto& n : order) {
      auto it = c.find(n);
      if (it == c.end() || !seen.insert(it->second).second) return cur;  // two aliases may name one array
      targets.insert(it->second);
    }
  }
  // the rest of the block must reach the arrays through the aliases only and leave the aliases alone
  bool clean = true;
  std::map<Name, Type> types;
  Stmts rest(cur.begin() + b, cur.end());
  visit_stmts(rest, [&](const S& st) {
    if (st->k == Stmt::Def && (targets.count(st->id) || std::count(order.begin(), order.end(), st->id))) clean = false;
    if (st->k == Stmt::Assign && st->dst->k == Expr::Var && std::count(order.begin(), order.end(), st->dst->name)) clean = false;
    if (wrap && (st->k == Stmt::Def || (st->k == Stmt::Assign && st->dst->k == Expr::Var)) && is_alias_type(st->k == Stmt::Def ? st->ty : st->dst->ty))
      clean = false;  // a further alias inside the scope could name the same arrays
    auto scan = [&](const E& e) {
      visit_exprs(e, [&](const E& x) {
        if (x->k != Expr::Var) return;
        if (wrap && targets.count(x->name)) clean = false;
        if (std::count(order.begin(), order.end(), x->name)) types[x->name] = x->ty;
      });
    };
    scan(st->dst); scan(st->expr); scan(st->lo); scan(st->hi);
    for (auto& e : st->args) scan(e);
  });
  if (!clean) return cur;
  std::vector<E> params;
  for (auto& n : order)
    if (types.count(n) && types[n].k == Type::Pointer) params.push_back(mk_var(n, types[n]));
  if (!wrap) {
    std::vector<Name> group;
    for (auto& n : order)
      if (types.count(n)) group.push_back(n);
    if (group.size() >= 2) k.distinct_pointers.push_back(group);
    return cur;
  }
  if (params.size() < 2) return cur;
  auto scope = std::make_shared<Stmt>();
  scope->k = Stmt::Scope;
  scope->args = params;
  scope->body = rest;
  Stmts out(cur.begin(), cur.begin() + b);
  out.push_back(scope);
  return out;
}

// ================================================================ read-only parameters
// A pointer parameter is read-only when nothing in the kernel stores through
// it, directly or through a local alias initialised from it.
void Pass::mark_read_only() {
  std::set<Name> written;
  std::map<Name, std::set<Name>> alias_of;
  std::function<void(const E&, std::set<Name>&)> bases = [&](const E& e, std::set<Name>& out) {
    if (!e) return;
    if (e->k == Expr::Var) {
      auto it = alias_of.find(e->name);
      if (it != alias_of.end()) out.insert(it->second.begin(), it->second.end());
      else out.insert(e->name);
      return;
    }
    if (e->k == Expr::AddrOf || e->k == Expr::Index) { bases(e->args[0], out); return; }
    if (e->k == Expr::IfExpr) { bases(e->args[1], out); bases(e->args[2], out); }
  };
  for (int sweep = 0; sweep < 2; ++sweep) {
    visit_stmts(k.body, [&](const S& s) {
      if (s->k == Stmt::Def && (s->ty.is_array() || s->ty.is_pointer())) bases(s->expr, alias_of[s->id]);
      if (s->k == Stmt::Assign && s->dst->k == Expr::Var && (s->dst->ty.is_array() || s->dst->ty.is_pointer()))
        bases(s->expr, alias_of[s->dst->name]);
      if (s->k == Stmt::Assign && s->dst->k == Expr::Index) bases(s->dst->args[0], written);
      // an array handed to an external device function may be written by it, one handed to the device-scope store is
      auto calls = [&](const E& root) {
        visit_exprs(root, [&](const E& x) {
          if (x->k != Expr::Call || !(x->ext || x->sval == "parpy_device_store")) return;
          for (auto& a : x->args)
            if (a->k == Expr::AddrOf || (a->k == Expr::Var && !a->ty.is_scalar())) bases(a, written);
        });
      };
      calls(s->expr); calls(s->dst); calls(s->lo); calls(s->hi);
    });
  }
  for (auto& p : k.params) p.read_only = p.ty.is_pointer() && !written.count(p.id);
}

// Large inputs whose elements a launch reads once each.  One access in the kernel, each of its dimensions indexed by a
// loop of its own, every loop around it one of these or a division of one of these into shares: nothing is read again
// that a cache could keep, and reads from HBM are faster with non-temporal loads (10 rows of 10^7 floats 69.9 -> 64.8 us,
// 1024 of 65536 45.2 -> 42.2; a plain reading kernel reaches 6.0 and 6.75 TB/s).  Only from the 256 MB on that the
// memory-side cache holds: a smaller array that has just been written or read is found there or in L2, and non-temporal
// loads are the slower ones then (1000 rows of 20000 floats, 80 MB: 14.8 and 17.2 us, read again and again 12.2 and 15.0;
// 2000 of 10000 doubles, 160 MB: 27.4 and 26.1, 22.9 and 23.7; at 256 MB read again and again 39.3 and 40.2).  And only in
// kernels that write little and gather nothing: five million indices and values of a sparse product 38.9 us with plain
// loads, 49.0 with these (rows share lines), 671744 sampled products 33.6 and 37.5; a copy of 200 MB takes 76 and 71 us from HBM, but 50 and 69 between the same two arrays.
void Pass::mark_read_once() {
  struct Site { int count = 0; bool ok = false; int64_t bytes = 0; };
  std::map<Name, Site> reads;
  int64_t stored = 0;
  std::set<Name> barred;   // written, aliased or handed to a call
  auto size = [](const E& x) {
    int64_t n = elem_bytes(x->ty.sz);
    for (int64_t d : x->dim_shape) n *= d;
    return n;
  };
  std::vector<S> loops;
  bool seen_while = false, gathers = false;
  std::set<Name> loop_vars;
  visit_stmts(k.body, [&](const S& s) { if (s->k == Stmt::For) loop_vars.insert(s->id); });
  auto once = [&](const E& x) {
    if (seen_while || x->dim_idx.empty() || x->dim_idx.size() != x->dim_shape.size() || x->ty.sz == ElemSize::Bool) return false;
    std::set<Name> used;
    for (E d : x->dim_idx) {
      while (d->k == Expr::Convert) d = d->args[0];
      if (d->k != Expr::Var || !used.insert(d->name).second) return false;
    }
    // innermost first: a loop counts when its variable indexes a dimension or bounds a loop that counts
    for (size_t q = loops.size(); q-- > 0;) {
      if (!used.count(loops[q]->id)) return false;
      if (has_load(loops[q]->lo) || has_load(loops[q]->hi)) return false;
      for (const E& b : {loops[q]->lo, loops[q]->hi})
        visit_exprs(b, [&](const E& y) { if (y->k == Expr::Var) used.insert(y->name); });
    }
    return true;
  };
  auto scan = [&](const E& root, bool is_dst) {
    if (!root) return;
    visit_exprs(root, [&](const E& x) {
      if (x->k == Expr::Index) visit_exprs(x->args[1], [&](const E& y) { if (y->k == Expr::Index || (y->k == Expr::Var && !loop_vars.count(y->name))) gathers = true; });
      if (x->k == Expr::Index && x->args[0]->k == Expr::Var) {
        if (is_dst && x == root) { barred.insert(x->args[0]->name); stored = std::max(stored, size(x)); return; }
        Site& s = reads[x->args[0]->name];
        s.ok = ++s.count == 1 && once(x);
        s.bytes = size(x);
      }
      if (x->k == Expr::AddrOf || x->k == Expr::Call || x->k == Expr::Raw)
        for (auto& a : x->args) visit_exprs(a, [&](const E& y) { if (y->k == Expr::Var && !y->ty.is_scalar()) barred.insert(y->name); });
    });
  };
  std::function<void(const Stmts&)> walk = [&](const Stmts& ss) {
    for (auto& s : ss) {
      scan(s->dst, s->k == Stmt::Assign);
      scan(s->expr, false);
      scan(s->lo, false);
      scan(s->hi, false);
      if ((s->k == Stmt::Def && !s->ty.is_scalar()) || (s->k == Stmt::Assign && s->dst->k == Expr::Var && !s->dst->ty.is_scalar()))
        visit_exprs(s->expr, [&](const E& y) { if (y->k == Expr::Var) barred.insert(y->name); });
      const bool outer = seen_while;
      seen_while = seen_while || s->k == Stmt::While;
      if (s->k == Stmt::For) loops.push_back(s);
      walk(s->body);
      walk(s->els);
      if (s->k == Stmt::For) loops.pop_back();
      seen_while = outer;
    }
  };
  walk(k.body);
  k.read_once.clear();
  if (gathers) return;
  for (auto& p : k.params) {
    auto r = reads.find(p.id);
    if (!p.ty.is_pointer() || r == reads.end() || !r->second.ok || barred.count(p.id)) continue;
    if (r->second.bytes >= (int64_t(256) << 20) && stored <= r->second.bytes / 8) k.read_once.insert(p.id);
  }
}

}  // namespace hipopt
}  // namespace parpy
