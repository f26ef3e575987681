// gfx950 memory passes, helpers over the kernel IR.
#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

bool mentions(const E& e, const Name& v) {
  bool m = false;
  visit_exprs(e, [&](const E& x) { if (x->k == Expr::Var && x->name == v) m = true; });
  return m;
}

bool has_load(const E& e) {
  bool m = false;
  visit_exprs(e, [&](const E& x) { if (x->k == Expr::Index || x->k == Expr::AddrOf || x->k == Expr::RegElem) m = true; });
  return m;
}

// idx == rest + d with rest free of d
bool affine_unit(const E& idx, const Name& d, E* rest) {
  if (idx->k == Expr::Var && idx->name == d) { *rest = mk_int(0, idx->ty.sz); return true; }
  if (idx->k == Expr::BinOpE && (idx->bop == BinOp::Add || idx->bop == BinOp::Sub)) {
    E r;
    if (affine_unit(idx->args[0], d, &r) && !mentions(idx->args[1], d)) {
      *rest = fold_expr(mk_binop(idx->bop, r, idx->args[1], idx->ty));
      return true;
    }
    if (idx->bop == BinOp::Add && affine_unit(idx->args[1], d, &r) && !mentions(idx->args[0], d)) {
      *rest = fold_expr(mk_binop(BinOp::Add, idx->args[0], r, idx->ty));
      return true;
    }
  }
  return false;
}

int64_t const_extent(const S& loop) {
  if (loop->lo->k != Expr::Int || loop->hi->k != Expr::Int || loop->step <= 0) return -1;
  return (loop->hi->iv - loop->lo->iv + loop->step - 1) / loop->step;
}

// iterations every thread runs in a thread-mapped loop, when that is a compile-time constant
int64_t per_thread_trips(const S& loop) {
  return counted_trips(const_extent(loop), loop->map.n);
}

// the per-thread iteration counter of a mapped loop as the printer names it
E counter_var(const S& loop, ElemSize isz) {
  if (per_thread_trips(loop) == 1) return mk_int(0, isz);
  return mk_var(Name{loop->id.str() + "_k", 0}, Type::scalar(isz));
}

E subst_vars(const E& e, const std::map<Name, E>& m) {
  if (!e) return e;
  if (e->k == Expr::Var) {
    auto it = m.find(e->name);
    return it == m.end() ? e : it->second;
  }
  return map_children(e, [&](const E& c) { return subst_vars(c, m); });
}

E arrays_disjoint(const Program& p, const std::vector<HostArray>& arrays) {
  std::set<Name> made_here;   // temporaries of the plan meet nothing
  visit_stmts(p.host, [&](const S& s) { if (s->k == Stmt::Alloc) made_here.insert(s->id); });
  const Type bty = Type::scalar(ElemSize::Bool);
  E all;
  for (size_t x = 0; x < arrays.size(); ++x)
    for (size_t y = x + 1; y < arrays.size(); ++y) {
      const HostArray &a = arrays[x], &b = arrays[y];
      if (!(a.written || b.written) || made_here.count(a.name) || made_here.count(b.name)) continue;
      auto c = std::make_shared<Expr>();
      c->k = Expr::Call;
      c->ty = bty;
      c->sval = "parpy_disjoint";
      c->args = {mk_var(a.name, Type::pointer(ElemSize::I8)), mk_int(a.bytes), mk_var(b.name, Type::pointer(ElemSize::I8)), mk_int(b.bytes)};
      all = all ? mk_binop(BinOp::And, all, E(c), bty) : E(c);
    }
  return all;
}

int64_t temporaries(const Stmts& host) {
  int64_t bytes = 0;
  visit_stmts(host, [&](const S& s) { if (s->k == Stmt::Alloc) bytes += (s->iv * elem_bytes(s->ty.sz) + 255) / 256 * 256; });
  return bytes;
}

}  // namespace hipopt
}  // namespace parpy
