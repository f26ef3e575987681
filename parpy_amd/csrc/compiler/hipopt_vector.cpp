// gfx950 memory passes, several consecutive elements per thread; MFMA dot products.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

// ================================================================ vectorised iteration remap
// Elements per thread that turn the unit-stride accesses of `loop` into 16-byte accesses, 0 when the
// rewrite does not pay.  It does not pay when such an access goes through a local pointer into global
// memory (`src = a if t & 1 else b`): loads and stores through pointers that may coincide cannot be
// merged, so every lane would issue four 4-byte accesses 16 bytes apart from its neighbour's -- a
// quarter of each cache line per request -- where the plain loop has neighbouring lanes on
// neighbouring words.  (Measured on a 262144-state HMM step kept in global memory: 158 us per step
// with the rewrite, 60 us without.)  Pointers into LDS have no such cost.
int Pass::vector_width(const S& loop) {
  int v = 0;
  bool through_global_alias = false, owns_runs = false;
  std::set<Name> params = param_names();
  std::function<void(const E&)> scan = [&](const E& e) {
    visit_exprs(e, [&](const E& x) {
      if (x->k != Expr::Index) return;
      E rest;
      if (!affine_unit(x->args[1], loop->id, &rest)) {
        // an iteration that already owns a run of 16 bytes or more (`a[4*d + c]`): neighbouring lanes sit on
        // neighbouring runs, and giving a thread V consecutive iterations would put them V runs apart
        if (strided_run(x->args[1], loop->id) * elem_bytes(x->ty.sz) >= 16) owns_runs = true;
        return;
      }
      const E& base = x->args[0];
      if (base->k == Expr::Var && !params.count(base->name) && base->ty.mem != Mem::LDS) through_global_alias = true;
      // (the same holds for every global array when the call passed one that is not 16-byte aligned)
      if (base->k == Expr::Var && base->ty.mem != Mem::LDS && !opts.assume_aligned) through_global_alias = true;
      int w = 16 / elem_bytes(x->ty.sz);
      v = v == 0 ? w : std::min(v, w);
    });
  };
  visit_stmts(loop->body, [&](const S& s) { scan(s->dst); scan(s->expr); scan(s->lo); scan(s->hi); });
  return through_global_alias || owns_runs ? 0 : v;
}

// c when idx == c * d + rest with rest free of d and c a constant > 1, else 0
int64_t Pass::strided_run(const E& idx, const Name& d) {
  if (idx->k != Expr::BinOpE) return 0;
  const E &a = idx->args[0], &b = idx->args[1];
  if (idx->bop == BinOp::Mul) {
    if (a->k == Expr::Int && b->k == Expr::Var && b->name == d) return a->iv > 1 ? a->iv : 0;
    if (b->k == Expr::Int && a->k == Expr::Var && a->name == d) return b->iv > 1 ? b->iv : 0;
    return 0;
  }
  if (idx->bop == BinOp::Add || idx->bop == BinOp::Sub) {
    if (!mentions(b, d)) return strided_run(a, d);
    if (idx->bop == BinOp::Add && !mentions(a, d)) return strided_run(b, d);
  }
  return 0;
}

// Whether a loop over elements of four bytes and more takes vectors that do not divide it.  In rows that stand in LDS it does
// where neighbouring elements are read by neighbouring iterations: 300 rows of 1001 / 4099 floats, 128 / 256 threads, 100 steps
// of `d[j] = f(s[j], s[(j + 1) % M])` 66 -> 36 / 102 -> 80 us, of `s[j / 2]` 54 -> 34 / 98 -> 64, and 300 steps with a row of a
// table 151 -> 87 / 258 -> 140; of `s[4 j % M]` 76 -> 96 / 127 -> 371, whose lanes then meet in the banks (`s[M - 1 - j]` and
// `s[p[j]]` gain on short rows and lose on long ones).  In rows that stand in memory it does where another loop walks the same
// elements, which then stay in registers (20 000 000 floats: x / sum(x), rows of 1001 on 64 threads 36 -> 30, of 4099 on 256
// 31 -> 28; two element-wise loops over two arrays 55 -> 46 and 46 -> 41); one loop alone is bound by memory and loses by
// accesses that share lines (x + 1, rows of 4099 30 -> 38, a sum of three neighbours 30 -> 51, x[M - 1 - j] 30 -> 67).
bool Pass::part_of_a_vector_pays(const S& loop) {
  // neighbours of the loop's elements, wherever the row starts or wraps around
  std::function<bool(const E&)> follows = [&](const E& x) {
    if (x->k == Expr::Convert) return follows(x->args[0]);
    if (x->k == Expr::Var) return x->name == loop->id;
    if (x->k != Expr::BinOpE) return false;
    const bool left = mentions(x->args[0], loop->id), right = mentions(x->args[1], loop->id);
    if (left && right) return false;
    if (x->bop == BinOp::Add) return follows(x->args[left ? 0 : 1]);
    return left && (x->bop == BinOp::Sub || x->bop == BinOp::FloorDiv || x->bop == BinOp::Rem) && follows(x->args[0]);
  };
  std::map<Name, E> named;
  std::vector<std::pair<Name, E>> rows;   // arrays in memory, and where the row starts
  bool in_lds = false, ok = true;
  visit_stmts(loop->body, [&](const S& c) {
    for (const E& e : {c->expr, c->dst})
      visit_exprs(e, [&](const E& x) {
        if (x->k != Expr::Index) return;
        const E at = subst_vars(x->args[1], named);
        E rest;
        if (x->args[0]->ty.mem == Mem::LDS) {
          in_lds = true;
          ok = ok && (!mentions(at, loop->id) || follows(at));
        } else if (affine_unit(at, loop->id, &rest)) {
          if (x->args[0]->k == Expr::Var) rows.push_back({x->args[0]->name, rest});
        } else {
          ok = ok && !mentions(at, loop->id);
        }
      });
    if (c->k == Stmt::Def && c->expr) named[c->id] = subst_vars(c->expr, named);
  });
  if (!ok || in_lds) return ok;
  bool shared = false;
  visit_stmts(k.body, [&](const S& o) {
    if (o == loop || !thread_mapped(o) || o->map.n != loop->map.n || !expr_eq(o->lo, loop->lo) || !expr_eq(o->hi, loop->hi)) return;
    visit_stmts(o->body, [&](const S& c) {
      for (const E& e : {c->expr, c->dst})
        visit_exprs(e, [&](const E& x) {
          E rest;
          if (x->k != Expr::Index || x->args[0]->k != Expr::Var || !affine_unit(x->args[1], o->id, &rest)) return;
          for (auto& r : rows) shared = shared || (r.first == x->args[0]->name && expr_eq(r.second, rest));
        });
    });
  });
  return shared;
}

// A long loop over a row that is no whole number of vectors: rows start anywhere.  The vectors begin where a line of the
// memory does, so that no two accesses share a line, and what stands in front of them and behind them (less than a line and
// a vector) is a loop of its own, one element to a thread.  Sums of 542 rows of 115 669 floats on 128 threads 70.5 -> 49.9 us,
// 300 of 100 001 on 512 34.8 -> 26.9, 16 of 1 000 001 on 1024 79.7 -> 44.4; with vectors that start where the row does 27.8 on
// the second, and 55.0 instead of 51.7 for 2000 of 40 001 on 256.  Doubles stay as they are: vectors of two were slower by the
// clock (200 rows of 200 001: 53.8 -> 63.1 us, 1500 of 33 001: 64.9 -> 66.9).
Stmts Pass::whole_lines(const S& s, int V) {
  const int64_t extent = const_extent(s), N = s->map.n;
  if (!s->els.empty() || s->lo->iv != 0 || extent % V == 0 || counted_trips(extent, N) > 0 || extent < 2 * V * N) return {};
  // the first element of the row, by the first array that is walked
  E row;
  int64_t line = 0;
  bool ok = true;
  // what the body names on the way (`base = i * M`) is written out: the names mean nothing in front of the loop
  std::map<Name, E> named;
  std::set<Name> assigned;
  for (auto& c : s->body) {
    if (c->k != Stmt::Def && c->k != Stmt::Assign) ok = false;
    if (c->k == Stmt::Def && c->expr) named[c->id] = subst_vars(c->expr, named);
    if (c->k == Stmt::Assign && c->dst->k == Expr::Var) assigned.insert(c->dst->name);
  }
  for (auto& n : assigned) named.erase(n);
  visit_stmts(s->body, [&](const S& c) {
    for (const E& e : {c->expr, c->dst})
      visit_exprs(e, [&](const E& x) {
        E rest;
        if (row || x->k != Expr::Index || x->args[0]->ty.mem == Mem::LDS || !affine_unit(x->args[1], s->id, &rest)) return;
        row = rest;
        line = 128 / elem_bytes(x->ty.sz);
      });
  });
  if (!ok || !row || N < line + V) return {};
  row = fold_expr(subst_vars(row, named));
  if (has_load(row) || mentions(row, s->id)) return {};
  for (auto& n : assigned)
    if (mentions(row, n)) return {};
  visit_exprs(row, [&](const E& x) { if (x->k != Expr::Var && x->k != Expr::Int && x->k != Expr::BinOpE && x->k != Expr::Convert) ok = false; });
  if (!ok) return {};
  Type ity = Type::scalar(isz), bty = Type::scalar(ElemSize::Bool);
  auto num = [&](int64_t v) { return mk_int(v, isz); };
  auto bin = [&](BinOp op, E a, E b) { return mk_binop(op, a, b, ity); };
  const Name front = gen.fresh(s->id.s + "_front"), vectors = gen.fresh(s->id.s + "_vectors"), q = gen.fresh(s->id.s + "_q"), u = gen.fresh(s->id.s + "_u"), o = gen.fresh(s->id.s + "_o");
  const E fv = mk_var(front, ity), nv = mk_var(vectors, ity), qv = mk_var(q, ity), ov = mk_var(o, ity);
  Stmts out;
  out.push_back(mk_def(front, ity, bin(BinOp::Min, bin(BinOp::Max, bin(BinOp::Rem, bin(BinOp::Sub, num(line), bin(BinOp::Rem, row, num(line))), num(line)), num(0)), num(line - 1)), s->i));
  out.push_back(mk_def(vectors, ity, bin(BinOp::FloorDiv, bin(BinOp::Sub, num(extent), fv), num(V)), s->i));
  Stmts ib{mk_def(s->id, ity, bin(BinOp::Add, fv, bin(BinOp::Add, bin(BinOp::Mul, qv, num(V)), mk_var(u, ity))), s->i)};
  ib.insert(ib.end(), s->body.begin(), s->body.end());
  auto inner = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(u, num(0), num(V), 1, ib, LoopPar(), s->i)));
  inner->unroll = true;
  inner->iv = 1;   // (the vectors are not known to be aligned)
  auto main = clone(s);
  main->id = q;
  main->hi = nv;
  main->body = {S(inner)};
  out.push_back(main);
  // the other elements, numbered: those in front, then those behind the vectors
  auto rest = clone(s);
  rest->id = o;
  rest->hi = num(line + V - 2);
  const E at = mk_ifexpr(mk_binop(BinOp::Lt, ov, fv, bty), ov, bin(BinOp::Add, ov, bin(BinOp::Mul, nv, num(V))), ity);
  rest->body = {mk_def(s->id, ity, at, s->i), mk_if(mk_binop(BinOp::Lt, mk_var(s->id, ity), num(extent), bty), s->body, {})};
  out.push_back(rest);
  return out;
}

Stmts Pass::vectorize(const Stmts& ss) {
  bool stores_rows = false;   // a loop of the kernel writes element after element of an array
  visit_stmts(k.body, [&](const S& s) {
    if (thread_mapped(s))
      visit_stmts(s->body, [&](const S& c) {
        E rest;
        if (c->k == Stmt::Assign && c->dst->k == Expr::Index && c->dst->args[0]->ty.mem != Mem::LDS && affine_unit(c->dst->args[1], s->id, &rest)) stores_rows = true;
      });
  });
  Stmts out;
  for (auto& s : ss) {
    bool done = false;
    // grid-wide loops qualify too when the launch has no partial block (no bounds guard)
    bool grid_wide = s->k == Stmt::For && s->map.k == GpuMap::ThreadBlock && s->map.tpb > 0 && s->map.n % s->map.tpb == 0;
    if ((thread_mapped(s) || grid_wide) && s->step == 1 && s->lo->k == Expr::Int && s->hi->k == Expr::Int) {
      int64_t extent = const_extent(s);
      const int widest = vector_width(s);
      bool nested = false;
      visit_stmts(s->body, [&](const S& c) { if (c->k == Stmt::For && c->map.k != GpuMap::None) nested = true; });
      // A block-level loop only needs whole vectors (threads may run different trip counts); a grid-wide one must also
      // fill its launch exactly, since it has no bounds guard.  Where 16-byte vectors would leave more than a quarter of
      // the threads without one, narrower vectors are taken.  Elements of four bytes and more move 256 bytes per
      // wavefront and access as they are, so only narrower ones take vectors that do not divide the loop: the last one
      // is then tested element by element.  So do wider ones where rows are written, threads take two vectors and more and
      // `part_of_a_vector_pays` (softmax, floats on 256 threads: 30000 rows of 501 / 999 / 1001 21.3 / 57.9 / 58.1 -> 19.2 / 40.3 / 40.0 us, 2000 of 20001
      // 182 -> 61; 63305 rows of 202 on one vector a thread 20.7 -> 25.7; sums of 20000 rows of 999 13.9 -> 15.6).  (Rows need not start on 16 bytes: the memory instructions take any
      // element-aligned address.  Softmax over 1000 rows of 20001 halves on 512 threads per row: 40.2 -> 21.6 us, over
      // 3000 rows of 999 on 256: 10.3 -> 6.7.)
      int V = 0;
      for (int v = widest; v >= 2 && V == 0 && !nested; v /= 2) {
        const int64_t vectors = (extent + v - 1) / v;
        const bool whole = extent % v == 0;
        if (grid_wide ? whole && extent % (s->map.n * v) == 0 : (extent % widest == 0 || widest > 4 || (stores_rows && v == widest && vectors > s->map.n && part_of_a_vector_pays(s))) && 4 * vectors >= 3 * s->map.n) V = v;
        if (grid_wide) break;
      }
      // (a long loop whose trip count is not the same for all threads is not counted: its last vector would put a test
      // into every iteration)
      const bool partial = V > 0 && extent % V != 0;
      if (partial && counted_trips((extent + V - 1) / V, s->map.n) < 0) V = 0;
      if (V == 0 && !grid_wide && !nested && widest >= 4) {
        Stmts lines = whole_lines(s, widest);
        if (!lines.empty()) {
          out.insert(out.end(), lines.begin(), lines.end());
          continue;
        }
      }
      if (V > 0) {
        Type ity = Type::scalar(isz), bty = Type::scalar(ElemSize::Bool);
        Name q = gen.fresh(s->id.s + "_q"), u = gen.fresh(s->id.s + "_u");
        E first = mk_binop(BinOp::Mul, mk_var(q, ity), mk_int(V, isz), ity);
        E d = fold_expr(mk_binop(BinOp::Add, s->lo, mk_binop(BinOp::Add, first, mk_var(u, ity), ity), ity));
        Stmts ib;
        ib.push_back(mk_def(s->id, ity, d, s->i));
        for (auto& b : s->body) ib.push_back(b);
        auto inner = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(
            mk_for(u, mk_int(0, isz), mk_int(V, isz), 1, ib, LoopPar(), s->i)));
        inner->unroll = true;
        if (partial) inner->iv = 1;   // (rows that are no whole vectors start anywhere)
        if (partial)   // (whole vector, element in range, end): printed as two loops
          inner->args = {mk_binop(BinOp::Leq, first, mk_int(extent - V, isz), bty), mk_binop(BinOp::Lt, mk_var(s->id, ity), s->hi, bty), s->hi};
        auto outer = clone(s);
        outer->id = q;
        outer->lo = mk_int(0, isz);
        outer->hi = mk_int((extent + V - 1) / V, isz);
        outer->body = {S(inner)};
        out.push_back(outer);
        done = true;
      }
    }
    if (done) continue;
    auto r = clone(s);
    r->body = vectorize(s->body);
    r->els = vectorize(s->els);
    out.push_back(r);
  }
  return out;
}

// ================================================================ sums of halves in single precision
// A reduction of halves adds up a thread's elements, then the threads'.  The running value is kept in single precision
// and rounded to a half once, when the reduction is complete: a thread that takes many elements then loses nothing
// against many threads that take a few each, and a mixed-precision multiply-add takes the half as it is.
Stmts Pass::widen_half_sums(const Stmts& ss) {
  Stmts out;
  for (auto& s : ss) {
    auto r = clone(s);
    r->body = widen_half_sums(s->body);
    r->els = widen_half_sums(s->els);
    out.push_back(r);
  }
  for (size_t q = 0; q < out.size(); ++q) {
    const S red = out[q];
    if (red->k != Stmt::WaveReduce || red->ty.sz != ElemSize::F16 || !(red->bop == BinOp::Add || red->bop == BinOp::Mul)) continue;
    const Name t = red->id;
    size_t def = q;
    for (size_t d = 0; d < q; ++d) if (out[d]->k == Stmt::Def && out[d]->id == t) def = d;
    if (def == q) continue;
    // between its definition and the reduction the value may only be added to (multiplied by) something
    bool ok = true;
    auto term_of = [&](const S& s, E* term) {
      if (!(s->k == Stmt::Assign && s->dst->k == Expr::Var && s->dst->name == t && s->expr->k == Expr::BinOpE && s->expr->bop == red->bop)) return false;
      const E &a = s->expr->args[0], &b = s->expr->args[1];
      *term = a->k == Expr::Var && a->name == t ? b : b->k == Expr::Var && b->name == t ? a : E();
      return *term && !mentions(*term, t);
    };
    Stmts between(out.begin() + def + 1, out.begin() + q);
    visit_stmts(between, [&](const S& s) {
      E term;
      if (term_of(s, &term)) return;
      if ((s->k == Stmt::Def || s->k == Stmt::WaveReduce) && s->id == t) ok = false;
      for (const E& e : {s->expr, s->dst, s->lo, s->hi}) if (e && mentions(e, t)) ok = false;
    });
    if (!ok) continue;
    const Type f32 = Type::scalar(ElemSize::F32);
    const Name w = gen.fresh(t.s + "_wide");
    std::function<Stmts(const Stmts&)> widen = [&](const Stmts& b) {
      Stmts o;
      for (auto& s : b) {
        E term;
        if (term_of(s, &term)) {
          o.push_back(mk_assign(mk_var(w, f32), mk_binop(red->bop, mk_var(w, f32), mk_convert(term, ElemSize::F32), f32), s->i));
          continue;
        }
        auto r = clone(s);
        r->body = widen(s->body);
        r->els = widen(s->els);
        o.push_back(r);
      }
      return o;
    };
    Stmts next(out.begin(), out.begin() + def + 1);
    next.push_back(mk_def(w, f32, mk_convert(mk_var(t, red->ty), ElemSize::F32), red->i));
    for (auto& s : widen(between)) next.push_back(s);
    auto wide = clone(red);
    wide->id = w;
    wide->ty = f32;
    next.push_back(wide);
    next.push_back(mk_assign(mk_var(t, red->ty), mk_convert(mk_var(w, f32), ElemSize::F16), red->i));
    const size_t at = next.size();
    next.insert(next.end(), out.begin() + q + 1, out.end());
    out = next;
    q = at - 1;
  }
  return out;
}

// ================================================================ dot products on the matrix cores
// `t = t + X[..] * Y[..]` in an innermost sequential f32 loop of constant length is a dot
// product that every thread computes for itself.  v_mfma_f32_4x4x1 multiplies, for each group
// of four lanes, the four X values by the four Y values of the group (a 4 x 4 outer product
// accumulated over the loop); the product a thread wants is element [lane % 4] of its own
// column.  Three quarters of the multiplications are thrown away and the instruction takes two
// passes, so this is no faster than v_fmac on the vector ALU: there is no operand reuse between
// the dot products of different threads for a matrix unit to exploit.  Kept as an option so
// that the comparison can be measured.
Stmts Pass::mfma_dot(const Stmts& ss) {
  Stmts out;
  for (auto& s : ss) {
    bool inner = s->k == Stmt::For && s->map.k == GpuMap::None && s->step == 1 && s->hi->k == Expr::Int && s->lo->k == Expr::Int &&
                 s->body.size() == 1 && s->body[0]->k == Stmt::Assign && s->body[0]->dst->k == Expr::Var;
    if (inner) {
      const S& a = s->body[0];
      const E& t = a->dst;
      E mul;
      if (a->expr->k == Expr::BinOpE && a->expr->bop == BinOp::Add) {
        const E &l = a->expr->args[0], &r = a->expr->args[1];
        if (l->k == Expr::Var && l->name == t->name) mul = r;
        else if (r->k == Expr::Var && r->name == t->name) mul = l;
      }
      bool ok = mul && mul->k == Expr::BinOpE && mul->bop == BinOp::Mul && t->ty.is_scalar() && t->ty.sz == ElemSize::F32 &&
                mul->args[0]->k == Expr::Index && mul->args[1]->k == Expr::Index && mul->args[0]->ty.sz == ElemSize::F32 &&
                mul->args[1]->ty.sz == ElemSize::F32 && !mentions(mul, t->name);
      if (ok) {
        Name acc = gen.fresh(t->name.s + "_acc");
        Type f32 = Type::scalar(ElemSize::F32);
        out.push_back(mk_rawstmt("parpy_f32x4 " + acc.str() + " = {0.0f, 0.0f, 0.0f, 0.0f};"));
        auto call = std::make_shared<Expr>();
        call->k = Expr::Call;
        call->ty = f32;
        call->sval = "__builtin_amdgcn_mfma_f32_4x4x1f32";
        call->args = {mul->args[0], mul->args[1], mk_var(acc, f32), mk_raw("0", f32), mk_raw("0", f32), mk_raw("0", f32)};
        auto loop = clone(s);
        loop->body = {mk_assign(mk_var(acc, f32), call)};
        out.push_back(loop);
        out.push_back(mk_assign(t, mk_binop(BinOp::Add, t, mk_raw(acc.str() + "[parpy_lane_id() & 3]", f32), f32)));
        continue;
      }
    }
    auto r = clone(s);
    r->body = mfma_dot(s->body);
    r->els = mfma_dot(s->els);
    out.push_back(r);
  }
  return out;
}

}  // namespace hipopt
}  // namespace parpy
