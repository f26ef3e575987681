// gfx950 memory passes, rewrites that change a launch: two steps of a host-side time loop in one pass over two arrays that
// change places.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

namespace {

// ================================================================ two steps per launch
// `for t: dst[r, s] = f(src[r, ...], t)` with two arrays that change places, one launch per step, reads and writes a whole
// state vector per step.  Where a thread computes several elements, s = g, g + N, g + 2N, ..., and f takes most of what it reads
// of `src` from the thread's own elements, the element of the next step needs from other threads only the few values that f
// takes from elsewhere.  Those are computed a second time by who needs them, and two steps run in one launch: the values
// of the step between stay in registers, half of the traffic and half of the launches go away.
//
//   * Four neighbouring threads that need the same four values of others (s / 4 in their places) compute one each and pass it
//     on (DPP within four lanes); otherwise each computes its own, where those are a quarter of its elements at most.
//   * Rows that end: `if t < len[r]: step, else if t == len[r]: dst = src` leaves the last values in both arrays.  A launch
//     for the steps t and t + 1 makes one step where the row ends between them, and copies where it ended in the step before
//     the launch's first or in that one; a launch of copies behind the last of them makes up for the rows that end there.
//   * Launches come in pairs, so that the arrays are where the loop of single steps has them, and the last one to four steps
//     run as single steps: both arrays end as they would.
//   * The arithmetic of an element is that of the statements as written: same operations, same order, and the value of the step
//     between is rounded as the store of it would.
//
// The step of a model of 16 layers of 16 384 states (`forward_kernel`, one thread per state of a layer, 100 rows of 1 MB that
// fit the memory-side cache): 31 us as a launch of its own, of which a copy of the arrays takes 25.6 and the vector ALU 24; two
// steps 55 to 61 us, of which vector instructions are active for 54 (counted, 89 % of the cycles; four recomputed values per
// thread instead of one: 4 us more).  100 reads of 500 to 1500 samples 36.2 -> 28.6 ms, 37 of them 18.2 -> 14.4; 98 of 666 to 2000 over 16 layers of 4096 states 19.2 -> 15.2.
struct TwoSteps {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;
  Type ity;
  Type bty = Type::scalar(ElemSize::Bool);

  TwoSteps(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()), ity(Type::scalar(o.int_size())) {}

  E iint(int64_t v) { return mk_int(v, isz); }
  E add(E a, E b) { return mk_binop(BinOp::Add, a, b, ity); }

  // the launch, taken apart
  struct Step {
    S root;                 // loop over the rows, one to a block of the grid's y dimension
    Name src, dst;          // pointer variables
    Name even, odd;         // the parameter that `src` names in even and in odd steps
    Stmts defs;             // scalars of the row
    E until;                // the row ends here; null: never
    S loop;                 // the elements, a thread's shared part in `els`
    Name g, k;              // the thread's number, the number of its element
    int64_t N = 0, per = 0; // threads of a row, elements of a thread
    ElemSize sz = ElemSize::F32;
    int64_t row = 0;        // elements of a row
  };

  static E bare(E e) {
    while (e && e->k == Expr::Convert) e = e->args[0];
    return e;
  }
  // an element of the arrays: row r, element `at`
  static bool element(const E& x, const Name& array, const Name& row, E* at) {
    if (!(x->k == Expr::Index && x->args[0]->k == Expr::Var && x->args[0]->name == array)) return false;
    if (!(x->dim_idx.size() == 2 && x->dim_shape.size() == 2 && x->dim_idx[0]->k == Expr::Var && x->dim_idx[0]->name == row)) return false;
    *at = x->dim_idx[1];
    return true;
  }

  // reads nothing but parameters that the kernel never writes, calls nothing
  static bool pure(const E& e, const std::set<Name>& never_written) {
    bool ok = true;
    visit_exprs(e, [&](const E& x) {
      if (x->k == Expr::Call || x->k == Expr::Raw || x->k == Expr::RegElem || x->k == Expr::AddrOf || x->k == Expr::ThreadIdx || x->k == Expr::BlockIdx) ok = false;
      if (x->k == Expr::Index && !(x->args[0]->k == Expr::Var && never_written.count(x->args[0]->name))) ok = false;
    });
    return ok;
  }

  bool match(const Kernel& k, const S& time, Step& st) {
    if (k.body.size() != 1 || k.grid.z != 1 || k.block.y != 1 || k.block.z != 1) return false;
    st.root = k.body[0];
    if (!(st.root->k == Stmt::For && st.root->map.k == GpuMap::Block && st.root->map.dim == 1 && st.root->map.mult == 1 && st.root->map.per == 1 &&
          st.root->map.n == k.grid.y && st.root->step == 1 && st.root->lo->k == Expr::Int && st.root->lo->iv == 0 && const_extent(st.root) == k.grid.y &&
          st.root->els.empty()))
      return false;
    const Stmts& ss = st.root->body;
    if (ss.size() < 4) return false;
    // which array is which
    std::vector<Name> pointers;
    for (auto& s : ss) if (s->k == Stmt::Def && Pass::is_alias_type(s->ty)) pointers.push_back(s->id);
    if (pointers.size() != 2) return false;
    Pass::AliasDef a = Pass::alias_definition(ss, ss.size() - 1, pointers[0]), b = Pass::alias_definition(ss, ss.size() - 1, pointers[1]);
    if (!a.ok || !b.ok || !(a.a == b.b) || !(a.b == b.a) || a.a == a.b || !expr_eq(a.cond, b.cond) || !Pass::alternates(a.cond, time)) return false;
    std::set<Name> params, never_written;
    for (auto& q : k.params) if (q.ty.is_pointer() || q.ty.is_array()) params.insert(q.id);
    if (!params.count(a.a) || !params.count(a.b)) return false;
    never_written = params;
    never_written.erase(a.a);
    never_written.erase(a.b);
    // everything else in front of the elements: scalars of the row
    for (size_t q = 0; q + 1 < ss.size(); ++q) {
      const S& s = ss[q];
      if (s->k == Stmt::Def && Pass::is_alias_type(s->ty)) continue;
      if (s->k == Stmt::If && s->els.empty()) {
        for (auto& c : s->body)
          if (!(c->k == Stmt::Assign && c->dst->k == Expr::Var && (c->dst->name == pointers[0] || c->dst->name == pointers[1]))) return false;
        continue;
      }
      if (!(s->k == Stmt::Def && s->ty.is_scalar() && pure(s->expr, never_written))) return false;
      st.defs.push_back(s);
    }
    st.loop = ss.back();
    S copy;
    if (st.loop->k == Stmt::If) {
      const S test = st.loop;
      const E& c = test->expr;
      if (!(c->k == Expr::BinOpE && (c->bop == BinOp::Lt || c->bop == BinOp::Gt) && test->body.size() == 1 && test->els.size() == 1)) return false;
      const E now = bare(c->bop == BinOp::Lt ? c->args[0] : c->args[1]);
      st.until = c->bop == BinOp::Lt ? c->args[1] : c->args[0];
      if (!(now->k == Expr::Var && now->name == time->id) || mentions(st.until, time->id) || st.until->ty.sz != isz || !pure(st.until, never_written)) return false;
      for (auto& d : st.defs) if (mentions(st.until, d->id)) return false;
      st.loop = test->body[0];
      copy = test->els[0];
    }
    const S& L = st.loop;
    if (!(L->k == Stmt::For && L->map.k == GpuMap::ThreadBlock && L->map.dim == 0 && L->step == 1 && L->lo->k == Expr::Int && L->lo->iv == 0 && !L->els.empty() &&
          L->map.tpb == k.block.x && L->map.n == k.grid.x * k.block.x))
      return false;
    st.row = const_extent(L);
    st.N = L->map.n;
    if (st.row <= 0 || st.row % st.N != 0 || st.N % WAVE_SIZE != 0) return false;
    st.per = st.row / st.N;
    // (a thread's elements of the step between are registers)
    if (st.per < 4 || st.per > (k.block.x > 512 ? 16 : 32)) return false;
    st.g = Name{L->id.str() + "_g", 0};
    st.k = Name{L->id.str() + "_k", 0};
    // the elements: definitions and assignments, one store, to the thread's own element
    E at;
    const S& last = L->body.back();
    if (!(last->k == Stmt::Assign && last->dst->k == Expr::Index && last->dst->args[0]->k == Expr::Var)) return false;
    st.dst = last->dst->args[0]->name;
    if (!(st.dst == pointers[0] || st.dst == pointers[1])) return false;
    st.src = st.dst == pointers[0] ? pointers[1] : pointers[0];
    st.even = st.src == pointers[0] ? a.a : b.a;
    st.odd = st.src == pointers[0] ? a.b : b.b;
    st.sz = last->dst->ty.sz;
    if (!is_float(st.sz) || !element(last->dst, st.dst, st.root->id, &at) || last->dst->dim_shape[1] != st.row) return false;
    for (int64_t e = 0; e < st.per; ++e) {
      E rest;
      if (!affine_unit(fold_expr(subst_vars(at, {{st.k, iint(e)}})), st.g, &rest) || rest->k != Expr::Int || rest->iv != e * st.N) return false;
    }
    std::set<Name> local;
    auto reads = [&](const E& e) {
      bool ok = true;
      visit_exprs(e, [&](const E& x) {
        if (x->k == Expr::Call || x->k == Expr::Raw || x->k == Expr::RegElem || x->k == Expr::AddrOf || x->k == Expr::ThreadIdx || x->k == Expr::BlockIdx) ok = false;
        if (x->k == Expr::Var && (x->name == L->id || (x->name == st.src && Pass::is_alias_type(x->ty) == false))) ok = false;
        if (x->k != Expr::Index) return;
        E where;
        if (x->args[0]->k != Expr::Var || (!never_written.count(x->args[0]->name) && !element(x, st.src, st.root->id, &where))) ok = false;
        else if (x->args[0]->name == st.src && (x->dim_shape[1] != st.row || x->ty.sz != st.sz)) ok = false;
      });
      return ok;
    };
    for (auto* part : {&L->els, &L->body})
      for (auto& s : *part) {
        if (s == last) { if (!reads(s->expr)) return false; continue; }
        if (!reads(s->expr)) return false;
        if (s->k == Stmt::Def && s->ty.is_scalar()) { local.insert(s->id); continue; }
        if (!(part == &L->body && s->k == Stmt::Assign && s->dst->k == Expr::Var && s->dst->ty.is_scalar() && local.count(s->dst->name))) return false;
      }
    if (!st.until) return true;
    // where a row has ended: its elements are copied in the step `until`, and nothing happens behind it
    if (!(copy->k == Stmt::For && copy->map.k == L->map.k && copy->map.dim == 0 && copy->map.n == L->map.n && copy->map.tpb == L->map.tpb && copy->step == 1 &&
          copy->lo->k == Expr::Int && copy->lo->iv == 0 && const_extent(copy) == st.row && copy->els.empty() && copy->body.size() == 1))
      return false;
    const S& when = copy->body[0];
    if (!(when->k == Stmt::If && when->els.empty() && when->body.size() == 1 && when->expr->k == Expr::BinOpE && when->expr->bop == BinOp::Eq)) return false;
    for (int side = 0; side < 2; ++side) {
      const E now = bare(when->expr->args[side]);
      if (!(now->k == Expr::Var && now->name == time->id && expr_eq(when->expr->args[1 - side], st.until))) continue;
      const S& move = when->body[0];
      E to, from;
      return move->k == Stmt::Assign && element(move->dst, st.dst, st.root->id, &to) && element(move->expr, st.src, st.root->id, &from) && to->k == Expr::Var &&
             to->name == copy->id && expr_eq(to, from) && move->dst->dim_shape[1] == st.row && move->expr->dim_shape[1] == st.row;
    }
    return false;
  }

  // a copy of a thread's statements: what stands for their names, what they store
  struct Copy {
    std::map<Name, E> names;                             // of the statements, the thread's number, the element's
    std::map<Name, E> numbers;                           // whole numbers among them, by the thread's number alone
    std::function<E(const E& x, const E& at)> source;    // what stands for an element of `src`, given its place
    Stmts out;
    E stored;
  };

  RangeEnv ranges;   // of the thread's number

  // whole numbers by the thread's number: names resolved, conversions that change nothing left out
  E number(const Copy& c, const E& e) {
    return fold_expr(rewrite_expr(fold_expr(subst_vars(e, c.numbers)), [&](const E& x) -> E {
      if (x->k != Expr::Convert || !x->ty.is_scalar() || !x->args[0]->ty.is_scalar() || !is_int(x->args[0]->ty.sz)) return x;
      if (x->ty.sz != ElemSize::I32 && x->ty.sz != ElemSize::I64) return x;
      const Interval r = expr_range(x->args[0], ranges);
      return r.known && r.lo >= 0 && r.hi <= INT32_MAX ? x->args[0] : x;
    }));
  }

  E copied(Copy& c, const Step& st, const E& e) {
    if (!e) return e;
    if (e->k == Expr::Var) {
      auto it = c.names.find(e->name);
      return it == c.names.end() ? e : it->second;
    }
    E at;
    if (e->k == Expr::Index && element(e, st.src, st.root->id, &at)) return c.source(e, at);
    return fold_expr(map_children(e, [&](const E& x) { return copied(c, st, x); }));
  }

  void copy_of(Copy& c, const Step& st, const Stmts& ss) {
    for (auto& s : ss) {
      E v = copied(c, st, s->expr);
      if (s->k == Stmt::Assign && s->dst->k == Expr::Index) { c.stored = v; continue; }
      const Name id = s->k == Stmt::Def ? s->id : s->dst->name;
      const Type ty = s->k == Stmt::Def ? s->ty : s->dst->ty;
      if (is_int(ty.sz) && !has_load(s->expr)) c.numbers[id] = number(c, s->expr); else c.numbers.erase(id);
      if (s->k == Stmt::Def) {
        const Name n = gen.fresh(s->id.s);
        c.out.push_back(mk_def(n, ty, v, s->i));
        c.names[id] = mk_var(n, ty);
      } else {
        c.out.push_back(mk_assign(c.names.at(id), v, s->i));
      }
    }
  }

  // the same for every four neighbouring threads
  static bool same_in_four(const E& e, const Name& g) {
    if (e->k == Expr::Var) return !(e->name == g);
    if (e->k == Expr::BinOpE && e->bop == BinOp::FloorDiv && e->args[0]->k == Expr::Var && e->args[0]->name == g && e->args[1]->k == Expr::Int)
      return e->args[1]->iv > 0 && e->args[1]->iv % 4 == 0;
    for (auto& a : e->args) if (a && !same_in_four(a, g)) return false;
    return true;
  }
  static void constant_part(const E& e, int64_t* c, E* rest) {
    *c = 0;
    *rest = e;
    if (e->k == Expr::Int) { *c = e->iv; *rest = E(); return; }
    if (e->k != Expr::BinOpE || e->bop != BinOp::Add) return;
    for (int side = 0; side < 2; ++side)
      if (e->args[side]->k == Expr::Int) { *c = e->args[side]->iv; *rest = e->args[1 - side]; return; }
  }

  Stmts together(const S& time) {
    if (!(time->k == Stmt::For && time->map.k == GpuMap::None && time->step == 1 && time->lo->k == Expr::Int && time->hi->k == Expr::Int && time->body.size() == 1 &&
          time->body[0]->k == Stmt::Launch))
      return {};
    const int64_t first = time->lo->iv, steps = time->hi->iv - first, pairs = (steps - 1) / 4;
    if (pairs < 2) return {};
    const S launch = time->body[0];
    const Kernel* k = nullptr;
    for (auto& kk : p.kernels) if (kk.name == launch->fname) k = &kk;
    if (!k || k->opaque_body) return {};
    for (size_t q = 0; q < k->params.size(); ++q)
      if (!(launch->args[q]->k == Expr::Var && launch->args[q]->name == k->params[q].id)) return {};

    // the kernel with what a thread's elements have in common taken out
    Kernel kc = *k;
    Options o = opts;
    o.opt_prefetch_steps = false;
    Pass pass(kc, o, gen);
    kc.body = pass.propagate_constants(kc.body);
    if (opts.opt_expand_short_loops) kc.body = pass.expand_short_loops(kc.body, false);
    if (opts.opt_unswitch_uniform) kc.body = pass.hoist_uniform_conditions(kc.body);
    if (opts.opt_if_convert) kc.body = pass.if_convert(kc.body);
    kc.distinct_pointers.clear();
    pass.noalias_scopes(kc.body, false);
    kc.body = pass.share_own_iterations(kc.body);
    Step st;
    if (!match(kc, time, st)) return {};

    const Type vty = Type::scalar(st.sz), pty = Type::pointer(st.sz);
    const Name from = gen.fresh("from"), to = gen.fresh("to"), g = gen.fresh("own"), t = time->id;
    const E gv = mk_var(g, ity), tv = mk_var(t, ity);
    auto element_of = [&](const Name& array, const E& at) {
      const E row = mk_var(st.root->id, ity);
      auto x = std::make_shared<Expr>(*mk_index(mk_var(array, pty), add(mk_binop(BinOp::Mul, row, iint(st.row), ity), at), vty));
      x->dim_idx = {row, at};
      x->dim_shape = {const_extent(st.root), st.row};
      return E(x);
    };
    ranges.clear();
    Interval gr;
    gr.known = true;
    gr.lo = 0;
    gr.hi = st.N - 1;
    ranges[g] = gr;

    // scalars of the row in the launch's first and second step
    std::map<Name, E> in_step[2];
    Stmts defs[2];
    for (int s = 0; s < 2; ++s) {
      if (s == 1) in_step[1][t] = add(tv, iint(1));
      for (auto& d : st.defs) {
        const Name n = s == 0 ? d->id : gen.fresh(d->id.s);
        defs[s].push_back(mk_def(n, d->ty, subst_vars(d->expr, in_step[s]), d->i));
        in_step[s][d->id] = mk_var(n, d->ty);
      }
    }
    // the elements of a step: those of the thread itself, or element `slot` of thread `who`
    auto begin = [&](int step, const E& who) {
      Copy c;
      c.names = in_step[step];
      c.names[st.g] = c.numbers[st.g] = who;
      c.source = [&, who](const E&, const E&) { return E(); };
      return c;
    };
    auto set_slot = [&](Copy& c, int64_t slot) { c.names[st.k] = c.numbers[st.k] = iint(slot); };

    // what the second step takes from other threads: places by the thread's number
    std::vector<E> others;
    bool ok = true;
    auto own_slot = [&](const E& place) -> int64_t {
      E rest;
      if (!affine_unit(place, g, &rest) || rest->k != Expr::Int || rest->iv % st.N != 0) return -1;
      const int64_t s = rest->iv / st.N;
      return s >= 0 && s < st.per ? s : -1;
    };
    std::vector<E> taken;   // what stands for them in the second step
    std::vector<Stmts> later;       // the second step: the thread's shared part, its elements
    std::vector<int64_t> needs;     // the last of the thread's own elements that each takes
    auto second = [&](bool known) {
      Copy c = begin(1, gv);
      int64_t last = -1;
      c.source = [&](const E&, const E& at) -> E {
        const E place = number(c, at);
        const int64_t s = own_slot(place);
        last = std::max(last, s);
        if (s >= 0) return known ? taken[others.size() + s] : mk_float(0.0, st.sz);
        bool plain = true;
        visit_exprs(place, [&](const E& x) {
          if (x->k == Expr::Var && !(x->name == g)) plain = false;
          if (x->k == Expr::Index) plain = false;
        });
        const Interval r = expr_range(place, ranges);
        if (!plain || !r.known || r.lo < 0 || r.hi >= st.row || r.lo / st.N != r.hi / st.N) ok = false;
        size_t q = 0;
        while (q < others.size() && !expr_eq(others[q], place)) ++q;
        if (q == others.size()) { if (known) ok = false; others.push_back(place); }
        return known && ok ? taken[q] : mk_float(0.0, st.sz);
      };
      copy_of(c, st, st.loop->els);
      if (last >= 0) ok = false;   // (what is shared by all elements takes nothing of a single one)
      later = {c.out};
      needs.clear();
      for (int64_t s = 0; s < st.per; ++s) {
        c.out.clear();
        last = -1;
        set_slot(c, s);
        copy_of(c, st, st.loop->body);
        c.out.push_back(mk_assign(element_of(to, s == 0 ? gv : add(gv, iint(s * st.N))), c.stored));
        later.push_back(c.out);
        needs.push_back(last);
      }
    };
    second(false);
    if (!ok) return {};

    // (A product of the first step must not become part of a sum of the second.  What ends in a sum is left alone, since no
    // operation takes one in: kept apart all the same, 1500 steps of 16 layers of 7-mers take 29.6 ms instead of 29.1.)
    auto rounded = [&](const E& v) {
      if (v->k == Expr::BinOpE && (v->bop == BinOp::Add || v->bop == BinOp::Sub) && v->ty.sz == st.sz) return v;
      auto call = std::make_shared<Expr>();
      call->k = Expr::Call;
      call->ty = vty;
      call->sval = "parpy_rounded";
      call->args = {v->ty.sz == st.sz ? v : mk_convert(v, st.sz)};
      return E(call);
    };
    // the first step: own elements, then those of others that the second one takes
    Stmts body;
    std::map<int64_t, E> loaded;   // own elements of `from`, all of them in front
    Copy own = begin(0, gv);
    own.source = [&](const E&, const E& at) -> E {
      const E place = number(own, at);
      const int64_t s = own_slot(place);
      if (s < 0) return element_of(from, copied(own, st, at));
      if (!loaded.count(s)) {
        const Name n = gen.fresh("state");
        body.push_back(mk_def(n, vty, element_of(from, s == 0 ? gv : add(gv, iint(s * st.N)))));
        loaded[s] = mk_var(n, vty);
      }
      return loaded[s];
    };
    copy_of(own, st, st.loop->els);
    std::vector<Stmts> sooner{own.out};
    std::vector<E> mids;
    for (int64_t s = 0; s < st.per; ++s) {
      own.out.clear();
      set_slot(own, s);
      copy_of(own, st, st.loop->body);
      const Name n = gen.fresh("between");
      own.out.push_back(mk_def(n, vty, rounded(own.stored)));
      mids.push_back(mk_var(n, vty));
      sooner.push_back(own.out);
    }
    auto of_other = [&](const E& place) {   // place: in terms of g
      const Interval r = expr_range(place, ranges);
      const int64_t slot = r.lo / st.N;
      const Name who = gen.fresh("other");
      body.push_back(mk_def(who, ity, fold_expr(slot == 0 ? place : mk_binop(BinOp::Sub, place, iint(slot * st.N), ity))));
      Copy c = begin(0, mk_var(who, ity));
      c.source = [&](const E&, const E& at) -> E { return element_of(from, copied(c, st, at)); };
      copy_of(c, st, st.loop->els);
      set_slot(c, slot);
      copy_of(c, st, st.loop->body);
      body.insert(body.end(), c.out.begin(), c.out.end());
      const Name n = gen.fresh("between");
      body.push_back(mk_def(n, vty, rounded(c.stored)));
      return mk_var(n, vty);
    };
    // four values, the same for four neighbouring threads and evenly apart: one for each of them
    bool four = others.size() == 4;
    int64_t c0 = 0, apart = 0;
    E rest0;
    for (size_t q = 0; q < others.size() && four; ++q) {
      int64_t c = 0;
      E rest;
      constant_part(others[q], &c, &rest);
      if (q == 0) { c0 = c; rest0 = rest; four = rest && same_in_four(rest, g); continue; }
      if (q == 1) apart = c - c0;
      four = rest && expr_eq(rest, rest0) && c == c0 + (int64_t)q * apart;
    }
    if (four) {
      const E lane = mk_binop(BinOp::Rem, gv, iint(4), ity);
      const E place = fold_expr(add(rest0, add(iint(c0), mk_binop(BinOp::Mul, lane, iint(apart), ity))));
      const Interval r = expr_range(place, ranges);
      four = r.known && r.lo >= 0 && r.hi < st.row && r.lo / st.N == r.hi / st.N;
      if (four) {
        const E mine = of_other(place);
        for (int q = 0; q < 4; ++q) {
          auto call = std::make_shared<Expr>();
          call->k = Expr::Call;
          call->ty = vty;
          call->sval = "parpy_dpp<" + std::to_string(q * 0x55) + ">";   // quad_perm [q,q,q,q]
          call->args = {mine};
          const Name n = gen.fresh("between");
          body.push_back(mk_def(n, vty, call));
          taken.push_back(mk_var(n, vty));
        }
      }
    }
    if (!four) {
      if ((int64_t)others.size() * 4 > st.per) return {};
      for (auto& place : others) taken.push_back(of_other(place));
    }
    taken.insert(taken.end(), mids.begin(), mids.end());
    second(true);
    if (!ok) return {};
    // every element of the second step as soon as those it takes are there: few values between are alive at a time
    auto put = [&](const Stmts& part) { body.insert(body.end(), part.begin(), part.end()); };
    put(sooner[0]);
    put(later[0]);
    std::vector<bool> done(st.per);
    for (int64_t s = 0; s < st.per; ++s) {
      put(sooner[s + 1]);
      for (int64_t q = 0; q < st.per; ++q)
        if (!done[q] && needs[q] <= s) { put(later[q + 1]); done[q] = true; }
    }
    auto both_steps = clone(st.loop);
    both_steps->id = g;
    both_steps->lo = iint(0);
    both_steps->hi = iint(st.N);
    both_steps->els.clear();
    both_steps->unroll = false;
    both_steps->body = body;

    // ---- kernels: the two steps, and the copies behind the last pair
    auto kernel = [&](const char* what, const Stmts& row) {
      Kernel f;
      f.name = p.name + what + std::to_string(gen.next++);
      f.grid = kc.grid;
      f.block = kc.block;
      f.cached_stores = true;
      f.finished = true;
      auto root = clone(st.root);
      root->body = row;
      f.body = {S(root)};
      // parameters: the two arrays, and what the statements name
      std::set<Name> used;
      visit_stmts(f.body, [&](const S& s) { visit_stmt_exprs(s, [&](const E& x) { if (x->k == Expr::Var) used.insert(x->name); }); });
      KernelParam q;
      q.ty = pty;
      q.id = from;
      f.params.push_back(q);
      q.id = to;
      f.params.push_back(q);
      for (auto& kp : kc.params) if (used.count(kp.id) && !(kp.id == st.even) && !(kp.id == st.odd)) f.params.push_back(kp);
      return f;
    };
    auto launch_of = [&](const Kernel& f, bool odd, const E& now) {
      auto l = clone(launch);
      l->fname = f.name;
      l->args.clear();
      l->args.push_back(mk_var(odd ? st.odd : st.even, pty));
      l->args.push_back(mk_var(odd ? st.even : st.odd, pty));
      for (size_t q = 2; q < f.params.size(); ++q) l->args.push_back(f.params[q].id == t ? now : mk_var(f.params[q].id, f.params[q].ty));
      return S(l);
    };
    auto is_now = [&](int64_t before) { return mk_binop(BinOp::Eq, before == 0 ? tv : mk_binop(BinOp::Sub, tv, iint(before), ity), st.until, bty); };
    Stmts row = defs[0];
    if (!st.until) {
      row.insert(row.end(), defs[1].begin(), defs[1].end());
      row.push_back(both_steps);
    } else {
      Stmts two = defs[1];
      two.push_back(both_steps);
      const std::map<Name, E> arrays{{st.src, mk_var(from, pty)}, {st.dst, mk_var(to, pty)}};
      const Stmts one = rewrite_stmts({st.loop}, [&](const E& x) { return x->k == Expr::Var && arrays.count(x->name) ? arrays.at(x->name) : x; });
      row.push_back(mk_if(mk_binop(BinOp::Lt, add(tv, iint(1)), st.until, bty), two,
                          {mk_if(mk_binop(BinOp::Lt, tv, st.until, bty), one,
                                 {mk_if(mk_binop(BinOp::Or, is_now(0), mk_binop(BinOp::And, is_now(1), mk_binop(BinOp::Gt, tv, iint(first), bty), bty), bty), {copies(st, from, to, element_of)}, {})})}));
    }
    const Kernel f = kernel("_two_steps_", row);
    p.kernels.push_back(f);
    const Name pair = gen.fresh("pair");
    const E at = add(iint(first), mk_binop(BinOp::Mul, mk_var(pair, ity), iint(4), ity));
    const bool odd = first & 1;
    Stmts host{mk_for(pair, iint(0), iint(pairs), 1, {launch_of(f, odd, at), launch_of(f, !odd, add(at, iint(2)))}, LoopPar(), time->i)};
    if (st.until) {
      const Kernel c = kernel("_ends_", {mk_if(is_now(1), {copies(st, from, to, element_of)}, {})});
      p.kernels.push_back(c);
      host.push_back(launch_of(c, odd, iint(first + 4 * pairs)));
    }
    auto singles = clone(time);
    singles->lo = iint(first + 4 * pairs);
    host.push_back(singles);
    // Elements of the step between are never stored, so nothing may see them under another name.
    std::vector<HostArray> ranges_of;
    for (auto& q : kc.params) {
      if (!q.ty.is_pointer() && !q.ty.is_array()) continue;
      HostArray a{q.id, INT64_MAX, q.id == st.even || q.id == st.odd};   // (of unknown length unless it is an argument)
      for (auto& e : p.entry_params) if (e.id == q.id) a.bytes = e.ty.numel() * elem_bytes(e.ty.sz);
      ranges_of.push_back(a);
    }
    const E disjoint = arrays_disjoint(p, ranges_of);
    if (!disjoint) return host;
    auto either = clone(mk_if(disjoint, host, {time}));
    either->fname = "one launch per step";
    return {S(either)};
  }

  template <class F> S copies(const Step& st, const Name& from, const Name& to, F element_of) {
    auto l = clone(st.loop);
    l->id = gen.fresh("ended");
    l->els.clear();
    l->unroll = false;
    const E e = mk_var(l->id, ity);
    l->body = {mk_assign(element_of(to, e), element_of(from, e))};
    return l;
  }

  Stmts walk(const Stmts& ss) {
    Stmts out;
    for (auto& s : ss) {
      const Stmts both = together(s);
      if (!both.empty()) { out.insert(out.end(), both.begin(), both.end()); continue; }
      auto r = clone(s);
      if (s->k == Stmt::For || s->k == Stmt::While || s->k == Stmt::If) {
        r->body = walk(s->body);
        r->els = walk(s->els);
      }
      out.push_back(r);
    }
    return out;
  }

  void run() { p.host = walk(p.host); }
};

}  // namespace

void two_steps(Program& p, const Options& opts, NameGen& gen) { TwoSteps(p, opts, gen).run(); }

}  // namespace hipopt
}  // namespace parpy
