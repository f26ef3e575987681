// gfx950 memory passes, rewrites that change a launch: reductions spread over several workgroups.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

namespace {

// ================================================================ reductions over several workgroups
// A reduction on more threads than a workgroup holds arrives here as two launches: `blocks` workgroups per result, each
// over a contiguous share of the elements, write partial results to a temporary, and a second launch reduces those.
//
//   * The shares are cut at whole vectors, so that the elements are loaded 16 bytes at a time; the last workgroup takes
//     what is left over one by one.  (Shares of 312 500 floats were read one element per access.)
//   * Long shares are split further: workgroups of 256 threads, four times as many.  320 workgroups of 1024 threads put
//     two on a quarter of the compute units; 1280 smaller ones fill all of them alike.
//   * The second launch goes: the workgroup that finishes last (a counter per result, back at zero afterwards) reduces
//     the partial results itself.  They are stored and loaded at device scope, past the caches of the dies.
//
// Sums of 10 rows of 10^7 floats on 32768 threads each: 78.9 -> 70.5 us (5.7 TB/s); 12 rows of 390 000: 12.6 -> 7.8 us; 5 of
// 200 001: 12.7 -> 4.8 us; one of 10^7 on 8192 threads: 100 -> 29.5 us; 3 of 3 000 001 doubles on 8192: 45 -> 24 us.
struct Stages {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;
  Type ity;

  Stages(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()), ity(Type::scalar(o.int_size())) {}

  E iint(int64_t v) { return mk_int(v, isz); }
  E add(E a, E b) { return mk_binop(BinOp::Add, a, b, ity); }
  E mul(E a, E b) { return mk_binop(BinOp::Mul, a, b, ity); }

  Kernel* find(const std::string& name) {
    for (auto& k : p.kernels) if (k.name == name) return &k;
    return nullptr;
  }
  static bool block_loop(const S& s) {
    return s->k == Stmt::For && s->map.k == GpuMap::Block && s->map.mult == 1 && s->map.per == 1 && s->step == 1 && s->lo->k == Expr::Int && s->lo->iv == 0 &&
           s->hi->k == Expr::Int && s->map.n == s->hi->iv && s->els.empty();
  }
  static bool first_thread(const S& s) {   // if (threadIdx.x == 0): assignments
    if (!(s->k == Stmt::If && s->els.empty() && s->expr->k == Expr::BinOpE && s->expr->bop == BinOp::Eq && s->expr->args[0]->k == Expr::ThreadIdx &&
          s->expr->args[0]->iv == 0 && s->expr->args[1]->k == Expr::Int && s->expr->args[1]->iv == 0))
      return false;
    for (auto& b : s->body) if (b->k != Stmt::Assign || b->dst->k != Expr::Index) return false;
    return true;
  }

  // the first launch of such a pair
  struct First {
    std::vector<S> outer;       // loops over the results, outermost first
    Stmts prefix;               // in front of the loop over workgroups
    S blocks;                   // loop over the workgroups of a result
    S init, loop, reduce, name; // running value, share of the elements, its reduction, its name
    S store;                    // the partial result's store
    Name tmp;
    int64_t nb = 0, elements = 0;
  };

  bool match_first(const Kernel& k, First& f) {
    if (k.opaque_body || k.body.size() != 1 || k.block.y != 1 || k.block.z != 1) return false;
    S s = k.body[0];
    int64_t grid = 1;
    for (;;) {
      if (!block_loop(s)) return false;
      grid *= s->map.n;
      // the loop over workgroups is the one whose body holds the reduction
      bool reduces = false;
      for (auto& b : s->body) if (b->k == Stmt::WaveReduce) reduces = true;
      if (reduces) break;
      f.outer.push_back(s);
      S next;
      for (auto& b : s->body) {
        if (b->k == Stmt::For) {
          if (next) return false;
          next = b;
        } else if (next) {
          if (b->k != Stmt::Sync) return false;
        } else {
          if (!(b->k == Stmt::Sync || (b->k == Stmt::Def && b->ty.is_scalar()) || first_thread(b))) return false;
          f.prefix.push_back(b);
        }
      }
      if (!next) return false;
      if (!f.prefix.empty() && !(next->k == Stmt::For && [&] { for (auto& b : next->body) if (b->k == Stmt::WaveReduce) return true; return false; }())) return false;
      s = next;
    }
    if (grid != k.grid.x * k.grid.y * k.grid.z) return false;
    f.blocks = s;
    f.nb = s->hi->iv;
    Stmts body;
    for (auto& b : s->body) if (b->k != Stmt::Sync) body.push_back(b);
    if (body.size() != 5) return false;
    f.init = body[0];
    f.loop = body[1];
    f.reduce = body[2];
    f.name = body[3];
    f.store = body[4];
    if (f.init->k != Stmt::Def || !thread_mapped(f.loop) || f.reduce->k != Stmt::WaveReduce || f.name->k != Stmt::Def || !first_thread(f.store) || f.store->body.size() != 1)
      return false;
    const Name t = f.init->id;
    if (f.reduce->id != t || f.reduce->iv != k.block.x || f.loop->map.n != k.block.x || f.loop->map.dim != 0) return false;
    if (!(f.name->expr->k == Expr::Var && f.name->expr->name == t)) return false;
    const S& st = f.store->body[0];
    E rest;
    if (!(st->expr->k == Expr::Var && st->expr->name == f.name->id && st->dst->args[0]->k == Expr::Var && affine_unit(st->dst->args[1], s->id, &rest))) return false;
    f.tmp = st->dst->args[0]->name;
    // one update of the running value per element, from nothing that this kernel writes
    if (f.loop->body.size() != 1 || f.loop->step != 1 || f.loop->els.size()) return false;
    const S& u = f.loop->body[0];
    if (!(u->k == Stmt::Assign && u->dst->k == Expr::Var && u->dst->name == t)) return false;
    std::set<Name> written{f.tmp};
    for (auto& b : f.prefix) if (b->k == Stmt::If) for (auto& a : b->body) written.insert(a->dst->args[0]->name);
    bool ok = true;
    visit_exprs(u->expr, [&](const E& x) {
      if (x->k == Expr::Call || x->k == Expr::Raw || x->k == Expr::AddrOf) ok = false;
      if (x->k == Expr::Var && written.count(x->name)) ok = false;
    });
    // shares: chunk * b .. min(chunk * b + chunk, elements)
    const E &lo = f.loop->lo, &hi = f.loop->hi;
    if (!(lo->k == Expr::BinOpE && lo->bop == BinOp::Mul && hi->k == Expr::BinOpE && hi->bop == BinOp::Min && hi->args[1]->k == Expr::Int)) return false;
    const E chunk = lo->args[0]->k == Expr::Int ? lo->args[0] : lo->args[1], var = lo->args[0]->k == Expr::Int ? lo->args[1] : lo->args[0];
    if (!(chunk->k == Expr::Int && var->k == Expr::Var && var->name == s->id)) return false;
    f.elements = hi->args[1]->iv;
    return ok && chunk->iv == (f.elements + f.nb - 1) / f.nb;
  }

  // the second launch: the same results, the partial results over the threads of a workgroup, then what is done with them
  bool match_second(const Kernel& k, const First& f, std::map<Name, E>* rename, Stmts* body, S* partials) {
    if (k.opaque_body || k.body.size() != 1 || k.block.y != 1 || k.block.z != 1) return false;
    S s = k.body[0];
    int64_t grid = 1;
    for (size_t q = 0; q < f.outer.size(); ++q) {
      if (!block_loop(s) || s->hi->iv != f.outer[q]->hi->iv) return false;
      grid *= s->map.n;
      (*rename)[s->id] = mk_var(f.outer[q]->id, ity);
      if (q + 1 < f.outer.size()) {
        Stmts inner;
        for (auto& b : s->body) if (b->k != Stmt::Sync) inner.push_back(b);
        if (inner.size() != 1) return false;
        s = inner[0];
      }
    }
    if (f.outer.empty() || grid != k.grid.x * k.grid.y * k.grid.z) return false;
    int reduces = 0;
    for (auto& b : s->body) {
      if (b->k == Stmt::Sync) continue;
      if (b->k == Stmt::For) {
        if (*partials || !thread_mapped(b) || b->map.dim != 0 || b->lo->k != Expr::Int || b->lo->iv != 0 || b->hi->k != Expr::Int || b->hi->iv != f.nb || b->step != 1 || b->els.size())
          return false;
        *partials = b;
      } else if (b->k == Stmt::WaveReduce) {
        if (b->iv != k.block.x || ++reduces > 1) return false;
      } else if (!((b->k == Stmt::Def && b->ty.is_scalar()) || (b->k == Stmt::Assign && b->dst->k == Expr::Var) || first_thread(b))) {
        return false;
      }
      body->push_back(b);
    }
    if (!*partials || reduces != 1) return false;
    // the temporary is only read, where the loop over the partial results stands
    bool ok = true;
    visit_stmts(s->body, [&](const S& b) {
      if (b->k == Stmt::RawStmt) ok = false;
      for (const E& e : {b->expr, b->dst, b->lo, b->hi})
        if (e) visit_exprs(e, [&](const E& x) {
          if (x->k == Expr::Call || x->k == Expr::Raw || x->k == Expr::AddrOf) ok = false;
          E rest;
          if (x->k == Expr::Index && x->args[0]->k == Expr::Var && x->args[0]->name == f.tmp && !affine_unit(x->args[1], (*partials)->id, &rest)) ok = false;
        });
    });
    return ok;
  }

  // number of uses of a temporary on the host
  int launches_with(const Name& n) {
    int c = 0;
    visit_stmts(p.host, [&](const S& s) {
      if (s->k == Stmt::Launch || s->k == Stmt::PersistentLaunch) for (auto& a : s->args) if (mentions(a, n)) { ++c; break; }
    });
    return c;
  }

  bool apply(Stmts& host, size_t at) {
    auto l1 = std::make_shared<Stmt>(*host[at]);
    Kernel* k1 = find(l1->fname);
    First f;
    if (!k1 || !match_first(*k1, f)) return false;
    Name tmp_arg;
    for (size_t q = 0; q < k1->params.size(); ++q)
      if (k1->params[q].id == f.tmp) { if (l1->args[q]->k != Expr::Var) return false; tmp_arg = l1->args[q]->name; }
    size_t alloc = host.size(), second = at + 1;
    for (size_t q = 0; q < at; ++q) if (host[q]->k == Stmt::Alloc && host[q]->id == tmp_arg) alloc = q;
    if (alloc == host.size() || second >= host.size() || host[second]->k != Stmt::Launch || launches_with(tmp_arg) != 2) return false;
    auto l2 = std::make_shared<Stmt>(*host[second]);
    Kernel* k2 = find(l2->fname);
    if (!k2) return false;
    std::map<Name, E> rename;
    Stmts tail;
    S partials;
    // (parameters carry the name of the host variable they are given)
    for (auto* kl : {&l1, &l2}) {
      Kernel* k = kl == &l1 ? k1 : k2;
      for (size_t q = 0; q < k->params.size(); ++q) if (!((*kl)->args[q]->k == Expr::Var && (*kl)->args[q]->name == k->params[q].id)) return false;
    }
    if (!match_second(*k2, f, &rename, &tail, &partials)) return false;

    // ---- shares of whole vectors
    const int64_t V = opts.opt_vectorize ? std::max(1, Pass(*k1, opts, gen).vector_width(f.loop)) : 1;
    const int64_t vectors = f.elements / V;
    int64_t threads = k1->block.x, nb = f.nb, split = 1;
    // (each thread of a long share: at least sixteen vectors)
    if (threads == 1024 && vectors / (nb * threads) >= 16) { split = 4; threads /= 4; nb *= 4; }
    // Few results leave most of the chip idle: twice the workgroups, and again, up to 128 (one row of 10^7 floats on 8192
    // threads: 29.5 us on 32 workgroups, 11.0 on 128, 13.7 on 256, 18.6 on 512 -- all of them count in one word).
    int64_t results = 1;
    for (auto& o : f.outer) results *= o->hi->iv;
    // Workgroups of fewer than 256 threads are there only because the program names that size: the split it names with it,
    // two launches and the temporary between them, stay.  Split further and in one launch they are no faster on the whole:
    // 100 rows of 65536 floats on 1024 threads in workgroups of 128 6.8 us as named, 11.2 so; 10 of 10^6 on 8192 in 128 12.6
    // and 16.3; 1000 of 65536 on 512 in 128 40.3 and 40.9; 37 of 3000 on 256 in 128 6.3 and 5.2; 10 of 10^6 on 2048 in 64
    // 17.9 and 16.5; one of 10^7 on 8192 in 64 28.5 and 26.2.
    const bool named = threads < 256;
    while (!named && nb < 128 && results * nb * threads < 2048 * WAVE_SIZE && vectors / (nb * threads) >= 16) { split *= 2; nb *= 2; }
    const int64_t share = (vectors + nb - 1) / nb;
    const E bv = mk_var(f.blocks->id, ity);
    auto mapped = [&](const Name& id, E lo, E hi, const Stmts& body) {
      auto l = clone(f.loop);
      l->id = id;
      l->lo = lo;
      l->hi = hi;
      l->body = body;
      l->map.n = threads;
      return S(l);
    };
    Stmts elements;
    if (V > 1) {
      Name q = gen.fresh(f.loop->id.s + "_q"), u = gen.fresh(f.loop->id.s + "_u");
      Stmts ib{mk_def(f.loop->id, ity, add(mul(mk_var(q, ity), iint(V)), mk_var(u, ity)))};
      ib.insert(ib.end(), f.loop->body.begin(), f.loop->body.end());
      auto inner = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(u, iint(0), iint(V), 1, ib, LoopPar())));
      inner->unroll = true;
      inner->iv = f.elements % V != 0 || V > 4;   // rows start anywhere, or several elements to a word
      E lo = mul(iint(share), bv);
      elements.push_back(mapped(q, lo, mk_binop(BinOp::Min, add(lo, iint(share)), iint(vectors), ity), {S(inner)}));
      if (f.elements % V != 0)
        elements.push_back(mk_if(mk_binop(BinOp::Eq, bv, iint(nb - 1), Type::scalar(ElemSize::Bool)),
                                 {mapped(f.loop->id, iint(vectors * V), iint(f.elements), f.loop->body)}, {}));
    } else {
      E lo = mul(iint(share), bv);
      elements.push_back(mapped(f.loop->id, lo, mk_binop(BinOp::Min, add(lo, iint(share)), iint(f.elements), ity), f.loop->body));
    }
    // ---- the temporary's index with the new number of workgroups: b + rest, rest a multiple of the old number
    auto reindex = [&](const E& e, const Name& b) {
      return rewrite_expr(e, [&](const E& x) -> E {
        if (split == 1 || x->k != Expr::Index || x->args[0]->k != Expr::Var || x->args[0]->name != f.tmp) return x;
        E rest;
        affine_unit(x->args[1], b, &rest);
        auto n = std::make_shared<Expr>(*x);
        n->args = {x->args[0], fold_expr(add(mk_var(b, ity), mul(rest, iint(split))))};
        n->dim_idx.clear();
        n->dim_shape.clear();
        return n;
      });
    };
    auto reduce1 = clone(f.reduce);
    reduce1->iv = threads;
    const E partial_dst = reindex(f.store->body[0]->dst, f.blocks->id);

    // ---- whether the second launch can go
    // Results that the first launch initialises and the second one reads back must be values known by then: the last
    // workgroup takes the value itself, the initialising stores disappear.  (Workgroups on different dies must not store
    // to one element.)  From five elements per thread on; with fewer, a share is little more than one access, the time
    // is that of the launches themselves and both forms stay as they are.
    bool fuse = !named && f.elements >= 5 * nb * threads && elem_bytes(f.reduce->ty.sz) >= 4 && !opts.persistent_loops;
    std::vector<std::pair<E, E>> known;   // element -> value
    std::map<Name, E> defs;
    for (auto& b : f.prefix) {
      if (b->k == Stmt::Def) { if (b->expr->k == Expr::Float || b->expr->k == Expr::Int) defs[b->id] = b->expr; else fuse = false; }
      if (b->k == Stmt::If)
        for (auto& a : b->body) {
          E v = subst_vars(a->expr, defs);
          if (v->k != Expr::Float && v->k != Expr::Int) fuse = false;
          known.push_back({a->dst, v});
        }
    }
    Stmts finish;
    if (fuse) {
      auto device_load = [&](const E& x) {
        auto a = std::make_shared<Expr>(*x);
        a->k = Expr::AddrOf;
        auto c = std::make_shared<Expr>();
        c->k = Expr::Call;
        c->ty = x->ty;
        c->sval = "parpy_device_load";
        c->args = {E(a)};
        return E(c);
      };
      std::set<Name> stored;   // elements this kernel initialised: every read of them must be a known one
      for (auto& kv : known) stored.insert(kv.first->args[0]->name);
      auto value = [&](const E& e0) {
        E e = reindex(subst_vars(e0, rename), partials->id);
        return rewrite_expr(e, [&](const E& x) -> E {
          if (x->k != Expr::Index || x->args[0]->k != Expr::Var) return x;
          if (x->args[0]->name == f.tmp) return device_load(x);
          for (auto& kv : known) if (expr_eq(kv.first, x)) return kv.second;
          if (stored.count(x->args[0]->name)) fuse = false;
          return x;
        });
      };
      std::function<Stmts(const Stmts&)> take = [&](const Stmts& ss) {
        Stmts out;
        for (auto& s : ss) {
          auto r = clone(s);
          if (s->expr && s->k != Stmt::If) r->expr = value(s->expr);
          if (s->dst && s->dst->k == Expr::Index) r->dst = subst_vars(s->dst, rename);
          if (s->k == Stmt::For) { r->map.n = threads; r->hi = iint(nb); }
          if (s->k == Stmt::WaveReduce) r->iv = threads;
          r->body = take(s->body);
          out.push_back(r);
        }
        return out;
      };
      finish = take(tail);
      // a result that is initialised and then not written by the second launch would be lost
      for (auto& kv : known) {
        bool again = false;
        visit_stmts(finish, [&](const S& s) { if (s->k == Stmt::Assign && s->dst->k == Expr::Index && expr_eq(s->dst, kv.first)) again = true; });
        if (!again) fuse = false;
      }
    }

    // ---- the new first launch
    Stmts body{f.init};
    body.insert(body.end(), elements.begin(), elements.end());
    body.push_back(reduce1);
    body.push_back(f.name);
    if (fuse) {
      auto addr = std::make_shared<Expr>(*partial_dst);
      addr->k = Expr::AddrOf;
      auto store = std::make_shared<Expr>();
      store->k = Expr::Call;
      store->ty = Type::scalar(ElemSize::Bool);
      store->sval = "parpy_device_store";
      store->args = {E(addr), f.store->body[0]->expr};
      body.push_back(mk_if(f.store->expr, {mk_def(gen.fresh("stored"), Type::scalar(ElemSize::Bool), store)}, {}));
      E which = iint(0);
      for (auto& o : f.outer) which = add(mul(which, o->hi), mk_var(o->id, ity));
      const std::string counters = p.name + "_done_" + std::to_string(gen.next++);
      p.preamble.push_back("static __device__ unsigned " + counters + "[" + std::to_string(results) + "];   // workgroups that are done, per result; zero between launches");
      auto last = std::make_shared<Expr>();
      last->k = Expr::Call;
      last->ty = Type::scalar(ElemSize::Bool);
      last->sval = "parpy_last_workgroup";
      last->args = {mk_raw(counters, Type::pointer(ElemSize::U32)), fold_expr(which), mk_raw(std::to_string(nb) + "u", Type::scalar(ElemSize::U32))};
      Name is_last = gen.fresh("last");
      body.push_back(mk_def(is_last, Type::scalar(ElemSize::Bool), last));
      body.push_back(mk_if(mk_var(is_last, Type::scalar(ElemSize::Bool)), finish, {}));
    } else {
      body.push_back(mk_if(f.store->expr, {mk_assign(partial_dst, f.store->body[0]->expr)}, {}));
    }
    auto blocks = clone(f.blocks);
    blocks->hi = iint(nb);
    blocks->map.n = nb;
    blocks->body = body;
    S nest = blocks;
    for (size_t q = f.outer.size(); q-- > 0;) {
      auto o = clone(f.outer[q]);
      Stmts inner;
      if (q + 1 == f.outer.size() && !fuse) inner = f.prefix;
      inner.push_back(nest);
      o->body = inner;
      nest = o;
    }
    k1->body = {nest};
    k1->block.x = threads;
    (f.blocks->map.dim == 0 ? k1->grid.x : f.blocks->map.dim == 1 ? k1->grid.y : k1->grid.z) = nb;
    l1->grid = k1->grid;
    l1->block = k1->block;
    auto a = std::make_shared<Stmt>(*host[alloc]);
    a->iv *= split;
    host[alloc] = a;
    if (fuse) {
      for (size_t q = 0; q < k2->params.size(); ++q) {
        bool has = false;
        for (auto& kp : k1->params) if (kp.id == k2->params[q].id) { has = true; if (!k2->params[q].read_only) kp.read_only = false; }
        if (!has) { k1->params.push_back(k2->params[q]); l1->args.push_back(l2->args[q]); }
      }
      // parameters that nothing mentions any more would only be copied
      host[at] = l1;
      host.erase(host.begin() + second);
      const std::string gone = k2->name;
      p.kernels.erase(std::remove_if(p.kernels.begin(), p.kernels.end(), [&](const Kernel& k) { return k.name == gone; }), p.kernels.end());
    } else {
      host[at] = l1;
      if (split > 1) {
        std::function<Stmts(const Stmts&)> widen = [&](const Stmts& ss) {
          Stmts out;
          for (auto& s : ss) {
            auto r = clone(s);
            if (s->expr) r->expr = reindex(s->expr, partials->id);
            if (s == partials) r->hi = iint(nb);
            r->body = widen(s->body);
            r->els = widen(s->els);
            out.push_back(r);
          }
          return out;
        };
        k2->body = widen(k2->body);
      }
    }
    return true;
  }

  void walk(Stmts& host) {
    for (size_t q = 0; q < host.size(); ++q)
      if (host[q]->k == Stmt::Launch) apply(host, q);
  }

  void run() { walk(p.host); }
};

}  // namespace

void reduction_stages(Program& p, const Options& opts, NameGen& gen) { Stages(p, opts, gen).run(); }

}  // namespace hipopt
}  // namespace parpy
