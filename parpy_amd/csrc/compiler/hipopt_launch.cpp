// gfx950 memory passes, rewrites that change a launch: transposed staging of column gathers, lane groups, coarsened element-wise launches.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

namespace {

// ================================================================ transposed staging of column gathers
// A read-only matrix X[K, N] that a kernel only reads as X[d, c] with d the
// variable of an innermost sequential loop over all K rows and c fixed per
// thread is a column gather: every step of the loop touches one 4-byte word
// in each of up to 64 different cache lines per wavefront.  Staging X^T once
// in a device temporary turns each thread's column into K contiguous words
// (dwordx4 loads, whole cache lines used).  The transposition costs two
// passes over X; it is applied to kernels launched once per call.
struct GatherTranspose {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;

  GatherTranspose(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()) {}

  struct Cand { Name arr; int64_t K = 0, N = 0, pitch = 0; ElemSize sz = ElemSize::F32; bool ok = true; bool seen = false; };

  void scan_expr(const E& e, const std::vector<std::pair<Name, int64_t>>& seq_loops, std::map<Name, Cand>& cands) {
    if (!e) return;
    if ((e->k == Expr::Index || e->k == Expr::AddrOf) && e->args[0]->k == Expr::Var && cands.count(e->args[0]->name)) {
      Cand& c = cands[e->args[0]->name];
      bool good = e->k == Expr::Index && e->dim_idx.size() == 2 && e->dim_idx[0]->k == Expr::Var && !seq_loops.empty() &&
                  e->dim_idx[0]->name == seq_loops.back().first && e->dim_shape[0] == seq_loops.back().second &&
                  !mentions(e->dim_idx[1], seq_loops.back().first) && !has_load(e->dim_idx[1]);
      if (good && c.seen && (c.K != e->dim_shape[0] || c.N != e->dim_shape[1])) good = false;
      if (!good) c.ok = false;
      else { c.seen = true; c.K = e->dim_shape[0]; c.N = e->dim_shape[1]; c.sz = e->ty.sz; }
      scan_expr(e->args[1], seq_loops, cands);
      return;
    }
    if (e->k == Expr::Var && cands.count(e->name)) { cands[e->name].ok = false; return; }
    for (auto& a : e->args) scan_expr(a, seq_loops, cands);
  }

  void scan(const Stmts& ss, std::vector<std::pair<Name, int64_t>>& seq_loops, std::map<Name, Cand>& cands) {
    for (auto& s : ss) {
      scan_expr(s->dst, seq_loops, cands);
      scan_expr(s->expr, seq_loops, cands);
      scan_expr(s->lo, seq_loops, cands);
      scan_expr(s->hi, seq_loops, cands);
      for (auto& a : s->args) scan_expr(a, seq_loops, cands);
      bool seq = s->k == Stmt::For && s->map.k == GpuMap::None && s->step == 1 && s->lo->k == Expr::Int && s->lo->iv == 0 &&
                 s->hi->k == Expr::Int;
      // only innermost loops qualify: a nested loop hides the enclosing one
      if (seq) seq_loops.emplace_back(s->id, s->hi->iv);
      else if (s->k == Stmt::For || s->k == Stmt::While) seq_loops.emplace_back(Name{"", -1}, -1);
      scan(s->body, seq_loops, cands);
      if (s->k == Stmt::For || s->k == Stmt::While) seq_loops.pop_back();
      scan(s->els, seq_loops, cands);
    }
  }

  static constexpr int64_t CACHE_LINE = 128, FIXED_MEMORY = int64_t(16) << 20;   // (PARPY_HIP_SCRATCH_BYTES)
  static bool tiles(const Cand& c) { return c.K >= 16 && c.N >= 64 && elem_bytes(c.sz) >= 4; }

  Kernel make_transpose(const Name& x, const Name& xt, const Cand& c) {
    KernelParam px, pxt;
    px.id = x;
    px.ty = Type::pointer(c.sz);
    px.read_only = true;
    pxt.id = xt;
    pxt.ty = Type::pointer(c.sz);
    if (tiles(c)) {
      // tiles turned round in LDS by a device helper, whole lines on both sides (edge tiles are guarded)
      const int64_t rows = 256 / elem_bytes(c.sz);
      Kernel k;
      k.name = p.name + "_transpose_" + x.s + "_" + std::to_string(gen.next++);
      k.grid.x = (c.N + 63) / 64;
      k.grid.y = (c.K + rows - 1) / rows;
      k.block.x = 256;
      k.lds_bytes = rows * 65 * elem_bytes(c.sz);
      k.cached_stores = true;
      k.opaque_body = true;
      k.body = {mk_rawstmt("parpy_transpose_tile<" + std::string(elem_ctype(c.sz)) + ", " + std::to_string(c.K) + ", " +
                           std::to_string(c.N) + (c.pitch == c.K ? "" : ", " + std::to_string(c.pitch)) + ">(" + x.str() + ", " + xt.str() + ");")};
      k.params = {px, pxt};
      return k;
    }
    // one thread per column c; reads are coalesced across the wavefront, each thread writes its own row of X^T
    Type ity = Type::scalar(isz);
    Type elem = Type::scalar(c.sz);
    Name cv = gen.fresh("c"), dv = gen.fresh("d");
    E ce = mk_var(cv, ity), de = mk_var(dv, ity);
    E src = mk_index(mk_var(x, Type::pointer(c.sz)), fold_expr(mk_binop(BinOp::Add, mk_binop(BinOp::Mul, de, mk_int(c.N, isz), ity), ce, ity)), elem);
    E dst = mk_index(mk_var(xt, Type::pointer(c.sz)), fold_expr(mk_binop(BinOp::Add, mk_binop(BinOp::Mul, ce, mk_int(c.K, isz), ity), de, ity)), elem);
    S inner = mk_for(dv, mk_int(0, isz), mk_int(c.K, isz), 1, {mk_assign(dst, src)}, LoopPar());
    LoopPar par;
    par.nthreads = c.N;
    par.tpb = 256;
    auto outer = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(cv, mk_int(0, isz), mk_int(c.N, isz), 1, {inner}, par)));
    int64_t n = (c.N + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    Kernel k;
    k.name = p.name + "_transpose_" + x.s + "_" + std::to_string(gen.next++);
    if (n > 256) {
      outer->map.k = GpuMap::ThreadBlock;
      outer->map.n = n;
      outer->map.tpb = 256;
      k.grid.x = (n + 255) / 256;
      k.block.x = 256;
    } else {
      outer->map.k = GpuMap::Thread;
      outer->map.n = n;
      k.block.x = n;
    }
    outer->map.dim = 0;
    k.body = {S(outer)};
    k.cached_stores = true;
    k.params = {px, pxt};
    return k;
  }

  // the matrices that a launch reads in this way, rows of their copies on cache lines where `pitch` says so
  std::map<Name, Cand> candidates(const Kernel& k) {
    std::map<Name, Cand> cands;
    std::set<Name> written;
    visit_stmts(k.body, [&](const S& st) {
      if (st->k == Stmt::Assign && st->dst->k == Expr::Index)
        visit_exprs(st->dst->args[0], [&](const E& x) { if (x->k == Expr::Var) written.insert(x->name); });
      if ((st->k == Stmt::Def && !st->ty.is_scalar()) || (st->k == Stmt::Assign && st->dst->k == Expr::Var && !st->dst->ty.is_scalar()))
        visit_exprs(st->expr, [&](const E& x) { if (x->k == Expr::Var) written.insert(x->name); });  // aliased: leave alone
    });
    for (auto& q : k.params)
      if (q.ty.is_pointer() && !written.count(q.id)) { Cand c; c.arr = q.id; cands[q.id] = c; }
    std::vector<std::pair<Name, int64_t>> seq_loops;
    scan(k.body, seq_loops, cands);
    std::map<Name, Cand> out;
    for (auto& kv : cands) {
      Cand c = kv.second;
      // worth it when the stride is at least a cache line and the matrix is re-read many times
      if (!c.ok || !c.seen || c.N < 32 || c.K < 8 || c.K * c.N * elem_bytes(c.sz) > (int64_t(1) << 30)) continue;
      const int64_t line = CACHE_LINE / elem_bytes(c.sz);
      c.pitch = tiles(c) && c.K >= 8 * line ? (c.K + line - 1) / line * line : c.K;
      out[kv.first] = c;
    }
    return out;
  }

  // Rows of the copies start on cache lines where they are longer than eight of them: eight lanes that read 128 bytes of a row
  // then ask for one line, not for two (2500 rows of 1000 doubles, 50 000 products 51.7 -> 42.5 us, 9000 of 780 floats, 270 000:
  // 119 -> 107, 12 000 of 331 doubles, 720 000: 262 -> 253; shorter rows do not repay the lines that are added: 8192 of 97
  // floats 30.6 -> 31.4).
  // A run that may allocate nothing has a fixed amount of memory for the program's temporaries at a time, and a captured one
  // what the plan keeps for all of them: where they fit without the lines they fit with them.
  static bool lines_fit(int64_t plain, int64_t lined, int64_t others, int64_t of_program) {
    return of_program <= KEPT_MEMORY && (plain > FIXED_MEMORY || others + lined <= FIXED_MEMORY / 8 * 7);
  }

  void run() {
    Stmts host;
    std::vector<Kernel> extra;
    auto kernel_of = [&](const S& s) -> Kernel* {
      if (s->k != Stmt::Launch) return nullptr;
      Kernel* k = nullptr;
      for (auto& kk : p.kernels)
        if (kk.name == s->fname) k = &kk;
      return k;
    };
    const int64_t others = temporaries(p.host);
    auto bytes_of = [](const Cand& c, int64_t pitch) { return (pitch * c.N * elem_bytes(c.sz) + 255) / 256 * 256; };
    int64_t of_program = others;
    for (auto& s : p.host)
      if (const Kernel* k = kernel_of(s))
        for (auto& kv : candidates(*k)) of_program += bytes_of(kv.second, kv.second.pitch);
    for (auto& s : p.host) {
      Kernel* k = kernel_of(s);
      if (!k) { host.push_back(s); continue; }
      std::map<Name, Cand> cands = candidates(*k);
      std::map<Name, Name> staged;
      Stmts pre, post;
      int64_t plain = 0, lined = 0;
      for (auto& kv : cands) {
        plain += bytes_of(kv.second, kv.second.K);
        lined += bytes_of(kv.second, kv.second.pitch);
      }
      const bool lines = lines_fit(plain, lined, others, of_program);
      for (auto& kv : cands) {
        Cand& c = kv.second;
        if (!lines) c.pitch = c.K;
        Name xt = gen.fresh(c.arr.s + "_T");
        staged[c.arr] = xt;
        auto a = std::make_shared<Stmt>();
        a->k = Stmt::Alloc;
        a->id = xt;
        a->ty = Type::scalar(c.sz);
        a->iv = c.pitch * c.N;
        pre.push_back(a);
        Kernel tk = make_transpose(c.arr, xt, c);
        auto l = std::make_shared<Stmt>();
        l->k = Stmt::Launch;
        l->fname = tk.name;
        l->grid = tk.grid;
        l->block = tk.block;
        // the launch argument is whatever the consumer was given for this parameter
        E src_arg;
        for (size_t i = 0; i < k->params.size(); ++i)
          if (k->params[i].id == c.arr) src_arg = s->args[i];
        l->args = {src_arg, mk_var(xt, Type::pointer(c.sz))};
        pre.push_back(l);
        extra.push_back(tk);
        auto f = std::make_shared<Stmt>();
        f->k = Stmt::Free;
        f->id = xt;
        post.insert(post.begin(), f);   // (the last one first, as fixed memory is given back)
      }
      if (staged.empty()) { host.push_back(s); continue; }
      Type ity = Type::scalar(isz);
      k->body = rewrite_stmts(k->body, [&](const E& e) -> E {
        if (e->k == Expr::Index && e->args[0]->k == Expr::Var && staged.count(e->args[0]->name)) {
          const Cand& c = cands[e->args[0]->name];
          auto n = std::make_shared<Expr>(*e);
          E idx = fold_expr(mk_binop(BinOp::Add, mk_binop(BinOp::Mul, e->dim_idx[1], mk_int(c.pitch, isz), ity), e->dim_idx[0], ity));
          n->args = {mk_var(staged.at(e->args[0]->name), Type::tensor(c.sz, {c.N, c.pitch}), e->i), idx};
          n->dim_idx = {e->dim_idx[1], e->dim_idx[0]};
          n->dim_shape = {c.N, c.pitch};
          return n;
        }
        return e;
      });
      auto ns = std::make_shared<Stmt>(*s);
      for (size_t i = 0; i < k->params.size(); ++i)
        if (staged.count(k->params[i].id)) {
          Name xt = staged.at(k->params[i].id);
          ns->args[i] = mk_var(xt, Type::pointer(k->params[i].ty.sz));
          k->params[i].id = xt;
        }
      for (auto& q : pre) host.push_back(q);
      host.push_back(ns);
      for (auto& q : post) host.push_back(q);
    }
    for (auto& e : extra) p.kernels.push_back(e);
    p.host = host;
  }
};

// ================================================================ lane groups for per-thread dot products
// A grid-wide loop whose every iteration runs a long sequential sum over unit-stride rows
// (`t += X[a*K + d] * Y[b*K + d]`, d = 0..K) makes each lane walk its own rows: one wavefront load
// touches 64 different cache lines and uses 16 bytes of each, and the line is fetched again for
// each of the following iterations unless it survives in L1.  Here G = 8 adjacent lanes share one
// iteration instead: lane g takes the g-th 16-byte piece of every 128-byte line, so each line is
// requested once, and the eight partial sums are added with three DPP steps.  The launch grows by
// G; statements after the sum that store to memory are executed by lane 0 of each group.
struct LaneSplit {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;
  static constexpr int64_t G = 8;
  Stmts in_slabs;              // what takes the place of the launch at hand where `room` says so
  E room;
  std::vector<Kernel> extra;
  std::vector<StmtP> wholes;   // their launches that add parts up
  int64_t taken = 0;           // bytes of the program's temporaries

  LaneSplit(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()) {}

  // the sum loop: a sequential loop over [0, K) whose body is `acc = acc + e`, where acc is a scalar
  // variable or an array element that does not depend on d, and all d-dependent accesses are unit-stride
  bool sum_loop(const S& s, int* vec, E* term_out) {
    if (!(s->k == Stmt::For && s->map.k == GpuMap::None && !s->unroll && s->step == 1 && s->body.size() == 1)) return false;
    if (!(s->lo->k == Expr::Int && s->lo->iv == 0 && s->hi->k == Expr::Int)) return false;
    const S& a = s->body[0];
    if (a->k != Stmt::Assign) return false;
    const E& acc = a->dst;
    bool scalar_acc = acc->k == Expr::Var && acc->ty.is_scalar();
    bool elem_acc = acc->k == Expr::Index && acc->args[0]->k == Expr::Var && !mentions(acc->args[1], s->id) && !has_load(acc->args[1]);
    if (!(scalar_acc || elem_acc) || !is_float(acc->ty.sz)) return false;
    if (!(a->expr->k == Expr::BinOpE && a->expr->bop == BinOp::Add)) return false;
    const E &l = a->expr->args[0], &r = a->expr->args[1];
    E term;
    if (expr_eq(l, acc)) term = r;
    else if (expr_eq(r, acc)) term = l;
    if (!term) return false;
    const Name& acc_name = scalar_acc ? acc->name : acc->args[0]->name;
    if (mentions(term, acc_name)) return false;
    int v = 0, loads = 0;
    bool ok = true;
    visit_exprs(term, [&](const E& x) {
      if (x->k == Expr::Call || x->k == Expr::AddrOf) ok = false;
      if (x->k != Expr::Index) return;
      if (!mentions(x->args[1], s->id)) return;
      E rest;
      if (!affine_unit(x->args[1], s->id, &rest)) { ok = false; return; }
      int w = elem_bytes(x->ty.sz) == 4 ? 4 : elem_bytes(x->ty.sz) == 8 ? 2 : 0;
      if (w == 0) { ok = false; return; }
      v = v == 0 ? w : std::min(v, w);
      ++loads;
    });
    if (!ok || loads < 1) return false;
    // Two vectors for every lane; one for products of two rows, where a lane on its own would walk twice as many lines.
    // (A product over 33 doubles, 204 600 of them: 21.5 us one thread each, 15.2 shared; over 777 floats, 150 050 of
    // them, no whole number of vectors: 294 and 56 us.)
    if (s->hi->iv < v * G * (loads >= 2 ? 1 : 2)) return false;
    *vec = v;
    *term_out = term;
    return true;
  }

  static constexpr int64_t ROW_REGISTERS = 48, L2_OF_A_DIE = int64_t(4) << 20;   // (registers for 16 bytes per lane and round of three rows)

  // the two rows of a product: the one that neighbouring iterations may have in common, and the other
  bool rows_of(const S& loop, const E& term, E* common, E* other, bool* swapped) {
    const E& acc = loop->body[0]->dst;
    if (!(term->k == Expr::BinOpE && term->bop == BinOp::Mul)) return false;
    E x = term->args[0], y = term->args[1];
    for (const E& e : {x, y})
      if (e->k != Expr::Index || e->args[0]->k != Expr::Var || e->ty.sz != acc->ty.sz || !mentions(e->args[1], loop->id) || has_load(e->args[1])) return false;
    // (in common: of the array that the program passes, where the other is a copy made for this launch)
    auto passed = [&](const E& e) {
      for (auto& q : p.entry_params) if (q.id == e->args[0]->name) return true;
      return false;
    };
    *swapped = !passed(x) && passed(y);
    *common = *swapped ? y : x;
    *other = *swapped ? x : y;
    return true;
  }

  // The products of iterations `fv` and the one behind it over `len` elements of two rows, from vector `start` of them on (from the
  // first where it is null): `names` of each iteration's values, `sum` of its products in all lanes.  Where that is no whole
  // number of rounds of the group, it ends with the rows: their last vector is moved to end there, and what it has of the one in
  // front of it and what lies behind counts as zero.
  Stmts two_sums(const S& root, size_t pos, int vec, const E& x, const E& y, bool swapped, const E& fv, const E& gv, const E& start, int64_t len,
                 std::map<Name, E>* names, Name* sum) {
    const S& loop = root->body[pos];
    const E& acc = loop->body[0]->dst;
    const int64_t N = root->hi->iv, K = loop->hi->iv;
    const Type ity = Type::scalar(isz), bty = Type::scalar(ElemSize::Bool), ety = Type::scalar(acc->ty.sz);
    auto iint = [&](int64_t v) { return mk_int(v, isz); };
    auto add = [&](const E& a, const E& b) { return mk_binop(BinOp::Add, a, b, ity); };
    auto mul = [&](const E& a, int64_t b) { return mk_binop(BinOp::Mul, a, iint(b), ity); };
    Stmts body;
    auto reg = [&](const Name& name, const E& c) {
      auto e = std::make_shared<Expr>();
      e->k = Expr::RegElem;
      e->ty = ety;
      e->name = name;
      e->args = {c};
      return E(e);
    };
    auto unrolled = [&](const Name& id, int64_t n, const Stmts& ss) {
      auto l = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(id, iint(0), iint(n), 1, ss, LoopPar(), loop->i)));
      l->unroll = true;
      return l;
    };
    // Pieces of as many rounds as registers hold of three rows.  The place of each follows from the sums of the one in front of it
    // as far as the device compiler can tell, which would load them all in front otherwise (eight rounds of doubles in 135 registers,
    // 83 so) and in a loop lose track of which elements are one vector.  Two rounds of doubles, which leave a SIMD more
    // wavefronts (300 000 products over 900 doubles 193 us, 214 with four, over 1024 114.5 and 115.8).
    const int64_t chunk = vec * G, rounds = (len + chunk - 1) / chunk, most = ROW_REGISTERS / 12, of_piece = rounds <= most ? rounds : vec == 2 ? 2 : most;
    const bool single = rounds <= of_piece;
    auto declare = [&](const Name& name) {
      auto d = std::make_shared<Stmt>();
      d->k = Stmt::RegDecl;
      d->id = name;
      d->ty = ety;
      d->iv = of_piece * vec;
      body.push_back(S(d));
    };
    for (int u = 0; u < 2; ++u) {
      Name i = gen.fresh(root->id.s);
      E at = u == 0 ? fv : add(fv, iint(1));
      if (u == 1 && N % 2 != 0) at = mk_binop(BinOp::Min, at, iint(N - 1), ity);   // (the last one again, not stored)
      body.push_back(mk_def(i, ity, at, root->i));
      names[u][root->id] = mk_var(i, ity);
      sum[u] = gen.fresh(acc->name.s);
      for (size_t q = 0; q < pos; ++q) {
        const S& st = root->body[q];
        const bool total = st->id == acc->name;
        Name n = total ? sum[u] : gen.fresh(st->id.s);
        E e = total ? mk_float(0.0, acc->ty.sz) : subst_vars(st->expr, names[u]);
        names[u][st->id] = mk_var(n, st->ty);
        body.push_back(mk_def(n, st->ty, e, st->i));
      }
    }
    Name xs = gen.fresh("row"), ys[2] = {gen.fresh("other"), gen.fresh("other")};
    declare(xs);
    declare(ys[0]);
    declare(ys[1]);
    auto total = [&](int u) { return mk_assign(mk_var(sum[u], ety), mk_raw("parpy_sum8(" + sum[u].str() + ")", ety)); };
    // `n` rounds behind the first `from`; `ends`: the rows end in the last of them
    auto piece = [&](const E& from, int64_t n, bool ends) {
      Stmts ss;
      // the first element of round c's vector, and where it stands
      auto vector = [&](const E& c) {
        E v = add(mul(c, G), gv);
        if (from) v = add(mul(from, G), v);
        return mul(start ? add(start, v) : v, vec);
      };
      auto place = [&](const E& c) { return ends ? mk_binop(BinOp::Min, vector(c), iint(K - vec), ity) : vector(c); };
      // the group's pieces of a row into registers
      auto load = [&](const Name& name, const E& e) {
        Name c = gen.fresh("c"), u = gen.fresh(loop->id.s + "_u"), d = gen.fresh(loop->id.s);
        auto each = unrolled(u, vec, {mk_def(d, ity, add(place(mk_var(c, ity)), mk_var(u, ity)), loop->i),
                                      mk_assign(reg(name, add(mul(mk_var(c, ity), vec), mk_var(u, ity))), subst_vars(e, {{loop->id, mk_var(d, ity)}}))});
        if (K % vec != 0) each->iv = 1;   // (rows that start at any element)
        return S(unrolled(c, n, {S(each)}));
      };
      ss.push_back(load(xs, subst_vars(x, names[0])));
      for (int u = 0; u < 2; ++u) ss.push_back(load(ys[u], subst_vars(y, names[u])));
      for (int u = 0; u < 2; ++u) {
        if (u == 1) {
          E a = subst_vars(subst_vars(x, names[0])->args[1], {{loop->id, iint(0)}}), b = subst_vars(subst_vars(x, names[1])->args[1], {{loop->id, iint(0)}});
          ss.push_back(mk_if(mk_binop(BinOp::Neq, fold_expr(a), fold_expr(b), bty), {load(xs, subst_vars(x, names[1]))}, {}));
        }
        Name c = gen.fresh("c");
        const E cv = mk_var(c, ity), sv = mk_var(sum[u], ety);
        E l = reg(xs, cv), r = reg(ys[u], cv);
        if (swapped) std::swap(l, r);
        E product = mk_binop(BinOp::Mul, l, r, ety);
        if (ends) {
          const E round = mk_binop(BinOp::FloorDiv, cv, iint(vec), ity);
          const E own = mk_binop(BinOp::Geq, add(place(round), mk_binop(BinOp::Rem, cv, iint(vec), ity)), vector(round), bty);
          product = mk_ifexpr(own, product, mk_float(0.0, acc->ty.sz), ety);
        }
        ss.push_back(S(unrolled(c, n * vec, {mk_assign(sv, mk_binop(BinOp::Add, sv, product, ety), loop->i)})));
        if (single) ss.push_back(total(u));
      }
      return ss;
    };
    for (int64_t from = 0; from < rounds; from += of_piece) {
      const int64_t n = std::min(of_piece, rounds - from);
      if (from > 0) body.push_back(mk_rawstmt("asm(\"\" : \"+v\"(" + gv->name.str() + "), \"+v\"(" + sum[0].str() + "), \"+v\"(" + sum[1].str() + "));"));
      const Stmts ss = piece(from > 0 ? iint(from) : E(), n, len % chunk != 0 && from + n == rounds);
      body.insert(body.end(), ss.begin(), ss.end());
    }
    if (!single) for (int u = 0; u < 2; ++u) body.push_back(total(u));
    return body;
  }

  // Two neighbouring iterations per group for products of two short rows, `t += X[a*K + d] * Y[b*K + d]` with a and b from
  // memory.  Neighbours mostly have one row in common (non-zeros sorted by rows or columns): the group loads it once and
  // tests whether the second iteration's is another one; a quarter of the 16-byte pieces that pass through L1 go away.
  // 655360 products over 128 floats out of a 4 MiB table: 27.9 -> 21.6 us (four iterations 22.4), over 64 floats 19.4 ->
  // 15.1, 262144 over 128 out of 1 MiB 10.7 -> 8.8.  Three rows are in registers at a time, 16 bytes of each per lane and
  // round, and 48 registers of them leave a SIMD its wavefronts: not for rows of more than 512 bytes (256 floats: 37.4 ->
  // 43.1).  Nor for tables that the 4 MiB L2 of a die does not hold, where the pieces come from farther than L1 anyway (8 MiB:
  // 43.9 -> 45.7), nor for launches that run at once as they are.
  bool pair(Kernel& k, const StmtP& launch, const S& root, size_t pos, int vec, const E& term) {
    const S& loop = root->body[pos];
    const E& acc = loop->body[0]->dst;
    const int64_t N = root->hi->iv, K = loop->hi->iv, rounds = K / (vec * G);
    if (acc->k != Expr::Var || K % (vec * G) != 0 || 3 * rounds * 4 > ROW_REGISTERS || N * G <= 2 * 256 * 2048) return false;
    E x, y;
    bool swapped = false;
    if (!rows_of(loop, term, &x, &y, &swapped)) return false;
    int64_t table = elem_bytes(y->ty.sz);
    for (int64_t d : y->dim_shape) table *= d;
    if (y->dim_shape.empty() || table > L2_OF_A_DIE) return false;
    std::set<Name> from_memory;
    bool zero = false;
    for (size_t q = 0; q < pos; ++q) {
      const S& st = root->body[q];
      if (st->k != Stmt::Def || !st->ty.is_scalar()) return false;
      if (st->id == acc->name) { zero = st->expr->k == Expr::Float && st->expr->fv == 0.0; continue; }
      if (mentions(st->expr, acc->name)) return false;
      if (has_load(st->expr)) from_memory.insert(st->id);
    }
    bool stores = false;
    for (size_t q = pos + 1; q < root->body.size(); ++q) {
      const S& st = root->body[q];
      if (st->k == Stmt::Assign && st->dst->k == Expr::Index) stores = true;
      else if (st->k != Stmt::Def || stores) return false;
    }
    auto selected = [&](const E& e) { bool f = false; visit_exprs(e->args[1], [&](const E& v) { if (v->k == Expr::Var && from_memory.count(v->name)) f = true; }); return f; };
    if (!zero || !stores || !selected(x) || !selected(y)) return false;

    const Type ity = Type::scalar(isz), bty = Type::scalar(ElemSize::Bool);
    Name lane = gen.fresh(root->id.s + "_lane"), g = gen.fresh("g"), first = gen.fresh(root->id.s + "_pair");
    E gv = mk_var(g, ity), fv = mk_var(first, ity);
    Stmts body;
    body.push_back(mk_def(first, ity, mk_binop(BinOp::Mul, mk_binop(BinOp::FloorDiv, mk_var(lane, ity), mk_int(G, isz), ity), mk_int(2, isz), ity), root->i));
    body.push_back(mk_def(g, ity, mk_binop(BinOp::Rem, mk_var(lane, ity), mk_int(G, isz), ity), root->i));
    std::map<Name, E> names[2];
    Name sum[2];
    const Stmts sums = two_sums(root, pos, vec, x, y, swapped, fv, gv, E(), K, names, sum);
    body.insert(body.end(), sums.begin(), sums.end());
    for (int u = 0; u < 2; ++u) {
      Stmts ss;
      for (size_t q = pos + 1; q < root->body.size(); ++q) {
        const S& st = root->body[q];
        if (st->k == Stmt::Def) {
          Name n = gen.fresh(st->id.s);
          E e = subst_vars(st->expr, names[u]);
          names[u][st->id] = mk_var(n, st->ty);
          ss.push_back(mk_def(n, st->ty, e, st->i));
        } else {
          ss.push_back(mk_assign(subst_vars(st->dst, names[u]), subst_vars(st->expr, names[u]), st->i));
        }
      }
      E mine = mk_binop(BinOp::Eq, gv, mk_int(u, isz), bty);
      if (u == 1 && N % 2 != 0) mine = mk_binop(BinOp::And, mine, mk_binop(BinOp::Lt, fv, mk_int(N - 1, isz), bty), bty);
      body.push_back(mk_if(mine, ss, {}));
    }
    auto nr = clone(root);
    const int64_t pairs = (N + 1) / 2;
    nr->id = lane;
    nr->hi = mk_int(pairs * G, isz);
    nr->body = body;
    nr->map.n = (pairs * G + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    k.body = {S(nr)};
    k.grid.x = (nr->map.n + root->map.tpb - 1) / root->map.tpb;
    launch->grid = k.grid;
    return true;
  }

  // `t += term` for those of the sum's iterations start * vec .. start * vec + len - 1 that lane g of a group has: every G-th vector
  Stmts share(const S& loop, int vec, const E& term, const E& t, const E& gv, const E& start, int64_t len) {
    const Type ity = Type::scalar(isz);
    const Name d0 = gen.fresh(loop->id.s + "_c"), u = gen.fresh(loop->id.s + "_u");
    // d = (start + d0 * G + g) * V + u
    E piece = mk_binop(BinOp::Add, mk_binop(BinOp::Mul, mk_var(d0, ity), mk_int(G, isz), ity), gv, ity);
    auto element = [&](const E& v, const E& u) {
      return mk_binop(BinOp::Add, mk_binop(BinOp::Mul, start ? mk_binop(BinOp::Add, start, v, ity) : v, mk_int(vec, isz), ity), u, ity);
    };
    const S add = mk_assign(t, mk_binop(BinOp::Add, t, term, t->ty), loop->i);
    auto inner = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(
        u, mk_int(0, isz), mk_int(vec, isz), 1, {mk_def(loop->id, ity, element(piece, mk_var(u, ity)), loop->i), add}, LoopPar(), loop->i)));
    inner->unroll = true;
    const bool whole = loop->hi->iv % vec == 0;
    const int64_t chunk = vec * G, rounds = len / chunk, vectors = len / vec;
    auto outer = clone(loop);
    outer->id = d0;
    auto part_of = [&](int64_t lanes, const Stmts& ss) {
      return mk_if(mk_binop(BinOp::Lt, gv, mk_int(lanes, isz), Type::scalar(ElemSize::Bool)), ss, {});
    };
    if (!whole) inner->iv = 1;   // (rows that start at any element)
    if (len % chunk == 0 || !whole) {
      outer->hi = mk_int(rounds, isz);
      outer->body = {S(inner)};
    } else {
      // the last round covers only part of the group: lanes whose vector starts past the end sit it out
      outer->hi = mk_int(rounds + 1, isz);
      outer->body = {mk_if(mk_binop(BinOp::Lt, mk_binop(BinOp::Mul, piece, mk_int(vec, isz), ity), mk_int(len, isz), Type::scalar(ElemSize::Bool)), {S(inner)}, {})};
    }
    Stmts body{outer};
    if (!whole && len % chunk != 0) {
      // whole rounds of the group, then a round that covers part of it, then what is left of a vector, an element per lane
      if (vectors % G != 0) {
        auto tail = clone(S(inner));
        tail->id = gen.fresh(loop->id.s + "_u");
        tail->body = {mk_def(loop->id, ity, start ? element(mk_binop(BinOp::Add, mk_int(rounds * G, isz), gv, ity), mk_var(tail->id, ity))
                                                  : mk_binop(BinOp::Add, mk_int(rounds * chunk, isz), element(gv, mk_var(tail->id, ity)), ity), loop->i),
                      add};
        body.push_back(part_of(vectors % G, {S(tail)}));
      }
      if (len % vec != 0) body.push_back(part_of(len % vec, {mk_def(loop->id, ity, start ? element(mk_int(vectors, isz), gv) : mk_binop(BinOp::Add, mk_int(vectors * vec, isz), gv, ity), loop->i), add}));
    }
    return body;
  }

  // Sums over long rows that memory selects out of large tables, cut into slabs along the rows.  Whole rows come from the memory
  // side: 270 MB to 2.7 GB of them at 6 to 8 TB/s.  Here a workgroup takes a slab of its rows, and the slabs are dealt out to
  // the dies (a workgroup's number modulo 8; slabs beyond the eighth follow when all workgroups of the first eight have
  // started), so that a die's L2 sees an eighth of the table or less: 11 to 14 TB/s.  The parts of a sum go to memory, and a
  // second launch adds them up and does the rest of the iteration.  A group of lanes takes two iterations, which mostly have a row
  // in common, as above.  Microseconds of the whole call, in one piece, in slabs an iteration at a time, and so; masks whose
  // columns lie anywhere, and within 32 of the row:
  //   225 000 products over 1024 floats, 61 MB table     157, 104, 104       94,  80,  74
  //    81 000 over 1024 floats, 37 MB                     62,  41,  41       51,  37,  36
  //   640 000 over 512 floats, 33 MB                     178, 127, 125       85,  95,  78
  //   300 000 over 512 floats, 10 MB                      66,  52,  48       43,  46,  39
  //   300 000 over 1024 floats, 12 MB                    122,  86,  73       76,  80,  65
  //   300 000 over 777 floats, 16 MB                     114,  89,  83       64,  79,  66
  //   324 000 over 1024 doubles, 74 MB                   383, 244, 202      170, 232, 178
  //   324 000 over 1000 doubles, 72 MB                   386, 256, 190      177, 192, 173
  //   300 000 over 900 doubles, 43 MB                    293, 191, 163      145, 189, 139
  //    16 000 over 1024 doubles, 131 MB                   94,  81,  82       99,  78,  79
  // Rows next to each other that select neighbouring rows find them in L2 as they are, which the program does not say: there the
  // requests to L1 are what bounds it (77 % of its cycles, counted), and a row in common is a quarter of them.
  // The bounds: tables below 9 MiB gain nothing (8192 x 256 floats 55.6 -> 54.5 without the second table's passes, 1000 x 1024
  // 26.7 -> 28.5), nor do launches that read less than 96 MiB of rows, which the added launch costs more, or less than half as much again
  // of 4 KB and more out of tables below 16 MiB (26 400 products over 1024 floats, 10 MB: 19.7 in one piece, 22.9; 48 000: 27.5 and 26.3;
  // 27 000 and 60 000 of 12 MB: 21.8 and 23.3, 32.6 and 29.1; 15 600 and 52 000 over 1024 doubles, 11 MB: 21.2 and 22.1, 45.5 and
  // 36.6; but 60 000 over 512 floats, 10 MB: 24.1 and 23.4).  Slabs are halved
  // while theirs of the table is above 5 MiB, down to 512 bytes on average, a sixteenth less will do: four 16-byte pieces for each of
  // eight lanes (the first product above in slabs of 1024, 512, 256 and 128 bytes 108, 86, 96 and 156, the main launches alone; 3000 rows
  // of 4 KB, 12 MB: 49, 58, 75 and 122).
  static constexpr int64_t DIES = 8, SLAB_ROW = 512, SLAB_TABLE = int64_t(5) << 20, WHOLE_TABLE = int64_t(9) << 20, LARGE_TABLE = int64_t(16) << 20, LONG_ROW = 4096, GATHERED = int64_t(96) << 20;
  void slabs(const Kernel& k, const StmtP& launch, const S& root, size_t pos, int vec, const E& term) {
    const S& loop = root->body[pos];
    const E& acc = loop->body[0]->dst;
    const int64_t N = root->hi->iv, K = loop->hi->iv, es = elem_bytes(acc->ty.sz), chunk = vec * G, tpb = root->map.tpb;
    if (acc->k != Expr::Var || tpb % WAVE_SIZE != 0) return;
    // straight iterations: definitions, the sum, definitions and stores to arrays that the sum does not read
    std::set<Name> from_memory, read, stored;
    auto reads = [&](const E& e) { visit_exprs(e, [&](const E& v) { if (v->k == Expr::Var) read.insert(v->name); }); };
    for (size_t q = 0; q < root->body.size(); ++q) {
      const S& st = root->body[q];
      if (q == pos) { reads(term); continue; }
      if (st->k == Stmt::Def && st->ty.is_scalar()) {
        if (q < pos) {
          if (st->id != acc->name && mentions(st->expr, acc->name)) return;
          bool loads = has_load(st->expr);
          visit_exprs(st->expr, [&](const E& v) { if (v->k == Expr::Var && from_memory.count(v->name)) loads = true; });
          if (loads) from_memory.insert(st->id);
          reads(st->expr);
        }
      } else if (q > pos && st->k == Stmt::Assign && st->dst->k == Expr::Index && st->dst->args[0]->k == Expr::Var) {
        stored.insert(st->dst->args[0]->name);
      } else {
        return;
      }
    }
    if (stored.empty()) return;
    for (auto& n : stored) if (read.count(n)) return;
    // the smallest of the tables that the rows are selected from
    int64_t table = 0;
    bool ok = true;
    visit_exprs(term, [&](const E& e) {
      if (e->k != Expr::Index || !mentions(e->args[1], loop->id)) return;
      bool selected = false;
      visit_exprs(e->args[1], [&](const E& v) { if (v->k == Expr::Var && from_memory.count(v->name)) selected = true; });
      if (!selected) return;
      int64_t bytes = elem_bytes(e->ty.sz);
      for (int64_t d : e->dim_shape) bytes *= d;
      if (e->dim_shape.empty() || e->ty.sz != acc->ty.sz) ok = false;
      table = table == 0 ? bytes : std::min(table, bytes);
    });
    if (!ok || table <= WHOLE_TABLE || N * K * es < (table < LARGE_TABLE && K * es >= LONG_ROW ? GATHERED / 2 * 3 : GATHERED)) return;
    int64_t cut = 1;
    const int64_t chunks = (K + chunk - 1) / chunk;
    auto divides = [&](int64_t n) { return (n - 1) * ((chunks + n - 1) / n) < chunks; };
    while (cut < 64 && chunks * chunk * es / (2 * cut) >= SLAB_ROW / 16 * 15 && table / cut > SLAB_TABLE && divides(2 * cut)) cut *= 2;
    if (cut == 1 || taken + cut * N * es > KEPT_MEMORY || N * G * cut > (int64_t(1) << 30)) return;
    taken += cut * N * es;
    const int64_t width = (chunks + cut - 1) / cut * chunk, last = K - (cut - 1) * width;

    const Type ity = Type::scalar(isz), bty = Type::scalar(ElemSize::Bool), ety = Type::scalar(acc->ty.sz), pty = Type::pointer(acc->ty.sz);
    auto iint = [&](int64_t v) { return mk_int(v, isz); };
    const Name parts = gen.fresh(acc->name.s + "_parts"), slab = gen.fresh("slab"), place = gen.fresh("place"), g = gen.fresh("g"), tid = gen.fresh("t");
    auto index = [&](Expr::Kind kind) {
      auto e = std::make_shared<Expr>();
      e->k = kind;
      e->ty = ity;
      e->iv = 0;
      return E(e);
    };
    const E bx = index(Expr::BlockIdx), tv = mk_var(tid, ity), gv = mk_var(g, ity);
    // two products to a group of lanes, as above
    E x, y;
    bool swapped = false;
    const bool twice = width / chunk <= 32 && rows_of(loop, term, &x, &y, &swapped);   // (written out)
    const int64_t of_group = tpb / G * (twice ? 2 : 1), groups = (N + of_group - 1) / of_group;
    auto div = [&](const E& a, int64_t b) { return mk_binop(BinOp::FloorDiv, a, iint(b), ity); };
    auto rem = [&](const E& a, int64_t b) { return mk_binop(BinOp::Rem, a, iint(b), ity); };
    auto part = [&](const E& i, const E& s) { return mk_index(mk_var(parts, pty), fold_expr(mk_binop(BinOp::Add, mk_binop(BinOp::Mul, s, iint(N), ity), i, ity)), ety); };
    Stmts top;
    if (cut <= DIES) {
      top.push_back(mk_def(slab, ity, rem(bx, cut)));
      top.push_back(mk_def(place, ity, div(bx, cut)));
    } else {
      top.push_back(mk_def(slab, ity, mk_binop(BinOp::Add, mk_binop(BinOp::Mul, div(bx, DIES * groups), iint(DIES), ity), rem(bx, DIES), ity)));
      top.push_back(mk_def(place, ity, rem(div(bx, DIES), groups)));
    }
    top.push_back(mk_def(tid, ity, index(Expr::ThreadIdx)));
    top.push_back(mk_def(g, ity, rem(tv, G)));
    const E team = div(tv, G);
    top.push_back(mk_def(root->id, ity, mk_binop(BinOp::Add, mk_binop(BinOp::Mul, mk_var(place, ity), iint(of_group), ity), twice ? mk_binop(BinOp::Mul, team, iint(2), ity) : team, ity), root->i));
    const E first = mk_var(root->id, ity);
    // the slab that starts with vector `from`, `len` elements of it
    auto sum_of = [&](const E& from, int64_t len) {
      Stmts ss;
      if (twice) {
        std::map<Name, E> names[2];
        Name sums[2];
        ss = two_sums(root, pos, vec, x, y, swapped, first, gv, from, len, names, sums);
        for (int u = 0; u < 2; ++u) {
          E mine = mk_binop(BinOp::Eq, gv, iint(u), bty);
          if (u == 1 && N % 2 != 0) mine = mk_binop(BinOp::And, mine, mk_binop(BinOp::Lt, first, iint(N - 1), bty), bty);
          ss.push_back(mk_if(mine, {mk_assign(part(u == 0 ? first : mk_binop(BinOp::Add, first, iint(1), ity), mk_var(slab, ity)), mk_var(sums[u], ety), loop->i)}, {}));
        }
        return ss;
      }
      const Name sum = gen.fresh(acc->name.s);
      const E sv = mk_var(sum, ety);
      for (size_t q = 0; q < pos; ++q)
        if (root->body[q]->id != acc->name) ss.push_back(root->body[q]);
      ss.push_back(mk_def(sum, ety, mk_float(0.0, acc->ty.sz), loop->i));
      for (const S& st : share(loop, vec, term, sv, gv, from, len)) ss.push_back(st);
      ss.push_back(mk_assign(sv, mk_raw("parpy_sum8(" + sum.str() + ")", ety)));
      ss.push_back(mk_if(mk_binop(BinOp::Eq, gv, iint(0), bty), {mk_assign(part(first, mk_var(slab, ity)), sv, loop->i)}, {}));
      return ss;
    };
    Stmts own = sum_of(mk_binop(BinOp::Mul, mk_var(slab, ity), iint(width / vec), ity), width);
    if (last != width) own = {mk_if(mk_binop(BinOp::Lt, mk_var(slab, ity), iint(cut - 1), bty), own, sum_of(iint((cut - 1) * width / vec), last))};
    if (N % of_group == 0) top.insert(top.end(), own.begin(), own.end());
    else top.push_back(mk_if(mk_binop(BinOp::Lt, mk_var(root->id, ity), iint(N), bty), own, {}));

    Kernel sums = k;
    sums.name = k.name + "_slabs_" + std::to_string(gen.next++);
    sums.body = top;
    sums.grid.x = groups * cut;
    sums.cached_stores = true;
    sums.read_once.clear();   // (by every slab)

    // the iterations once more, a thread each, with the parts in place of the sum
    Kernel whole = k;
    whole.name = k.name + "_whole_" + std::to_string(gen.next++);
    auto nr = clone(root);
    nr->map.tpb = 256;
    nr->map.n = (N + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    std::set<Name> needed{acc->name};
    auto uses = [](const E& e, std::set<Name>& names) { if (e) visit_exprs(e, [&](const E& v) { if (v->k == Expr::Var) names.insert(v->name); }); };
    Stmts from_last;
    for (size_t q = root->body.size(); q-- > 0;) {
      const S& st = root->body[q];
      if (q == pos) {
        for (int64_t n = cut; n-- > 0;) from_last.push_back(mk_assign(acc, mk_binop(BinOp::Add, acc, part(mk_var(root->id, ity), iint(n)), ety), loop->i));
      } else if (st->k != Stmt::Def || needed.count(st->id)) {
        uses(st->expr, needed);
        uses(st->dst, needed);
        from_last.push_back(st);
      }
    }
    nr->body = Stmts(from_last.rbegin(), from_last.rend());
    whole.body = {S(nr)};
    whole.block.x = 256;
    whole.grid.x = (nr->map.n + 255) / 256;

    auto launch_of = [&](Kernel& kernel) {
      auto l = std::make_shared<Stmt>(*launch);
      l->fname = kernel.name;
      l->grid = kernel.grid;
      l->block = kernel.block;
      l->args.clear();
      std::set<Name> used;
      visit_stmts(kernel.body, [&](const S& st) { for (const E& e : {st->dst, st->expr, st->lo, st->hi}) uses(e, used); });
      std::vector<KernelParam> params;
      for (size_t i = 0; i < kernel.params.size(); ++i)
        if (used.count(kernel.params[i].id)) { params.push_back(kernel.params[i]); l->args.push_back(launch->args[i]); }
      KernelParam q;
      q.id = parts;
      q.ty = pty;
      params.push_back(q);
      l->args.push_back(mk_var(parts, pty));
      kernel.params = params;
      return l;
    };
    auto alloc = std::make_shared<Stmt>(), give = std::make_shared<Stmt>();
    alloc->k = Stmt::Alloc;
    alloc->id = parts;
    alloc->ty = ety;
    alloc->iv = N * cut;
    give->k = Stmt::Free;
    give->id = parts;
    const StmtP a = launch_of(sums), b = launch_of(whole);
    in_slabs = {S(alloc), S(a), S(b), S(give)};
    // (the call must not fail for the parts: what the device has left, or the fixed amount of memory of a run that may
    // allocate nothing, may not hold them)
    auto fits = std::make_shared<Expr>(*mk_raw("parpy_temporaries_fit(" + std::to_string(N * cut * es) + ")", bty));
    fits->iv = N * cut * es;
    room = fits;
    extra.push_back(sums);
    extra.push_back(whole);
    wholes.push_back(b);
  }

  bool apply(Kernel& k, const StmtP& launch) {
    if (k.body.size() != 1) return false;
    const S root = k.body[0];
    // the iterations of the whole launch: spread over the grid, or over the threads of a single workgroup
    // (which then becomes a grid, since eight times as many threads may not fit one workgroup)
    bool one_group = root->k == Stmt::For && root->map.k == GpuMap::Thread && k.grid.x == 1;
    if (!(root->k == Stmt::For && (root->map.k == GpuMap::ThreadBlock || one_group) && root->map.dim == 0 && root->step == 1 &&
          root->lo->k == Expr::Int && root->lo->iv == 0 && root->hi->k == Expr::Int))
      return false;
    int64_t N = root->hi->iv;
    if (one_group && N > root->map.n) return false;  // a strided loop inside the workgroup: iterations are not one per thread
    if (N < 64 || k.grid.y != 1 || k.grid.z != 1 || k.block.y != 1 || k.block.z != 1) return false;  // (less than a wavefront of iterations: nothing to share)
    int pos = -1, vec = 0;
    E term;
    for (size_t q = 0; q < root->body.size(); ++q) {
      const S& st = root->body[q];
      int v = 0;
      E t;
      if (sum_loop(st, &v, &t)) {
        if (pos >= 0) return false;
        pos = (int)q;
        vec = v;
        term = t;
        continue;
      }
      bool simple = st->k == Stmt::Def || (st->k == Stmt::Assign && (st->dst->k == Expr::Index || st->dst->k == Expr::Var));
      if (!simple) return false;
    }
    if (pos < 0) return false;
    const S& loop = root->body[pos];
    const E& acc = loop->body[0]->dst;
    bool elem_acc = acc->k == Expr::Index;
    // an array element as accumulator: nothing else in the iteration may touch that array but plain
    // stores to the very element in front of the loop (its initialisation)
    if (elem_acc)
      for (size_t q = 0; q < root->body.size(); ++q) {
        if ((int)q == pos) continue;
        const S& st = root->body[q];
        bool init = (int)q < pos && st->k == Stmt::Assign && expr_eq(st->dst, acc) && !mentions(st->expr, acc->args[0]->name);
        if (init) continue;
        bool touches = false;
        auto scan = [&](const E& e) { if (e && mentions(e, acc->args[0]->name)) touches = true; };
        scan(st->dst); scan(st->expr);
        if (touches) return false;
      }
    if (!one_group && pair(k, launch, root, (size_t)pos, vec, term)) return true;
    for (int q = 0; q < pos; ++q)   // other stores in front of the sum would be repeated by every lane of a group: harmless, same value
      if (root->body[q]->k == Stmt::Assign && root->body[q]->dst->k == Expr::Index && !expr_eq(root->body[q]->dst, acc)) return false;
    Type ity = Type::scalar(isz);
    Name gi = gen.fresh(root->id.s + "_lane"), g = gen.fresh("g");
    E giv = mk_var(gi, ity), gv = mk_var(g, ity);
    E lane0 = mk_binop(BinOp::Eq, gv, mk_int(0, isz), Type::scalar(ElemSize::Bool));
    Stmts body;
    body.push_back(mk_def(root->id, ity, mk_binop(BinOp::FloorDiv, giv, mk_int(G, isz), ity), root->i));
    body.push_back(mk_def(g, ity, mk_binop(BinOp::Rem, giv, mk_int(G, isz), ity), root->i));
    for (int q = 0; q < pos; ++q) {
      const S& st = root->body[q];
      if (st->k == Stmt::Assign && st->dst->k == Expr::Index) body.push_back(mk_if(lane0, {st}, {}));
      else body.push_back(st);
    }
    // the lanes of a group add up their shares apart from what the sum starts from (which only counts once)
    bool from_zero = false;
    for (int q = 0; q < pos; ++q)
      if (!elem_acc && root->body[q]->k == Stmt::Def && root->body[q]->id == acc->name) from_zero = root->body[q]->expr->k == Expr::Float && root->body[q]->expr->fv == 0.0;
    for (int q = 0; q < pos; ++q)
      if (!elem_acc && root->body[q]->k == Stmt::Assign && root->body[q]->dst->k == Expr::Var && root->body[q]->dst->name == acc->name) from_zero = false;
    E t = acc;
    if (!from_zero) {
      Name tn = gen.fresh(elem_acc ? "part" : acc->name.s + "_part");
      body.push_back(mk_def(tn, acc->ty, mk_float(0.0, acc->ty.sz), loop->i));
      t = mk_var(tn, acc->ty);
    }
    for (const S& st : share(loop, vec, term, t, gv, E(), loop->hi->iv)) body.push_back(st);
    body.push_back(mk_assign(t, mk_raw("parpy_sum8(" + t->name.str() + ")", t->ty)));
    if (!elem_acc && !from_zero) body.push_back(mk_assign(acc, mk_binop(BinOp::Add, acc, t, acc->ty), loop->i));
    Stmts stores;
    if (elem_acc) {
      // a group that lies wholly in one lane-0 store: the synchronisation between the initialising store
      // and this read-modify-write is program order of lane 0
      stores.push_back(mk_assign(acc, mk_binop(BinOp::Add, acc, t, acc->ty), loop->i));
    }
    for (size_t q = pos + 1; q < root->body.size(); ++q) {
      const S& st = root->body[q];
      if (st->k == Stmt::Assign && st->dst->k == Expr::Index) stores.push_back(st);
      else {
        if (!stores.empty()) return false;  // a definition after a store: not the shape this pass handles
        body.push_back(st);
      }
    }
    if (!stores.empty()) body.push_back(mk_if(lane0, stores, {}));
    auto nr = clone(root);
    nr->id = gi;
    nr->hi = mk_int(N * G, isz);
    nr->body = body;
    int64_t tpb = one_group ? 256 : root->map.tpb;
    nr->map.k = GpuMap::ThreadBlock;
    nr->map.tpb = tpb;
    nr->map.n = (N * G + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    if (!one_group) slabs(k, launch, root, (size_t)pos, vec, term);
    k.body = {S(nr)};
    k.block.x = tpb;
    k.grid.x = (nr->map.n + tpb - 1) / tpb;
    launch->grid = k.grid;
    launch->block = k.block;
    return true;
  }

  void run() {
    Stmts host;
    taken = temporaries(p.host);
    for (auto& s : p.host) {
      if (s->k != Stmt::Launch) { host.push_back(s); continue; }
      Kernel* k = nullptr;
      for (auto& kk : p.kernels)
        if (kk.name == s->fname) k = &kk;
      auto ns = std::make_shared<Stmt>(*s);
      in_slabs.clear();
      if (k && !k->opaque_body) apply(*k, ns);
      if (in_slabs.empty()) { host.push_back(ns); continue; }
      auto either = clone(mk_if(room, in_slabs, {ns}));
      either->fname = "whole sums";
      host.push_back(S(either));
    }
    for (auto& k : extra) p.kernels.push_back(k);
    p.host = host;
  }
};

// ================================================================ four elements per thread for element-wise launches
// `parpy.threads(n)` on a loop of n iterations gives every thread one element, and a thread cannot
// turn one 4-byte access into a 16-byte one.  When the iteration is nothing but straight-line
// element-wise work on unit-stride data, the launch is cut to n/4 threads; the vectorised remap then
// gives each of them four consecutive elements (y = a*x + y on 2^28 floats: 5.5 -> 5.9 TB/s).  Launches
// that would drop below 64 threads per CU keep their shape, as do iterations that contain loops (those
// want more threads, not fewer: see the lane groups below).
struct Coarsen {
  Program& p;
  const Options& opts;
  NameGen& gen;
  Coarsen(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g) {}

  bool apply(Kernel& k, const StmtP& launch) {
    if (k.body.size() != 1) return false;
    const S& root = k.body[0];
    if (!(root->k == Stmt::For && root->map.k == GpuMap::ThreadBlock && root->map.dim == 0 && root->step == 1 &&
          root->lo->k == Expr::Int && root->lo->iv == 0 && root->hi->k == Expr::Int))
      return false;
    const int64_t n = root->hi->iv, tpb = root->map.tpb;
    const int64_t launched = (n + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    if (launched != root->map.n || tpb <= 0 || n / 4 < 256 * 64) return false;   // exactly one iteration per thread, and plenty
    if (k.grid.y != 1 || k.grid.z != 1 || k.block.y != 1 || k.block.z != 1) return false;
    bool straight = true;
    visit_stmts(root->body, [&](const S& c) {
      if (c->k == Stmt::For || c->k == Stmt::While || c->k == Stmt::Sync || c->k == Stmt::RawStmt) straight = false;
    });
    if (!straight) return false;
    Pass probe(k, opts, gen);
    if (probe.vector_width(root) != 4) return false;   // 4-byte elements through parameters only
    if (n % (4 * tpb) == 0) {
      // whole workgroups of whole vectors: shrink the launch and let the vectorised remap do the rest
      auto nr = clone(root);
      nr->map.n = n / 4;
      k.body = {S(nr)};
      k.grid.x = n / 4 / tpb;
      launch->grid = k.grid;
      return true;
    }
    // any other n: thread q takes elements 4q .. 4q+3; the last thread may hold fewer and tests each of its own
    ElemSize isz = opts.int_size();
    Type ity = Type::scalar(isz);
    const int64_t quads = (n + 3) / 4;
    Name q = gen.fresh(root->id.s + "_q");
    E qv = mk_var(q, ity);
    auto elements = [&](bool guarded) {
      Name u = gen.fresh(root->id.s + "_u");
      E d = mk_binop(BinOp::Add, mk_binop(BinOp::Mul, qv, mk_int(4, isz), ity), mk_var(u, ity), ity);
      Stmts ib;
      ib.push_back(mk_def(root->id, ity, d, root->i));
      for (auto& b : root->body) ib.push_back(b);
      if (guarded) {
        Stmts inner = {ib.begin() + 1, ib.end()};
        ib = {ib[0], mk_if(mk_binop(BinOp::Lt, mk_var(root->id, ity), mk_int(n, isz), Type::scalar(ElemSize::Bool)), inner, {})};
      }
      auto loop = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(
          mk_for(u, mk_int(0, isz), mk_int(4, isz), 1, ib, LoopPar(), root->i)));
      loop->unroll = true;
      return S(loop);
    };
    Stmts body;
    if (n % 4 == 0) {
      body = {elements(false)};
    } else {
      E whole = mk_binop(BinOp::Leq, mk_binop(BinOp::Add, mk_binop(BinOp::Mul, qv, mk_int(4, isz), ity), mk_int(4, isz), ity), mk_int(n, isz),
                         Type::scalar(ElemSize::Bool));
      body = {mk_if(whole, {elements(false)}, {elements(true)})};
    }
    auto nr = clone(root);
    nr->id = q;
    nr->hi = mk_int(quads, isz);
    nr->body = body;
    nr->map.n = (quads + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    k.body = {S(nr)};
    k.grid.x = (nr->map.n + tpb - 1) / tpb;
    launch->grid = k.grid;
    return true;
  }

  void run() {
    Stmts host;
    for (auto& s : p.host) {
      if (s->k != Stmt::Launch) { host.push_back(s); continue; }
      Kernel* k = nullptr;
      for (auto& kk : p.kernels)
        if (kk.name == s->fname) k = &kk;
      auto ns = std::make_shared<Stmt>(*s);
      if (k && !k->opaque_body) apply(*k, ns);
      host.push_back(ns);
    }
    p.host = host;
  }
};

// ================================================================ threads for short rows
// `{'N': threads(n), 'M': threads(512)}` on rows of 300 elements starts eight wavefronts per row, most of them for one
// element per lane or none, and each takes part in every reduction: cross-lane steps, a round trip through LDS and a
// barrier, around a hundred instructions per wavefront and reduction.  A row that is reduced and then needs no more than
// a vector per thread gets fewer threads; a row that fits one wavefront reduces without LDS or barriers, and several
// such rows share a workgroup.
struct RowThreads {
  Program& p;
  const Options& opts;
  NameGen& gen;
  RowThreads(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g) {}

  bool apply(Kernel& k, const StmtP& launch) {
    if (k.body.size() != 1 || k.block.y != 1 || k.block.z != 1 || k.opaque_body) return false;
    const S& root = k.body[0];
    if (!(root->k == Stmt::For && root->map.k == GpuMap::Block && root->map.mult == 1 && root->step == 1 && root->lo->k == Expr::Int &&
          root->lo->iv == 0 && root->hi->k == Expr::Int && root->els.empty()))
      return false;
    const int64_t rows = root->hi->iv, threads = k.block.x;
    if (root->map.n != rows || k.grid.x * k.grid.y * k.grid.z != rows) return false;
    if (share_starts(k, root, launch, rows, threads)) return true;
    // straight through the row: element loops and reductions over the whole workgroup, no loop around them
    bool ok = true, reduces = false, strided = false;
    bool meets_in_test = false;   // a barrier under a test that not all rows of a workgroup need pass
    int64_t longest = 0, bytes = 0, loops = 0;
    Pass probe(k, opts, gen);
    std::function<void(const Stmts&, bool)> walk = [&](const Stmts& ss, bool tested) {
      for (auto& s : ss) {
        switch (s->k) {
          case Stmt::Def: case Stmt::Assign: break;
          case Stmt::Sync: meets_in_test = meets_in_test || tested; break;
          case Stmt::WaveReduce:
            reduces = true;
            meets_in_test = meets_in_test || tested;
            if (s->iv != threads) ok = false;
            break;
          case Stmt::If: walk(s->body, true); walk(s->els, true); break;
          case Stmt::For: {
            if (!thread_mapped(s) || s->map.dim != 0 || s->map.n != threads || !s->els.empty()) { ok = false; break; }
            const int64_t extent = const_extent(s);
            if (extent <= 0) { ok = false; break; }
            visit_stmts(s->body, [&](const S& c) { if (c->k == Stmt::For || c->k == Stmt::While || c->k == Stmt::Sync || c->k == Stmt::RawStmt || c->k == Stmt::WaveReduce) ok = false; });
            longest = std::max(longest, extent);
            ++loops;
            strided = strided || s->step != 1;
            if (const int v = probe.vector_width(s)) bytes = std::max<int64_t>(bytes, 16 / v);
            break;
          }
          default: ok = false;
        }
      }
    };
    walk(root->body, false);
    if (!ok || !reduces || longest == 0 || bytes == 0) return false;
    int64_t want = threads;
    if (rows * (threads / WAVE_SIZE) > 4096) {
      // At least 24 bytes of the row per thread: 16384 rows of 1000 floats 27.6 us on 512 threads, 20.0 / 20.8 / 21.5 on
      // 256 / 128 / 64 (softmax); 1000 halves 20.2 us on 256 threads, 15.0 on 64; 300 doubles 23.6 and 14.7; sums of 20000
      // rows of 300 floats 31.4 us on 1024 threads, 14.4 on 64.
      want = WAVE_SIZE;
      while (want * 2 * 24 <= longest * bytes) want *= 2;
      want = std::min(want, threads);
    } else {
      // A launch of less than two wavefronts per SIMD, and rows of four 16-byte vectors per thread and more: twice the
      // threads, and again.  Sums of one row of 100000 floats 15.8 us on 64 threads, 5.0 on 1024; of 30 such rows 19.1 and 5.9; of 100
      // rows of 150000 29.5 us on 128, 13.7 on 1024; softmax over 300 rows of 30000 doubles 75 us on 256, 39 on 512.
      // (With a limit of four per SIMD 300 rows of 100000 took 23.9 us instead of 22.2.)
      while (!strided && want < 1024 && rows * (want / WAVE_SIZE) < 2048 && longest * bytes >= 64 * want) want *= 2;
    }
    // Rows that several loops walk stay in registers where a thread runs 32 vectors of them at most (softmax, doubles, 256
    // threads asked for: 644 rows of 29553 165 -> 78 us, 2000 of 20001 349 -> 138, 1000 of 17001 147 -> 57).
    while (loops > 1 && !strided && want < 1024 && longest * bytes > 32 * 16 * want) want *= 2;
    // Workgroups start at about two per nanosecond, which is what small ones wait for: four rows each where a row is a
    // wavefront's (the sums above 7.1 us, 6.7 with eight; softmax over 30000 rows of 200 floats 16.0 -> 8.7 us).
    // Fewer of them start at once in time where a wavefront has more than four vectors per lane to move; below that they
    // share workgroups too (softmax over 4000 rows of 700 floats 5.4 -> 5.0 us, over 3000 of 300 3.85 -> 3.57).
    int64_t group = want == WAVE_SIZE && (rows > 4096 || (rows > 256 && longest * bytes <= 64 * want)) ? 4 : 1;
    // Rows of one loop, four vectors per thread at most: what such a workgroup moves is over before the next has started, and
    // what they wait for is the start.  Up to eight rows and 1024 threads each, the rows still on threads of their own: the
    // order of a row's sum stays.  Floats, rows x length, one row against this: 400 x 4000 5.0 -> 3.5 us, 1000 x 1708 4.8 -> 3.4,
    // 5000 x 1000 7.9 -> 5.0, 5000 x 1001 7.5 -> 5.4, 9001 x 1777 14.0 -> 12.1, 12000 x 1500 15.0 -> 11.8, 16384 x 3000
    // 35.0 -> 33.2; doubles 4001 x 333 5.3 -> 3.5, 16384 x 500 12.3 -> 11.2 (11.0 with four wavefronts' rows, but 5000 x 1000
    // floats 5.3).  At most 256 rows start at once.  Where memory is the bound it is no gain: 7602 x 2236 doubles 23.9 and 23.9
    // us, 512 threads and 134 MB 24.2 and 24.6.  Rows that several loops walk lose by waiting for each other at the barriers:
    // softmax over 8000 x 1024 floats 11.6 us alone, 12.9 in eights; over 16384 x 1500 32.3 and 34.4.
    const int64_t total = rows * longest * bytes;
    if (loops == 1 && rows > 256 && !meets_in_test && longest * bytes <= 64 * want && total < (int64_t(1) << (want > 256 ? 27 : 28)))
      group = std::max<int64_t>(group, std::min<int64_t>(8, 1024 / want));
    if (want == threads && group == 1) return false;
    std::function<Stmts(const Stmts&)> cut = [&](const Stmts& ss) {
      Stmts out;
      for (auto& s : ss) {
        auto r = clone(s);
        if (s->k == Stmt::WaveReduce) r->iv = want;
        if (s->k == Stmt::For) r->map.n = want;
        r->body = cut(s->body);
        r->els = cut(s->els);
        out.push_back(r);
      }
      return out;
    };
    auto nr = clone(root);
    nr->body = cut(root->body);
    k.block = Dim3{want, group, 1};
    if (group > 1) k.wave_rows = want == WAVE_SIZE;
    several(k, nr, launch, rows, group);
    return true;
  }

  static void several(Kernel& k, const StmtP& root, const StmtP& launch, int64_t rows, int64_t group) {
    if (group > 1) {
      const int64_t blocks = (rows + group - 1) / group;
      root->map.per = group;
      root->map.n = blocks * group;
      (root->map.dim == 0 ? k.grid.x : root->map.dim == 1 ? k.grid.y : k.grid.z) = blocks;
    }
    k.body = {S(root)};
    launch->grid = k.grid;
    launch->block = k.block;
  }

  // Rows on a wavefront or two whose threads never meet share workgroups where those are still as many as the device has
  // compute units: short rows wait for the starts.  The row numbers of a compressed matrix, written to its elements (how long
  // a row is stands in memory), 64 threads: 20 000 rows of 3 / 30 / 100 10.6 / 10.3 / 10.6 -> 3.5 / 3.8 / 5.0 us, 100 000 of 30
  // 22.6 -> 11.8, 2048 the same; of 600 each up to 13 % slower, 600 on average 5 % faster.  Within SDDMM, 8192 rows of 82, 128
  // deep, 34.8 -> 32.1 us; 2491 rows of 5, 174 deep, doubles 13.8 -> 13.0.  Element-wise rows of floats, halves and doubles,
  // 20 000 of 20 / 64 / 100 10.2 / 9.8 / 10.5 -> 3.8 / 3.7 / 4.5; 8192 of 256 4.9 -> 3.4; 100 000 of 256 and 20 000 of 500 are
  // bound by memory: 0.95 to 1.08 of the time.  Not with a loop inside the thread's element, where the row's own values
  // are scalar loads as long as a workgroup has one row: products of half-precision sparse matrices 1.2 times as slow in the
  // median (5000 rows of 60 times 128 columns 29.7 -> 54.2 us), dense products by rows 1.2 (5000 x 256 x 64 38.7 -> 56.7).
  bool share_starts(Kernel& k, const S& root, const StmtP& launch, int64_t rows, int64_t threads) {
    bool apart = threads <= 128 && rows >= 2048 && rows < (int64_t(1) << 30);
    visit_stmts(root->body, [&](const S& s) {
      bool plain = s->k == Stmt::Def || s->k == Stmt::Assign || s->k == Stmt::If;
      if (s->k == Stmt::For && s->map.k == GpuMap::Thread && s->map.dim == 0 && s->map.n == threads && !s->par.reduction) {
        const int64_t extent = const_extent(s);
        plain = extent <= 128 || rows * extent <= 6000000;   // (-1 where it is not constant)
      }
      apart = apart && plain;
    });
    if (!apart) return false;
    const int64_t group = 512 / threads;
    k.block = Dim3{threads, group, 1};
    several(k, clone(root), launch, rows, group);
    return true;
  }

  void run() {
    Stmts host;
    for (auto& s : p.host) {
      if (s->k != Stmt::Launch) { host.push_back(s); continue; }
      Kernel* k = nullptr;
      for (auto& kk : p.kernels)
        if (kk.name == s->fname) k = &kk;
      auto ns = std::make_shared<Stmt>(*s);
      if (k) apply(*k, ns);
      host.push_back(ns);
    }
    p.host = host;
  }
};

}  // namespace

void row_threads(Program& p, const Options& opts, NameGen& gen) { RowThreads(p, opts, gen).run(); }
void gather_transpose(Program& p, const Options& opts, NameGen& gen) { GatherTranspose(p, opts, gen).run(); }
void lane_split(Program& p, const Options& opts, NameGen& gen) {
  LaneSplit split(p, opts, gen);
  split.run();
  if (!opts.opt_vectorize) return;
  for (auto& l : split.wholes)
    for (auto& k : p.kernels)
      if (k.name == l->fname) Coarsen(p, opts, gen).apply(k, l);
}
void coarsen(Program& p, const Options& opts, NameGen& gen) { Coarsen(p, opts, gen).run(); }

}  // namespace hipopt
}  // namespace parpy
