// gfx950 memory passes, rewrites that change a launch: several steps of a host-side time loop in one pass over memory.
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

namespace {

// ================================================================ time loops over stencils, several steps per launch
// `for t: B[1:-1] = f(A[:-2], A[1:-1], A[2:]); A[1:-1] = f(B[:-2], ...)` runs as one launch per statement and step:
// each launch reads and writes whole arrays and waits for the one before it, a few microseconds for some tens of
// nanoseconds of work per compute unit.  When every launch of the loop updates arrays element by element from
// elements a fixed distance away, a stretch of the arrays can be carried through several steps on its own, provided it
// starts with a margin of (steps x distance) elements on either side that is computed along and thrown away.
//
//   * A wavefront owns a stretch of 64 * E elements, E neighbouring ones per lane, in registers: own elements and
//     those of the neighbouring lanes (DPP wave shifts by one lane) are all a step needs, so the steps take neither
//     LDS nor barriers.
//   * Stretches overlap, so a launch must not overwrite what its neighbours still read: it writes to a second set of
//     arrays, and the next launch brings the values back.  The number of launches is even; their steps differ by at
//     most one.
//   * The arithmetic of an element is that of the statement as written: same operations, same order.
//
//   * A lane's neighbouring elements come and go through LDS where they are more than 16 bytes, so that memory is read and
//     written in whole lines; a wavefront's part of LDS is its own, without barriers.
//   * At the ends of the arrays an update covers a part of a stretch: there the new value is blended with the old one under
//     a mask kept in a register, for the elements of a lane that may be such.
//   * Divisions by constants leave infinite dividends out where a NaN at the end shows them; such a stretch is computed again,
//     one that loads infinities or NaN without them from the start.
//
// A three-point average back and forth over 10^6 float64 elements, 98 updates, two launches of 25 steps: 447 us as launches
// of 4.5 us each, 45.6 on eight elements per lane with their own accesses and a division of four instructions one of which
// takes as long as four, 39.1 with blends for all elements of a stretch at the ends and divisions of any dividend, 31.6 with
// both arrays loaded and stored by every launch, 28.9 as it is: 1852 wavefronts, 1.8 to a SIMD.  The vector ALU and its latency bound it: 5.7 instructions per update and element of a
// stretch, of whose 640 elements 100 are margins.  A launch is over with its slowest stretches, those at the ends.
struct TimeTile {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;
  Type ity;
  Type bty = Type::scalar(ElemSize::Bool);

  TimeTile(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()), ity(Type::scalar(o.int_size())) {}

  struct Arr { Name host; ElemSize sz = ElemSize::F32; int64_t n = 0; bool written = false; int64_t left = 0, right = 0; };
  struct Update {                 // one launch of the loop
    int64_t lo = 0, hi = 0;       // elements it writes, in array coordinates
    int64_t c = 0;                // array coordinate = iteration + c
    Name id;
    Stmts body;
    std::map<Name, Name> host;    // parameter -> host variable
    int64_t radius = 0;
  };

  E iint(int64_t v) { return mk_int(v, isz); }
  E add(E a, E b) { return mk_binop(BinOp::Add, a, b, ity); }

  // Vector instructions for one element of an update: a product and the sum that it goes into are one, a division by a
  // constant is five and a half (`DevicePrinter` has which constants), neighbours and own elements are registers.  `waits`
  // counts what those that depend on each other wait where a SIMD has nothing else to issue.
  static double instructions(const E& e, double* waits) {
    if (!e->ty.is_scalar() || e->k == Expr::Index) return 0;
    const bool f32 = e->ty.sz == ElemSize::F32, integer = is_int(e->ty.sz);
    const double words = integer && elem_bytes(e->ty.sz) == 8 ? 2 : 1;
    if (e->k == Expr::Convert) {
      const E& d = e->args[0];
      // float32(float64(x) / c) is a division in single precision
      if (f32 && d->k == Expr::BinOpE && d->bop == BinOp::Div && d->args[1]->k == Expr::Float && d->args[0]->k == Expr::Convert && d->args[0]->args[0]->ty.sz == ElemSize::F32)
        return instructions(mk_binop(BinOp::Div, d->args[0]->args[0], d->args[1], e->ty), waits);
      if (d->k == Expr::Int || d->k == Expr::Float || d->k == Expr::Bool) return 0;
      return instructions(d, waits) + (d->ty.sz == e->ty.sz ? 0 : words);
    }
    double n = 0;
    for (auto& a : e->args) n += instructions(a, waits);
    auto product = [](const E& x) { return x->k == Expr::BinOpE && x->bop == BinOp::Mul && x->ty.is_scalar() && is_float(x->ty.sz); };
    if (e->k == Expr::IfExpr) return n + 1 + elem_bytes(e->ty.sz) / 4;
    if (e->k == Expr::UnOpE) return n + (e->uop == UnOp::Sub || e->uop == UnOp::Abs || e->uop == UnOp::Not || e->uop == UnOp::BitNeg ? words : f32 ? 4 : 40);
    if (e->k != Expr::BinOpE) return n;
    switch (e->bop) {
      case BinOp::Add: case BinOp::Sub: return n + (product(e->args[0]) || product(e->args[1]) ? 0 : words);
      case BinOp::Mul: return n + (integer ? 4 * words : 1);
      case BinOp::Div: case BinOp::FloorDiv: case BinOp::Rem:
        if (integer) return n + 20 * words;
        *waits += f32 ? 5 : 3;
        return n + (e->args[1]->k != Expr::Float ? 12 : f32 ? 5 : 5.5);
      case BinOp::Pow: case BinOp::Atan2: return n + 40;
      default: return n + words;
    }
  }

  // Divisions by constants that may give NaN for an infinite dividend are an instruction shorter, two in single precision
  // (`parpy_div_const`).  A stretch may take them where everything that follows from a NaN is one, so that the elements which
  // would have been other values are NaN at the end: sums, differences, products and quotients, no selections, comparisons,
  // maxima or integers made of what was divided.
  static bool carries_nan(const E& e, bool* divides) {
    if (!e->ty.is_scalar()) return false;
    if (e->k == Expr::Index || e->k == Expr::Float || e->k == Expr::Int) return true;
    if (is_int(e->ty.sz) || e->ty.sz == ElemSize::Bool) {   // integers of integers: iteration numbers, arrays of integers
      bool ok = true;
      visit_exprs(e, [&](const E& x) {
        if (x->ty.is_scalar() && is_float(x->ty.sz)) ok = false;
        if (x->k == Expr::Call || x->k == Expr::Raw) ok = false;
      });
      return ok;
    }
    if (!is_float(e->ty.sz)) return false;
    if (e->k == Expr::Var) return true;   // (its definition is looked at by itself)
    if (e->k == Expr::Convert || (e->k == Expr::UnOpE && e->uop == UnOp::Sub)) return carries_nan(e->args[0], divides);
    if (e->k != Expr::BinOpE || !(e->bop == BinOp::Add || e->bop == BinOp::Sub || e->bop == BinOp::Mul || e->bop == BinOp::Div)) return false;
    if (e->bop == BinOp::Div && e->args[1]->k == Expr::Float) *divides = true;
    return carries_nan(e->args[0], divides) && carries_nan(e->args[1], divides);
  }

  // how far an update reads each array to the left and to the right
  static std::map<Name, std::pair<int64_t, int64_t>> need_of(const Update& u) {
    std::map<Name, std::pair<int64_t, int64_t>> need;
    for (auto& st : u.body)
      visit_exprs(st->expr, [&](const E& x) {
        if (x->k != Expr::Index) return;
        E rest;
        affine_unit(x->args[1], u.id, &rest);
        const int64_t d = rest->iv - u.c;
        auto& nd = need[u.host.at(x->args[0]->name)];
        nd.first = std::max(nd.first, -d);
        nd.second = std::max(nd.second, d);
      });
    return need;
  }

  bool update_of(const Kernel& k, const S& launch, Update& u, std::vector<Arr>& arrays) {
    if (k.opaque_body || k.body.size() != 1 || k.grid.y != 1 || k.grid.z != 1 || k.block.y != 1 || k.block.z != 1) return false;
    const S& root = k.body[0];
    if (!(root->k == Stmt::For && root->step == 1 && root->lo->k == Expr::Int && root->hi->k == Expr::Int && root->hi->iv > root->lo->iv && root->els.empty()))
      return false;
    if (!(root->map.dim == 0 && (root->map.k == GpuMap::ThreadBlock || (root->map.k == GpuMap::Thread && k.grid.x == 1)))) return false;
    for (size_t q = 0; q < k.params.size(); ++q) {
      if (!k.params[q].ty.is_pointer() && !k.params[q].ty.is_array()) return false;
      const E& a = launch->args[q];
      if (a->k != Expr::Var) return false;
      for (auto& kv : u.host) if (kv.second == a->name) return false;
      u.host[k.params[q].id] = a->name;
    }
    auto arr = [&](const Name& host) -> Arr& {
      for (auto& a : arrays) if (a.host == host) return a;
      arrays.push_back(Arr());
      arrays.back().host = host;
      return arrays.back();
    };
    u.id = root->id;
    u.body = root->body;
    bool first = true;
    std::set<Name> written;
    for (auto& st : root->body) {
      if (st->k == Stmt::Def && st->ty.is_scalar()) continue;
      if (st->k != Stmt::Assign || st->dst->k != Expr::Index || st->dst->args[0]->k != Expr::Var || !u.host.count(st->dst->args[0]->name)) return false;
      E rest;
      if (st->dst->dim_shape.size() != 1 || !affine_unit(st->dst->args[1], root->id, &rest) || rest->k != Expr::Int) return false;
      if (!first && rest->iv != u.c) return false;
      u.c = rest->iv;
      first = false;
      written.insert(u.host[st->dst->args[0]->name]);
    }
    if (first) return false;
    u.lo = root->lo->iv + u.c;
    u.hi = root->hi->iv + u.c;
    bool ok = true;
    auto access = [&](const E& x, bool store) {
      if (x->k == Expr::Call || x->k == Expr::Raw || x->k == Expr::AddrOf || x->k == Expr::RegElem) { ok = false; return; }
      if (x->k != Expr::Index) return;
      if (x->args[0]->k != Expr::Var || !u.host.count(x->args[0]->name) || x->dim_shape.size() != 1) { ok = false; return; }
      Arr& a = arr(u.host[x->args[0]->name]);
      const int bytes = elem_bytes(x->ty.sz);
      if ((a.n != 0 && (a.n != x->dim_shape[0] || a.sz != x->ty.sz)) || (bytes != 4 && bytes != 8)) { ok = false; return; }
      a.n = x->dim_shape[0];
      a.sz = x->ty.sz;
      E rest;
      if (!affine_unit(x->args[1], root->id, &rest) || rest->k != Expr::Int) { ok = false; return; }
      const int64_t d = rest->iv - u.c;
      if (d != 0 && written.count(a.host)) ok = false;   // reads what other iterations of the same launch write
      if (store) a.written = true;
      a.left = std::max(a.left, -d);
      a.right = std::max(a.right, d);
      u.radius = std::max(u.radius, std::abs(d));
    };
    for (auto& st : root->body) {
      visit_exprs(st->expr, [&](const E& x) { access(x, false); });
      if (st->dst) access(st->dst, true);
    }
    return ok;
  }

  S tile(const S& loop) {
    if (!(loop->k == Stmt::For && loop->map.k == GpuMap::None && loop->step == 1 && loop->lo->k == Expr::Int && loop->hi->k == Expr::Int && !loop->body.empty()))
      return S();
    const int64_t steps = loop->hi->iv - loop->lo->iv;
    std::vector<Arr> arrays;
    std::vector<Update> ups;
    for (auto& l : loop->body) {
      if (l->k != Stmt::Launch) return S();
      const Kernel* k = nullptr;
      for (auto& kk : p.kernels) if (kk.name == l->fname) k = &kk;
      for (auto& a : l->args) if (mentions(a, loop->id)) return S();
      Update u;
      if (!k || !update_of(*k, l, u, arrays)) return S();
      ups.push_back(u);
    }
    int64_t per_step = 0, reach = 0, n = 0, words = 0, second_set = 0, lo = 0, hi = INT64_MAX;
    for (auto& u : ups) {
      per_step += u.radius;
      lo = std::max(lo, u.lo);
      hi = std::min(hi, u.hi);
      if (u.lo < 0) return S();
    }
    for (auto& a : arrays) {
      reach = std::max(reach, std::max(a.left, a.right));
      n = std::max(n, a.n);
      hi = std::min(hi, a.n);
      words += elem_bytes(a.sz) / 4;
      if (a.written) second_set += (a.n * elem_bytes(a.sz) + 255) / 256 * 256;
      for (auto& u : ups) if (u.hi > a.n) { bool w = false; for (auto& st : u.body) if (st->dst && st->dst->k == Expr::Index && u.host[st->dst->args[0]->name] == a.host) w = true; if (w) return S(); }
    }
    // Four updates cost what two launches save, except for long arrays of float64, where the launches move as much as the
    // updates did and the division's arithmetic comes on top (Jacobi, tiled and as launches: 1000 6.8 and 12.0 us, 300 000
    // 8.6 and 11.6, 10^6 21.3 and 17.9, 2 * 10^6 34.8 and 26.6, 4 * 10^6 59 and 62, 3 * 10^7 470 and 417; six updates of
    // 10^6 21.0 and 26.2; float32 12.7 and 13.6 for 10^6, 205 and 285 for 3 * 10^7).
    bool wide = false;
    for (auto& a : arrays) wide = wide || elem_bytes(a.sz) == 8;
    const int64_t updates = steps * (int64_t)ups.size();
    if (n < 512 || n > (int64_t(1) << 30) || steps < 2 || updates < (wide && n >= 800000 ? 6 : 4)) return S();
    // The second set is kept between runs up to 1 GiB per plan; a larger one is obtained and given back by every call, out of
    // the device's pool, which costs a tenth of a millisecond up to some size and then hundreds (ten Jacobi steps, float64,
    // tiled and as launches: 1.6 GB 1.6 and 6.6 ms, 4.3 GB 5.2 and 17.9, 6.4 GB 6.7 and 26.3, 9.6 GB 10 and 39 with single
    // calls of 149, 14.4 GB 390 and 58.6).
    if (second_set > (int64_t(6) << 30)) return S();
    // Elements per lane, and with them steps per launch (a margin of up to a quarter of the stretch on either side) and
    // wavefronts: what is expected to be over first.  A step is `work` instructions for every element, `taken` words from the
    // neighbouring lanes and, next to the ends, a blend of `kept` words for every element.  A wavefront issues one in 1.0 ns,
    // where a word from another lane counts as three and a blended one as four, and waits for the steps of a division; a SIMD
    // takes 1.05 ns for each of its share, a whole number of wavefronts, and 1.5 for a lane's word.  A launch costs 2.4 us,
    // 15 ns times the square of the elements (the ends of the arrays are loaded and stored one by one) and its bytes,
    // margins included, at 8 TB/s.
    // Fitted to 2040 times: two updates a step that copy, average three neighbours with and without a division, and add 2, 5,
    // 10, 20 and 33 products and three far ones, floats and doubles, 2000 to 4 * 10^6 elements, 3 to 93 steps, each on 1 to 32
    // elements per lane.  The choice then takes 1.2 % longer than the best of them on average and 16 % at most; a time
    // per element that knows nothing of the update took 2.8 % and 39 % longer (98 updates, its choice and this one: copies of
    // 403 337 doubles 14.0 and 10.1 us, ten products over 403 337 floats 66.8 and 52.2, over 10 007 doubles 42.5 and 35.5;
    // 186 of 403 337 floats with a division 36.7 and 32.0; the one that loses most, five over 403 337 doubles, 25.8 and 29.9).
    double work = 0, waits = 0;
    int64_t taken = 0, kept = 0;
    for (auto& u : ups) {
      for (auto& st : u.body) {
        const double v = instructions(st->expr, &waits);
        work += st->k == Stmt::Assign ? std::max(1.0, v) : v;
        if (st->k == Stmt::Assign) kept += elem_bytes(st->dst->ty.sz) / 4;
      }
      for (auto& kv : need_of(u))
        for (auto& a : arrays) if (a.host == kv.first) taken += (kv.second.first + kv.second.second) * (elem_bytes(a.sz) / 4);
    }
    int64_t Es = 0;
    double best = 0;
    auto consider = [&](int64_t e) {
      if (e * words > 64 || e < reach || per_step > 8 * e) return;
      const int64_t most = per_step > 0 ? 16 * e / per_step : steps, pairs = (steps + 2 * most - 1) / (2 * most);
      const int64_t margin = ((steps + 2 * pairs - 1) / (2 * pairs) * per_step + e - 1) / e * e, useful = WAVE_SIZE * e - 2 * margin;
      if (useful < WAVE_SIZE * e / 4) return;
      const int64_t waves = (n + useful - 1) / useful, share = (waves + 1023) / 1024;
      const double lane = (work + waits + 4.0 * (double)kept) * (double)e + 3.0 * (double)taken;
      const double simd = 1.05 * (double)share * (work * (double)e + 1.5 * (double)taken);
      const double bytes = (double)(n * words * 4) * (1.0 + (double)(WAVE_SIZE * e) / (double)useful);
      const double time = std::max(lane, simd) * (double)steps + (double)(2 * pairs) * (2400.0 + 15.0 * (double)(e * e) + bytes / 8000.0);
      if (Es == 0 || time < best) Es = e, best = time;
    };
    for (int64_t e : {1, 2, 3, 4, 6, 8, 10, 12}) consider(e);
    // Updates that reach further than 12 elements take up to 32, where that beats a launch per update by a tenth: those take
    // 3 us each behind the first, or their arrays at 3.6 TB/s or loads at 15.  Steps of two updates, tiled and as launches,
    // three products 13 elements apart, doubles: three steps over 30 000 elements 13.5 and 15.3 us, over 4 * 10^6 52 and 94,
    // ten over 30 000 16.6 and 57, fifty over 10^6 98 and 447; 32 apart, floats: three over 30 000 29.7 and 16.4 (stays
    // launches), ten over 30 000 35 and 57, over 4 * 10^6 62 and 161; 33 neighbouring ones, ten over 10^6 doubles 61 and 349.
    if (Es == 0) {
      for (int64_t e : {14, 16, 20, 24, 28, 32}) consider(e);
      double launches = -3000.0;
      for (auto& u : ups) {
        double loaded = 0, moved = 0;
        std::set<Name> seen;
        auto count = [&](const E& e) {
          visit_exprs(e, [&](const E& x) {
            if (x->k != Expr::Index) return;
            loaded += elem_bytes(x->ty.sz);
            if (seen.insert(x->args[0]->name).second) moved += elem_bytes(x->ty.sz);
          });
        };
        for (auto& st : u.body) { count(st->expr); count(st->dst); }
        launches += std::max({3000.0, (double)n * moved / 3600.0, (double)n * loaded / 15000.0}) * (double)steps;
      }
      if (1.1 * best > launches) return S();
    }
    if (Es == 0) return S();
    const int64_t most = per_step > 0 ? 16 * Es / per_step : steps;
    const int64_t pairs = (steps + 2 * most - 1) / (2 * most), launches = 2 * pairs;
    const int64_t base_steps = steps / launches, extra = steps % launches;
    const int64_t margin = ((base_steps + (extra > 0)) * per_step + Es - 1) / Es * Es;
    const int64_t width = WAVE_SIZE * Es, useful = width - 2 * margin;
    const int64_t tpb = 256;

    // ---- the kernel
    Kernel f;
    f.name = p.name + "_steps_" + std::to_string(gen.next++);
    f.block.x = tpb;
    f.grid.x = ((n + useful - 1) / useful + tpb / WAVE_SIZE - 1) / (tpb / WAVE_SIZE);
    f.cached_stores = true;
    f.aligned_params = opts.assume_aligned;
    std::map<Name, Name> reg, dst;
    for (auto& a : arrays) {
      KernelParam q;
      q.id = a.host;
      q.ty = Type::pointer(a.sz);
      f.params.push_back(q);
      reg[a.host] = gen.fresh(a.host.s + "_r");
    }
    for (auto& a : arrays)
      if (a.written) {
        KernelParam q;
        q.id = dst[a.host] = gen.fresh(a.host.s + "_to");
        q.ty = Type::pointer(a.sz);
        f.params.push_back(q);
      }
    KernelParam count;
    count.id = gen.fresh("steps");
    count.ty = Type::scalar(ElemSize::I32);
    f.params.push_back(count);
    auto slot = [&](const Arr& a, int64_t e) {
      auto x = std::make_shared<Expr>();
      x->k = Expr::RegElem;
      x->ty = Type::scalar(a.sz);
      x->name = reg[a.host];
      x->args = {iint(e)};
      return E(x);
    };
    auto arr_of = [&](const Name& host) -> const Arr& {
      for (auto& a : arrays) if (a.host == host) return a;
      return arrays[0];
    };
    Name lane = gen.fresh("lane"), wave = gen.fresh("wave"), at = gen.fresh("at");
    E lv = mk_var(lane, ity), wv = mk_var(wave, ity), av = mk_var(at, ity);
    auto index_reg = [&](Expr::Kind kk) {
      auto x = std::make_shared<Expr>();
      x->k = kk;
      x->ty = ity;
      x->iv = 0;
      return E(x);
    };
    Stmts top;
    top.push_back(mk_def(lane, ity, mk_binop(BinOp::Rem, index_reg(Expr::ThreadIdx), iint(WAVE_SIZE), ity)));
    top.push_back(mk_def(wave, ity, add(mk_binop(BinOp::Mul, index_reg(Expr::BlockIdx), iint(tpb / WAVE_SIZE), ity),
                                        mk_binop(BinOp::FloorDiv, index_reg(Expr::ThreadIdx), iint(WAVE_SIZE), ity))));
    const Name first = gen.fresh("start"), meeting = gen.fresh("stretch");
    top.push_back(mk_def(first, ity, mk_binop(BinOp::Sub, mk_binop(BinOp::Mul, wv, iint(useful), ity), iint(margin), ity)));
    E start = mk_var(first, ity);
    int64_t widest = 4;
    for (auto& a : arrays) widest = std::max<int64_t>(widest, elem_bytes(a.sz));
    const int64_t part = WAVE_SIZE * (Es * widest + 16);   // bytes of LDS for a wavefront
    top.push_back(mk_rawstmt("__shared__ __attribute__((aligned(16))) unsigned char " + meeting.str() + "[" + std::to_string(part * (tpb / WAVE_SIZE)) + "];"));
    f.lds_bytes = part * (tpb / WAVE_SIZE);
    auto through_lds = [&](const Arr& a) {
      return std::string("parpy_stretch<") + elem_ctype(a.sz) + ", " + std::to_string(Es) + ">::";
    };
    auto lds_of_wave = [&](const Arr& a) {
      return std::string("(") + elem_ctype(a.sz) + "*)(" + meeting.str() + " + threadIdx.x / 64 * " + std::to_string(part) + "), " + lane.str();
    };
    top.push_back(mk_def(at, ity, add(start, mk_binop(BinOp::Mul, lv, iint(Es), ity))));
    for (auto& a : arrays) {
      auto d = std::make_shared<Stmt>();
      d->k = Stmt::RegDecl;
      d->id = reg[a.host];
      d->ty = Type::scalar(a.sz);
      d->iv = Es;
      top.push_back(d);
    }
    auto elem = [&](const Name& array, const Arr& a, int64_t e) {
      auto x = std::make_shared<Expr>(*mk_index(mk_var(array, Type::pointer(a.sz)), fold_expr(add(av, iint(e))), Type::scalar(a.sz)));
      return E(x);
    };
    auto lt = [&](E a, E b) { return mk_binop(BinOp::Lt, a, b, bty); };
    auto le = [&](E a, E b) { return mk_binop(BinOp::Leq, a, b, bty); };
    auto both = [&](E a, E b) { return mk_binop(BinOp::And, a, b, bty); };
    auto within = [&](int64_t e, int64_t from, int64_t to) {   // from <= at + e < to
      E g = fold_expr(add(av, iint(e)));
      return both(le(iint(from), g), lt(g, iint(to)));
    };

    // Stretches whose results hold no NaN keep them, the others are computed again with divisions of any dividend; those that
    // load a NaN or an infinity are computed with these from the start.  98 updates of 10^6 doubles that are all NaN: 39.6 us
    // with divisions of any dividend alone, 63.0 with one attempt for all and the tests of the ends when it was in vain, 36.4 as
    // it is; with a NaN in every 10 000 40.0, 47.7 and 35.0, of 300 000 doubles, 58 updates, 11.8, 14.4 and 12.4; with none 41.8,
    // 30.6 and 30.3.  Short launches pay up to 0.1 us each for the look at what they load.
    // Steps of two three-point averages before this and the masks for some elements only, with this, and with both: 98 updates of
    // 10^6 doubles 39.1, 32.7 and 31.6 us, 198 of 4 * 10^6 doubles 228, 190 and 183, of as many floats 153, 114 and 109, 118 of
    // 1500 doubles 13.5, 11.7 and 10.6.
    bool divides = false, nan_stays = true;
    for (auto& u : ups)
      for (auto& st : u.body) nan_stays = nan_stays && is_float(st->k == Stmt::Def ? st->ty.sz : st->dst->ty.sz) && carries_nan(st->expr, &divides);
    const bool hopeful = divides && nan_stays;
    const Name lost = hopeful ? gen.fresh("lost") : Name();

    // Arrays that every step writes before it reads them: where updates cover all of a stretch, nothing of them is taken from
    // one launch to the next, so only stretches at the ends load them, and the launches into the second set of arrays
    // store them there alone (98 updates of 10^6 doubles 31.6 -> 28.9 us, 40 instead of 64 MB; 58 of 300 000 11.6 -> 10.5).
    std::set<Name> scratch;
    for (auto& a : arrays) {
      bool read = false, written = false;
      for (auto& u : ups) {
        for (auto& st : u.body) {
          visit_exprs(st->expr, [&](const E& x) { if (x->k == Expr::Index && u.host.at(x->args[0]->name) == a.host) read = true; });
          if (st->dst && st->dst->k == Expr::Index && u.host.at(st->dst->args[0]->name) == a.host) written = true;
        }
        if (read || written) break;
      }
      if (written && !read && base_steps > 0) scratch.insert(a.host);
    }
    KernelParam keep;
    keep.ty = Type::scalar(ElemSize::I32);
    if (!scratch.empty()) {
      keep.id = gen.fresh("keep");
      f.params.push_back(keep);
    }

    // is one of the elements from .. to - 1 element e of its lane
    auto some_of = [&](int64_t from, int64_t to, int64_t e) { return from < to && (e - from % Es + Es) % Es < to - from; };

    auto no_number = [&](const Arr& a) { return "parpy_no_number<" + std::to_string(Es) + ">(" + reg[a.host].str() + ")"; };

    // the path of a stretch: `edge` tests every element against the bounds of the arrays and of the updates
    // (`any`: with divisions of any dividend)
    auto path = [&](bool edge, bool any) {
      Stmts ss;
      for (auto& a : arrays) {
        if (!edge && scratch.count(a.host)) continue;
        if (!edge && Es * elem_bytes(a.sz) > 16) {
          ss.push_back(mk_rawstmt(through_lds(a) + "in(" + reg[a.host].str() + ", " + a.host.str() + " + " + first.str() + ", " + lds_of_wave(a) + ");"));
          continue;
        }
        for (int64_t e = 0; e < Es; ++e) {
          S ld = mk_assign(slot(a, e), elem(a.host, a, e));
          ss.push_back(!edge ? ld : mk_if(within(e, 0, a.n), {ld}, {mk_assign(slot(a, e), is_float(a.sz) ? mk_float(0.0, a.sz) : mk_int(0, a.sz))}));
        }
      }
      if (!any) {
        // (not for values that are no numbers to begin with)
        std::string some = "false";
        for (auto& a : arrays) if (is_float(a.sz) && !scratch.count(a.host)) some += " || " + no_number(a);
        ss.push_back(mk_rawstmt("if (__builtin_amdgcn_ballot_w64(" + some + ") == 0) {"));
      }
      Stmts step, masks;
      std::vector<std::pair<std::vector<int64_t>, E>> known;
      auto covered = [&](int64_t e, int64_t from, int64_t to) {
        for (auto& kn : known) if (kn.first == std::vector<int64_t>{e, from, to}) return kn.second;
        auto call = std::make_shared<Expr>();
        call->k = Expr::Call;
        call->ty = Type::scalar(ElemSize::I32);
        call->sval = "parpy_mask";
        call->args = {within(e, from, to)};
        Name m = gen.fresh("covered");
        masks.push_back(mk_def(m, call->ty, E(call)));
        known.push_back({{e, from, to}, mk_var(m, call->ty)});
        return known.back().second;
      };
      for (auto& u : ups) {
        // what the neighbouring lanes hold
        std::map<std::pair<Name, int64_t>, E> from;
        for (auto& kv : need_of(u)) {
          const Arr& a = arr_of(kv.first);
          auto fetch = [&](int64_t pos, int64_t own, const char* fn) {
            Name nm = gen.fresh(a.host.s + (pos < 0 ? "_left" : "_right"));
            auto call = std::make_shared<Expr>();
            call->k = Expr::Call;
            call->ty = Type::scalar(a.sz);
            call->sval = fn;
            call->args = {slot(a, own)};
            step.push_back(mk_def(nm, Type::scalar(a.sz), call));
            from[{a.host, pos}] = mk_var(nm, Type::scalar(a.sz));
          };
          for (int64_t q = 1; q <= kv.second.first; ++q) fetch(-q, Es - q, "parpy_lane_before");
          for (int64_t q = 0; q < kv.second.second; ++q) fetch(Es + q, q, "parpy_lane_after");
        }
        for (int64_t e = 0; e < Es; ++e) {
          std::map<Name, E> names{{u.id, fold_expr(add(av, iint(e - u.c)))}};
          auto value = [&](const E& x0) {
            E x1 = rewrite_expr(x0, [&](const E& x) -> E {
              if (x->k != Expr::Index) return x;
              E rest;
              affine_unit(x->args[1], u.id, &rest);
              const int64_t pos = e + rest->iv - u.c;
              const Arr& a = arr_of(u.host[x->args[0]->name]);
              return pos >= 0 && pos < Es ? slot(a, pos) : from.at({a.host, pos});
            });
            return subst_vars(x1, names);
          };
          Stmts one;
          for (auto& st : u.body) {
            E v = value(st->expr);
            if (!any) {
              auto call = std::make_shared<Expr>();
              call->k = Expr::Call;
              call->ty = v->ty;
              call->sval = "parpy_no_infinities";
              call->args = {v};
              v = E(call);
            }
            if (st->k == Stmt::Def) {
              Name nm = gen.fresh(st->id.s);
              one.push_back(mk_def(nm, st->ty, v, st->i));
              names[st->id] = mk_var(nm, st->ty);
            } else {
              E to = slot(arr_of(u.host[st->dst->args[0]->name]), e);
              // computed for every element and kept where the update covers it, bit by bit: of a selection the device compiler
              // makes a branch around the element, and the stretches at the ends took twice as long as the others.  Only for
              // the elements of a lane that somewhere are elements of the array which the update leaves alone: stretches start
              // at multiples of Es, and what lies outside the array is read by no element that an update covers.
              if (edge && (some_of(0, u.lo, e) || some_of(u.hi, arr_of(u.host[st->dst->args[0]->name]).n, e))) {
                auto blend = std::make_shared<Expr>();
                blend->k = Expr::Call;
                blend->ty = to->ty;
                blend->sval = std::string("parpy_blend<") + elem_ctype(to->ty.sz) + ">";   // (integers may be computed in 32 bits)
                blend->args = {covered(e, u.lo, u.hi), v, to};
                v = E(blend);
              }
              one.push_back(mk_assign(to, v, st->i));
            }
          }
          step.insert(step.end(), one.begin(), one.end());
        }
      }
      ss.insert(ss.end(), masks.begin(), masks.end());
      Name s = gen.fresh("s");
      ss.push_back(mk_for(s, mk_int(0, ElemSize::I32), mk_var(count.id, Type::scalar(ElemSize::I32)), 1, step, LoopPar()));
      const int64_t outer = margin / Es;
      if (!any) {
        // (elements outside the arrays may be NaN, quotients of the zeros that stand there)
        const std::string l = lost.str(), place = at.str() + " + e";
        ss.push_back(mk_rawstmt("bool " + l + " = false;"));
        for (auto& a : arrays)
          if (a.written)
            ss.push_back(mk_rawstmt(!edge ? l + " = " + l + " || " + no_number(a) + ";" :
                                    "for (int e = 0; e < " + std::to_string(Es) + "; ++e) " + l + " = " + l + " || (" + reg[a.host].str() + "[e] != " + reg[a.host].str() + "[e] && " +
                                    place + " >= 0 && " + place + " < " + std::to_string(a.n) + ");"));
        ss.push_back(mk_rawstmt("if (__builtin_amdgcn_ballot_w64(" + l + " && " + lane.str() + " >= " + std::to_string(outer) + " && " + lane.str() + " < " + std::to_string(WAVE_SIZE - outer) + ") == 0) {"));
      }
      Stmts put, put_kept;
      for (auto& a : arrays) {
        if (!a.written) continue;
        const bool only_kept = !edge && scratch.count(a.host);
        if (!edge && Es * elem_bytes(a.sz) > 16) {
          ss.push_back(mk_rawstmt((only_kept ? "if (" + keep.id.str() + ") " : "") + through_lds(a) + "out(" + reg[a.host].str() + ", " + dst[a.host].str() + " + " + first.str() + ", " + lds_of_wave(a) + ", " + std::to_string(margin) + ");"));
          continue;
        }
        for (int64_t e = 0; e < Es; ++e) {
          S stt = mk_assign(elem(dst[a.host], a, e), slot(a, e));
          (only_kept ? put_kept : put).push_back(edge ? mk_if(within(e, 0, a.n), {stt}, {}) : stt);
        }
      }
      if (!put_kept.empty()) put.push_back(mk_if(mk_raw(keep.id.str(), bty), put_kept, {}));
      if (!put.empty()) ss.push_back(mk_if(both(le(iint(outer), lv), lt(lv, iint(WAVE_SIZE - outer))), put, {}));
      if (!any) ss.push_back(mk_rawstmt("return; } }"));
      return ss;
    };
    // A stretch that lies inside all bounds takes the plain path.  Values next to the bounds of a stretch are wrong (its
    // outermost lanes have no neighbour) and stay within the margin.
    E inside = both(le(iint(lo), start), le(add(start, iint(width)), iint(hi)));
    top.push_back(mk_if(inside, path(false, !hopeful), path(true, !hopeful)));
    if (hopeful) top.push_back(mk_if(inside, path(false, true), path(true, true)));
    f.body = top;
    p.kernels.push_back(f);

    // ---- the host side
    Stmts tiled;
    std::map<Name, Name> tmp;
    for (auto& a : arrays)
      if (a.written) {
        auto al = std::make_shared<Stmt>();
        al->k = Stmt::Alloc;
        al->id = tmp[a.host] = gen.fresh(a.host.s + "_next");
        al->ty = Type::scalar(a.sz);
        al->iv = a.n;
        tiled.push_back(al);
      }
    Name pair = gen.fresh("pair");
    auto launch = [&](int64_t which) {
      auto l = std::make_shared<Stmt>();
      l->k = Stmt::Launch;
      l->fname = f.name;
      l->grid = f.grid;
      l->block = f.block;
      l->i = loop->i;
      for (auto& a : arrays) l->args.push_back(mk_var(which == 1 && a.written ? tmp[a.host] : a.host, Type::pointer(a.sz)));
      for (auto& a : arrays) if (a.written) l->args.push_back(mk_var(which == 1 ? a.host : tmp[a.host], Type::pointer(a.sz)));
      E number = add(mk_binop(BinOp::Mul, mk_var(pair, ity), iint(2), ity), iint(which));
      const E number_of_steps = extra == 0 ? iint(base_steps) : add(iint(base_steps), mk_binop(BinOp::Lt, number, iint(extra), bty));
      l->args.push_back(number_of_steps);
      if (!scratch.empty()) l->args.push_back(iint(which));
      return S(l);
    };
    tiled.push_back(mk_for(pair, iint(0), iint(pairs), 1, {launch(0), launch(1)}, LoopPar(), loop->i));
    for (auto& kv : tmp) {
      auto fr = std::make_shared<Stmt>();
      fr->k = Stmt::Free;
      fr->id = kv.second;
      tiled.push_back(fr);
    }
    // The tiled loop carries every array in registers of its own and in a second set of memory, so an element must not be
    // reachable under two names when one of them is written: `C is B`, or views that overlap, is legal in a loop of
    // launches none of which writes an array that it reads under another name.  Names say nothing about that and a plan
    // serves any pointers, so it tests the address ranges and holds the loop of launches for those that meet.
    std::vector<HostArray> ranges;
    for (auto& a : arrays) ranges.push_back({a.host, a.n * elem_bytes(a.sz), a.written});
    const E apart = arrays_disjoint(p, ranges);
    // Nor must the call fail for the second set: what the device has left, or the fixed amount of scratch memory of a run
    // that may allocate nothing, may not hold it.
    auto fits = std::make_shared<Expr>(*mk_raw("parpy_temporaries_fit(" + std::to_string(second_set) + ")", bty));
    fits->iv = second_set;
    auto either = clone(mk_if(apart ? both(apart, E(fits)) : E(fits), tiled, {loop}));
    either->fname = "one launch per update";
    return mk_scope({S(either)});
  }

  Stmts walk(const Stmts& ss) {
    Stmts out;
    for (auto& s : ss) {
      if (S t = tile(s)) { for (auto& q : t->body) out.push_back(q); continue; }
      auto r = clone(s);
      if (s->k == Stmt::For || s->k == Stmt::While || s->k == Stmt::If) {
        r->body = walk(s->body);
        r->els = walk(s->els);
      }
      out.push_back(r);
    }
    return out;
  }

  void run() {
    p.host = walk(p.host);
    // kernels that nothing launches any more
    std::set<std::string> used;
    visit_stmts(p.host, [&](const S& s) { if (s->k == Stmt::Launch) used.insert(s->fname); });
    std::vector<Kernel> keep;
    for (auto& k : p.kernels) if (used.count(k.name)) keep.push_back(k);
    p.kernels = keep;
  }
};

}  // namespace

void time_tile(Program& p, const Options& opts, NameGen& gen) { TimeTile(p, opts, gen).run(); }

}  // namespace hipopt
}  // namespace parpy
