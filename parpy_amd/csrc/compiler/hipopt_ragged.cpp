// gfx950 memory passes, rewrites that change a launch: sums whose bounds are data (rows of a sparse matrix).
#include <algorithm>
#include <functional>

#include "hipopt_pass.hpp"

namespace parpy {
namespace hipopt {

namespace {

// ================================================================ teams of lanes for sums of uneven length
// `for row: for i in rows[row] .. rows[row + 1]: y[row] += f(i)` and the same with a column loop around the sum
// (`C[row, j] += f(i, j)`): how long a row is stands in memory, a few rows may hold a thousand times the average,
// and each element costs two dependent loads (its column, then what the column selects).  Two things bound such a
// kernel when a fixed group of lanes walks each row one element at a time: the round trips of the longest row, and
// one element in flight per lane.
//
//   * A row belongs to a team of T = L * P adjacent lanes of a wavefront: L lanes lie along the columns (16 bytes
//     each where the columns allow it), P subteams take every P-th element of the row.
//   * A subteam issues U elements at a time: index loads first, then what they select.  The last batch is clamped to
//     the row's last element instead of branching, so that its loads are issued together as well.
//   * A row longer than `longest` elements is shared by all waves of a workgroup: by one of those in front of the others,
//     which look for such rows and queue them in LDS, or, where there are none, by that of its own team.
//   * Columns are divided into slabs, one to every second, fourth or eighth workgroup (`slabs`).
//
// Measured (100 000 rows of 50 non-zeros on average, the longest 15 800, float64): eight lanes per row, one element in
// flight 547 us, in teams 34 us.  The gathers out of L2 are then what bounds it: 5.5 million lines requested (counted, 87 %
// of them hits), 158 per nanosecond.  20 000 rows of 24 on average (longest 3400)
// times a 128-column matrix: one workgroup per row with the sum read and written back in LDS per element 840 us, in
// teams 42 us, with the long rows in front (below) 34: the longest pulled 1.7 MB through one compute unit, and 165 of the 261 MB
// that the L2s deliver came from behind them, since the 10 MB matrix does not fit a die's 4 MB.  In two slabs 26.6 us.
struct RaggedSum {
  Program& p;
  const Options& opts;
  NameGen& gen;
  ElemSize isz;
  Type ity;
  Type bty = Type::scalar(ElemSize::Bool);

  RaggedSum(Program& prog, const Options& o, NameGen& g) : p(prog), opts(o), gen(g), isz(o.int_size()), ity(Type::scalar(o.int_size())) {}

  // a launch of this shape, taken apart
  struct Rows {
    Name row;
    int64_t n = 0;            // rows
    bool has_col = false;
    Name col;
    int64_t cols = 1;
    Stmts pre;                // definitions of the row in front of the sum
    S loop;                   // the sum loop
    Stmts defs;               // definitions inside it
    E acc, term, start;       // accumulator, summand, value the sum starts from
    Stmts post;               // statements after the sum
    int64_t elements = 0;     // length of the array that the loop variable walks, 0 when there is none
    bool bounded = false;     // the loop variable stays below it (not when all its accesses are under tests)
    int64_t tpb = 0;          // threads per workgroup
    bool one_group = false;   // the launch was a single workgroup
  };

  E iint(int64_t v) { return mk_int(v, isz); }
  E add(E a, E b) { return mk_binop(BinOp::Add, a, b, a->ty); }

  // `acc = acc + term` with definitions in front of it, bounds that are not both constants
  bool sum_loop(const S& s, Rows& r) {
    if (!(s->k == Stmt::For && s->map.k == GpuMap::None && !s->unroll && s->step == 1 && !s->body.empty() && !s->par.reduction)) return false;
    if (s->lo->k == Expr::Int && s->hi->k == Expr::Int) return false;
    std::set<Name> inner;
    for (size_t q = 0; q + 1 < s->body.size(); ++q) {
      const S& d = s->body[q];
      if (d->k != Stmt::Def || !d->ty.is_scalar()) return false;
      inner.insert(d->id);
    }
    const S& a = s->body.back();
    if (a->k != Stmt::Assign) return false;
    const E& acc = a->dst;
    bool scalar_acc = acc->k == Expr::Var && acc->ty.is_scalar() && !inner.count(acc->name);
    bool elem_acc = acc->k == Expr::Index && acc->args[0]->k == Expr::Var && !mentions(acc->args[1], s->id) && !has_load(acc->args[1]);
    if (!(scalar_acc || elem_acc) || !(acc->ty.sz == ElemSize::F32 || acc->ty.sz == ElemSize::F64)) return false;
    if (elem_acc)
      for (auto& n : inner) if (mentions(acc->args[1], n)) return false;
    if (!(a->expr->k == Expr::BinOpE && a->expr->bop == BinOp::Add)) return false;
    const E &l = a->expr->args[0], &rr = a->expr->args[1];
    E term = expr_eq(l, acc) ? rr : expr_eq(rr, acc) ? l : E();
    if (!term) return false;
    const Name& acc_name = scalar_acc ? acc->name : acc->args[0]->name;
    bool ok = !mentions(term, acc_name) && !mentions(s->lo, acc_name) && !mentions(s->hi, acc_name);
    int loads = 0;
    std::function<void(const E&, bool)> scan = [&](const E& x, bool always) {
      if (x->k == Expr::Call || x->k == Expr::AddrOf || x->k == Expr::Raw || x->k == Expr::RegElem) ok = false;
      E rest;
      if (x->k == Expr::Index) {
        ++loads;
        if (x->dim_shape.size() == 1 && affine_unit(x->args[1], s->id, &rest) && rest->k == Expr::Int) {
          r.elements = std::max(r.elements, x->dim_shape[0]);
          r.bounded = r.bounded || always;
        }
      }
      for (size_t q = 0; q < x->args.size(); ++q)
        if (x->args[q]) scan(x->args[q], always && !may_skip(x, q));
    };
    scan(term, true);
    for (size_t q = 0; q + 1 < s->body.size(); ++q) {
      scan(s->body[q]->expr, true);
      if (mentions(s->body[q]->expr, acc_name)) ok = false;
    }
    if (!ok || loads < 1) return false;
    r.loop = s;
    r.acc = acc;
    r.term = term;
    r.defs = Stmts(s->body.begin(), s->body.end() - 1);
    return true;
  }

  // statements of one row (or of one row and column): definitions, the sum, what is done with it
  bool row_body(const Stmts& body, Rows& r) {
    int pos = -1;
    for (size_t q = 0; q < body.size(); ++q) {
      const S& st = body[q];
      if (st->k == Stmt::For) {
        if (pos >= 0 || !sum_loop(st, r)) return false;
        pos = (int)q;
        continue;
      }
      bool simple = (st->k == Stmt::Def && st->ty.is_scalar()) ||
                    (st->k == Stmt::Assign && (st->dst->k == Expr::Index || (st->dst->k == Expr::Var && st->dst->ty.is_scalar())));
      if (!simple) return false;
      bool raw = false;
      auto scan = [&](const E& e) { visit_exprs(e, [&](const E& x) { if (x->k == Expr::Call || x->k == Expr::AddrOf || x->k == Expr::Raw) raw = true; }); };
      scan(st->expr);
      scan(st->dst);
      if (raw) return false;
    }
    if (pos < 0) return false;
    const bool elem = r.acc->k == Expr::Index;
    const Name& acc_name = elem ? r.acc->args[0]->name : r.acc->name;
    for (int q = 0; q < (int)body.size(); ++q) {
      if (q == pos) continue;
      const S& st = body[q];
      if (q < pos) {
        // what the sum starts from: the last store to the element, or the definition of the scalar
        bool init = elem ? st->k == Stmt::Assign && expr_eq(st->dst, r.acc) : st->k == Stmt::Def && st->id == acc_name;
        if (init && !r.start && !mentions(st->expr, acc_name)) { r.start = st->expr; continue; }
        if (st->k == Stmt::Assign && st->dst->k == Expr::Index) return false;
        if (mentions(st->expr, acc_name) || (st->dst && mentions(st->dst, acc_name))) return false;
        if (r.start && st->k == Stmt::Assign && mentions(r.start, st->dst->name)) return false;   // (the start value is evaluated behind the sum)
        r.pre.push_back(st);
      } else {
        if (elem && (mentions(st->expr, acc_name) || (st->dst && mentions(st->dst, acc_name)))) return false;
        if (st->k == Stmt::Assign && st->dst->k == Expr::Index && st->dst->args[0]->k != Expr::Var) return false;
        r.post.push_back(st);
      }
    }
    if (!r.start) {
      if (!elem) return false;
      r.start = r.acc;
    }
    // a store behind the sum to an array that the start value reads would be reordered with it only across rows; inside
    // the row the start value is read first, as written
    return true;
  }

  bool match(const Kernel& k, Rows& r) {
    if (k.body.size() != 1 || k.block.y != 1 || k.block.z != 1) return false;
    const S& root = k.body[0];
    if (!(root->k == Stmt::For && root->step == 1 && root->lo->k == Expr::Int && root->lo->iv == 0 && root->hi->k == Expr::Int)) return false;
    r.row = root->id;
    r.n = root->hi->iv;
    if (r.n < 64) return false;   // (less than a wavefront of rows)
    const bool one_group = root->map.k == GpuMap::Thread && k.grid.x == 1;
    if ((root->map.k == GpuMap::ThreadBlock || one_group) && root->map.dim == 0) {
      // one thread per row
      if (k.grid.y != 1 || k.grid.z != 1 || (one_group && r.n > root->map.n)) return false;
      r.tpb = one_group ? 256 : root->map.tpb;
      r.one_group = one_group;
      return row_body(root->body, r);
    }
    if (root->map.k == GpuMap::Block && k.grid.x * k.grid.y * k.grid.z == r.n && root->map.n == r.n) {
      // one workgroup per row, its threads along the columns
      S inner;
      Stmts before;
      for (auto& st : root->body) {
        if (st->k == Stmt::Sync) continue;
        if (st->k == Stmt::Def && st->ty.is_scalar() && !inner) { before.push_back(st); continue; }
        if (inner || !thread_mapped(st)) return false;
        inner = st;
      }
      if (!inner || inner->step != 1 || inner->lo->k != Expr::Int || inner->lo->iv != 0 || inner->hi->k != Expr::Int || inner->par.reduction) return false;
      r.has_col = true;
      r.col = inner->id;
      r.cols = inner->hi->iv;
      r.tpb = 1024;   // the threads that share a long row (3000 rows of 60 times 256 columns: 256 / 512 / 1024 threads 107 / 67 / 57 us)
      if (r.cols < 1 || !row_body(inner->body, r)) return false;
      // everything in front of the sum belongs to the row; its bounds are the same for all columns
      for (auto& st : r.pre)
        if (st->k != Stmt::Def || mentions(st->expr, r.col)) return false;
      if (mentions(r.loop->lo, r.col) || mentions(r.loop->hi, r.col)) return false;
      if (r.acc->k == Expr::Index && !mentions(r.acc->args[1], r.col)) return false;
      before.insert(before.end(), r.pre.begin(), r.pre.end());
      r.pre = before;
      return true;
    }
    return false;
  }

  static int64_t average(const Rows& r) { return r.elements > 0 ? std::max<int64_t>(1, r.elements / r.n) : 32; }

  // Rows that are no whole number of vectors: the last vector ends with the row, and what it shares with the one in front of it
  // is summed and stored twice, in the same order, by lanes of one wavefront, which has read what a sum reads before it stores
  // any.  Not where the end of a row reads memory: the element that one of the two has
  // stored may be what the other reads.  A quarter of the load instructions, and as many more rows to a wavefront.  Floats, a
  // column per lane before and four now, us: 20 000 rows of 24 times 33 / 65 / 101 / 162 / 255 columns 26.1 -> 19.7, 33.2 -> 27.7,
  // 43.0 -> 32.0, 64.8 -> 50.8, 69.4 -> 62.9, 3000 of 40 times 33 / 65 / 101 / 199 14.6 -> 9.1, 18.3 -> 11.8, 15.0 -> 12.1, 20.5 -> 17.1,
  // 60 000 of 6 times 17 / 65 / 101 20.9 -> 14.5, 34.2 -> 28.5, 36.2 -> 32.2.  Rows of a wavefront each gain less, and lose
  // where they are short (60 000 of 6 times 162 46.6 -> 47.6, 255 67.5 -> 67.7; 8000 of 10 times 162 15.2 -> 16.4, but times 250
  // 17.4 -> 15.0) or leave lanes idle (20 000 of 24 times 129 / 145
  // 43.0 -> 45.4, 45.8 -> 47.3).  Doubles, of which the device compiler makes two loads again, stay a column per lane.
  static bool whole_vectors_pay(const Rows& r, int64_t v) {
    const int64_t slots = (r.cols + v - 1) / v, lanes = (slots + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
    if (v != 4 || r.cols < 4 * v || has_load(r.start)) return false;
    if (slots > WAVE_SIZE / 2 && (average(r) < 8 || 1000 - 1000 * slots / lanes > (average(r) < 24 ? 130 : 420))) return false;
    for (auto& st : r.post) {
      if (has_load(st->expr)) return false;
      if (st->dst && st->dst->k == Expr::Index && has_load(st->dst->args[1])) return false;
    }
    return true;
  }

  // columns a lane takes side by side: 16 bytes when every access along the columns is unit-stride through an aligned parameter
  int64_t column_vector(const Kernel& k, const Rows& r) {
    if (!r.has_col || !opts.assume_aligned) return 1;
    int64_t v = 0;
    bool ok = true;
    std::set<Name> params;
    for (auto& q : k.params) if (q.ty.is_pointer()) params.insert(q.id);
    auto scan = [&](const E& e) {
      visit_exprs(e, [&](const E& x) {
        if (x->k != Expr::Index || !mentions(x->args[1], r.col)) return;
        E rest;
        if (!affine_unit(x->args[1], r.col, &rest) || x->args[0]->k != Expr::Var || !params.count(x->args[0]->name)) { ok = false; return; }
        int64_t w = 16 / elem_bytes(x->ty.sz);
        if (w != 4 && w != 2) { ok = false; return; }
        v = v == 0 ? w : std::min(v, w);
      });
    };
    scan(r.term);
    scan(r.acc);
    for (auto& d : r.defs) scan(d->expr);
    if (!ok || v <= 0) return 1;
    return r.cols % v == 0 || whole_vectors_pay(r, v) ? v : 1;
  }

  // does a row read, in front of its columns, an array that they store, or one that may be the same memory: of the same type,
  // and large enough to have an element in every row
  static bool reads_first(const Rows& r) {
    std::vector<E> stored;
    if (r.acc->k == Expr::Index) stored.push_back(r.acc);
    for (auto& st : r.post) if (st->dst && st->dst->k == Expr::Index) stored.push_back(st->dst);
    auto elements = [](const E& x) {
      if (x->dim_shape.empty()) return INT64_MAX;
      int64_t n = 1;
      for (int64_t d : x->dim_shape) n *= d;
      return n;
    };
    bool found = false;
    auto scan = [&](const E& e) {
      visit_exprs(e, [&](const E& x) {
        if (x->k != Expr::Index) return;
        for (auto& q : stored) found = found || expr_eq(x->args[0], q->args[0]) || (x->ty.sz == q->ty.sz && elements(x) > (r.n - 1) * r.cols);
      });
    };
    for (auto& st : r.pre) scan(st->expr);
    scan(r.loop->lo);
    scan(r.loop->hi);
    return found;
  }

  static int64_t pow2_at_least(int64_t n) { int64_t q = 1; while (q < n) q *= 2; return q; }

  // Slabs of columns: workgroups b, b + n, b + 2n, ... sum the rows over one n-th of the columns.  Workgroups are dealt to the
  // eight dies in turn, so with two, four or eight slabs a die's L2 holds its slab of the selected rows only (pieces of 512 / 256
  // / 128 bytes out of 10 MB: 24.1 us in one slab, 15.8 in two, 12.8 in four; where they end up is a matter of speed alone), and
  // the longest rows are shared by as many workgroups.  Rows go to as many slabs as leave a wavefront one batch of loads for a
  // row of average length, 64 lanes with four times 16 bytes (an eighth less will do).  Rows of uneven length, in one slab and
  // in 2 / 4 / 8, us: 20 000 of 24 times 128 columns 43.7 (33.8 on 1024 threads) and 26.3 / 27.0 (6 KB and 3 KB a wavefront);
  // 16 000 of 24 times 256: 77.9 (61.3) and 47.5 / 35.0 / 46.9; 8192 of 20 times 128: 19.1 and 11.9 / 13.7 / 22.0; 40 000 of 16
  // times 128: 50.1 (45.7) and 39.3 / 53.5; 60 000 of 20 times 64: 41.8 and 45.6; 100 000 of 4 times 256: 73.7 and 86.3.
  // A last vector that is moved is not the first of its slab: what it shares with the one in front of it would be columns of two
  // workgroups, and one of them may read what the other has stored (`t += A[k] * (B[cols[k], j] - E[i, j])`, `E[i, j] = t`).  Nor
  // is a row divided that reads in front of its columns what they store (`x = E[i, 0]`), under whatever name.
  static int64_t slabs(const Rows& r, int64_t V, int64_t avg) {
    if (!r.has_col || reads_first(r)) return 1;
    const int64_t slots = (r.cols + V - 1) / V;
    int64_t row = 0;   // bytes of a selected row
    auto scan = [&](const E& e) {
      visit_exprs(e, [&](const E& x) { if (x->k == Expr::Index && mentions(x->args[1], r.col)) row = std::max(row, r.cols * elem_bytes(x->ty.sz)); });
    };
    scan(r.term);
    for (auto& d : r.defs) scan(d->expr);
    // thousandths of the lanes along the columns that have none: no more than in one slab, or than 420 (65 columns on 128 lanes,
    // two slabs of 13 895 rows of 21 times 129: 33.3 us instead of 28.8; 77 on 128, 3616 of 21 times 153: 13.8 instead of 15.7)
    auto idle = [&](int64_t n) {
      const int64_t own = (slots + n - 1) / n, lanes = std::min<int64_t>(WAVE_SIZE, pow2_at_least(own)), taken = (own + lanes - 1) / lanes * lanes;
      return 1000 - 1000 * own / taken;
    };
    int64_t best = 1;
    for (int64_t n = 2; n <= 8 && r.cols >= 16 * n && slots >= n && r.n * WAVE_SIZE * n <= (int64_t(1) << 30) && avg * row >= 3584 * n; n *= 2)
      if (idle(n) <= std::max<int64_t>(idle(1), 420) && !(r.cols % V != 0 && (slots - 1) % ((slots + n - 1) / n) == 0)) best = n;
    return best;
  }

  // a[v + c] and a[v + c + 1]
  static bool adjacent(E a, E b, const Name& v) {
    while (a->k == Expr::Convert) a = a->args[0];
    while (b->k == Expr::Convert) b = b->args[0];
    if (a->k != Expr::Index || b->k != Expr::Index || !expr_eq(a->args[0], b->args[0])) return false;
    E ra, rb;
    return affine_unit(a->args[1], v, &ra) && affine_unit(b->args[1], v, &rb) && ra->k == Expr::Int && rb->k == Expr::Int && rb->iv == ra->iv + 1;
  }

  // Loads of every element that depend on its number alone (`cols[i]`, `values[i]`): each is executed for all elements of
  // a row, and nothing in the kernel writes there.
  std::vector<E> element_loads(const Kernel& k, const Rows& r) {
    std::set<Name> params, written;
    for (auto& q : k.params) if (q.ty.is_pointer()) params.insert(q.id);
    visit_stmts(k.body, [&](const S& c) {
      if (c->k == Stmt::Assign && c->dst->k == Expr::Index && c->dst->args[0]->k == Expr::Var) written.insert(c->dst->args[0]->name);
    });
    std::vector<E> out;
    std::function<void(const E&, bool)> scan = [&](const E& x, bool always) {
      if (!x) return;
      E rest;
      if (always && x->k == Expr::Index && x->args[0]->k == Expr::Var && params.count(x->args[0]->name) && !written.count(x->args[0]->name) &&
          !k.no_restrict && x->ty.is_scalar() && x->ty.sz != ElemSize::Bool && affine_unit(x->args[1], r.loop->id, &rest) &&
          rest->k == Expr::Int) {
        bool known = false;
        for (auto& e : out) known = known || expr_eq(e, x);
        if (!known) out.push_back(x);
        return;
      }
      for (size_t q = 0; q < x->args.size(); ++q) scan(x->args[q], always && !may_skip(x, q));
    };
    for (auto& d : r.defs) scan(d->expr, true);
    scan(r.term, true);
    return out;
  }

  bool apply(Kernel& k, const StmtP& launch) {
    Rows r;
    if (!match(k, r)) return false;
    const int64_t V = column_vector(k, r);
    const int64_t words = elem_bytes(r.acc->ty.sz) / 4;
    const int64_t avg = average(r);
    const int64_t SL = slabs(r, V, avg);
    const bool moved = r.cols % V != 0;                     // the last vector of columns, to end with the row
    const int64_t all_slots = (r.cols + V - 1) / V, slots = (all_slots + SL - 1) / SL;   // vectors along the columns: all, of a slab
    const int64_t wide = slots * V;                                            // columns of a slab
    const int64_t L = std::min<int64_t>(WAVE_SIZE, pow2_at_least(slots));
    const int64_t chunks = (slots + L - 1) / L;
    const int64_t K = chunks * V;                           // sums a lane holds
    if (K * words > 16) return false;
    // Subteams: two elements of an average row per lane, at least four lanes so that they share cache lines.  (100 000
    // rows of 50 non-zeros, float64: 4 / 8 / 16 / 32 / 64 lanes 53 / 47 / 40 / 38 / 45 us; 300 000 rows of 16: 41.7 us
    // on four lanes, 36.0 on eight and sixteen; 50 000 rows of 200: 110 us on 16, 94 on 64; 50 000 rows of 8 times 32
    // columns: 22.4 / 17.7 / 17.4 / 20.9 us for 1 / 2 / 4 / 8 subteams.)  Rows that were the threads of one workgroup
    // are too few to fill the chip in any case and take eight lanes, but for long ones, of which the others' round trips are what
    // they wait for (1000 rows of 50 doubles on 8 / 16 / 32 / 64 lanes 5.1 / 4.2 / 4.0 / 4.0 us, of 100 6.9 / 5.3 / 4.5 / 4.2, of 200 11.2 /
    // 8.0 / 6.3 / 5.6, of 200 floats 9.4 / 6.8 / 5.4 / 5.0, of 20 3.9 on any; sums of columns have lanes enough).
    auto subteams = [&](int64_t lanes) {
      if (r.one_group && (r.has_col || avg < 48)) return int64_t(8);
      return std::min<int64_t>(WAVE_SIZE / lanes, std::max<int64_t>(pow2_at_least((avg + 1) / 2), r.has_col ? 1 : 4));
    };
    // more wavefronts than run at once
    constexpr int64_t RESIDENT = 256 * 2048;
    // Elements in flight per lane: up to sixteen registers of what they select; four for single sums, but where many wavefronts
    // follow each other, as many as an average row has for 32 lanes: every load of a batch is issued for all of its lanes.
    // (100 000 rows of 33 / 40 / 50 / 64 doubles on 32 lanes, two and four: 23.5 and 27.1 us, 26.7 and 30.1, 32.5 and 34.0, 50.4
    // and 53.6, but 40 000 of 64 20.9 and 19.4, and floats 20.1 and 20.5, 23.2 and 23.2, 29.8 and 28.1, 36.1 and 34.6.  40 000
    // rows of 200 doubles with eight on 32 lanes 63.0, four on 64 72.7, as many floats 56.1 and 63.4, 50 000 of 200 doubles 74.9 and
    // 83.5, of 150 61.5 and 61.7, of 150 floats 44.3 and 46.4; 60 000 of 130 doubles 65.8 and 64.4.)
    const bool two = !r.has_col && words == 2 && subteams(L) == 32 && r.n * 32 > 7 * RESIDENT / 2, eight = !r.has_col && avg >= (words == 2 ? 160 : 128) && r.n * 64 > 4 * RESIDENT;
    const int64_t U = r.has_col ? std::max<int64_t>(2, std::min<int64_t>(8, 16 / (K * words))) : two ? 2 : eight ? 8 : 4;
    const int64_t P = eight ? 32 : subteams(L), T = L * P;
    const int64_t lanes0 = std::min<int64_t>(WAVE_SIZE, pow2_at_least(all_slots)), T0 = lanes0 * subteams(lanes0);   // a team of the whole row
    if ((all_slots + lanes0 - 1) / lanes0 * V * words > 16 || (r.has_col && r.tpb < r.cols)) return false;
    const bool queues = r.n * T0 > RESIDENT;
    // Single sums: a workgroup is over with its slowest wavefront; 1024 / 512 / 256 threads 36.6 / 34.2 / 34.2 us for the 50
    // non-zeros above, 29.9 / 28.2 / 30.2 in floats, 99.8 / 91.2 / 91.9 for 10^6 rows of 10 floats.  Where all wavefronts run at
    // once: 16 000 rows of 60 floats 12.5 / 10.6 / 10.4, doubles 15.2 / 14.0 / 13.0, 20 000 of 7 floats 6.6 / 5.8 / 5.6, 10 000 of
    // 100 10.5 / 10.5 / 10.2, 12 000 of 200 doubles 26.2 / 26.1 / 26.5.  Up to 5000 rows doubles gain (1100 of 100 4.6 / 4.0, 2500
    // of 150 7.0 / 6.4, 3000 of 200 12.1 / 11.0, 4000 of 100 7.8 / 6.9, 4900 of 60 5.9 / 5.4; where the time is that of one longest row
    // it depends on the matrix: 4500 of 180 12.0 / 11.5 and 11.9 / 12.2, 2000 of 100 5.1 / 5.1), and floats, which gain or lose,
    // keep the threads they have (2000 of 100 3.8 / 4.0, 4000 of 199 7.7 / 8.1, 5000 of 150 8.3 / 8.5; 3000 of 200 8.7 / 8.2, 4500 of
    // 180 8.6 / 8.2).
    // Rows of columns: 512 threads, unless a row of average length is more than one batch of its team and cannot be divided into
    // slabs, whose longest rows take 1024 (7794 rows of 45 times 32 columns: 13.5 us and 12.6; 3000 of 200 times 20: 25.8 and
    // 20.2; but 100 000 of 20 times 32: 39.7 and 50.9, 58 973 of 27 times 32: 29.7 and 38.1).
    const bool fewer = r.has_col ? wide <= 512 && (SL > 1 || 8 * avg < 7 * P * U || r.n * T0 > 4 * RESIDENT) : queues || words == 2 || r.n > 5000;
    const int64_t tpb = fewer ? std::min<int64_t>(r.tpb, 512) : r.tpb;
    if (tpb % WAVE_SIZE != 0 || tpb < L * V || r.n * T * SL > (int64_t(1) << 30)) return false;
    const int64_t teams = tpb / T, waves = tpb / WAVE_SIZE;
    if (r.has_col && (tpb < wide || waves * L * K * elem_bytes(r.acc->ty.sz) > 64 * 1024)) return false;
    // Rows longer than this are shared by the workgroup.  A shared row costs two barriers and a round trip of its own,
    // and the waves that have no such row wait for it: 256 elements for single sums (128 costs 5 to 20 %), fewer when
    // every element moves a row of columns (64 against 256 elements: 17.4 and 20.1 us for the 32-column product above).
    const int64_t longest = r.has_col ? std::max<int64_t>(64, 2 * avg) : std::max<int64_t>(256, 4 * avg);
    // The rows longer than that go to workgroups in front of the others, which look for them and share each as above: started
    // in order, the longest may start last, and in the others' workgroups sixteen wavefronts would wait for them.  Where more
    // wavefronts are launched than run at once (slabs not counted), 1024 such workgroups for rows of columns (30 978 rows of 19
    // on average times 32 columns: 14.5 us, 15.9 with 512, 17.5 with 256; 20 000 of 24 times 128 in two slabs: 26.9, 30.1, 33.8;
    // 100 000 of 4 times 256: 74.6, 74.4) and 512 for single sums (100 000 rows of 50, doubles: 36.3, 37.5 with 1024; 39.5 us
    // with every long row shared where it is).  Fewer rows of columns: one for 160 elements, up to 512 (5835 of 40 times 128:
    // 29.8 us with 148 in front, 20.0 / 15.9 / 15.3 with 256 / 512 / 1024; 1000 of 64 times 256: 12.4 / 9.1 / 8.8 with 125 / 256
    // / 512; 1045 of 10 times 256: 4.4 / 4.5 / 5.3 with 130 / 256 / 1024), but for a launch whose undivided rows fill the device
    // exactly.  Fewer single sums: one for sixteen rows where there is room beside the others (3000 rows of 60, doubles 6.3 ->
    // 4.9 us, 5.5 with one for four; 20 000 of 30: 9.8 -> 9.0), else 256 for doubles, whose others then start a little later
    // (none / 64 / 128 / 256 / 512: 16 000 rows of 60 14.1 / 14.4 / 13.1 / 11.6 / 12.4, 15 500 of 40 10.3 / 10.2 / 8.9 / 8.5 / 9.1, 7800
    // of 80 10.4 / 11.0 / 9.5 / 9.0 / 9.2, 8000 of 150 16.0 / 17.5 / 15.4 / 15.5 / 15.6).  Floats keep the queues of the others'
    // workgroups there, as the tests of this rule have it; 256 in front would be worth -2 to 20 % (none / 256: 16 000 of 40 7.3 / 6.3,
    // 14 400 of 60 9.7 / 8.9, 16 300 of 64 10.8 / 11.0, 8100 of 100 9.0 / 8.7, 8000 of 150 13.6 / 11.4, 31 000 of 25 7.9 / 7.2).
    const int64_t room = RESIDENT / r.tpb - (r.n * T0 + r.tpb - 1) / r.tpb;
    const int64_t scouts = queues ? std::max<int64_t>(r.has_col ? 1024 : 512, (r.n * SL + 1023) / 1024)
                           : r.one_group ? 0
                           : r.has_col ? (room > 0 ? std::max(SL, std::min<int64_t>(512, r.n * avg / 160)) : 0)
                           : room >= 64 ? std::max<int64_t>(1, std::min<int64_t>(room, r.n / 16))
                           : words == 2 ? 256
                                        : 0;
    const int64_t slices = scouts / SL;
    const int64_t looked = scouts ? (r.n + slices - 1) / slices : 0;   // rows for each of them
    const int64_t groups = (r.n + teams - 1) / teams;                  // workgroups of the others, per slab
    // element numbers in 32 bits when the array they walk is known to be small enough
    const bool small = r.bounded && r.elements < (int64_t(1) << 29);
    const ElemSize esz = small && isz == ElemSize::I64 ? ElemSize::I32 : isz;
    const Type ety = Type::scalar(esz);
    auto eint = [&](int64_t v) { return mk_int(v, esz); };
    auto narrow = [&](const E& e) { return e->ty.sz == esz ? e : mk_convert(e, esz); };
    auto widen = [&](const E& e) { return e->ty.sz == isz ? e : mk_convert(e, isz); };

    const Name reg = gen.fresh(r.acc->k == Expr::Var ? r.acc->name.s + "_part" : "part");
    const Type sty = Type::scalar(r.acc->ty.sz);
    auto part = [&](const E& c) {
      auto e = std::make_shared<Expr>();
      e->k = Expr::RegElem;
      e->ty = sty;
      e->name = reg;
      e->args = {c};
      return E(e);
    };
    // for (c = 0; c < K; ++c) unrolled around the statements that f makes for slot c
    auto per_slot = [&](std::function<Stmts(const E&)> f) {
      Name c = gen.fresh("c");
      auto loop = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(
          mk_for(c, iint(0), iint(K), 1, f(mk_var(c, ity)), LoopPar())));
      loop->unroll = true;
      if (moved) loop->iv = 1;   // (rows that start at any element)
      return S(loop);
    };
    auto to_end = [&](const E& first) { return moved ? mk_binop(BinOp::Min, first, iint(r.cols - V), ity) : first; };
    // the column of slot c of lane l, counted from the start of the slab
    const Name slab = SL > 1 ? gen.fresh("slab") : Name();
    E sv = mk_var(slab, ity);
    auto slab_column = [&](const E& c, const E& l) {
      E chunk = mk_binop(BinOp::FloorDiv, c, iint(V), ity), v = mk_binop(BinOp::Rem, c, iint(V), ity);
      E base = chunks == 1 ? l : add(mk_binop(BinOp::Mul, chunk, iint(L), ity), l);
      return V == 1 ? base : add(mk_binop(BinOp::Mul, base, iint(V), ity), v);
    };
    // the column itself; past the slab's last vector of columns that vector again
    auto column = [&](const E& c, const E& l) {
      E chunk = mk_binop(BinOp::FloorDiv, c, iint(V), ity), v = mk_binop(BinOp::Rem, c, iint(V), ity);
      E base = chunks == 1 ? l : add(mk_binop(BinOp::Mul, chunk, iint(L), ity), l);
      if (L * chunks != slots) base = mk_binop(BinOp::Min, base, iint(slots - 1), ity);
      if (SL > 1) base = add(mk_binop(BinOp::Mul, sv, iint(slots), ity), base);
      if (slots * SL != all_slots) base = mk_binop(BinOp::Min, base, iint(all_slots - 1), ity);
      return V == 1 ? base : add(to_end(mk_binop(BinOp::Mul, base, iint(V), ity)), v);
    };
    // is column `at` of the slab (a number below `upto`) one, and one of the array
    auto in_slab = [&](const E& at, int64_t upto) {
      E c;
      if (upto > wide) c = mk_binop(BinOp::Lt, at, iint(wide), bty);
      if (wide * SL != r.cols) {
        E whole = mk_binop(BinOp::Lt, SL == 1 ? at : add(mk_binop(BinOp::Mul, sv, iint(wide), ity), at), iint(r.cols), bty);
        c = c ? mk_binop(BinOp::And, c, whole, bty) : whole;
      }
      return c;
    };
    // statements that add the elements first, first + stride, ... of the row to the lane's sums
    // (staged: loads of the elements that stand in LDS, from element `lo` on)
    struct Staged { E load; Name lds; };
    auto sums_from_zero = [&](Stmts& out) {
      out.push_back([&] {
        auto d = std::make_shared<Stmt>();
        d->k = Stmt::RegDecl;
        d->id = reg;
        d->ty = sty;
        d->iv = K;
        return S(d);
      }());
      out.push_back(per_slot([&](const E& c) { return Stmts{mk_assign(part(c), mk_float(0.0, sty.sz))}; }));
    };
    auto walk = [&](Stmts& out, const E& lo, const E& hi, const E& first, int64_t stride, const E& l, int64_t U, const std::vector<Staged>& staged = {}) {
      Name b = gen.fresh(r.loop->id.s + "_b"), at = gen.fresh(r.loop->id.s + "_at");
      E bv = mk_var(b, ety), iv = mk_var(r.loop->id, ety), atv = mk_var(at, ety);
      Stmts batch;
      batch.push_back(mk_def(at, ety, mk_binop(BinOp::Min, iv, mk_binop(BinOp::Sub, hi, eint(1), ety), ety), r.loop->i));
      std::map<Name, E> to_clamped{{r.loop->id, widen(atv)}};
      // Loaded values that select other elements get a name, which lets them take part in 32-bit address arithmetic.  A
      // name is evaluated in front of the term whatever the term's tests say, so operands that a selection or a
      // short-circuit operator may skip make none (`x[perm[c]] if c >= 0 else 0`: c may be anything where it is not used).
      std::vector<std::pair<E, Name>> named;
      auto bind = [&](const E& e0, Stmts& to) {
        E e = rewrite_expr(e0, [&](const E& x) -> E {
          for (auto& st : staged)
            if (expr_eq(st.load, x)) return mk_index(mk_var(st.lds, Type::pointer(x->ty.sz, Mem::LDS)), widen(mk_binop(BinOp::Sub, atv, lo, ety)), x->ty);
          return x;
        });
        e = subst_vars(e, to_clamped);
        std::function<E(const E&, bool, bool)> go = [&](const E& x, bool inside, bool always) -> E {
          if (!x) return x;
          size_t q = 0;
          E y = map_children(x, [&](const E& ch) { return go(ch, inside || x->k == Expr::Index, always && !may_skip(x, q++)); });
          if (!(inside && y->k == Expr::Index && is_int(y->ty.sz))) return y;
          for (auto& nv : named) if (expr_eq(nv.first, y)) return mk_var(nv.second, y->ty);
          if (!always) return y;
          Name nm = gen.fresh("sel");
          named.push_back({y, nm});
          to.push_back(mk_def(nm, y->ty, y, r.loop->i));
          return mk_var(nm, y->ty);
        };
        return go(e, false, true);
      };
      auto summand = [&](const E& c) {
        Stmts ss;
        named.clear();
        if (r.has_col) {
          ss.push_back(mk_def(r.col, ity, fold_expr(column(c, l)), r.loop->i));
        }
        for (auto& d : r.defs) { E e = bind(d->expr, ss); ss.push_back(mk_def(d->id, d->ty, e, d->i)); }
        Name tv = gen.fresh("term");
        E te = bind(r.term, ss);
        ss.push_back(mk_def(tv, sty, te, r.loop->i));
        E masked = mk_ifexpr(mk_binop(BinOp::Lt, iv, hi, bty), mk_var(tv, sty), mk_float(0.0, sty.sz), sty);
        ss.push_back(mk_assign(part(c), mk_binop(BinOp::Add, part(c), masked, sty), r.loop->i));
        return ss;
      };
      batch.push_back(per_slot(summand));
      auto inner = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(
          mk_for(r.loop->id, bv, mk_binop(BinOp::Add, bv, eint(U * stride), ety), stride, batch, LoopPar(), r.loop->i)));
      inner->unroll = true;
      out.push_back(mk_for(b, mk_binop(BinOp::Add, lo, first, ety), hi, U * stride, {S(inner)}, LoopPar(), r.loop->i));
    };
    auto team_sum = [&](const std::string& fn) {
      return per_slot([&](const E& c) {
        auto call = std::make_shared<Expr>();
        call->k = Expr::Call;
        call->ty = sty;
        call->sval = fn;
        call->args = {part(c)};
        return Stmts{mk_assign(part(c), call)};
      });
    };
    // what is done with a finished sum
    auto finish = [&](const E& sum) {
      Stmts ss;
      E whole = r.start->k == Expr::Float && r.start->fv == 0.0 ? sum : mk_binop(BinOp::Add, r.start, sum, sty);
      if (r.acc->k == Expr::Index) ss.push_back(mk_assign(r.acc, whole, r.loop->i));
      else ss.push_back(mk_def(r.acc->name, sty, whole, r.loop->i));
      ss.insert(ss.end(), r.post.begin(), r.post.end());
      return ss;
    };
    auto finish_slots = [&](const E& l) {
      if (!r.has_col) return finish(part(iint(0)));
      return Stmts{per_slot([&](const E& c) {
        // (lanes and slots past the slab's last column, or past the array's, store nothing)
        // (of vectors that may be moved the first column tells)
        auto of_row = [&](const E& at) { return SL == 1 ? at : add(mk_binop(BinOp::Mul, sv, iint(wide), ity), at); };
        const E v = mk_binop(BinOp::Rem, c, iint(V), ity), own = slab_column(c, l), head = moved ? slab_column(mk_binop(BinOp::Sub, c, v, ity), l) : own;
        Stmts f{mk_def(r.col, ity, fold_expr(moved ? add(to_end(of_row(head)), v) : of_row(own)), r.loop->i)};
        Stmts g = finish(part(c));
        E some = in_slab(fold_expr(head), L * K);
        if (some && moved) {
          f.insert(f.end(), g.begin(), g.end());
          return Stmts{mk_if(some, f, {})};
        }
        if (!some) { f.insert(f.end(), g.begin(), g.end()); return f; }
        if (SL == 1) { f.push_back(mk_if(mk_binop(BinOp::Lt, mk_var(r.col, ity), iint(r.cols), bty), g, {})); return f; }
        f.insert(f.end(), g.begin(), g.end());
        return Stmts{mk_if(some, f, {})};
      })};
    };
    auto limits = [&](Stmts& ss, E* lo, E* hi) {
      Name lw = gen.fresh("lo"), hw = gen.fresh("hi");
      // (`rows[row] .. rows[row + 1]` in the plain form of an index, whose neighbours the device compiler joins to one load: with
      // 32-bit offsets two loads of eight bytes, 52.0 us for SpMV with 100 000 rows of 50, 50.4 so, 50.0 unchecked)
      std::map<Name, E> plain;
      if (adjacent(r.loop->lo, r.loop->hi, r.row)) plain[r.row] = mk_raw(r.row.str(), ity);
      ss.push_back(mk_def(lw, ity, subst_vars(r.loop->lo, plain), r.loop->i));
      ss.push_back(mk_def(hw, ity, subst_vars(r.loop->hi, plain), r.loop->i));
      *lo = mk_var(lw, ity);
      *hi = mk_var(hw, ity);
    };
    auto bounds = [&](Stmts& ss, E* lo, E* hi) {
      for (auto& st : r.pre) ss.push_back(st);
      // (the bounds of a row without elements may be anything, a marker like 2^63 - 1 and 0: what is cut to 32 bits of them, or
      // passes the largest integer when a lane's place is added, must not become a row)
      Name any = gen.fresh("any"), ln = gen.fresh("first"), hn = gen.fresh("end");
      E l, h, some = mk_var(any, bty);
      limits(ss, &l, &h);
      ss.push_back(mk_def(any, bty, mk_binop(BinOp::Lt, l, h, bty), r.loop->i));
      ss.push_back(mk_def(ln, ety, narrow(mk_ifexpr(some, l, iint(0), ity)), r.loop->i));
      ss.push_back(mk_def(hn, ety, narrow(mk_ifexpr(some, h, iint(0), ity)), r.loop->i));
      *lo = mk_var(ln, ety);
      *hi = mk_var(hn, ety);
    };

    Name queue = gen.fresh("long_rows"), count = gen.fresh("long_count");
    Stmts top;
    {
      auto d = std::make_shared<Stmt>();
      d->k = Stmt::LdsDecl;
      d->id = queue;
      d->ty = Type::scalar(ElemSize::I32);
      d->iv = std::max(teams, looked);
      top.push_back(d);
      auto e = std::make_shared<Stmt>(*d);
      e->id = count;
      e->iv = 1;
      top.push_back(e);
    }
    top.push_back(mk_rawstmt("if (threadIdx.x == 0) " + count.str() + "[0] = 0;"));
    top.push_back(mk_sync());

    // every team its row
    Name lane = gen.fresh(r.row.s + "_lane"), q = gen.fresh("g");
    E lv = mk_var(lane, ity), qv = mk_var(q, ity);
    {
      Stmts body;
      E team = mk_binop(BinOp::FloorDiv, lv, iint(T), ity);
      E behind = lv;
      if (scouts && SL == 1) team = mk_binop(BinOp::Max, mk_binop(BinOp::Sub, team, iint(scouts * teams), ity), iint(0), ity);   // (known not to be negative)
      if (SL > 1) {
        if (scouts) {
          Name at = gen.fresh("behind");
          behind = mk_var(at, ity);
          body.push_back(mk_def(at, ity, mk_binop(BinOp::Max, mk_binop(BinOp::Sub, lv, iint(scouts * tpb), ity), iint(0), ity), r.loop->i));
        }
        // (every SL-th workgroup is one of the same slab)
        team = mk_binop(BinOp::FloorDiv, add(mk_binop(BinOp::Mul, mk_binop(BinOp::FloorDiv, behind, iint(SL * tpb), ity), iint(tpb), ity), mk_binop(BinOp::Rem, behind, iint(tpb), ity)), iint(T), ity);
      }
      body.push_back(mk_def(r.row, ity, team, r.loop->i));
      body.push_back(mk_def(q, ity, mk_binop(BinOp::Rem, lv, iint(T), ity), r.loop->i));
      if (SL > 1) body.push_back(mk_def(slab, ity, mk_binop(BinOp::Rem, mk_binop(BinOp::FloorDiv, behind, iint(tpb), ity), iint(SL), ity), r.loop->i));
      const size_t placed = body.size();
      E lo, hi;
      bounds(body, &lo, &hi);
      Stmts own;
      E l = L == 1 ? iint(0) : mk_binop(BinOp::Rem, qv, iint(L), ity), sub = L == 1 ? qv : mk_binop(BinOp::FloorDiv, qv, iint(L), ity);
      if (r.has_col && L > 1) {
        Name ln = gen.fresh("l");
        own.push_back(mk_def(ln, ity, l));
        l = mk_var(ln, ity);
      }
      sums_from_zero(own);
      walk(own, lo, hi, narrow(sub), P, l, U);
      if (P > 1) own.push_back(team_sum(L == 1 && P == 8 ? "parpy_sum8" : "parpy_team_sum<" + std::to_string(L) + ", " + std::to_string(T) + ">"));
      Stmts f = finish_slots(l);
      if (P > 1) own.push_back(mk_if(mk_binop(BinOp::Lt, qv, iint(L), bty), f, {}));
      else own.insert(own.end(), f.begin(), f.end());
      const S enqueue = mk_rawstmt(queue.str() + "[atomicAdd(&" + count.str() + "[0], 1)] = (int)" + r.row.str() + ";");
      Stmts defer;
      if (!scouts) defer = {mk_if(mk_binop(BinOp::Eq, qv, iint(0), bty), {enqueue}, {})};
      body.push_back(mk_if(mk_binop(BinOp::Leq, mk_binop(BinOp::Sub, hi, lo, ety), eint(longest), bty), own, defer));
      if (SL > 1 && groups * teams != r.n) {
        // (the last workgroup of every slab may hold teams without a row)
        Stmts rest(body.begin() + placed, body.end());
        body.resize(placed);
        body.push_back(mk_if(mk_binop(BinOp::Lt, mk_var(r.row, ity), iint(r.n), bty), rest, {}));
      }
      auto nr = clone(k.body[0]);
      nr->id = lane;
      const int64_t lanes = SL == 1 ? r.n * T + scouts * tpb : (groups * SL + scouts) * tpb;
      nr->hi = iint(lanes);
      nr->body = body;
      if (scouts) {
        Name at = gen.fresh(r.row.s + "_at"), slice = gen.fresh("slice");
        const E first = mk_binop(BinOp::Mul, mk_var(slice, ity), iint(looked), ity);
        Stmts look{mk_def(r.row, ity, mk_var(at, ity), r.loop->i)};
        for (auto& st : r.pre) look.push_back(st);
        E a, b;
        limits(look, &a, &b);
        const E more = mk_binop(BinOp::Gt, mk_binop(BinOp::Sub, b, a, ity), iint(longest), bty);
        look.push_back(mk_if(mk_binop(BinOp::And, mk_binop(BinOp::Lt, a, b, bty), more, bty), {enqueue}, {}));
        nr->body = {mk_if(mk_binop(BinOp::Lt, lv, iint(scouts * tpb), bty),
                          {mk_def(slice, ity, mk_binop(BinOp::FloorDiv, lv, iint(SL * tpb), ity)),
                           mk_for(at, add(first, mk_binop(BinOp::Rem, lv, iint(tpb), ity)), mk_binop(BinOp::Min, add(first, iint(looked)), iint(r.n), ity), tpb, look, LoopPar(), r.loop->i)},
                          body)};
      }
      nr->els.clear();
      nr->map = GpuMap();
      nr->map.k = GpuMap::ThreadBlock;
      nr->map.tpb = tpb;
      nr->map.n = (lanes + WAVE_SIZE - 1) / WAVE_SIZE * WAVE_SIZE;
      top.push_back(nr);
    }
    if (scouts) top.push_back(mk_rawstmt("if (blockIdx.x >= " + std::to_string(scouts) + ") return;"));
    top.push_back(mk_sync());

    // long rows, one after the other, by all threads of the workgroup
    {
      Name h = gen.fresh("h"), tid = gen.fresh("tid");
      E tv = mk_var(tid, ity);
      auto tx = std::make_shared<Expr>();
      tx->k = Expr::ThreadIdx;
      tx->ty = ity;
      tx->iv = 0;
      Stmts body;
      body.push_back(mk_def(r.row, ity, mk_raw("((int64_t)" + queue.str() + "[" + h.str() + "])", ity), r.loop->i));
      body.push_back(mk_def(tid, ity, tx));
      if (SL > 1) {
        auto bx = std::make_shared<Expr>(*tx);
        bx->k = Expr::BlockIdx;
        body.push_back(mk_def(slab, ity, mk_binop(BinOp::Rem, E(bx), iint(SL), ity)));
      }
      E lo, hi;
      bounds(body, &lo, &hi);
      E l = L == 1 ? iint(0) : mk_binop(BinOp::Rem, tv, iint(L), ity), sub = L == 1 ? tv : mk_binop(BinOp::FloorDiv, tv, iint(L), ity);
      sums_from_zero(body);
      // An element costs two dependent round trips, its column and what the column selects, and the longest row makes them one
      // batch after the other.  Where lanes along the columns leave few elements to a batch, the workgroup loads the columns
      // and values of as many elements as it has threads at once, those of the next piece while this one is summed, and the
      // batches wait for the selected rows alone.  The order of the sum stays.  9529 rows of 41 on average times 101 columns
      // 40.7 -> 31.8 us, 1021 of 35 times 256 23.2 -> 20.3, 20 000 of 24 times 128 35.4 -> 34.5; twice the elements in a batch
      // instead of that or beside it are registers: 75 and 46 us for the first and the last.
      std::vector<Staged> staged;
      int64_t bytes = 0;
      if (r.has_col && U <= L)
        for (auto& e : element_loads(k, r)) {
          staged.push_back({e, gen.fresh("staged")});
          bytes += elem_bytes(e->ty.sz);
        }
      if (!r.has_col) {
        // Single sums: eight in flight for each thread while the row fills them (10 468 rows of 185 on average, the longest of 18 900,
        // doubles 21.1 -> 19.9 us, floats 18.2 -> 16.4, 30 000 of 100 floats 22.0 -> 20.0), then four.  Sixteen take more registers
        // than leave the other rows their wavefronts.
        const Name full = gen.fresh("full");
        const E fv = mk_var(full, ety), piece = eint(8 * tpb);
        auto minus = [&](const E& a, const E& b) { return mk_binop(BinOp::Sub, a, b, ety); };
        body.push_back(mk_def(full, ety, mk_binop(BinOp::Add, lo, mk_binop(BinOp::Mul, mk_binop(BinOp::FloorDiv, minus(hi, lo), piece, ety), piece, ety), ety)));
        walk(body, lo, fv, narrow(sub), tpb, l, 8);
        walk(body, fv, hi, narrow(sub), tpb, l, 4);
      } else if (staged.empty() || bytes > 16) {
        walk(body, lo, hi, narrow(sub), tpb / L, l, U);
      } else {
        Name from = gen.fresh("from"), upto = gen.fresh("upto");
        E fv = mk_var(from, ety), uv = mk_var(upto, ety);
        Stmts put;
        Stmts fetch_next;
        for (auto& st : staged) {
          auto d = std::make_shared<Stmt>();
          d->k = Stmt::LdsDecl;
          d->id = st.lds;
          d->ty = st.load->ty;
          d->iv = tpb;
          top.push_back(d);
          k.lds_bytes += tpb * elem_bytes(st.load->ty.sz);
          Name next = gen.fresh(st.lds.s + "_next");
          auto load_at = [&](const E& start, int64_t ahead) {
            // (the last element where the thread has none: loads without a test, which the walk does not wait for)
            E i = mk_binop(BinOp::Min, mk_binop(BinOp::Add, narrow(tv), eint(ahead), ety), mk_binop(BinOp::Sub, mk_binop(BinOp::Sub, hi, eint(1), ety), start, ety), ety);
            std::map<Name, E> at{{r.loop->id, widen(mk_binop(BinOp::Add, start, i, ety))}};
            return subst_vars(st.load, at);
          };
          body.push_back(mk_def(next, st.load->ty, load_at(lo, 0)));
          fetch_next.push_back(mk_assign(mk_var(next, st.load->ty), load_at(fv, tpb)));
          put.push_back(mk_assign(mk_index(mk_var(st.lds, Type::pointer(st.load->ty.sz, Mem::LDS)), tv, st.load->ty), mk_var(next, st.load->ty)));
        }
        Stmts piece{mk_def(upto, ety, mk_binop(BinOp::Min, mk_binop(BinOp::Add, fv, eint(tpb), ety), hi, ety)), mk_sync()};
        piece.insert(piece.end(), put.begin(), put.end());
        piece.push_back(mk_sync());
        piece.insert(piece.end(), fetch_next.begin(), fetch_next.end());
        walk(piece, fv, uv, narrow(sub), tpb / L, l, U, staged);
        body.push_back(mk_for(from, lo, hi, tpb, piece, LoopPar(), r.loop->i));
      }
      if (!r.has_col) {
        Name w = gen.fresh("whole");
        body.push_back(mk_def(w, sty, part(iint(0))));
        auto red = std::make_shared<Stmt>();
        red->k = Stmt::WaveReduce;
        red->id = w;
        red->ty = sty;
        red->bop = BinOp::Add;
        red->iv = tpb;
        red->unroll = true;   // the slots are used again for the next row
        body.push_back(red);
        body.push_back(mk_if(mk_binop(BinOp::Eq, tv, iint(0), bty), finish(mk_var(w, sty)), {}));
      } else {
        if (L < WAVE_SIZE) body.push_back(team_sum("parpy_team_sum<" + std::to_string(L) + ", " + std::to_string(WAVE_SIZE) + ">"));
        Name shared = gen.fresh("long_sums");
        auto d = std::make_shared<Stmt>();
        d->k = Stmt::LdsDecl;
        d->id = shared;
        d->ty = sty;
        d->iv = waves * L * K;
        top.push_back(d);
        E base = mk_var(shared, Type::pointer(sty.sz, Mem::LDS));
        E wave = mk_binop(BinOp::FloorDiv, tv, iint(WAVE_SIZE), ity);
        Stmts put{per_slot([&](const E& c) {
          E at = add(mk_binop(BinOp::Mul, wave, iint(L * K), ity), slab_column(c, l));
          return Stmts{mk_assign(mk_index(base, fold_expr(at), sty), part(c))};
        })};
        body.push_back(mk_if(mk_binop(BinOp::Lt, mk_binop(BinOp::Rem, tv, iint(WAVE_SIZE), ity), iint(L), bty), put, {}));
        body.push_back(mk_sync());
        Name s = gen.fresh("whole"), w = gen.fresh("w");
        Stmts sum{mk_def(r.col, ity, SL == 1 ? tv : add(mk_binop(BinOp::Mul, sv, iint(wide), ity), tv)), mk_def(s, sty, mk_float(0.0, sty.sz))};
        // (columns of the last vector lie where it would without having been moved)
        E place = tv;
        if (moved) {
          Name at = gen.fresh("place");
          sum.push_back(mk_def(at, ity, mk_ifexpr(mk_binop(BinOp::Lt, mk_var(r.col, ity), iint((all_slots - 1) * V), bty), tv, add(tv, iint(all_slots * V - r.cols)), ity)));
          place = mk_var(at, ity);
        }
        auto over = std::const_pointer_cast<Stmt>(std::static_pointer_cast<const Stmt>(mk_for(
            w, iint(0), iint(waves), 1,
            {mk_assign(mk_var(s, sty), mk_binop(BinOp::Add, mk_var(s, sty),
                                                mk_index(base, add(mk_binop(BinOp::Mul, mk_var(w, ity), iint(L * K), ity), place), sty), sty))},
            LoopPar())));
        over->unroll = true;
        sum.push_back(over);
        Stmts f = finish(mk_var(s, sty));
        sum.insert(sum.end(), f.begin(), f.end());
        E some = in_slab(tv, tpb);
        if (some) body.push_back(mk_if(some, sum, {}));
        else body.insert(body.end(), sum.begin(), sum.end());
        body.push_back(mk_sync());
        k.lds_bytes += waves * L * K * elem_bytes(sty.sz);
      }
      top.push_back(mk_for(h, iint(0), mk_raw("((int64_t)" + count.str() + "[0])", ity), 1, body, LoopPar()));
    }
    k.lds_bytes += (std::max(teams, looked) + 1) * 4;
    k.body = top;
    k.block = Dim3{tpb, 1, 1};
    k.grid = Dim3{groups * SL + scouts, 1, 1};
    launch->grid = k.grid;
    launch->block = k.block;
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

}  // namespace

void ragged_sum(Program& p, const Options& opts, NameGen& gen) { RaggedSum(p, opts, gen).run(); }

}  // namespace hipopt
}  // namespace parpy
