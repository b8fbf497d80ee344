// Fused RK stage on the source lists (list.hpp): the lists of the current
// grid, the plan of a stage's sweeps, and the stage itself.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <climits>
#include <map>

#include "context.hpp"
#include "list.hpp"

namespace adg {

namespace {

template <class T>
void upload(DevBuf<T>& b, const std::vector<T>& h, hipStream_t s) {
  b.ensure(std::max<size_t>(h.size(), 1));
  if (!h.empty()) hip_check(hipMemcpyAsync(b.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s), "upload");
}

int prod_of(const int* sz, int D) {
  int p = 1;
  for (int d = 0; d < D; ++d) p *= sz[d];
  return p;
}

}  // namespace

// The sweeps of a stage, in launch order, as device descriptors.  They hold
// buffer addresses but nothing of the grid (its size is a kernel argument and
// the buffers keep room for more elements), so a plan outlives grid changes.
struct Context::ListPhase {
  int first = 0, n = 0, R = 0;
  double bytes = 0.;  // algorithmic bytes per element
};
using ListKey = std::array<uintptr_t, 16 + 6 * kMaxDim>;
struct Context::ListPlan {
  int64_t serial = 0;  // of this build (Context::plan_serial)
  ListKey key{};  // the addresses that the terms hold and what they were chosen by
  DevBuf<ListTerm> terms;
  DevBuf<int2> rofs;
  using Phase = ListPhase;
  std::vector<Phase> up, rhs;
  Phase up_final, rhs_final;
  // the volume (0) and flux (1) operators: all directions at once, or (split) one
  // after another in the same phase buffers
  struct Op {
    std::vector<Phase> phases;
    Phase last;
  };
  std::vector<Op> ops[2];
  bool split = false;
  int pen = 0;  // the D penalty sweeps (after rhs_final's terms in the stage's plan; not in eval_up's)
};

int64_t Context::list_stage_serial() const {
  return list_plans[LIST_STAGE] ? list_plans[LIST_STAGE]->serial : 0;
}

bool Context::list_stage_fits() const {
  if (E() == 0) return false;
  // the kernels use 32-bit work items and byte offsets into the lists, one
  // component of a sweep's input and the tables, 24-bit products of element
  // and slot numbers, and count a target's entries in 16 bits
  const int mx = std::max(k, m) + 1;
  int64_t T = 1;
  for (int d = 0; d < D; ++d) T *= mx;
  const int64_t lim = int64_t{1} << 32, ns = int64_t{1} << nmax;
  // the last sweeps keep every term value of an element in LDS (all but k = 3
  // in four dimensions fit: 68 terms of 256 values)
  const int64_t nord = D == 1 ? 1 : int64_t{1} << (D - 1);
  if ((2 * D * nord + D) * K > kFinalValues || nord * P > kFinalValues) return false;
  return E() < (1 << 24) && E() * T * 8 < lim && E() * (4 * nmax + 4) * 8 < lim && ns * ns * mx * mx * 8 < lim;
}

// Tables whose blocks decide which pairs a list holds.
void Context::list_nonzero_tables() {
  const int ns = 1 << nmax, kb = (k + 1) * (m + 1);
  for (int q = LIST_PT; q <= LIST_FLX; ++q) nz_tab[q].ensure(static_cast<size_t>(ns) * ((ns + 31) / 32));
  list_nonzero(nz_tab[LIST_VOL].p, nullptr, ns, 1, true, true, stream);
  list_nonzero(nz_tab[LIST_PT].p, t_pt.p, ns, kb, true, true, stream);
  list_nonzero(nz_tab[LIST_FLX].p, t_la_flx.p, ns, kb, false, true, stream);
  list_nonzero(nz_tab[LIST_FLX].p, t_aa[4].p, ns, (k + 1) * (k + 1), false, false, stream);
  nz_interp = interp;
}

// Room for the entries of a list of this kind.  An element of level l has at most
// l + 1 related cells at levels up to its own in a nested relation, 2 l + 1 in
// one that counts touching cells, and as many pairs (less itself) with it as the
// finer one are in the L parts: 2 l + 1 and 4 l + 1 entries an element.
int64_t Context::list_room(int kind, int lmax) const {
  return E() * (kind == LIST_FLX || kind == LIST_LIN ? 4 * lmax + 4 : 2 * lmax + 1);
}

int Context::deepest_level(int d) const {
  int lmax = 0;
  for (int i = 0; i < B(); ++i) lmax = std::max(lmax, inst_lmax[static_cast<size_t>(i) * D + d]);
  return lmax;
}

bool Context::lists_current(int kind0, int nkind) const {
  bool ok = true;
  for (int q = kind0; q < kind0 + nkind; ++q)
    ok = ok && list_version[q] == grid_version && list_level_cap[q] == lsum_cap && list_interp[q] == interp;
  return ok;
}

void Context::ensure_lists(int kind0, int nkind) {
  if (lists_current(kind0, nkind)) return;
  not_recording("source lists");
  HostTimer timer(*this, HOST_UPLOAD);
  if (kind0 != LIST_LIN && nz_interp != interp) list_nonzero_tables();
  ListBuildArgs a{};
  for (int d = 0; d < D; ++d) {
    a.slot[d] = g_slot[d].p;
    a.fbase[d] = g_fbase[d].p;
    a.fmaxl[d] = g_fmaxl[d].p;
    a.fmap[d] = g_fmap[d].p;
    a.fbits[d] = g_fbits[d].p;
  }
  a.lsum = g_lsum.p; a.inst = g_inst.p; a.err = err_flag.p;
  a.E = E(); a.D = D; a.ns = 1 << nmax; a.level_cap = lsum_cap;
  for (int q = 0; q < LIST_KINDS; ++q) a.nz[q] = nz_tab[q].p;
  l_total.ensure(LIST_KINDS * kMaxDim);
  a.total = l_total.p;
  int deepest = 0;
  for (int d = 0; d < D; ++d) {
    const int lmax = deepest_level(d);
    deepest = std::max(deepest, lmax);
    for (int q = kind0; q < kind0 + nkind; ++q) {
      const int l = q * D + d;
      l_meta[l].ensure(static_cast<size_t>(E()));
      l_ent[l].ensure(static_cast<size_t>(list_room(q, lmax)));
      a.meta[l] = l_meta[l].p;
      a.ent[l] = l_ent[l].p;
      a.cap[l] = static_cast<int64_t>(l_ent[l].cap);
    }
  }
  list_fill_totals(l_total.p + kind0 * D, nkind * D, stream);
  list_build(a, kind0, nkind, deepest, stream);
  for (int q = kind0; q < kind0 + nkind; ++q) {
    list_version[q] = grid_version;
    list_level_cap[q] = lsum_cap;
    list_interp[q] = interp;
  }
}

// Terms of a plan, with the places in the phase buffers still relative.
struct Context::ListTerms {
  std::vector<ListTerm> terms;
  std::vector<int2> rofs;
  size_t values = 0;                              // of the phase buffers, per element
  std::vector<std::pair<size_t, size_t>> outs;    // (term, first value of its output buffer)
  std::vector<std::pair<size_t, size_t>> ins;     // (term, first value of its input) where that is a phase buffer
  std::vector<size_t> rofs_of;                    // per term: first entry of its offsets
};

// form LIST_STAGE: volume and flux terms in one set of phases, in the storage
// of `precision`; the others: separate operators in FP64.
void Context::list_terms(ListForm form, ListPlan& pl, ListTerms& b) {
  const bool ops = form != LIST_STAGE, f32 = !ops && precision == 1;
  const bool same = ops ? form == LIST_OPS_SAME : same_flux;
  auto ptr = [](const void* q) { return reinterpret_cast<uintptr_t>(q); };
  const double* pen_coef = inst_alpha.empty() ? nullptr : d_pen_coef.p;
  std::vector<std::vector<int>> lus;
  const std::vector<std::vector<int>> dims = transform_orders(D, lus);
  const int nord = static_cast<int>(dims.size());
  const double w = f32 ? 4.0 : 8.0;
  std::vector<ListTerm>& flat = b.terms;
  std::vector<int2>& rofs = b.rofs;
  std::map<std::vector<int>, size_t> rofs_at;
  size_t tmp_used = 0;
  // per rest index (row-major over the dimensions other than dd): offsets in
  // tensors of input sizes sin with the given strides
  auto rest_offsets = [&](const int* sin, const int* stin, const int* stout, int dd) {
    std::vector<int> id(sin, sin + D);
    id.insert(id.end(), stin, stin + D);
    id.insert(id.end(), stout, stout + D);
    id.push_back(dd);
    auto it = rofs_at.find(id);
    if (it != rofs_at.end()) return it->second;
    const size_t at = rofs.size();
    rofs_at[id] = at;
    int R = 1;
    for (int d = 0; d < D; ++d) R *= d == dd ? 1 : sin[d];
    for (int r = 0; r < R; ++r) {
      int rem = r, bi = 0, bo = 0;
      for (int d = D - 1; d >= 0; --d) {
        if (d == dd) continue;
        bi += rem % sin[d] * stin[d];
        bo += rem % sin[d] * stout[d];
        rem /= sin[d];
      }
      rofs.push_back(int2{bi, bo});
    }
    return at;
  };
  // strides of a tensor of sizes sz: row-major, with dimension `inner` (if not
  // -1) moved to the innermost place
  auto strides = [&](const int* sz, int inner, int* st) {
    int n = 1;
    if (inner >= 0) {
      st[inner] = 1;
      n = sz[inner];
    }
    for (int d = D - 1; d >= 0; --d) {
      if (d == inner) continue;
      st[d] = n;
      n *= sz[d];
    }
  };
  // a term over lists of `kind`; sizes and strides before and after the sweep of dd
  auto make_term = [&](int kind, const double* in, const float* in32, int comp, const int* sin, const int* stin,
                       const int* sout, const int* stout, int dd, const double* M, int lu, double coef, bool split) {
    ListTerm t{};
    t.in = in; t.in32 = in32; t.M = M; t.ns = 1 << nmax; t.lu = lu; t.coef = coef;
    if (split) {
      const SplitTable& sp = split_table(M, (static_cast<size_t>(1) << (2 * nmax)) * sin[dd] * sout[dd]);
      t.Mh = sp.hi.p;
      t.Ml = sp.lo.p;
    }
    t.meta = l_meta[kind * D + dd].p;
    t.ent = l_ent[kind * D + dd].p;
    t.comp = comp;
    t.comp_size = prod_of(sin, D);
    t.Tin = prod_of(sin, D);
    t.Tout = prod_of(sout, D);
    t.R = t.Tin / sin[dd];
    t.sdd = stin[dd];
    t.sod = stout[dd];
    b.rofs_of.push_back(rest_offsets(sin, stin, stout, dd));
    return t;
  };
  auto in_bytes = [&](const ListTerm& t, bool phase_in) { return (phase_in || t.in32 || !f32) ? w : 8.0; };
  // Chains of partial sums as a prefix tree (one node per distinct leading
  // sequence of sweeps; Context::fused_plan states why sharing them and
  // where the coefficient 1/2 is applied leaves every value unchanged).
  struct Chain {
    int kind[kMaxDim], comp, o;
    const double* in;
    const float* in32;
    const double* tab[kMaxDim];
    double coef;
  };
  auto build = [&](const std::vector<Chain>& chains, int pf1, int pt1, std::vector<ListPlan::Phase>& phases,
                   ListPlan::Phase& last) {
    auto prefix = [&](const Chain& c, int st) {
      std::vector<uintptr_t> id = {ptr(c.in), static_cast<uintptr_t>(c.comp)};
      for (int j = 0; j <= st; ++j) {
        const int dd = dims[c.o][j];
        id.insert(id.end(), {static_cast<uintptr_t>(dd), ptr(c.tab[dd]), static_cast<uintptr_t>(lus[c.o][j])});
      }
      return id;
    };
    std::map<std::vector<uintptr_t>, std::vector<double>> coefs;  // coefficients of the chains through a node
    for (const Chain& c : chains)
      for (int st = 0; st + 1 < D; ++st) {
        std::vector<double>& v = coefs[prefix(c, st)];
        if (std::find(v.begin(), v.end(), c.coef) == v.end()) v.push_back(c.coef);
      }
    // the dimension most of a node's continuations sweep next (the later one on
    // a tie): innermost in its output, so that they read their values as one run
    std::map<std::vector<uintptr_t>, std::vector<int>> nexts;
    for (const Chain& c : chains)
      for (int st = 0; st + 1 < D; ++st) {
        std::vector<int>& v = nexts[prefix(c, st)];
        v.resize(D, 0);
        ++v[dims[c.o][st + 1]];
      }
    struct Node { size_t at; bool applied; int st[kMaxDim]; };  // output of a node; the coefficient is in it
    std::map<std::vector<uintptr_t>, Node> nodes;
    tmp_used = 0;
    phases.clear();
    for (int st = 0; st < D; ++st) {
      ListPlan::Phase ph{static_cast<int>(flat.size()), 0, 0, 0.};
      for (const Chain& c : chains) {
        const std::vector<uintptr_t> id = prefix(c, st);
        if (st + 1 < D && nodes.count(id)) continue;
        int sin[kMaxDim], sout[kMaxDim];
        for (int d = 0; d < D; ++d) sin[d] = pf1;
        for (int j = 0; j < st; ++j) sin[dims[c.o][j]] = pt1;
        std::copy(sin, sin + D, sout);
        const int dd = dims[c.o][st];
        sout[dd] = pt1;
        const Node* before = st ? &nodes.at(prefix(c, st - 1)) : nullptr;
        const bool applied = before && before->applied;
        const bool here = !applied && (st + 1 == D || coefs[id].size() == 1);
        int stin[kMaxDim], inner = -1;
        if (before) std::copy(before->st, before->st + D, stin);
        else strides(sin, -1, stin);
        if (st + 1 < D) {
          const std::vector<int>& v = nexts[id];
          inner = D - 1;
          for (int d = D - 1; d >= 0; --d)
            if (v[d] > v[inner]) inner = d;
        }
        Node node{tmp_used, applied || here, {}};
        strides(sout, inner, node.st);
        ListTerm t = make_term(c.kind[dd], before ? nullptr : c.in, before ? nullptr : c.in32, before ? 0 : c.comp, sin,
                               stin, sout, node.st, dd, c.tab[dd], lus[c.o][st], here ? c.coef : 1.0, f32);
        if (before) b.ins.push_back({flat.size(), before->at});
        ph.bytes += in_bytes(t, before != nullptr) * t.Tin;
        if (st + 1 < D) {
          nodes[id] = node;
          b.outs.push_back({flat.size(), tmp_used});
          tmp_used += t.Tout;
          ph.bytes += w * t.Tout;
        }
        ph.R = t.R;
        ++ph.n;
        flat.push_back(t);
      }
      if (st + 1 < D) phases.push_back(ph);
      else last = ph;
    }
    b.values = std::max(b.values, tmp_used);
  };
  std::vector<Chain> chains;
  if (form == LIST_STAGE || form == LIST_UP) {
    for (int o = 0; o < nord; ++o) {
      Chain c{};
      c.o = o;
      c.coef = 1.0;
      for (int d = 0; d < D; ++d) { c.kind[d] = LIST_PT; c.tab[d] = t_pt.p; }
      chains.push_back(c);
    }
    build(chains, k + 1, m + 1, pl.up, pl.up_final);
    const int nc = ops ? 0 : (same ? 1 : D);
    pl.up_final.bytes += w * P * (1 + nc) + (is_varcoef(flux_kind) ? 8.0 * P * nc : 0.);
    chains.clear();
  }
  // in the reference order: volume terms for d = 0..D-1, then flux terms
  const bool rhs = form == LIST_STAGE || form == LIST_OPS || form == LIST_OPS_SAME;
  auto build_op = [&](int ft) {
    pl.ops[ft].emplace_back();
    build(chains, m + 1, k + 1, pl.ops[ft].back().phases, pl.ops[ft].back().last);
    chains.clear();
  };
  for (int ft = 0; ft < 2 && rhs; ++ft) {
    for (int d = 0; d < D; ++d) {
      for (int o = 0; o < nord; ++o) {
        Chain c{};
        c.o = o;
        c.comp = same ? 0 : d;
        c.in = fucoe.p;
        c.in32 = f32 ? fucoe32.p : nullptr;
        c.coef = ft ? 0.5 : 1.0;
        for (int dd = 0; dd < D; ++dd) {
          c.kind[dd] = dd == d && ft ? LIST_FLX : LIST_VOL;
          c.tab[dd] = dd == d ? (ft ? t_la_flx.p : t_la_uvx.p) : t_la_uv.p;
        }
        chains.push_back(c);
      }
      if (pl.split) build_op(ft);
    }
    if (ops && !pl.split) build_op(ft);
  }
  if (form == LIST_STAGE) {
    build(chains, m + 1, k + 1, pl.rhs, pl.rhs_final);
    pl.rhs_final.bytes += 8.0 * K * (1 + 3 + D);
  }
  if (form == LIST_UP) return;
  pl.pen = static_cast<int>(flat.size());
  // the LF penalty stays FP64 in every precision
  int ksz[kMaxDim];
  int kst[kMaxDim];
  for (int d = 0; d < D; ++d) ksz[d] = k + 1;
  strides(ksz, -1, kst);
  for (int d = 0; d < D; ++d) {
    flat.push_back(make_term(LIST_FLX, nullptr, nullptr, 0, ksz, kst, ksz, kst, d, t_aa[4].p, LU_FULL, 0., false));
    if (pen_coef) flat.back().coef_inst = pen_coef + static_cast<size_t>(d) * B();
  }
}

// Element places of the phase buffers that a grid of this size needs.
int64_t Context::list_places() const {
  return E() > list_ecap ? (E() + E() / 4 + 1023) / 1024 * 1024 : list_ecap;
}

Context::ListPlan& Context::get_list_plan(ListForm form, bool split) {
  if (list_places() > list_ecap) {
    not_recording("stage buffers");
    list_ecap = list_places();
    for (auto& q : list_plans) q.reset();
  }
  const bool ops = form != LIST_STAGE, f32 = !ops && precision == 1;
  if (!ops) u_next.ensure(static_cast<size_t>(E()) * K);
  auto ptr = [](const void* q) { return reinterpret_cast<uintptr_t>(q); };
  const double* pen_coef = inst_alpha.empty() ? nullptr : d_pen_coef.p;
  ListKey key{};
  size_t n = 0;
  auto add = [&](uintptr_t v) { key[n++] = v; };
  add(ptr(list_tmp.p));
  add(static_cast<uintptr_t>(interp));
  add(static_cast<uintptr_t>(split));
  if (!ops) {
    add(static_cast<uintptr_t>(f32));
    add(static_cast<uintptr_t>(same_flux));
    add(static_cast<uintptr_t>(is_varcoef(flux_kind)));
    add(ptr(fucoe32.p));
  }
  add(ptr(fucoe.p));
  if (form != LIST_UP) {
    add(ptr(pen_coef));
    add(pen_coef ? static_cast<uintptr_t>(B()) : 0);
  }
  for (int q = form == LIST_STAGE || form == LIST_UP ? LIST_PT : LIST_VOL; q <= (form == LIST_UP ? LIST_PT : LIST_FLX); ++q)
    for (int d = 0; d < D; ++d) {
      add(ptr(l_meta[q * D + d].p));
      add(ptr(l_ent[q * D + d].p));
    }
  std::shared_ptr<ListPlan>& list_plan = list_plans[form];
  if (list_plan && list_plan->key == key) return *list_plan;
  not_recording("stage plan");
  HostTimer timer(*this, HOST_PLAN);
  list_plan.reset(new ListPlan());
  ListPlan& pl = *list_plan;
  pl.serial = ++plan_serial;
  pl.split = split;
  ListTerms b;
  list_terms(form, pl, b);
  list_tmp.ensure(std::max<size_t>(b.values * list_ecap, 1));
  key[0] = ptr(list_tmp.p);
  upload(pl.rofs, b.rofs, stream);
  for (const auto& o : b.outs) b.terms[o.first].out = list_tmp.p + o.second * list_ecap;
  for (const auto& i : b.ins) {
    b.terms[i.first].in = list_tmp.p + i.second * list_ecap;
    if (f32) b.terms[i.first].in32 = reinterpret_cast<const float*>(b.terms[i.first].in);
  }
  for (size_t i = 0; i < b.terms.size(); ++i) b.terms[i].rofs = pl.rofs.p + b.rofs_of[i];
  upload(pl.terms, b.terms, stream);
  sync();  // the host vectors are gone after this call
  pl.key = key;
  return pl;
}

template <class T>
void Context::list_phases(const ListPlan& pl, const std::vector<ListPhase>& phases, int cat, int pf1, int pt1) {
  for (const ListPhase& ph : phases) {
    prof_begin(cat, ph.bytes * E());
    list_phase<T>(pf1, pt1, pl.terms.p + ph.first, ph.n, E(), ph.R, u.p, stream);
    prof_end();
  }
}

template <class T>
void Context::stage_list(const StageProblem& p, int scheme, int stage, double dt, bool first) {
  ListPlan& pl = get_list_plan(LIST_STAGE);
  constexpr bool f32 = sizeof(T) == 4;
  const int up_kind = interp == 1 ? -1 : p.flux_kind;
  const int ncomp = same_flux ? 1 : D;
  T* upp;
  T* fpp;
  if constexpr (f32) { upp = up32.p; fpp = fp32.p; }
  else { upp = up.p; fpp = fp.p; }
  const int64_t n = E();
  list_phases<T>(pl, pl.up, PROF_SWEEP, k + 1, m + 1);
  prof_begin(PROF_FLUX, pl.up_final.bytes * n);
  list_up_final<T>(k + 1, m + 1, pl.terms.p + pl.up_final.first, pl.up_final.n, n, P, u.p, upp, fpp, vcoef.p, up_kind,
                   p.flux_param, ncomp, stream);
  ++stage_launches;
  if (interp == 1) {
    flux_herm<T>(upp, fpp, p.flux_kind, T(p.flux_param), ncomp);
    ++stage_launches;
  }
  prof_end();
  if constexpr (f32) surplus_transform32(fp32.p, fucoe32.p, interA32.p, interB32.p, ncomp);
  else surplus_transform(fp.p, fucoe.p, interA.p, interB.p, ncomp);
  stage_launches += D + static_cast<int64_t>(pl.up.size() + pl.rhs.size());
  list_phases<T>(pl, pl.rhs, PROF_RHS_PHASE, m + 1, k + 1);
  prof_begin(PROF_RK, pl.rhs_final.bytes * n);
  list_rhs_final<T>(m + 1, k + 1, pl.terms.p + pl.rhs_final.first, pl.rhs_final.n, D, n, K,
                    list_rhs(false, scheme, stage, dt, first, p.alpha), stream);
  ++stage_launches;
  prof_end();
  std::swap(u.p, u_next.p);
  std::swap(u.cap, u_next.cap);
}

// Arguments of a last-sweep launch that ends in an RK stage.
ListRhs Context::list_rhs(bool add, int scheme, int stage, double dt, bool first, const double* alpha) const {
  ListRhs r{rhs.p, add, u.p, u_next.p, first ? u.p : tn.p, first ? tn.p : nullptr, scheme, stage, dt,
            use_inst_dt ? d_inst_dt.p : nullptr, err_flag.p, {}};
  for (int d = 0; d < D; ++d) r.coef[d] = alpha ? -alpha[d] / 2. : 1.0;
  return r;
}

template void Context::stage_list<double>(const StageProblem&, int, int, double, bool);
template void Context::stage_list<float>(const StageProblem&, int, int, double, bool);

// ---- the single operators on lists (FP64) ----
// A partial-sum operator is its phases and one launch that adds the terms of
// an output in order: D launches where the sweep-by-sweep form takes
// D 2^(D-1) per term (2D: 28 launches of a right-hand side and stage become
// 12).  The sums are the same: the sweep-by-sweep form adds term after term to
// the output as well.

// The sweep-by-sweep form needs two buffers of an element's values and no
// lists.  Lists and phase buffers take more (bytes an element with k = 2, m = 3:
// 1.8 K beside 2.1 K of fields in 2D at level 9, 10 K beside 11 K in 3D at level
// 7, 108 K beside 52 K in 4D at level 8).  So past 1 GiB of phase buffers the
// volume and flux operators go direction by direction (4D: 33 K; the launches
// that this adds are nothing there, and equal fluxes share no sweeps between
// directions), and the operators run on lists while these need at most 16 GiB
// and half of the free memory, or where a stage holds them already; beyond, and
// where the offsets do not fit, sweep by sweep.  A right-hand side by operators:
// 4D level 8, 168 thousand elements, 82.6 ms sweep by sweep, 49.1 joined with 32.6
// GiB, 48.4 direction by direction with 8.5 GiB; 3D level 7, 109 thousand, 8.3 and
// 3.2 ms (1.2 GiB); 2D level 9, 180 thousand, 6.8 and 1.7 ms (0.4 GiB).
constexpr int64_t kListOpsJoined = int64_t{1} << 30, kListOpsBytes = int64_t{16} << 30;
constexpr int64_t kListOpsFree = int64_t{64} << 20;  // taken without a look at the free memory

Context::ListWay Context::list_ops_way(ListForm form, int kind0, int nkind) {
  // (Lagrange degree 5 has list kernels for the constant-coefficient operator only)
  if ((m > 4 && form != LIST_LINEAR) || !list_stage_fits()) return WAY_SWEEPS;
  if (lists_current(kind0, nkind)) {
    if (form == LIST_LINEAR) return WAY_JOINED;
    if (list_plans[form] && E() <= list_ecap) return list_plans[form]->split ? WAY_SPLIT : WAY_JOINED;
  }
  ListWay way = WAY_JOINED;
  int64_t all = 0, more = 0;  // bytes needed, and bytes of them not yet held
  auto bytes = [](auto& buf, int64_t n) {
    return static_cast<int64_t>(sizeof(*buf.p)) * static_cast<int64_t>(buf.grown(static_cast<size_t>(n)));
  };
  auto held = [](auto& buf, int64_t n) { return n <= static_cast<int64_t>(buf.cap); };
  auto need = [&](auto& buf, int64_t n) {
    all += bytes(buf, n);
    if (!held(buf, n)) more += bytes(buf, n);
  };
  for (int d = 0; d < D; ++d) {
    const int lmax = deepest_level(d);
    for (int q = kind0; q < kind0 + nkind; ++q) {
      need(l_meta[q * D + d], E());
      need(l_ent[q * D + d], list_room(q, lmax));
    }
  }
  const bool rhs = form == LIST_OPS || form == LIST_OPS_SAME;
  if (rhs || form == LIST_UP) {
    // every sweep of every chain in a buffer of its own: no plan takes more, and
    // on small grids that is little enough to count nothing
    const int64_t nord = D == 1 ? 1 : int64_t{1} << (D - 1);
    int64_t T = 1;
    for (int d = 0; d < D; ++d) T *= std::max(k, m) + 1;
    const int64_t most = std::max<int64_t>((rhs ? D * nord : nord) * (D - 1) * T, 1);
    if (all + bytes(list_tmp, most * list_places()) <= kListOpsFree) return way;
    auto values = [&](bool split) {
      int64_t& v = list_values[form][split];
      if (v < 0) {
        ListPlan pl;
        pl.split = split;
        ListTerms b;
        list_terms(form, pl, b);
        v = static_cast<int64_t>(b.values);
      }
      return v * list_places();
    };
    if (rhs && !held(list_tmp, values(false)) && bytes(list_tmp, values(false)) > kListOpsJoined) way = WAY_SPLIT;
    need(list_tmp, values(way == WAY_SPLIT));
  }
  if (more == 0 || all <= kListOpsFree) return way;
  if (all > kListOpsBytes) return WAY_SWEEPS;
  size_t free = 0, total = 0;
  hip_check(hipMemGetInfo(&free, &total), "hipMemGetInfo");
  return more <= static_cast<int64_t>(free / 2) ? way : WAY_SWEEPS;
}

void Context::eval_up_op() {
  if (list_ops_way(LIST_UP, LIST_PT, 1) == WAY_SWEEPS) { eval_up(); return; }
  ensure_lists(LIST_PT, 1);
  const ListPlan& pl = get_list_plan(LIST_UP);
  list_phases<double>(pl, pl.up, PROF_SWEEP, k + 1, m + 1);
  prof_begin(PROF_SWEEP, pl.up_final.bytes * E());
  list_up_final<double>(k + 1, m + 1, pl.terms.p + pl.up_final.first, pl.up_final.n, E(), P, u.p, up.p, fp.p, vcoef.p, -1,
                        0., 0, stream);
  prof_end();
}

void Context::rhs_lagr_op(bool flux_term) {
  const ListForm form = same_flux ? LIST_OPS_SAME : LIST_OPS;
  const ListWay way = list_ops_way(form, LIST_VOL, 2);
  if (way == WAY_SWEEPS) { rhs_lagr(flux_term); return; }
  ensure_lists(LIST_VOL, 2);
  const ListPlan& pl = get_list_plan(form, way == WAY_SPLIT);
  ListRhs r = list_rhs(true, 0, 0, 0., false, nullptr);
  r.u_next = nullptr;
  for (const ListPlan::Op& op : pl.ops[flux_term]) {
    list_phases<double>(pl, op.phases, PROF_RHS_PHASE, m + 1, k + 1);
    prof_begin(PROF_SWEEP, op.last.bytes * E());
    list_rhs_final<double>(m + 1, k + 1, pl.terms.p + op.last.first, op.last.n, 0, E(), K, r, stream);
    prof_end();
  }
}

void Context::rhs_penalty_op(const double* alpha) {
  // the right-hand side's plan holds the sweeps too; without one they need no phase buffers
  const ListForm rhs_form = same_flux ? LIST_OPS_SAME : LIST_OPS;
  const ListForm form = list_plans[rhs_form] && E() <= list_ecap ? rhs_form : LIST_PENALTY;
  const ListWay way = list_ops_way(form, LIST_VOL, 2);
  if (way == WAY_SWEEPS) { rhs_penalty(alpha); return; }
  ensure_lists(LIST_VOL, 2);
  const ListPlan& pl = get_list_plan(form, way == WAY_SPLIT);
  ListRhs r = list_rhs(true, 0, 0, 0., false, alpha);
  r.u_next = nullptr;
  prof_begin(PROF_SWEEP, 8.0 * E() * K * (2 + D));
  list_rhs_final<double>(m + 1, k + 1, pl.terms.p + pl.pen, 0, D, E(), K, r, stream);
  prof_end();
}

// The assembled constant-coefficient operator as D sweeps of one launch: added
// to the right-hand side, or with a whole RK stage (run = true).
void Context::linear_list(const double* coef, bool run, int scheme, int stage, double dt, bool first) {
  linear_tables(coef);
  ensure_lists(LIST_LIN, 1);
  u_next.ensure(static_cast<size_t>(E()) * K);
  ListKey key{};
  size_t n = 0;
  for (int d = 0; d < D; ++d)
    for (const void* q : {static_cast<const void*>(l_meta[LIST_LIN * D + d].p), static_cast<const void*>(l_ent[LIST_LIN * D + d].p),
                          static_cast<const void*>(t_lin[d].p)})
      key[n++] = reinterpret_cast<uintptr_t>(q);
  std::shared_ptr<ListPlan>& pl = list_plans[LIST_LINEAR];
  if (!pl || pl->key != key) {
    pl.reset(new ListPlan());
    std::vector<ListTerm> terms;
    std::vector<int2> rofs;
    const int k1 = k + 1, R = K / k1;
    for (int d = 0; d < D; ++d) {
      ListTerm t{};
      t.M = t_lin[d].p; t.meta = l_meta[LIST_LIN * D + d].p; t.ent = l_ent[LIST_LIN * D + d].p;
      t.coef = 1.0; t.comp_size = t.Tin = t.Tout = K; t.R = R; t.ns = 1 << nmax; t.lu = LU_FULL;
      t.sdd = 1;
      for (int q = d + 1; q < D; ++q) t.sdd *= k1;
      t.sod = t.sdd;
      terms.push_back(t);
      for (int r = 0; r < R; ++r) {
        const int o = (r / t.sdd) * t.sdd * k1 + r % t.sdd;
        rofs.push_back(int2{o, o});
      }
    }
    upload(pl->rofs, rofs, stream);
    for (int d = 0; d < D; ++d) terms[d].rofs = pl->rofs.p + static_cast<size_t>(d) * R;
    upload(pl->terms, terms, stream);
    sync();
    pl->key = key;
  }
  ListRhs r = list_rhs(!run, scheme, stage, dt, first, nullptr);
  if (!run) r.u_next = nullptr;
  prof_begin(PROF_SWEEP, 8.0 * E() * K * (run ? D + 4 : D + 2));
  list_rhs_final<double>(k + 1, k + 1, pl->terms.p, 0, D, E(), K, r, stream);
  prof_end();
  if (run) {
    std::swap(u.p, u_next.p);
    std::swap(u.cap, u_next.cap);
  }
}

// One RK stage of du/dt = A u; first: u^n <- u before it.
void Context::linear_stage(const double* coef, int scheme, int stage, double dt, bool first) {
  if (list_ops_way(LIST_LINEAR, LIST_LIN, 1) != WAY_SWEEPS) {
    linear_list(coef, true, scheme, stage, dt, first);
    return;
  }
  if (first) rk_init();
  rhs_zero();
  rhs_linear(coef);
  rk_stage(scheme, stage, dt);
}

void Context::rhs_linear_op(const double* coef) {
  if (list_ops_way(LIST_LINEAR, LIST_LIN, 1) != WAY_SWEEPS) linear_list(coef, false, 0, 0, 0., false);
  else rhs_linear(coef);
}

}  // namespace adg
