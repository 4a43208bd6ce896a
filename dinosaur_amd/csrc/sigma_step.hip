// Whole evaluations of the sigma equations behind one C call each: the explicit
// terms (modal prep, inverse transform, nodal terms, forcing, forward
// transform, epilogue) and an IMEX Runge-Kutta step (its stages, implicit solves
// and terms, explicit terms, output combination and filter).
//
// Host code only: the launches are those of the separate entry points, in the
// same order, on the caller's stream and workspace, so results are bitwise the
// same.  It exists for the small grids, where a step's 31 launches of 4-10 us
// each cost 18-20 us apiece from Python: T21 L12, one member, a SIL3 step with
// its filter, 641 us through the separate calls and 227 in one, with the same kernels;
// T42 L24 explicit terms 141 and 77 us.
#include <algorithm>
#include <vector>

#include "dino_common.h"

using namespace dino;

namespace {

// Bump allocator over the caller's workspace, in elements; base null: sizes only.
struct Arena {
  char* base;
  size_t es;
  int64_t used = 0;
  void* take(int64_t n) {
    void* p = base ? base + (size_t)used * es : nullptr;
    used += (n + 63) / 64 * 64;
    return p;
  }
};

struct ExplicitSizes {
  int64_t n_prep, n_epi, n_in, n_out, RL, RJ, IJ;
};

ExplicitSizes explicit_sizes(const dino_explicit_args* a) {
  ExplicitSizes s;
  s.n_prep = dino_modal_fields(a->modal, a->members, 1);
  s.n_epi = dino_modal_fields(a->modal, a->members, 2);
  s.n_in = dino_nodal_fields(a->nodal, a->members, 0);
  s.n_out = dino_nodal_fields(a->nodal, a->members, 1);
  s.RL = (int64_t)a->plan->R * a->plan->L;
  s.RJ = (int64_t)a->plan->R * a->plan->J;
  s.IJ = (int64_t)a->plan->I * a->plan->J;
  return s;
}

struct ExplicitWork {
  void *modal, *rows, *nodal_in, *nodal_out;
};

ExplicitWork explicit_work(const ExplicitSizes& s, Arena* w) {
  const int64_t n = std::max(s.n_prep, s.n_epi);
  return {w->take(n * s.RL), w->take(n * s.RJ), w->take(s.n_prep * s.IJ),
          w->take(s.n_epi * s.IJ)};
}

#define TRY(expr)                   \
  do {                              \
    const int rc_ = (expr);         \
    if (rc_ != DINO_OK) return rc_; \
  } while (0)

int check_explicit(const dino_explicit_args* a) {
  DINO_REQUIRE(a && a->plan && a->modal && a->nodal && a->orography, DINO_EINVAL,
               "explicit terms: NULL argument");
  DINO_REQUIRE(a->members >= 1 && a->members <= 65535, DINO_EINVAL, "members out of range");
  DINO_REQUIRE(a->dtype == DINO_F32 || a->dtype == DINO_F64, DINO_EINVAL, "unknown dtype %d",
               a->dtype);
  const ExplicitSizes s = explicit_sizes(a);
  const int64_t E = a->members, extra = a->forcing ? E : 0;
  DINO_REQUIRE(s.n_prep == s.n_in + extra && s.n_epi == s.n_out + extra * a->layers,
               DINO_ESHAPE, "explicit terms: the modal and nodal handles do not match");
  return DINO_OK;
}

int run_explicit(const dino_explicit_args* a, const ExplicitSizes& s, const ExplicitWork& w,
                 const void* state, void* tendency, void* stream) {
  const int64_t E = a->members, EK = E * a->layers;
  const int prec = a->dtype == DINO_F64 ? (int)DINO_PREC_NATIVE : a->precision;
  TRY(dino_modal_prep(a->modal, state, nullptr, w.modal, E, a->dtype, stream));
  TRY(dino_sht_inverse(a->plan, w.modal, w.nodal_in, w.rows, s.n_prep, a->dtype, prec, stream));
  TRY(dino_nodal_explicit(a->nodal, w.nodal_in, w.nodal_out, E, a->dtype, stream));
  if (a->forcing) {
    const int64_t in_groups[4] = {2 * EK, (3 + a->tracers) * EK, (4 + a->tracers) * EK, s.n_in};
    const int64_t out_groups[3] = {0, EK, s.n_out};
    TRY(dino_held_suarez_nodal(a->forcing, w.nodal_in, w.nodal_out, in_groups, out_groups, E,
                               a->dtype, stream));
  }
  TRY(dino_sht_forward(a->plan, w.nodal_out, w.modal, w.rows, s.n_epi, a->dtype,
                       prec | DINO_SHT_TRIANGLE_ONLY, stream));
  return dino_modal_epilogue(a->modal, w.modal, a->orography, tendency, E, a->dtype, stream);
}

// Which tendencies the step's formula contains (a later stage or the output).
void used_terms(int n, const double* a, const double* b, std::vector<char>* used) {
  used->assign(n, 0);
  for (int i = 0; i < n; ++i) {
    bool u = b[i] != 0;
    for (int j = i; j < n - 1; ++j) u = u || a[j * n + i] != 0;
    (*used)[i] = u;
  }
}

struct StepWork {
  ExplicitWork ex;
  std::vector<void*> f, g;
  void* y;
};

StepWork step_work(const dino_imex_step_args* a, const ExplicitSizes& s, Arena* w) {
  std::vector<char> fu, gu;
  used_terms(a->stages, a->a_ex, a->b_ex, &fu);
  used_terms(a->stages, a->a_im, a->b_im, &gu);
  StepWork r;
  r.ex = explicit_work(s, w);
  r.f.assign(a->stages, nullptr);
  r.g.assign(a->stages, nullptr);
  r.y = w->take(a->n);
  for (int i = 0; i < a->stages; ++i) {
    // stage 0's explicit tendency is always formed
    if (fu[i] || i == 0) r.f[i] = w->take(a->n);
    if (gu[i]) r.g[i] = w->take(a->im_end - a->g_origin);
  }
  return r;
}

size_t elem_size(int dtype) { return dtype == DINO_F64 ? 8 : 4; }

}  // namespace

extern "C" int64_t dino_explicit_workspace(const dino_explicit_args* a) {
  if (check_explicit(a) != DINO_OK) return -1;
  Arena w{nullptr, elem_size(a->dtype)};
  explicit_work(explicit_sizes(a), &w);
  return w.used;
}

extern "C" int dino_explicit_terms(const dino_explicit_args* a, const void* state,
                                   void* tendency, void* work, void* stream) {
  TRY(check_explicit(a));
  DINO_REQUIRE(state && tendency && work, DINO_EINVAL, "dino_explicit_terms: NULL buffer");
  Arena w{static_cast<char*>(work), elem_size(a->dtype)};
  const ExplicitSizes s = explicit_sizes(a);
  return run_explicit(a, s, explicit_work(s, &w), state, tendency, stream);
}

static int check_step(const dino_imex_step_args* a) {
  DINO_REQUIRE(a && a->a_ex && a->a_im && a->b_ex && a->b_im && a->terms && a->solve,
               DINO_EINVAL, "dino_imex_step: NULL argument");
  TRY(check_explicit(&a->explicit_args));
  DINO_REQUIRE(a->stages >= 2 && a->stages <= 7, DINO_EINVAL, "dino_imex_step: %d stages",
               a->stages);
  DINO_REQUIRE(0 <= a->g_origin && a->g_origin <= a->im_begin && a->im_begin <= a->im_end &&
                   a->im_end <= a->n,
               DINO_EINVAL, "dino_imex_step: invalid implicit range");
  return DINO_OK;
}

extern "C" int64_t dino_imex_step_workspace(const dino_imex_step_args* a) {
  if (check_step(a) != DINO_OK) return -1;
  Arena w{nullptr, elem_size(a->explicit_args.dtype)};
  step_work(a, explicit_sizes(&a->explicit_args), &w);
  return w.used;
}

extern "C" int dino_imex_step(const dino_imex_step_args* a, const void* y0, void* out, void* work,
                              void* stream) {
  TRY(check_step(a));
  DINO_REQUIRE(y0 && out && work, DINO_EINVAL, "dino_imex_step: NULL buffer");
  const dino_explicit_args* ex = &a->explicit_args;
  const ExplicitSizes s = explicit_sizes(ex);
  const size_t es = elem_size(ex->dtype);
  Arena arena{static_cast<char*>(work), es};
  StepWork w = step_work(a, s, &arena);
  const int n = a->stages, dt = ex->dtype;
  const int64_t E = ex->members, EK = E * ex->layers;
  const int stage_type = dt | (a->triangle_only && a->degrees ? DINO_STAGE_TRIANGLE_ONLY : 0);
  auto at = [&](const void* p, int64_t i) {
    return static_cast<void*>(const_cast<char*>(static_cast<const char*>(p)) + (size_t)i * es);
  };
  // divergence, temperature and ln ps of a state buffer or a compact one
  auto terms = [&](const void* y, void* g) {
    const int64_t o = a->im_begin - a->g_origin;
    return dino_implicit_terms(a->terms, at(y, EK * s.RL), at(y, 2 * EK * s.RL),
                               at(y, 3 * EK * s.RL), at(g, o), at(g, o + EK * s.RL),
                               at(g, o + 2 * EK * s.RL), E, dt, stream);
  };
  // terms with nonzero coefficients of one combination
  const void *fs[7], *gs[7];
  double ca[7], cb[7];
  auto collect = [&](const double* ca_, const double* cb_, int upto, int* n_ex, int* n_im) {
    *n_ex = *n_im = 0;
    for (int j = 0; j < upto; ++j) {
      if (ca_[j] != 0) { ca[*n_ex] = ca_[j]; fs[(*n_ex)++] = w.f[j]; }
      if (cb_[j] != 0) { cb[*n_im] = cb_[j]; gs[(*n_im)++] = w.g[j]; }
    }
  };
  int n_ex, n_im;
  TRY(run_explicit(ex, s, w.ex, y0, w.f[0], stream));
  if (w.g[0]) TRY(terms(y0, w.g[0]));
  for (int i = 1; i < n; ++i) {
    if (!w.f[i] && !w.g[i]) continue;
    collect(a->a_ex + (i - 1) * n, a->a_im + (i - 1) * n, i, &n_ex, &n_im);
    if (w.f[i]) {
      TRY(dino_imex_stage_ranged(y0, n_ex, fs, ca, n_im, gs, cb, a->dt, w.y, a->n, a->im_begin,
                                 a->im_end, a->g_origin, a->field_size, a->degrees, stage_type,
                                 stream));
    } else {  // only the implicit terms read this stage value
      for (int k = 0; k < n_ex; ++k) fs[k] = at(fs[k], a->im_begin);
      for (int k = 0; k < n_im; ++k) gs[k] = at(gs[k], a->im_begin - a->g_origin);
      const int64_t nr = a->im_end - a->im_begin;
      TRY(dino_imex_stage_ranged(at(y0, a->im_begin), n_ex, fs, ca, n_im, gs, cb, a->dt,
                                 at(w.y, a->im_begin), nr, 0, nr, 0, a->field_size, a->degrees,
                                 dt, stream));
    }
    void *d = at(w.y, EK * s.RL), *t = at(w.y, 2 * EK * s.RL), *l = at(w.y, 3 * EK * s.RL);
    TRY(dino_implicit_solve(a->solve[i - 1], d, t, l, d, t, l, E, dt, stream));
    if (w.f[i]) TRY(run_explicit(ex, s, w.ex, w.y, w.f[i], stream));
    if (w.g[i]) TRY(terms(w.y, w.g[i]));
  }
  collect(a->b_ex, a->b_im, n, &n_ex, &n_im);
  if (a->degree_scale)
    return dino_imex_stage_ranged_scaled(y0, n_ex, fs, ca, n_im, gs, cb, a->dt, out, a->n,
                                         a->im_begin, a->im_end, a->g_origin, a->field_size,
                                         a->degrees, a->degree_scale, a->scale_len, dt, stream);
  return dino_imex_stage_ranged(y0, n_ex, fs, ca, n_im, gs, cb, a->dt, out, a->n, a->im_begin,
                                a->im_end, a->g_origin, a->field_size, a->degrees, dt, stream);
}
