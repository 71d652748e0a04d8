// sd2d_adjhost.hpp - the adjoint entry points (sd2d_fwd, sd2d_vjp,
// sd2d_compresid_vjp in include/sd2d.h).  Included at the end of sd2d.hip.
//
// sd2d_fwd steps the context like sd2d_step (RK_S5P3, FP64, inviscid path),
// accumulates the time-averaged wall drag J = (1/nsteps) sum_n D(Q_n) and
// keeps a checkpoint (state and running maxima) every `ckpt` steps.
// sd2d_vjp runs backwards over the checkpoint segments: a segment's step
// inputs are recomputed from its checkpoint, then each step's five stage
// inputs and the GLM maxima before each stage are recomputed by the line kernel
// with M_TRACE (the forward's states bit for bit, whichever form of the stage
// kernel it took), and the step is reversed stage by stage:
//   Q1 = Q0 + b10 dt R(Q0)            Q0bar += Q1bar + (dR/dQ0)^T b10 dt Q1bar
//   Q2 = Q1 + b21 dt R(Q1)            ...
//   Q3 = a30 Q0 + a32 Q2 + b32 dt R(Q2)
//   Q4 = a40 Q0 + a43 Q3 + b43 dt R(Q3)
//   Q5 = a52 Q2 + a54 Q4 + b54 dt R(Q4)   (iterations.f90:158-213)
// with the drag's cotangent added to each step's output.  The lagged GLM
// speed c_h = sqrt(E(E - U)) of an evaluation comes from the running maxima
// E, U of the wave speeds over all earlier evaluations: its cotangent is
// carried backwards (pools PE, PU) to the last earlier evaluation that
// raised the maximum, and there to the flux point whose speed attained it
// (recorded by the recomputed stage, M_TRACE; adj_tail_kernel).

// Everything the reverse pass accumulates stays on the device (AdjCarry), so
// no stage waits for the host: per reversed stage one adj_stage_kernel (the
// residual's reverse sweep and the RK combination) and one adj_tail_kernel.

struct AdjState {
  int nsteps = 0, ckpt = 0;
  bool have_fwd = false;
  double J = 0.0;
  double *t[4] = {};          // stage states Q1..Q4 of one step (tile layout)
  double *b[6] = {};          // cotangents of Q0..Q5
  double *divb = nullptr;     // divB per point of the five evaluations of a step
  double *part = nullptr;     // per tile partial sums
  unsigned long long *gm = nullptr;   // the maxima read by each of the 5 stages (sets)
  double *tmax = nullptr;     // per evaluation and tile: largest speeds and where
  int *tloc = nullptr;
  AdjCarry *carry = nullptr;  // what goes from one reversed evaluation to the next
  double *chb = nullptr;      // c_h cotangents, 5 per step
  int chb_n = 0;
  double *dtile = nullptr;    // drag per tile
  double *Jd = nullptr;       // running sum of the drag
  double *wq = nullptr;       // face quadrature weights
  std::vector<double *> ck;   // checkpoint states (index = step / ckpt) + final state
  std::vector<std::array<double, 4>> ckm;   // their maxima
  std::vector<int32_t> cki;   // their iter and ctime
  std::vector<double> ckt;
  std::vector<double *> seg;  // step inputs of one segment and its output
  double *segm = nullptr;     // the maxima before each step of the segment (4 each)
  int segm_n = 0;
  double fin_ctime = 0.0;
  int fin_iter = 0;
};

static void adj_free(AdjState *A) {
  if (!A) return;
  for (double *p : A->t) if (p) (void)hipFree(p);
  for (double *p : A->b) if (p) (void)hipFree(p);
  for (void *p : {(void *)A->divb, (void *)A->part, (void *)A->gm, (void *)A->tmax,
                  (void *)A->tloc, (void *)A->carry, (void *)A->chb,
                  (void *)A->dtile, (void *)A->Jd, (void *)A->wq, (void *)A->segm})
    if (p) (void)hipFree(p);
  for (double *p : A->ck) if (p) (void)hipFree(p);
  for (double *p : A->seg) if (p) (void)hipFree(p);
  delete A;
}

static size_t state_len(const sd2d_ctx *c) { return (size_t)c->ntile * 9 * c->N * c->N * c->cpw; }

// The running maxima of one run (a set) to and from four doubles on the device:
// eigvmax, umax, eigvmax_g, umax_g.
__global__ void k_save_max(const unsigned long long *set, double *m) {
  m[0] = __longlong_as_double((long long)set[0]);
  m[1] = __longlong_as_double((long long)set[1]);
  set_pair(set, m[2], m[3]);
}
__global__ void k_load_max(const double *m, unsigned long long *set) {
  set[threadIdx.x] = as_bits(m[threadIdx.x]);
}

static int save_max(sd2d_ctx *c, double *m) {
  hipLaunchKernelGGL(k_save_max, dim3(1), dim3(1), 0, c->stream, max_set(c, c->mset), m);
  HIPCHK(c, hipGetLastError());
  return SD2D_OK;
}

static int adj_maxima_get(sd2d_ctx *c, std::array<double, 4> &m) {
  sd2d_maxima mx;
  const int r = sd2d_get_state(c, nullptr, &mx);
  m = {mx.eigvmax, mx.umax, mx.eigvmax_g, mx.umax_g};
  return r;
}

static int adj_maxima_set(sd2d_ctx *c, const std::array<double, 4> &m) {
  hipLaunchKernelGGL(k_set_max, dim3(1), dim3(1), 0, c->stream, max_set(c, c->mset), m[0], m[1],
                     m[2], m[3]);
  HIPCHK(c, hipGetLastError());
  return SD2D_OK;
}

// interpolatory quadrature weights on the solution-point positions xs of
// [0, 1]: w_i = integral of the Lagrange basis polynomial l_i
static std::vector<double> face_weights(const double *xs, int N) {
  std::vector<double> w(N, 0.0);
  for (int i = 0; i < N; ++i) {
    std::vector<double> c(1, 1.0);   // coefficients of prod_{j != i} (x - xj)/(xi - xj)
    for (int j = 0; j < N; ++j) {
      if (j == i) continue;
      std::vector<double> n(c.size() + 1, 0.0);
      for (size_t k = 0; k < c.size(); ++k) {
        n[k + 1] += c[k] / (xs[i] - xs[j]);
        n[k] -= c[k] * xs[j] / (xs[i] - xs[j]);
      }
      c = n;
    }
    for (size_t k = 0; k < c.size(); ++k) w[i] += c[k] / double(k + 1);
  }
  return w;
}

// What one residual's reverse sweep needs, and (steps) the whole reverse pass.
static int adj_alloc(sd2d_ctx *c, AdjState *A, int nck, bool steps) {
  const size_t n = state_len(c);
  const size_t np = (size_t)c->ntile * c->N * c->N * c->cpw;
  auto get = [&](auto *&p, size_t count) -> int {
    if (!p) HIPCHK(c, hipMalloc(&p, count * sizeof(*p)));
    return SD2D_OK;
  };
  int r;
#define ADJGET(p, count) do { if ((r = get(p, count))) return r; } while (0)
  for (int i = 0; i < (steps ? 6 : 2); ++i) ADJGET(A->b[i], n);
  ADJGET(A->divb, 5 * np);
  ADJGET(A->part, (size_t)c->ntile * ADJ_NPART);
  if (!steps) return SD2D_OK;
  ADJGET(A->carry, 1);
  ADJGET(A->gm, 5 * MSTRIDE);
  for (auto &p : A->t) ADJGET(p, n);
  ADJGET(A->tmax, 10 * (size_t)c->ntile);
  ADJGET(A->tloc, 10 * (size_t)c->ntile);
  ADJGET(A->dtile, c->ntile);
  ADJGET(A->Jd, 1);
  if (A->chb_n < 5 * A->nsteps) {
    if (A->chb) { HIPCHK(c, hipFree(A->chb)); A->chb = nullptr; A->chb_n = 0; }
    ADJGET(A->chb, (size_t)5 * A->nsteps);
    A->chb_n = 5 * A->nsteps;
  }
  const int nseg = std::min(A->ckpt, A->nsteps);
  if (A->segm_n < nseg) {
    if (A->segm) { HIPCHK(c, hipFree(A->segm)); A->segm = nullptr; A->segm_n = 0; }
    ADJGET(A->segm, (size_t)4 * nseg);
    A->segm_n = nseg;
  }
#undef ADJGET
  while ((int)A->ck.size() < nck) {
    double *p = nullptr;
    HIPCHK(c, hipMalloc(&p, n * sizeof(double)));
    A->ck.push_back(p);
  }
  A->ckm.resize(A->ck.size());
  while ((int)A->seg.size() < nseg + 1) {
    double *p = nullptr;
    HIPCHK(c, hipMalloc(&p, n * sizeof(double)));
    A->seg.push_back(p);
  }
  return SD2D_OK;
}

// The wall drag at state q added to A->Jd (sum), or with qbar its cotangent
// scale * dD/dq added to qbar.
static int drag_eval(sd2d_ctx *c, const double *q, bool sum, double *qbar, double scale) {
  AdjState *A = c->adj;
  const dim3 grid(c->ntile), block(64);
  switch (c->N) {
    case 3: hipLaunchKernelGGL(drag_kernel<3>, grid, block, 0, c->stream, q, c->ftab, c->met, c->mcomp, A->wq, c->ops, A->dtile, qbar, scale); break;
    case 4: hipLaunchKernelGGL(drag_kernel<4>, grid, block, 0, c->stream, q, c->ftab, c->met, c->mcomp, A->wq, c->ops, A->dtile, qbar, scale); break;
    default: hipLaunchKernelGGL(drag_kernel<5>, grid, block, 0, c->stream, q, c->ftab, c->met, c->mcomp, A->wq, c->ops, A->dtile, qbar, scale); break;
  }
  HIPCHK(c, hipGetLastError());
  if (sum) {
    hipLaunchKernelGGL(k_drag_sum, dim3(1), dim3(1024), 0, c->stream, A->dtile, c->ntile,
                       A->Jd);
    HIPCHK(c, hipGetLastError());
  }
  return SD2D_OK;
}

// the RK_S5P3 stages as s5p3_sequence runs them, on the six stage buffers:
// qin, aux, coefficients and the mode of the forward launch
struct AdjStage { int in, aux, out; double cin, ca, b; };
static const AdjStage kS5P3[5] = {
    {0, -1, 1, 1.0, 0.0, 0.377268915331368},
    {1, -1, 2, 1.0, 0.0, 0.377268915331368},
    {2, 0, 3, 0.644090224936674, 0.355909775063327, 0.242995220537396},
    {3, 0, 4, 0.632066208361863, 0.367933791638137, 0.238458932846290},
    {4, 2, 5, 0.762406163401431, 0.237593836598569, 0.287632146308408}};

// The five stages of one step from qs[0] (the forward's launches), its states
// into qs[1..5]; with trace, what the reverse sweep needs of each evaluation
// is recorded as well (divB, the maxima before it, and where each tile's largest
// speeds are attained).
static int adj_stages(sd2d_ctx *c, double *const *qs, bool trace) {
  AdjState *A = c->adj;
  const int av = (c->p.artiv == 1 && c->p.vismode == 1) ? M_AV : 0;
  const size_t np = (size_t)c->ntile * c->N * c->N * c->cpw;
  for (int s = 0; s < 5; ++s) {
    const AdjStage &st = kS5P3[s];
    StageArgs a = base_args(c);
    a.qin = qs[st.in];
    a.qout = qs[st.out];
    a.cin = st.cin;
    a.cr = st.b * c->p.dt;
    a.naux = st.aux >= 0 ? 1 : 0;
    a.aux[0] = st.aux >= 0 ? qs[st.aux] : nullptr;
    a.ca[0] = st.ca;
    a.rev = c->nlaunch++ & 1;
    int mode = M_RK | (a.naux ? M_AUX1 : 0) | (s == 4 ? av : 0);
    if (trace) {
      mode |= M_TRACE;
      a.divb = A->divb + s * np;
      a.gmrec = A->gm + MSTRIDE * s;
      a.tmax = A->tmax + 2 * (size_t)c->ntile * s;
      a.tloc = A->tloc + 2 * (size_t)c->ntile * s;
    }
    HIPCHK(c, launch_stage(c, a, mode));
    rotate_maxima(c);
  }
  return SD2D_OK;
}

// One evaluation backwards: adj_stage_kernel and, within a pass over steps (m1
// set), adj_tail_kernel with the maxima m1 after the evaluation.
template <int N>
static hipError_t adj_launch_n(sd2d_ctx *c, const AdjArgs &a, const double *tmax, const int *tloc,
                               const unsigned long long *m1, double *chbar) {
  AdjState *A = c->adj;
  static_assert(adj_lds_bytes<N>() <= 65536, "adjoint kernel LDS above 64 KiB");
  hipLaunchKernelGGL(adj_stage_kernel<N>, dim3(c->ntile), dim3(STAGE_THREADS), adj_lds_bytes<N>(),
                     c->stream, a, c->ops);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !m1) return e;
  hipLaunchKernelGGL(adj_tail_kernel<N>, dim3(1), dim3(ADJ_TAIL_THREADS), 0, c->stream, a, c->ops,
                     tmax, tloc, m1, A->carry, chbar);
  return hipGetLastError();
}
static int adj_launch(sd2d_ctx *c, const AdjArgs &a, const double *tmax = nullptr,
                      const int *tloc = nullptr, const unsigned long long *m1 = nullptr,
                      double *chbar = nullptr) {
  switch (c->N) {
    case 3: HIPCHK(c, adj_launch_n<3>(c, a, tmax, tloc, m1, chbar)); break;
    case 4: HIPCHK(c, adj_launch_n<4>(c, a, tmax, tloc, m1, chbar)); break;
    default: HIPCHK(c, adj_launch_n<5>(c, a, tmax, tloc, m1, chbar)); break;
  }
  return SD2D_OK;
}

static AdjArgs adj_args(sd2d_ctx *c) {
  AdjState *A = c->adj;
  AdjArgs a{};
  a.rscale = 1.0; a.met = c->met; a.mcomp = c->mcomp; a.ftab = c->ftab; a.tinfo = c->tinfo; a.phm = c->phm;
  a.part = A->part; a.alpha = c->ph.alpha; a.ntile = c->ntile;
  return a;
}

// Reverse one RK_S5P3 step: A->b[5] holds the cotangent of the step's
// output (Q5), on return A->b[0] that of its input (Q0).  qs[0..4] are the
// recomputed stage inputs (adj_stages with trace; the maxima after the last
// stage are still the context's).
static int adj_step_vjp(sd2d_ctx *c, double *const *qs, double *chbar5) {
  AdjState *A = c->adj;
  double **B = A->b;
  const size_t np = (size_t)c->ntile * c->N * c->N * c->cpw;
  bool have[5] = {false, false, false, false, false};   // cotangents already begun
  for (int s = 4; s >= 0; --s) {
    const AdjStage &st = kS5P3[s];
    // Q_out = cin Q_in + ca Q_aux + b dt R(Q_in)
    AdjArgs a = adj_args(c);
    a.q = qs[st.in];
    a.rbar = B[st.out];
    a.rscale = st.b * c->p.dt;
    a.cin = st.cin;
    a.ca = st.ca;
    a.divb = A->divb + s * np;
    a.gm = A->gm + MSTRIDE * s;
    a.qbar = B[st.in];
    a.qadd = have[st.in];
    have[st.in] = true;
    if (st.aux >= 0) {
      a.abar = B[st.aux];
      a.aadd = have[st.aux];
      have[st.aux] = true;
    }
    const unsigned long long *m1 = s == 4 ? max_set(c, c->mset) : A->gm + MSTRIDE * (s + 1);
    const int r = adj_launch(c, a, A->tmax + 2 * (size_t)c->ntile * s,
                             A->tloc + 2 * (size_t)c->ntile * s, m1, chbar5 + s);
    if (r) return r;
  }
  return SD2D_OK;
}

extern "C" {

// the wall-drag quadrature weights on the device, once per context
static int adj_weights(sd2d_ctx *c, AdjState *A) {
  if (A->wq) return SD2D_OK;
  const std::vector<double> w = face_weights(c->xs.data(), c->N);
  HIPCHK(c, hipMalloc(&A->wq, w.size() * sizeof(double)));
  HIPCHK(c, hipMemcpy(A->wq, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice));
  return SD2D_OK;
}

int sd2d_fwd(sd2d_ctx *c, int32_t nsteps, int32_t ckpt, double *objective) {
  if (!c) return fail(nullptr, SD2D_EINVAL, "ctx is NULL");
  if (nsteps <= 0 || ckpt <= 0) return fail(c, SD2D_EINVAL, "nsteps and ckpt must be positive");
  if (c->next_stage != 1)
    return fail(c, SD2D_EINVAL, "a step is in progress (sd2d_rk_stage): finish it first");
  if (c->p.precision != SD2D_FP64 || c->p.k_stage != 3 || c->vis || c->nmem > 1)
    return fail(c, SD2D_EUNSUPPORTED,
                "the adjoint covers the FP64 inviscid path with RK_S5P3 (k_stage 3)");
  if (!c->adj) c->adj = new (std::nothrow) AdjState();
  AdjState *A = c->adj;
  if (!A) return fail(c, SD2D_ENOMEM, "host allocation failed");
  A->nsteps = nsteps;
  A->ckpt = ckpt;
  A->have_fwd = false;
  const int nck = (nsteps + ckpt - 1) / ckpt + 1;   // segment starts + the final state
  int r = adj_alloc(c, A, nck, true);
  if (r) return r;
  if ((r = adj_weights(c, A))) return r;
  A->cki.assign(nck, 0);
  A->ckt.assign(nck, 0.0);
  const size_t nb = state_len(c) * sizeof(double);
  HIPCHK(c, hipMemsetAsync(A->Jd, 0, sizeof(double), c->stream));
  for (int n = 0; n < nsteps; ++n) {
    if (n % ckpt == 0) {
      HIPCHK(c, hipMemcpyAsync(A->ck[n / ckpt], c->q[c->cur], nb, hipMemcpyDeviceToDevice, c->stream));
      if ((r = adj_maxima_get(c, A->ckm[n / ckpt]))) return r;
      A->cki[n / ckpt] = c->iter;
      A->ckt[n / ckpt] = c->ctime;
    }
    c->iter += 1;
    if ((r = step_rk(c, false))) return r;
    c->have_av = c->p.artiv == 1 && c->p.vismode == 1;
    if ((r = drag_eval(c, c->q[c->cur], true, nullptr, 0.0))) return r;
  }
  double J = 0.0;
  HIPCHK(c, hipMemcpyAsync(&J, A->Jd, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(A->ck[nck - 1], c->q[c->cur], nb, hipMemcpyDeviceToDevice, c->stream));
  if ((r = adj_maxima_get(c, A->ckm[nck - 1]))) return r;
  A->fin_ctime = c->ctime;
  A->fin_iter = c->iter;
  A->cki[nck - 1] = c->iter;
  A->ckt[nck - 1] = c->ctime;
  A->J = J / nsteps;
  A->have_fwd = true;
  if (objective) *objective = A->J;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return SD2D_OK;
}

int sd2d_vjp(sd2d_ctx *c, const double *qbar_final, double jbar, double *qbar_init,
             double *pbar, double *chbar) {
  if (!c) return fail(nullptr, SD2D_EINVAL, "ctx is NULL");
  SD2D_NOT_MID_STEP(c, "sd2d_vjp");
  AdjState *A = c->adj;
  if (!A || !A->have_fwd) return fail(c, SD2D_EINVAL, "sd2d_vjp needs a preceding sd2d_fwd");
  const int nsteps = A->nsteps, ckpt = A->ckpt, nck = (nsteps + ckpt - 1) / ckpt + 1;
  const size_t nb = state_len(c) * sizeof(double);
  int r;
  // cotangent of the final state
  if (qbar_final) {
    const size_t n = (size_t)c->ncell * 9 * c->N * c->N;
    HIPCHK(c, to_device(c, c->stagef, qbar_final, n));
    if ((r = f2t(c, c->stagef, A->b[5]))) return r;
  } else {
    HIPCHK(c, hipMemsetAsync(A->b[5], 0, nb, c->stream));
  }
  HIPCHK(c, hipMemsetAsync(A->carry, 0, sizeof(AdjCarry), c->stream));
  for (int sg = (nsteps - 1) / ckpt; sg >= 0; --sg) {
    const int n0 = sg * ckpt, n1 = std::min(nsteps, n0 + ckpt), len = n1 - n0;
    // the segment's step inputs and the maxima before them, recomputed from
    // its checkpoint
    HIPCHK(c, hipMemcpyAsync(A->seg[0], A->ck[sg], nb, hipMemcpyDeviceToDevice, c->stream));
    if ((r = adj_maxima_set(c, A->ckm[sg]))) return r;
    auto step_states = [&](int i, double **qs) {
      qs[0] = A->seg[i];
      for (int k = 0; k < 4; ++k) qs[1 + k] = A->t[k];
      qs[5] = A->seg[i + 1];
    };
    double *qs[6];
    for (int i = 0; i < len; ++i) {
      if ((r = save_max(c, A->segm + 4 * i))) return r;
      if (i + 1 == len) break;   // the last step runs once, below
      step_states(i, qs);
      if ((r = adj_stages(c, qs, false))) return r;
    }
    for (int i = len - 1; i >= 0; --i) {
      const int n = n0 + i;   // step n takes Q_n to Q_{n+1}
      hipLaunchKernelGGL(k_load_max, dim3(1), dim3(MSTRIDE), 0, c->stream, A->segm + 4 * i,
                         max_set(c, c->mset));
      HIPCHK(c, hipGetLastError());
      step_states(i, qs);
      if ((r = adj_stages(c, qs, true))) return r;
      // the drag of the step's output enters the objective with weight 1/nsteps
      if (jbar != 0.0 && (r = drag_eval(c, qs[5], false, A->b[5], jbar / nsteps))) return r;
      if ((r = adj_step_vjp(c, qs, A->chb + 5 * n))) return r;
      std::swap(A->b[0], A->b[5]);
    }
  }
  if (qbar_init) {
    if ((r = t2f(c, A->b[5], c->stagef))) return r;
    const size_t n = (size_t)c->ncell * 9 * c->N * c->N;
    HIPCHK(c, to_host(c, qbar_init, c->stagef, n));
  }
  AdjCarry cy{};
  HIPCHK(c, hipMemcpyAsync(&cy, A->carry, sizeof(cy), hipMemcpyDeviceToHost, c->stream));
  if (chbar)
    HIPCHK(c, hipMemcpyAsync(chbar, A->chb, (size_t)5 * nsteps * sizeof(double), hipMemcpyDeviceToHost,
                             c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (pbar) for (int j = 0; j < 6; ++j) pbar[j] = cy.p[j];
  // the context returns to the final state of sd2d_fwd
  HIPCHK(c, hipMemcpyAsync(c->q[c->cur], A->ck[nck - 1], nb, hipMemcpyDeviceToDevice, c->stream));
  if ((r = adj_maxima_set(c, A->ckm[nck - 1]))) return r;
  c->ctime = A->fin_ctime;
  c->iter = A->fin_iter;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (cy.missed)
    return fail(c, SD2D_EINVAL, "adjoint: the flux point of a running maximum was not found");
  return SD2D_OK;
}

// The adjoint checkpoints of the last sd2d_fwd as files: <prefix>.NNNN.dat
// (NNNN = 0..nck-1) in the reference's restart format with the maxima
// sidecar of sd2d_write_checkpoint, and <prefix>.adj: 8 bytes "SD2DADJ1",
// int32 N, NCELL, nsteps, ckpt, final iter, float64 J, final ctime.
static std::string adj_ck_path(const char *prefix, int k) {
  char tail[16];
  std::snprintf(tail, sizeof(tail), ".%04d.dat", k);
  return std::string(prefix) + tail;
}

int sd2d_adj_save(sd2d_ctx *c, const char *prefix) {
  if (!c || !prefix) return fail(c, SD2D_EINVAL, "NULL argument");
  AdjState *A = c->adj;
  if (!A || !A->have_fwd) return fail(c, SD2D_EINVAL, "sd2d_adj_save needs a preceding sd2d_fwd");
  const int nck = (A->nsteps + A->ckpt - 1) / A->ckpt + 1;
  const size_t n = (size_t)c->ncell * 9 * c->N * c->N;
  std::vector<double> q(n);
  for (int k = 0; k < nck; ++k) {
    int r = t2f(c, A->ck[k], c->stagef);
    if (r) return r;
    HIPCHK(c, to_host(c, q.data(), c->stagef, n));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const std::string path = adj_ck_path(prefix, k);
    const sd2d_maxima m{A->ckm[k][0], A->ckm[k][1], A->ckm[k][2], A->ckm[k][3]};
    if (!write_restart_file(path.c_str(), A->cki[k], A->ckt[k], c->N, c->ncell, q.data(), nullptr) ||
        !write_max_file(path.c_str(), A->cki[k], A->ckt[k], m))
      return fail(c, SD2D_EINVAL, "write failed: " + path);
  }
  const std::string mp = std::string(prefix) + ".adj";
  FILE *fh = std::fopen(mp.c_str(), "wb");
  if (!fh) return fail(c, SD2D_EINVAL, "cannot write " + mp);
  const int32_t hv[5] = {c->N, c->ncell, A->nsteps, A->ckpt, A->fin_iter};
  const double dv[2] = {A->J, A->fin_ctime};
  const bool ok = std::fwrite("SD2DADJ1", 1, 8, fh) == 8 && std::fwrite(hv, sizeof(int32_t), 5, fh) == 5 &&
                  std::fwrite(dv, sizeof(double), 2, fh) == 2;
  if (std::fclose(fh) != 0 || !ok) return fail(c, SD2D_EINVAL, "write failed: " + mp);
  return SD2D_OK;
}

int sd2d_adj_load(sd2d_ctx *c, const char *prefix) {
  if (!c || !prefix) return fail(c, SD2D_EINVAL, "NULL argument");
  SD2D_NOT_MID_STEP(c, "sd2d_adj_load");
  if (c->p.precision != SD2D_FP64 || c->p.k_stage != 3 || c->vis || c->nmem > 1)
    return fail(c, SD2D_EUNSUPPORTED,
                "the adjoint covers the FP64 inviscid path with RK_S5P3 (k_stage 3)");
  const std::string mp = std::string(prefix) + ".adj";
  FILE *fh = std::fopen(mp.c_str(), "rb");
  if (!fh) return fail(c, SD2D_EINVAL, "cannot open " + mp);
  char magic[8];
  int32_t hv[5];
  double dv[2];
  const bool ok = std::fread(magic, 1, 8, fh) == 8 && std::fread(hv, sizeof(int32_t), 5, fh) == 5 &&
                  std::fread(dv, sizeof(double), 2, fh) == 2 && std::fgetc(fh) == EOF;
  std::fclose(fh);
  if (!ok || std::memcmp(magic, "SD2DADJ1", 8) != 0)
    return fail(c, SD2D_EINVAL, "not an adjoint checkpoint manifest: " + mp);
  if (hv[0] != c->N || hv[1] != c->ncell || hv[2] <= 0 || hv[3] <= 0)
    return fail(c, SD2D_EINVAL, "the adjoint checkpoints of " + mp + " belong to another mesh or order");
  if (!c->adj) c->adj = new (std::nothrow) AdjState();
  AdjState *A = c->adj;
  if (!A) return fail(c, SD2D_ENOMEM, "host allocation failed");
  A->have_fwd = false;
  A->nsteps = hv[2];
  A->ckpt = hv[3];
  const int nck = (A->nsteps + A->ckpt - 1) / A->ckpt + 1;
  int r = adj_alloc(c, A, nck, true);
  if (r) return r;
  if ((r = adj_weights(c, A))) return r;
  A->cki.assign(nck, 0);
  A->ckt.assign(nck, 0.0);
  const size_t n = (size_t)c->ncell * 9 * c->N * c->N;
  for (int k = 0; k < nck; ++k) {
    const std::string path = adj_ck_path(prefix, k);
    int32_t it = 0;
    double t = 0.0;
    std::vector<double> q;
    sd2d_maxima m{};
    std::string e = read_restart_file(path.c_str(), c->N, c->ncell, it, t, q);
    if (e.empty()) e = read_max_file(path.c_str(), it, t, m);
    if (!e.empty()) return fail(c, SD2D_EINVAL, e);
    HIPCHK(c, to_device(c, c->stagef, q.data(), n));
    if ((r = f2t(c, c->stagef, A->ck[k]))) return r;
    HIPCHK(c, hipStreamSynchronize(c->stream));   // q is reused by the next file
    A->ckm[k] = {m.eigvmax, m.umax, m.eigvmax_g, m.umax_g};
    A->cki[k] = it;
    A->ckt[k] = t;
  }
  A->J = dv[0];
  A->fin_ctime = dv[1];
  A->fin_iter = hv[4];
  if (A->cki[nck - 1] != A->fin_iter || std::memcmp(&A->ckt[nck - 1], &A->fin_ctime, sizeof(double)) != 0)
    return fail(c, SD2D_EINVAL, "the last adjoint checkpoint is not the final state of " + mp);
  A->have_fwd = true;
  // the context holds the final state of the forward run, as after sd2d_fwd
  HIPCHK(c, hipMemcpyAsync(c->q[c->cur], A->ck[nck - 1], state_len(c) * sizeof(double),
                           hipMemcpyDeviceToDevice, c->stream));
  if ((r = adj_maxima_set(c, A->ckm[nck - 1]))) return r;
  c->ctime = A->fin_ctime;
  c->iter = A->fin_iter;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return SD2D_OK;
}

int sd2d_compresid_vjp(sd2d_ctx *c, const double *rbar, double *qbar, double *chbar, double *pbar) {
  if (!c || !rbar) return fail(c, SD2D_EINVAL, "NULL argument");
  SD2D_NOT_MID_STEP(c, "sd2d_compresid_vjp");
  if (c->p.precision != SD2D_FP64 || c->vis || c->nmem > 1)
    return fail(c, SD2D_EUNSUPPORTED, "the adjoint covers the FP64 inviscid path");
  if (!c->adj) c->adj = new (std::nothrow) AdjState();
  AdjState *A = c->adj;
  if (!A) return fail(c, SD2D_ENOMEM, "host allocation failed");
  int r = adj_alloc(c, A, 0, false);
  if (r) return r;
  const size_t n = (size_t)c->ncell * 9 * c->N * c->N;
  const size_t np = (size_t)c->ntile * ADJ_NPART;
  const std::unique_ptr<double[]> part(new (std::nothrow) double[np]);
  if (!part) return fail(c, SD2D_ENOMEM, "host allocation failed");
  HIPCHK(c, to_device(c, c->stagef, rbar, n));
  if ((r = f2t(c, c->stagef, A->b[1]))) return r;
  // divB of the state as the stepping kernel forms it for the Powell source
  const double *q = c->q[c->cur];
  const unsigned long long *set = max_set(c, c->mset);
  StageArgs s = base_args(c);
  s.qin = q;
  s.mread = nullptr;
  s.gmax = reinterpret_cast<const double *>(set);   // (divB does not depend on c_h)
  s.divb = A->divb;
  HIPCHK(c, launch_stage(c, s, M_DIVB));
  AdjArgs a = adj_args(c);
  a.q = q;
  a.rbar = A->b[1];
  a.divb = A->divb;
  a.gm = set;
  a.qbar = A->b[0];
  if ((r = adj_launch(c, a))) return r;
  if (qbar) {
    if ((r = t2f(c, A->b[0], c->stagef))) return r;
    HIPCHK(c, to_host(c, qbar, c->stagef, n));
  }
  // The tiles' partial sums are added up here, 56 bytes a tile: a launch for the
  // sum and two to prepare it cost more than they save (7 x 5 cells, N = 3: 118 us
  // a pullback with them, 93 without; 97 x 163, N = 5: 2.05 ms either way).
  HIPCHK(c, hipMemcpyAsync(part.get(), A->part, np * sizeof(double), hipMemcpyDeviceToHost,
                           c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  double acc[ADJ_NPART] = {};
  for (int t = 0; t < c->ntile; ++t)
    for (int j = 0; j < ADJ_NPART; ++j) acc[j] += part[(size_t)t * ADJ_NPART + j];
  if (chbar) *chbar = acc[0];
  if (pbar) for (int j = 0; j < 6; ++j) pbar[j] = acc[1 + j];
  return SD2D_OK;
}

}  // extern "C"
