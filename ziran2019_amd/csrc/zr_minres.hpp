// zr_minres.hpp -- Minres::solve (Lib/Ziran/Math/Linear/Minres.h:69-178) on
// the device: the scalar recurrences (Lanczos alpha / beta, the Givens QR of
// the tridiagonal, the residual estimate and the termination test) run in
// every block of the node kernel that needs them, from the block partials of
// the kernel before, so the host only watches a mark.  Used by the ADMM global
// step and by the implicit Newton step.  Included by zr_engine.hip inside its
// anonymous namespace after zr_implicit.hpp.
//
// An iteration is four launches: operator apply, A z with the partials of
// alpha, the Lanczos step with those of beta, and the update.  One-block
// kernels for the two sums and the scalars took 2.2 to 4.7 us each, with the
// gaps to their neighbours a third of an iteration of 20k particles
// (frames: 40k ADMM 11.6 -> 9.6 ms, 20k implicit
// 9.2 -> 8.7).

// Device scalars (double) and flags (int32) of a MINRES solve.  The state
// that an iteration hands to the next is kept twice, in turn, so that the
// blocks of the update read one copy while block 0 writes the other.
enum {
  AD_LTOL = 0,     // local tolerance
  AD_ALPHA = 1,
  AD_STATE = 2,    // two of:
  AS_BETA = 0,     // beta_{k+1}
  AS_LT0 = 1,      // the last Givens-transformed right-hand side component
  AS_GK_C = 2, AS_GK_S = 3, AS_GKM1_C = 4, AS_GKM1_S = 5,
  AS_N = 6,
};
static_assert(AD_STATE + 2 * AS_N <= SC_N, "the solvers' scalars");
// whether the solve had ended before iteration k, at minres_flag(k)
enum { AI_DONE = 0, AI_ITERS = 1 };
constexpr int minres_flag(int k) { return AI_DONE + 2 * (k & 1); }
static_assert(minres_flag(1) < CI_N, "the solvers' flags");

__device__ __forceinline__ double* minres_state(double* sc, int k) { return sc + AD_STATE + AS_N * (k & 1); }

__device__ __forceinline__ void g2_rot(double c, double s, double v[2])
{
  const double t1 = v[0], t2 = v[1];
  v[0] = c * t1 - s * t2;
  v[1] = s * t1 + c * t2;
}

// the start (Minres.h:89-101) from the partials of z . q: beta_1 = |r0|_P on
// every thread and whether the solve ends there
__device__ __forceinline__ bool minres_start(const double* partial, uint32_t nb, double* sc, int32_t* ai, double tol,
                                             double rel, int max_it, double& beta)
{
  __shared__ double red[5];
  beta = sqrt(block_total256(partial, nb, red));
  const double lt = rel * beta < tol ? rel * beta : tol;
  const bool done = beta < lt || max_it <= 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double* st = minres_state(sc, 0);
    sc[AD_LTOL] = lt;
    st[AS_BETA] = beta;
    st[AS_LT0] = beta;
    st[AS_GK_C] = st[AS_GKM1_C] = 1.0;
    st[AS_GK_S] = st[AS_GKM1_S] = 0.0;
    ai[AI_ITERS] = 0;
    ai[minres_flag(0)] = ai[minres_flag(1)] = done ? 1 : 0;
  }
  return done;
}

// the sum alpha of iteration k on every thread
__device__ __forceinline__ double minres_alpha(const double* partial, uint32_t nb, double* sc)
{
  __shared__ double red[5];
  const double alpha = block_total256(partial, nb, red);
  if (blockIdx.x == 0 && threadIdx.x == 0) sc[AD_ALPHA] = alpha;
  return alpha;
}

// applyAllPreviousGivensRotationsAndDetermineNewGivens and the termination
// test of iteration k (Minres.h:131-178); block 0 records the state
struct MinresStep {
  double beta, gamma, delta, eps, tk;
};
__device__ __forceinline__ MinresStep minres_givens(const double* partial, uint32_t nb, double* sc, int32_t* ai, int k,
                                                    int max_it, SolveMark mark)
{
  __shared__ double red[5];
  const double v = block_total256(partial, nb, red);
  const double* st = minres_state(sc, k);
  MinresStep m;
  m.beta = sqrt(v > 0.0 ? v : 0.0);
  double ek[2] = { 0.0, st[AS_BETA] };
  g2_rot(st[AS_GKM1_C], st[AS_GKM1_S], ek);
  double dk[2] = { ek[1], sc[AD_ALPHA] };
  g2_rot(st[AS_GK_C], st[AS_GK_S], dk);
  double tv[2] = { dk[1], m.beta };
  double c = 1.0, s = 0.0;  // GivensRotation::compute (Givens.h:56-62)
  const double d = sqrt(tv[0] * tv[0] + tv[1] * tv[1]);
  if (d) {
    const double t = 1.0 / d;
    c = tv[0] * t;
    s = -tv[1] * t;
  }
  g2_rot(c, s, tv);
  double lt[2] = { st[AS_LT0], 0.0 };
  g2_rot(c, s, lt);
  m.eps = ek[0];
  m.delta = dk[0];
  m.gamma = tv[0];
  m.tk = lt[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double* nx = minres_state(sc, k + 1);
    nx[AS_BETA] = m.beta;
    nx[AS_LT0] = lt[1];
    nx[AS_GKM1_C] = st[AS_GK_C];
    nx[AS_GKM1_S] = st[AS_GK_S];
    nx[AS_GK_C] = c;
    nx[AS_GK_S] = s;
    const double res = lt[1] < 0.0 ? -lt[1] : lt[1];
    const bool done = res < sc[AD_LTOL] || k + 1 >= max_it;
    ai[AI_ITERS] = k + 1;
    if (done) ai[minres_flag(k + 1)] = 1;
    mark_solve(mark, k + 1, done);
  }
  return m;
}
// what the update of iteration k does past the end of a solve
__device__ __forceinline__ void minres_pass(int32_t* ai, int k, SolveMark mark)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ai[minres_flag(k + 1)] = 1;
    mark_solve(mark, ai[AI_ITERS], 1);
  }
}

// ---- the implicit Newton step's MINRES (BackwardEuler::computeStep with the
// reference's default linear solver, BackwardEuler.h:55-62,200-240): vectors
// in the operator's precision T (FP32 in the FP32-bulk form), inner products
// and scalars in FP64, the mass-lumped or Jacobi preconditioner ----

// start (Minres.h:69-101) with x = 0 as computeStep sets it: q = P(b - A 0) = b
// (the Newton residual is already projected), z = M^-1 q; q_k, m_k and m_{k-1}
// start at zero (Minres::reinitialize, :40-66); partials of z . q
template <class T>
__global__ __launch_bounds__(256) void k_imr_init(uint32_t nn, const double* __restrict__ gm, NodeVec3 b,
                                                  NodeVec<T> x, NodeVec<T> q, NodeVec<T> z, NodeVec<T> zero0,
                                                  NodeVec<T> zero1, NodeVec<T> zero2, NodeVec<T> pinv,
                                                  double* __restrict__ partial)
{
  double contrib = 0.0;
  for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < nn; k += gridDim.x * 256u) {
    const double m = gm[k];
    for (int d = 0; d < 3; ++d) {
      const T qv = (T)b(d, k);
      const T zv = m != 0.0 ? (pinv.p ? qv * pinv(d, k) : qv / (T)m) : (T)0;
      x(d, k) = (T)0;
      q(d, k) = qv;
      z(d, k) = zv;
      zero0(d, k) = (T)0;
      zero1(d, k) = (T)0;
      zero2(d, k) = (T)0;
      contrib += (double)qv * (double)zv;
    }
  }
  block_partial(contrib, partial);
}

// beta_1 from the start's partials; the start vectors divided by it
// (Minres.h:95-98)
template <class T>
__global__ __launch_bounds__(256) void k_imr_scale(uint32_t nn, const double* __restrict__ gm, NodeVec<T> q,
                                                   NodeVec<T> z, const double* __restrict__ partial, double* sc,
                                                   int32_t* ai, double tol, double rel, int max_it)
{
  double b;
  if (minres_start(partial, gridDim.x, sc, ai, tol, rel, max_it, b) || !(b > 0.0)) return;
  for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < nn; k += gridDim.x * 256u) {
    if (gm[k] == 0.0) continue;
    for (int d = 0; d < 3; ++d) {
      q(d, k) /= (T)b;
      z(d, k) /= (T)b;
    }
  }
}

// q -= alpha q_k; q -= beta_k q_{k-1}; z = M^-1 q; partials of z . q
// (Minres.h:123-130)
template <class T>
__global__ __launch_bounds__(256) void k_imr_lanczos(uint32_t nn, const double* __restrict__ gm, NodeVec<T> q,
                                                     NodeVec<T> qk, NodeVec<T> qkm1, NodeVec<T> z, NodeVec<T> pinv,
                                                     const double* __restrict__ apartial, double* sc,
                                                     const int32_t* ai, int it, double* partial)
{
  if (ai[minres_flag(it)]) return;
  const T alpha = (T)minres_alpha(apartial, gridDim.x, sc), beta = (T)minres_state(sc, it)[AS_BETA];
  double contrib = 0.0;
  for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < nn; k += gridDim.x * 256u) {
    const double m = gm[k];
    if (m == 0.0) continue;
    for (int d = 0; d < 3; ++d) {
      T v = q(d, k);
      v -= alpha * qk(d, k);
      v -= beta * qkm1(d, k);
      q(d, k) = v;
      const T zv = pinv.p ? v * pinv(d, k) : v / (T)m;
      z(d, k) = zv;
      contrib += (double)zv * (double)v;
    }
  }
  block_partial(contrib, partial);
}

// q, z divided by beta_{k+1}; m_k = (m_k - delta m_{k-1} - eps m_{k-2}) / gamma;
// x += t_k m_k (Minres.h:131-143)
template <class T>
__global__ __launch_bounds__(256) void k_imr_update(uint32_t nn, const double* __restrict__ gm, NodeVec<T> q,
                                                    NodeVec<T> z, NodeVec<T> mk, NodeVec<T> mkm1, NodeVec<T> mkm2,
                                                    NodeVec<T> x, const double* __restrict__ partial, double* sc,
                                                    int32_t* ai, int it, int max_it, SolveMark mark)
{
  if (ai[minres_flag(it)]) {
    minres_pass(ai, it, mark);
    return;
  }
  const MinresStep st = minres_givens(partial, gridDim.x, sc, ai, it, max_it, mark);
  const T gamma = (T)st.gamma, delta = (T)st.delta, eps = (T)st.eps, tk = (T)st.tk;
  for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < nn; k += gridDim.x * 256u) {
    if (gm[k] == 0.0) continue;
    for (int d = 0; d < 3; ++d) {
      if (st.beta > 0.0) {
        q(d, k) /= (T)st.beta;
        z(d, k) /= (T)st.beta;
      }
      const T m = (mk(d, k) - delta * mkm1(d, k) - eps * mkm2(d, k)) / gamma;
      mk(d, k) = m;
      x(d, k) += tk * m;
    }
  }
}
