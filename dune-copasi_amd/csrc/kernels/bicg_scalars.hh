// The BiCGSTAB scalars, their update after each reduction stage, and the
// arguments of a fused Krylov operator launch, as macros: the ahead-of-time
// kernels expand them, and the generated kernels (compiled at run time, which
// fuse the vector updates into the operator) get the same text as a string.
// DCG_DEV is the functions' qualifier, which the user of the text defines.
#pragma once

// Device-resident BiCGSTAB state shared by its kernels.
#define DCG_BICG_STRUCT                                          \
  struct BicgScalars {                                           \
    double rho, alpha, omega, beta, r0, rnorm, tol, abstol;      \
    int iter, maxit, done, half;                                 \
  };

// Arguments of one operator launch of a fused BiCGSTAB iteration.  mode 0:
// y = J a.  mode 1: p = a + beta (b - omega c) into d, y = J M^-1 p, partial
// y.w.  mode 2: s = a - alpha c, y = J M^-1 s, partials y.s, y.y, s.s.  Modes
// 1 and 2 first finish the previous launch's reduction: every workgroup of the
// leading launch sums the same partials (fin[j * fstride + i], i < nfin) in the
// same order and updates its copy of *in; its first workgroup stores it to
// *out, which the launches of further compartments and of the facet rows take
// as it is (in = out, nfin = 0).  part[j * pstride + off + workgroup] gets this launch's partials.
// jac: 0 no preconditioner, 1 a block per slot, 2 the diagonal (in dinv).
#define DCG_KRYLOV_OP_STRUCT                                     \
  struct KrylovOp {                                              \
    int mode, jac, nfin, fstride, pstride, off, lead, pad;       \
    const void *a, *b, *c;                                       \
    void *d, *y;                                                 \
    const void* w;                                               \
    const double* dinv;                                          \
    const BicgScalars* in;                                       \
    BicgScalars* out;                                            \
    const double* fin;                                           \
    double* part;                                                \
  };

// The same launch over the members of a batch: vectors by index, the scalars
// one per member (in[m], out[m]), frange[m] = member m's partials of the
// previous launch (null: none to finish) and range[m] of this one, whose work
// items are numbered from off.
#define DCG_BATCH_OP_STRUCT                                      \
  struct BatchOp {                                               \
    int mode, jac, fstride, pstride, off;                        \
    int a, b, c, d, y, w;                                        \
    const int2 *frange, *range;                                  \
    const BicgScalars* in;                                       \
    BicgScalars* out;                                            \
    const double* fin;                                           \
    double* part;                                                \
  };

// Updates the scalars after one reduction stage; v0/v1 are its reduced sums.
// 0: v0 = r.r at the start (rho = r.r since rh = r).  1: after v = A ph,
// alpha = rho / (rh.v).  2: after s, half-step convergence test.  3: after
// t = A sh, omega = (t.s)/(t.t).  4: after the x, r update, convergence and
// beta for the next iteration.
#define DCG_BICG_UPDATE                                                                  \
  DCG_DEV void bicg_update(BicgScalars* sc, int stage, double v0, double v1) { \
    switch (stage) {                                                                     \
      case 0: {                                                                          \
        sc->r0 = sqrt(v0);                                                               \
        sc->rnorm = sc->r0;                                                              \
        sc->rho = v0;                                                                    \
        sc->alpha = sc->omega = 1.0;                                                     \
        sc->beta = 0.0;                                                                  \
        sc->iter = 0;                                                                    \
        sc->half = 0;                                                                    \
        if (!(sc->r0 > 0.0)) sc->done = isfinite(sc->r0) ? 1 : 3;                        \
        if (sc->r0 <= sc->abstol) sc->done = 1;                                          \
        break;                                                                           \
      }                                                                                  \
      case 1: {                                                                          \
        if (v0 == 0.0 || !isfinite(v0)) {                                                \
          sc->done = isfinite(v0) ? 4 : 3;                                               \
          break;                                                                         \
        }                                                                                \
        sc->alpha = sc->rho / v0;                                                        \
        break;                                                                           \
      }                                                                                  \
      case 2: {                                                                          \
        const double ns = sqrt(v0);                                                      \
        sc->iter += 1;                                                                   \
        if (!isfinite(ns)) {                                                             \
          sc->done = 3;                                                                  \
          break;                                                                         \
        }                                                                                \
        if (ns <= sc->tol * sc->r0 || ns <= sc->abstol) {                                \
          sc->half = 1;                                                                  \
          sc->rnorm = ns;                                                                \
        }                                                                                \
        break;                                                                           \
      }                                                                                  \
      case 3: {                                                                          \
        if (sc->half) break;                                                             \
        sc->omega = v1 == 0.0 ? 0.0 : v0 / v1;                                           \
        break;                                                                           \
      }                                                                                  \
      case 4: {                                                                          \
        if (sc->half) {                                                                  \
          sc->done = 1;                                                                  \
          break;                                                                         \
        }                                                                                \
        const double nr = sqrt(v1);                                                      \
        sc->rnorm = nr;                                                                  \
        if (!isfinite(nr)) {                                                             \
          sc->done = 3;                                                                  \
          break;                                                                         \
        }                                                                                \
        if (nr <= sc->tol * sc->r0 || nr <= sc->abstol) {                                \
          sc->done = 1;                                                                  \
          break;                                                                         \
        }                                                                                \
        if (sc->omega == 0.0 || v0 == 0.0) {                                             \
          sc->done = 4;                                                                  \
          break;                                                                         \
        }                                                                                \
        sc->beta = (v0 / sc->rho) * (sc->alpha / sc->omega);                             \
        sc->rho = v0;                                                                    \
        if (sc->iter >= sc->maxit) sc->done = 2;                                         \
        break;                                                                           \
      }                                                                                  \
    }                                                                                    \
  }

// Sums over a workgroup of NT threads, the same in every thread (fixed order:
// lanes, then waves), and the previous launch's reduction: false when the
// solve is done.  NV: partial arrays; stage of the update (2 runs stages 2
// and 3 on the sums (s.s; t.s, t.t)).
#define DCG_KRYLOV_FINISH                                                                \
  template <int NT, int N>                                                               \
  DCG_DEV void group_sums(double (&v)[N], double* lds) {              \
    for (int i = 0; i < N; ++i)                                                          \
      for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o, 64);                  \
    __syncthreads();                                                                     \
    if ((threadIdx.x & 63) == 0)                                                         \
      for (int i = 0; i < N; ++i) lds[(threadIdx.x >> 6) * N + i] = v[i];                \
    __syncthreads();                                                                     \
    for (int i = 0; i < N; ++i) {                                                        \
      double s = 0.0;                                                                    \
      for (int w = 0; w < NT / 64; ++w) s += lds[w * N + i];                             \
      v[i] = s;                                                                          \
    }                                                                                    \
  }                                                                                      \
  template <int NT, int N>                                                               \
  DCG_DEV bool finish_stage(BicgScalars& sc, const BicgScalars* in, BicgScalars* out, bool lead, \
                                               const double* fin, int nfin, int fstride, int stage, double* lds) { \
    sc = *in;                                                                            \
    if (!sc.done && nfin > 0) {                                                          \
      double v[N];                                                                       \
      for (int j = 0; j < N; ++j) v[j] = 0.0;                                            \
      for (int i = threadIdx.x; i < nfin; i += NT)                                       \
        for (int j = 0; j < N; ++j) v[j] += fin[(size_t)j * fstride + i];                \
      group_sums<NT, N>(v, lds);                                                         \
      if (N == 3) {                                                                      \
        bicg_update(&sc, 2, v[N - 1], 0.0);                                              \
        if (!sc.done) bicg_update(&sc, 3, v[0], v[N > 1 ? 1 : 0]);                       \
      } else {                                                                           \
        bicg_update(&sc, stage, v[0], v[N > 1 ? 1 : 0]);                                 \
      }                                                                                  \
    }                                                                                    \
    if (lead && threadIdx.x == 0) *out = sc;                                             \
    return !sc.done;                                                                     \
  }
