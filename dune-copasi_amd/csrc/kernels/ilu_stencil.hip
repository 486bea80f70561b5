// Block ILU0 on 1D and 2D structured grids (3 x 3 vertex stencils, blocks of
// at most 2 species): the factorisation and both triangular solves as one
// workgroup each over the level schedule (a row's level is one more than the
// deepest row it depends on: n0 + 2 n1 levels on a 9-point stencil).
//
// What bounds them: the chain of levels.  A level is at most a few waves
// wide, so nothing but one CU can work on it and a level's own latency times
// the number of levels is the floor (385 levels per sweep on the 129^2 grid).
// So everything that does not belong to the chain is taken off it:
//   - the waves form groups of as many waves as a level is wide, and the
//     groups take the levels in turn.  While one group runs its level, the
//     others' loads for their next levels are in flight, so a level never
//     waits for memory (the streams lie in level order, consecutive lanes on
//     consecutive words, and are read once);
//   - results pass from level to level through a ring in LDS;
//   - the block's rows sit at places fixed by the stencil offset, so every
//     operand of the elimination is in a register with a compile-time index
//     and absent neighbours are zero blocks instead of branches;
//   - in the factorisation a row is spread over B lanes, one per column of
//     its blocks: each lane reads only its column of the operands from LDS
//     and takes the other column of its own blocks by lane exchange.
// Measured on the 129^2 grid with 2 species (385 levels of at most 65 rows):
// factorisation 3180 -> 324 us, both triangular solves 1000 -> 186 us against
// the table-driven sweeps of solver.hip, which stay for wider levels, larger
// blocks, 3D and unstructured patterns and rows with interface blocks.  Now a
// level is bound by its chain of LDS round trips (count, ring, result: 0.24 us
// in the solves at every size from 17^2 to 129^2) and in the factorisation by
// the ~300 FP64 instructions of a lane's row.
#include <hip/hip_runtime.h>

#include "common.hh"
#include "kernels.hh"

namespace dcopasi::k {

namespace {

constexpr int kIluBlock = 1024;             // 16 waves
constexpr int kIluWaves = kIluBlock / kWave;
constexpr int NP = kIluPlaces;              // neighbours below / above the diagonal
constexpr int NO = 2 * NP + 1;              // places of a row

// words (16 bytes) of a row in the solves' streams
template <int B>
constexpr int lower_words = (NP * B * B + 1) / 2;
template <int B>
constexpr int upper_words = ((NP + 1) * B * B + 1) / 2;

// The hand-over from level to level: a count of finished waves in LDS.  Level
// l may start when the waves of all earlier levels have finished, G per
// level.  A wave's LDS accesses take effect in its own order, so the count
// follows the wave's results; a level waits for earlier levels alone, so
// every wait ends.  (A barrier per level instead makes every level wait for
// the group that has just finished to issue its next loads: 0.45 against
// 0.24 us per level of the triangular solves on the 129^2 grid.)
__device__ __forceinline__ void wait_levels(const int* count, int want) {
  // uniform over the wave: every lane reads the same word
  while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < want) {
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
__device__ __forceinline__ void level_done(int* count, int lane) {
  asm volatile("" ::: "memory");  // the results' LDS stores are issued before the count's
  if (lane == 0) __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the value of the other lane of a pair (lane ^ 1), without LDS
__device__ __forceinline__ double pair_swap(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)u, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// the two columns of a block row from a lane's own column c and its partner's
template <int B>
__device__ __forceinline__ void both_columns(double own, int c, double (&row)[B]) {
  if constexpr (B == 1) {
    row[0] = own;
  } else {
    const double other = pair_swap(own);
    row[0] = c ? other : own;
    row[1] = c ? own : other;
  }
}

// inverse of a 1 x 1 or 2 x 2 block by Gauss-Jordan with partial pivoting
// (the steps of the row-by-row factorisation, with selects for the swaps)
template <int B>
__device__ __forceinline__ void invert(double (&a)[B][B], double (&inv)[B][B], bool on, int* __restrict__ status) {
  if constexpr (B == 1) {
    if (on && a[0][0] == 0.0) status[0] = 4;
    inv[0][0] = 1.0 / (a[0][0] == 0.0 ? 1.0 : a[0][0]);
  } else {
    const bool swap = fabs(a[1][0]) > fabs(a[0][0]);
    double p0 = swap ? a[1][0] : a[0][0], p1 = swap ? a[1][1] : a[0][1];
    const double q0 = swap ? a[0][0] : a[1][0];
    double q1 = swap ? a[0][1] : a[1][1];
    double i00 = swap ? 0.0 : 1.0, i01 = swap ? 1.0 : 0.0, i10 = swap ? 1.0 : 0.0, i11 = swap ? 0.0 : 1.0;
    if (p0 == 0.0) {
      if (on) status[0] = 4;
      p0 = 1.0;
    }
    const double d0 = 1.0 / p0;
    p1 *= d0;
    i00 *= d0;
    i01 *= d0;
    q1 -= q0 * p1;
    i10 -= q0 * i00;
    i11 -= q0 * i01;
    if (q1 == 0.0) {
      if (on) status[0] = 4;
      q1 = 1.0;
    }
    const double d1 = 1.0 / q1;
    i10 *= d1;
    i11 *= d1;
    i00 -= p1 * i10;
    i01 -= p1 * i11;
    inv[0][0] = i00;
    inv[0][1] = i01;
    inv[1][0] = i10;
    inv[1][1] = i11;
  }
}

// place of the stencil offset a + b (offsets o = (dx + 1) + 3 (dy + 1)), -1 outside
constexpr int add_offsets(int a, int b) {
  const int dx = a % 3 + b % 3 - 2, dy = a / 3 + b / 3 - 2;
  return dx < -1 || dx > 1 || dy < -1 || dy > 1 ? -1 : (dx + 1) + 3 * (dy + 1);
}

}  // namespace

// The matrix's blocks in the factorisation's order: entry (r, c) of place o
// of the row at position lr of a level of n rows that begins at position b0
// lies at [(b0 * NO + o * n) * B * B + (r * n + lr) * B + c].
template <int B>
__global__ void ilu_stencil_pack_k(int nrows, IluStencil t, const double* __restrict__ val,
                                   double* __restrict__ pack) {
  const long g = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (g >= (long)nrows * NO) return;
  const int q = (int)(g / NO), o = (int)(g % NO);
  const int4 f = t.frow[q];  // row, level's first position, level's rows, stencil mask
  const int lr = q - f.y, n = f.z;
  const bool has = (f.w >> o) & 1;
  const double* a = val + (size_t)(t.first[q] + (has ? __popc(f.w & ((1 << o) - 1)) : 0)) * (B * B);
  double* d = pack + ((size_t)f.y * NO + (size_t)o * n) * (B * B) + (size_t)lr * B;
#pragma unroll
  for (int r = 0; r < B; ++r)
#pragma unroll
    for (int c = 0; c < B; ++c) d[(size_t)r * n * B + c] = has ? a[r * B + c] : 0.0;
}

// Factorisation: L_ik <- A_ik U_kk^-1, A_ij -= L_ik U_kj for the blocks of
// the pattern, U_ii^-1.  The sums run in the order of the row-by-row kernel.
// G: waves per level.
extern __shared__ __align__(16) char ilu_stencil_lds[];
template <int B>
__global__ void __launch_bounds__(kIluBlock) ilu_stencil_factor_k(IluStencil t, int G,
                                                                  const double* __restrict__ pack,
                                                                  double* __restrict__ ls, double* __restrict__ us,
                                                                  int* __restrict__ status) {
  constexpr int BB = B * B, LW = lower_words<B>;
  const int RS = (t.ring * t.width + 1) * B;  // ring columns, the last slot is the zero row
  double* ring = reinterpret_cast<double*>(ilu_stencil_lds);          // [(NP + 1) * B][RS]
  int* sLev = reinterpret_cast<int*>(ring + (size_t)(NP + 1) * B * RS);  // nlo + 1, then the count
  int* count = sLev + t.nlo + 1;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int NG = kIluWaves / G, g = wave / G;
  const int item = (wave - g * G) * kWave + lane;
  const int lr = item / B, c = item % B;
  for (int l = tid; l <= t.nlo; l += kIluBlock) sLev[l] = t.lo_lev[l];
  for (int e = tid; e < (NP + 1) * B * B; e += kIluBlock) ring[(size_t)(e / B) * RS + RS - B + e % B] = 0.0;
  if (tid == 0) *count = 0;
  __syncthreads();
  if (g >= NG) return;  // waves beyond the last whole group
  // the row of the group's next level: its blocks' column c by place
  double A[NO][B];
  ushort4 src = make_ushort4(0, 0, 0, 0);
  int mask = 0;
  int2 up = make_int2(0, 0);
  bool has = false;
  auto fetch = [&](int l) {
    has = false;
    if (l >= t.nlo) return;
    const int b0 = sLev[l], n = sLev[l + 1] - b0;
    if (lr >= n) return;
    has = true;
    const double* p = pack + (size_t)b0 * NO * BB + item;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int r = 0; r < B; ++r) A[o][r] = p[(size_t)(o * B + r) * (n * B)];
    src = t.lo_src[b0 + lr];
    mask = t.frow[b0 + lr].w;
    up = t.upos[b0 + lr];
  };
  fetch(g);
  for (int l = g; l < t.nlo; l += NG) {
    double inv[B][B];
    // the neighbours of two and more levels ago are eliminated while the last
    // level runs (129^2 grid: 411 -> 324 us; the triangular solves, whose
    // level is a fifth of this work, gain nothing from a second wait)
    wait_levels(count, (l - 1) * G);
    if (has) {
      const int slot[NP] = {src.x, src.y, src.z, src.w};
#pragma unroll
      for (int a = 0; a < NP; ++a) {
        if (a == t.lo_early) {
          wait_levels(count, l * G);
          __builtin_amdgcn_s_setprio(3);
        }
        const double* k = ring + (size_t)slot[a] * B + c;  // the column of row k's blocks
        double L[B][B];
        {
          double d[B], tmp[B];
#pragma unroll
          for (int r = 0; r < B; ++r) d[r] = k[(size_t)r * RS];
#pragma unroll
          for (int r = 0; r < B; ++r) {
            double row[B];
            both_columns<B>(A[a][r], c, row);
            double sum = 0.0;
#pragma unroll
            for (int q = 0; q < B; ++q) sum += row[q] * d[q];
            tmp[r] = sum;
          }
#pragma unroll
          for (int r = 0; r < B; ++r) {
            A[a][r] = tmp[r];
            both_columns<B>(tmp[r], c, L[r]);
          }
        }
#pragma unroll
        for (int b = 0; b < NP; ++b) {
          const int m = add_offsets(a, NP + 1 + b);
          if (m < 0) continue;
          double u[B];
#pragma unroll
          for (int r = 0; r < B; ++r) u[r] = k[(size_t)((1 + b) * B + r) * RS];
          const bool keep = (mask >> m) & 1;
#pragma unroll
          for (int r = 0; r < B; ++r) {
            double sum = 0.0;
#pragma unroll
            for (int q = 0; q < B; ++q) sum += L[r][q] * u[q];
            A[m][r] -= keep ? sum : 0.0;
          }
        }
      }
      double d[B][B];
#pragma unroll
      for (int r = 0; r < B; ++r) both_columns<B>(A[NP][r], c, d[r]);
      invert<B>(d, inv, true, status);
      double* w = ring + (size_t)((l % t.ring) * t.width + lr) * B + c;
#pragma unroll
      for (int r = 0; r < B; ++r) w[(size_t)r * RS] = B == 1 ? inv[r][0] : c ? inv[r][B - 1] : inv[r][0];
#pragma unroll
      for (int b = 0; b < NP; ++b)
#pragma unroll
        for (int r = 0; r < B; ++r) w[(size_t)((1 + b) * B + r) * RS] = A[NP + 1 + b][r];
    }
    if (!__any(has)) wait_levels(count, l * G);  // a wave without rows counts in its turn too
    level_done(count, lane);
    __builtin_amdgcn_s_setprio(0);
    if (has) {
      // off the chain: the row into the solves' streams, the next loads
      const int b0 = sLev[l], n = sLev[l + 1] - b0;
      double* o = ls + 2 * ((size_t)b0 * LW + lr);
#pragma unroll
      for (int a = 0; a < NP; ++a)
#pragma unroll
        for (int r = 0; r < B; ++r) {
          const int q = a * BB + r * B + c;
          o[2 * (size_t)(q / 2) * n + q % 2] = A[a][r];
        }
      double* v = us + 2 * (size_t)up.x;
#pragma unroll
      for (int b = 0; b < NP; ++b)
#pragma unroll
        for (int r = 0; r < B; ++r) {
          const int q = b * BB + r * B + c;
          v[2 * (size_t)(q / 2) * up.y + q % 2] = A[NP + 1 + b][r];
        }
#pragma unroll
      for (int r = 0; r < B; ++r) {
        const int q = NP * BB + r * B + c;
        v[2 * (size_t)(q / 2) * up.y + q % 2] = B == 1 ? inv[r][0] : c ? inv[r][B - 1] : inv[r][0];
      }
    }
    fetch(l + NG);
  }
}

namespace {

// A lane's row of one level of a triangular solve.
template <int B, bool UPPER>
struct SolveRow {
  static constexpr int NW = UPPER ? upper_words<B> : lower_words<B>;
  int row = -1;
  ushort4 src;
  double2 w[NW];
  double in[B];
};

// One triangular solve: levels in turn over the wave groups, each group two
// of its levels ahead with the stream and one with the right-hand side.
template <int B, typename V, bool UPPER>
__device__ __forceinline__ void stencil_sweep(const IluStencil& t, int G, int nlev, const int* __restrict__ lev,
                                              const int* __restrict__ rows, const ushort4* __restrict__ src,
                                              const double2* __restrict__ stream, const V* __restrict__ rhs,
                                              V* __restrict__ res, V* ring, int* count, int* sLev) {
  constexpr int BB = B * B;
  using Row = SolveRow<B, UPPER>;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int NG = kIluWaves / G, g = wave / G;
  const int lr = (wave - g * G) * kWave + lane;
  for (int l = tid; l <= nlev; l += kIluBlock) sLev[l] = lev[l];
  if (tid < B) ring[(size_t)t.ring * t.width * B + tid] = V(0);  // the zero row
  if (tid == 0) *count = 0;
  __syncthreads();
  if (g >= NG) return;  // waves beyond the last whole group
  auto load = [&](int l, Row& R) {
    R.row = -1;
    if (l >= nlev) return;
    const int b0 = sLev[l], n = sLev[l + 1] - b0;
    if (lr >= n) return;
    R.row = rows[b0 + lr];
    R.src = src[b0 + lr];
    const double2* p = stream + (size_t)b0 * Row::NW + lr;
#pragma unroll
    for (int k = 0; k < Row::NW; ++k) R.w[k] = p[(size_t)k * n];
  };
  auto gather = [&](Row& R) {
    if (R.row >= 0)
#pragma unroll
      for (int a = 0; a < B; ++a) R.in[a] = (double)rhs[(size_t)R.row * B + a];
  };
  auto process = [&](int l, Row& R) {
    if (R.row < 0) return;
    const int slot[NP] = {R.src.x, R.src.y, R.src.z, R.src.w};
    double y[NP][B], sum[B];
#pragma unroll
    for (int k = 0; k < NP; ++k)
#pragma unroll
      for (int c = 0; c < B; ++c) y[k][c] = (double)ring[(size_t)slot[k] * B + c];
    auto word = [&](int q) { return q % 2 ? R.w[q / 2].y : R.w[q / 2].x; };
#pragma unroll
    for (int a = 0; a < B; ++a) sum[a] = R.in[a];
#pragma unroll
    for (int k = 0; k < NP; ++k)
#pragma unroll
      for (int a = 0; a < B; ++a)
#pragma unroll
        for (int c = 0; c < B; ++c) sum[a] -= word(k * BB + a * B + c) * y[k][c];
    V out[B];
#pragma unroll
    for (int a = 0; a < B; ++a) {
      if constexpr (UPPER) {
        double v = 0.0;
#pragma unroll
        for (int c = 0; c < B; ++c) v += word(NP * BB + a * B + c) * sum[c];
        out[a] = (V)v;
      } else {
        out[a] = (V)sum[a];
      }
    }
    V* o = ring + (size_t)((l % t.ring) * t.width + lr) * B;
#pragma unroll
    for (int a = 0; a < B; ++a) {
      o[a] = out[a];
      R.in[a] = (double)out[a];
    }
  };
  auto store = [&](Row& R) {
    if (R.row >= 0)
#pragma unroll
      for (int a = 0; a < B; ++a) res[(size_t)R.row * B + a] = (V)R.in[a];
  };
  Row r0, r1;
  load(g, r0);
  load(g + NG, r1);
  gather(r0);
  auto turn = [&](int l, Row& now, Row& next) {
    wait_levels(count, l * G);
    __builtin_amdgcn_s_setprio(3);
    process(l, now);
    level_done(count, lane);
    __builtin_amdgcn_s_setprio(0);
    store(now);
    gather(next);
    load(l + 2 * NG, now);
  };
  // two levels per pass, so that the two row buffers are fixed registers
  for (int l = g; l < nlev; l += 2 * NG) {
    turn(l, r0, r1);
    if (l + NG < nlev) turn(l + NG, r1, r0);
  }
}

}  // namespace

// out = U^-1 L^-1 in, tmp = L^-1 in.
template <int B, typename V>
__global__ void __launch_bounds__(kIluBlock) ilu_stencil_apply_k(IluStencil t, int G, const double* __restrict__ ls,
                                                                 const double* __restrict__ us,
                                                                 const V* __restrict__ in, V* __restrict__ tmp,
                                                                 V* __restrict__ out,
                                                                 const BicgScalars* __restrict__ sc) {
  if (sc && sc->done) return;
  V* ring = reinterpret_cast<V*>(ilu_stencil_lds);
  int* count = reinterpret_cast<int*>(ilu_stencil_lds + (((size_t)t.ring * t.width + 1) * B * sizeof(V) + 15) / 16 * 16);
  int* sLev = count + 1;
  stencil_sweep<B, V, false>(t, G, t.nlo, t.lo_lev, t.lo_rows, t.lo_src, reinterpret_cast<const double2*>(ls), in, tmp,
                             ring, count, sLev);
  __syncthreads();
  stencil_sweep<B, V, true>(t, G, t.nup, t.up_lev, t.up_rows, t.up_src, reinterpret_cast<const double2*>(us), tmp, out,
                            ring, count, sLev);
}

// ----------------------------------------------------------------- host side
int ilu_stencil_lower_words(int B) { return B == 1 ? lower_words<1> : lower_words<2>; }
int ilu_stencil_upper_words(int B) { return B == 1 ? upper_words<1> : upper_words<2>; }

size_t ilu_stencil_factor_lds(const IluStencil& t, int B) {
  return sizeof(double) * (NP + 1) * B * ((size_t)t.ring * t.width + 1) * B + sizeof(int) * ((size_t)t.nlo + 2);
}

static size_t apply_lds(const IluStencil& t, int B, size_t vbytes) {
  return (((size_t)t.ring * t.width + 1) * B * vbytes + 15) / 16 * 16 +
         sizeof(int) * ((size_t)(t.nlo > t.nup ? t.nlo : t.nup) + 2);
}

bool ilu_stencil_fits(const IluStencil& t, int B, size_t lds) {
  return B >= 1 && B <= 2 && t.width * B <= kIluBlock / 2 && t.ring * t.width < 65535 &&
         ilu_stencil_factor_lds(t, B) <= lds && apply_lds(t, B, sizeof(double)) <= lds;
}

template <int B>
static void factor_t(const IluStencil& t, const double* val, double* pack, double* ls, double* us, int* status,
                     hipStream_t s) {
  const long n = (long)t.nrows * NO;
  ilu_stencil_pack_k<B><<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, s>>>(t.nrows, t, val, pack);
  const size_t lds = ilu_stencil_factor_lds(t, B);
  static std::atomic<unsigned long long> raised{0};
  raise_lds(reinterpret_cast<const void*>(&ilu_stencil_factor_k<B>), lds, raised);
  const int G = (t.width * B + kWave - 1) / kWave;
  ilu_stencil_factor_k<B><<<1, kIluBlock, lds, s>>>(t, G, pack, ls, us, status);
}

void ilu_stencil_factor(int B, const IluStencil& t, const double* val, double* pack, double* ls, double* us,
                        int* status, hipStream_t s) {
  if (t.nrows <= 0) return;
  if (B == 1) factor_t<1>(t, val, pack, ls, us, status, s);
  else factor_t<2>(t, val, pack, ls, us, status, s);
}

template <int B, typename V>
static void apply_t(const IluStencil& t, const double* ls, const double* us, const V* in, V* tmp, V* out,
                    const BicgScalars* sc, hipStream_t s) {
  const size_t lds = apply_lds(t, B, sizeof(V));
  static std::atomic<unsigned long long> raised{0};
  raise_lds(reinterpret_cast<const void*>(&ilu_stencil_apply_k<B, V>), lds, raised);
  const int G = (t.width + kWave - 1) / kWave;
  ilu_stencil_apply_k<B, V><<<1, kIluBlock, lds, s>>>(t, G, ls, us, in, tmp, out, sc);
}

template <typename V>
void ilu_stencil_apply(int B, const IluStencil& t, const double* ls, const double* us, const V* in, V* tmp, V* out,
                       const BicgScalars* sc, hipStream_t s) {
  if (t.nrows <= 0) return;
  if (B == 1) apply_t<1, V>(t, ls, us, in, tmp, out, sc, s);
  else apply_t<2, V>(t, ls, us, in, tmp, out, sc, s);
}
template void ilu_stencil_apply<double>(int, const IluStencil&, const double*, const double*, const double*, double*,
                                        double*, const BicgScalars*, hipStream_t);
template void ilu_stencil_apply<float>(int, const IluStencil&, const double*, const double*, const float*, float*,
                                       float*, const BicgScalars*, hipStream_t);

}  // namespace dcopasi::k
