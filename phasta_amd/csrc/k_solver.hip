// Linear-solver kernels on gfx950 for the block-diagonal-preconditioned
// GMRES of SolGMRs (solgmr.f:368-744): the nodal work between assembly and
// Krylov loop (bc3res.f, bc3bdg.f, tnanq.f), 5x5 block LU of BDiag (i3lu.f),
// two-sided block scaling of the matrix (spsi3pre.f), the block-CSR matvec
// with the periodic gather (sparseap.f), the periodic fold (bc3per.f),
// Krylov-vector kernels with deterministic wavefront/grid reductions
// (sumgat, mpitools.f:104-138) and the itrCorrect/itrBC state update
// (itrPC.f:128-148, itrbc.f).
//
// Matrix layout ("slots"): rows are grouped by 64, one wavefront per group.
// Group g owns slots [grp_slot[g], grp_slot[g+1]); slot s holds one 5x5 block
// for every row of the group, entry e (reference order f + 5 g) of row r at
// vals[(s*25 + e)*64 + r].  Each matrix load of a wavefront is therefore one
// contiguous 512-byte (FP64) or 256-byte (FP32) segment.  Rows shorter than
// the group's slot count are padded with zero blocks.
#include <type_traits>

#include "phg_internal.h"

namespace {

constexpr int kRedThreads = 256;

// ---------------- block LU (i3lu.f) ----------------
// 25 planes, D[(i + 5 j) * n + node] = Diag(node, i+1, j+1)
// Doolittle: unit-lower L, upper U with its diagonal stored inverted.  As in
// the reference (i3lu.f:82-97) the entry U(4,5) is never reduced: row 4 of U
// only gets its diagonal, so (4,5) keeps the raw BDiag value and the
// forward/backward sweeps use it as such.
__device__ inline void lu_factor(double a[5][5]) {
#pragma unroll
  for (int p = 0; p < 5; ++p) {
#pragma unroll
    for (int j = p; j < 5; ++j) {
      if (p == 3 && j == 4) continue;
      double s = a[p][j];
#pragma unroll
      for (int m = 0; m < p; ++m) s -= a[p][m] * a[m][j];
      a[p][j] = s;
    }
    a[p][p] = 1.0 / a[p][p];
#pragma unroll
    for (int i = p + 1; i < 5; ++i) {
      double s = a[i][p];
#pragma unroll
      for (int m = 0; m < p; ++m) s -= a[i][m] * a[m][p];
      a[i][p] = a[p][p] * s;
    }
  }
}

__device__ inline void lu_solve_lower(const double a[5][5], double v[5]) {
#pragma unroll
  for (int i = 1; i < 5; ++i) {
    double s = v[i];
#pragma unroll
    for (int m = 0; m < i; ++m) s -= a[i][m] * v[m];
    v[i] = s;
  }
}

__global__ void k_lu_fact(double* D, long long n) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double a[5][5];
#pragma unroll
  for (int j = 0; j < 5; ++j)
#pragma unroll
    for (int i = 0; i < 5; ++i) a[i][j] = D[(i + 5 * j) * n + k];
  lu_factor(a);
#pragma unroll
  for (int j = 0; j < 5; ++j)
#pragma unroll
    for (int i = 0; i < 5; ++i) D[(i + 5 * j) * n + k] = a[i][j];
}

__global__ void k_lu_forward(const double* D, double* r, long long n) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double v[5], a[5][5];
#pragma unroll
  for (int i = 0; i < 5; ++i) v[i] = r[i * n + k];
#pragma unroll
  for (int i = 1; i < 5; ++i)
#pragma unroll
    for (int m = 0; m < i; ++m) a[i][m] = D[(i + 5 * m) * n + k];
  lu_solve_lower(a, v);
#pragma unroll
  for (int i = 1; i < 5; ++i) r[i * n + k] = v[i];
}

__global__ void k_lu_backward(const double* D, double* r, long long n) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double v[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) v[i] = r[i * n + k];
#pragma unroll
  for (int i = 4; i >= 0; --i) {
    double s = v[i];
#pragma unroll
    for (int m = 4; m > i; --m) s -= v[m] * D[(i + 5 * m) * n + k];
    v[i] = D[(i + 5 * i) * n + k] * s;
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) r[i * n + k] = v[i];
}

// i3LU 'product' (i3lu.f:150-167): r <- U r with U's diagonal stored
// inverted (so r_i / D_ii), rows in ascending order (each row reads the
// entries below it before they change)
__global__ void k_lu_product(const double* D, double* r, long long n) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double v[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) v[i] = r[i * n + k];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    double s = v[i] / D[(i + 5 * i) * n + k];
#pragma unroll
    for (int m = i + 1; m < 5; ++m) s += v[m] * D[(i + 5 * m) * n + k];
    v[i] = s;
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) r[i * n + k] = v[i];
}

// yshuffle (shuffle.f:1-30) from src into dst: new2old (u,v,w,p,T) ->
// (p,u,v,w,T), else back
__global__ void k_yshuffle(const double* src, double* dst, long long n, int new2old) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double v[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) v[i] = src[i * n + k];
  if (new2old) {
    dst[k] = v[3];
    dst[n + k] = v[0];
    dst[2 * n + k] = v[1];
    dst[3 * n + k] = v[2];
  } else {
    dst[k] = v[1];
    dst[n + k] = v[2];
    dst[2 * n + k] = v[3];
    dst[3 * n + k] = v[0];
  }
  dst[4 * n + k] = v[4];
}

// ---------------- two-sided block scaling (spsi3pre.f) ----------------
// lhsK(i,j) <- L_i^{-1} lhsK(i,j) U_j^{-1} with the factors of BDiag.  Reads
// the assembled blocks (reference order, one padded record per block) and writes
// the 64-row interleaved matvec layout.
// One workgroup of kPreWaves wavefronts per 64-row group; wavefront w takes
// the group's slots w, w + kPreWaves, ... (more independent loads in flight
// than one wavefront walking all slots of its group).
// A lane's record loaded by the lane itself, 16 bytes at a time from 64 places,
// kept the texture addresser 87 % busy; so an octet of lanes loads its records
// together, 128 bytes per load straight into LDS (load i the lines of the
// octet's lane i, piece p at place 64 i + 8 octet + (p ^ i), whose reads are
// free of bank conflicts), a slot ahead of the arithmetic: 1.53 -> 1.36 ms in double
// at 100^3 hexes (4.6 TB/s), 1.77 -> 1.66 in float at 128^3 (4.2).
constexpr int kPreWaves = 4;

template <typename TI, typename TO>
__global__ void __launch_bounds__(kPreWaves * kGroup) k_spsi3pre(
    const TI* __restrict__ aos, TO* __restrict__ vals, const int* __restrict__ s2c,
    const int* __restrict__ scol, const long long* __restrict__ grp_slot,
    const int* __restrict__ rowmap, const double* __restrict__ D, long long n) {
  constexpr int kPieces = aos_stride<TI>() * (int)sizeof(TI) / 16;  // of a record: 7 or 13
  constexpr int kLines = (kPieces + 7) / 8;
  constexpr int kWave = kLines * 512 + 16;  // pieces of LDS: the lines, the lanes' records
  static_assert(kWave % 8 == 0, "a wavefront's lines begin at a multiple of 128 bytes");
  __shared__ LdsPieces<kPreWaves * kWave> lds_all;
  typedef __attribute__((address_space(3))) phg_i4* lp;
  typedef const __attribute__((address_space(1))) void* gp;
  const long long g = blockIdx.x;
  const int w = threadIdx.x / kGroup, r = threadIdx.x % kGroup;
  const lp lds = (lp)lds_all.p + w * kWave;
  const unsigned base = (unsigned)(size_t)lds;
  const unsigned at = base + 16 * (64 * (r & 7) + (r & 56) + (r & 7));
  const int row = max(rowmap[g * kGroup + r], 0);  // (a lane without a row has only padding)
  double lo[5][5];
#pragma unroll
  for (int i = 1; i < 5; ++i)
#pragma unroll
    for (int m = 0; m < i; ++m) lo[i][m] = D[(i + 5 * m) * n + row];
  // starts the loads of the lanes' records k (padding: record 0)
  auto start = [&](int k) {
    reinterpret_cast<__attribute__((address_space(3))) int*>(lds + kLines * 512)[r] = max(k, 0);
    const unsigned c = base + 16 * kLines * 512 + 4 * (r & 56);
    const phg_i4 k0 = lds_i4(c), k1 = lds_i4(c + 16);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const phg_i4* rec = reinterpret_cast<const phg_i4*>(aos) +
                          (size_t)kPieces * (unsigned)(i < 4 ? k0[i & 3] : k1[i & 3]);
#pragma unroll
      for (int h = 0; h < kLines; ++h)
        __builtin_amdgcn_global_load_lds((gp)(rec + min(8 * h + ((r & 7) ^ i), kPieces - 1)),
                                         lds + 512 * h + 64 * i, 16, 0, 0);
    }
  };
  const long long s1 = grp_slot[g + 1];
  long long s = grp_slot[g] + w;
  if (s >= s1) return;
  int k = s2c[s * kGroup + r], j = scol[s * kGroup + r];
  start(k);
  for (; s < s1; s += kPreWaves) {
    const bool more = s + kPreWaves < s1;
    const int kn = more ? s2c[(s + kPreWaves) * kGroup + r] : -1;
    const int jn = more ? scol[(s + kPreWaves) * kGroup + r] : 0;
    double up[5][5];
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int m = 0; m <= c; ++m) up[m][c] = k < 0 ? 0.0 : D[(m + 5 * c) * n + j];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    double a[4 * 4 * 16 / sizeof(TI)];
#pragma unroll
    for (int u = 0; u < (kPieces + 3) / 4; ++u) {
      unsigned from[4];
      phg_i4 x[4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        from[t] = (at ^ (16 * ((4 * u + t) & 7))) + 16 * 512 * ((4 * u + t) >> 3);
      lds_i4(from, x);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (sizeof(TI) == 4) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int v = x[t][q];
            a[16 * u + 4 * t + q] = __builtin_bit_cast(float, v);
          }
        } else {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const unsigned l = (unsigned)x[t][2 * q];
            const long long v = ((long long)x[t][2 * q + 1] << 32) | l;
            a[8 * u + 2 * t + q] = __builtin_bit_cast(double, v);
          }
        }
      }
    }
    if (more) start(kn);
    const int here = k;
    k = kn;
    j = jn;
    if (here < 0) continue;  // padding stays zero
    double b[5][5];
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int f = 0; f < 5; ++f) b[f][c] = a[f + 5 * c];
    // left: L_i^{-1} on every column
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int f = 1; f < 5; ++f) {
        double acc = b[f][c];
#pragma unroll
        for (int m = 0; m < f; ++m) acc -= lo[f][m] * b[m][c];
        b[f][c] = acc;
      }
    // right: U_j^{-1} on every row (columns in order)
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        double acc = b[f][c];
#pragma unroll
        for (int m = 0; m < c; ++m) acc -= up[m][c] * b[f][m];
        b[f][c] = up[c][c] * acc;
      }
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int f = 0; f < 5; ++f) a[f + 5 * c] = b[f][c];
    store_slot(vals + s * (25 * kGroup), r, a);
  }
}

// ---------------- block-CSR matvec (sparseap.f) ----------------
// q = K p(iper(:)); one lane per row of a 64-row group in each wavefront.
// T: stored value type; Acc: type of the products and row sums.  The mixed
// path stores float values and sums rows in double: float row sums of the
// scaled system lose digits to cancellation (on the 16^3 box the refinement
// loop then needed 12 instead of 10 Krylov iterations), while the kernel is
// bound by the matrix bytes, which float storage halves either way.
// One workgroup of W wavefronts per 64-row group: wavefront w takes the group's
// slots w, w + W, ..., so the wavefronts of a workgroup stream adjacent slots
// together and each runs a short loop; the partial row sums are added in
// wavefront order through LDS (fixed order, deterministic), a component per
// wavefront.  With at most a group per CU the loop's latency is the product's
// time, and W = 16 leaves one or two slots to each wavefront; above, the slots
// of a workgroup in flight should be some 13 to 25 KB.  us per product for W = 4
// | 8 | 16, float and double: 16^3 hexes (77 groups) 7.1 | 6.1 | 5.6 and 8.7 | 7.3 |
// 6.9; 24^3 (245) 7.9 | 7.1 | 6.8 and 10.9 | 9.7 | 9.6; 28^3 (382) 10.3 | 9.9 | 11.6
// and 15.5 | 15.6 | 16.4; 64^3 81.0 | 82.8 | 98.0 and 142.3 | 138.2 | 151.6; 128^3 644
// | 655 | 768 and 1138 | 1101 | 1209.
// The grid is a multiple of 8: consecutive workgroups go to different XCDs
// (round robin), so workgroup b takes group (b % 8) * per + b / 8 and each
// XCD sweeps one contiguous eighth of the rows, whose column neighbours
// (rows +-1, +-(N+1), +-(N+1)^2 on the box) then stay in that XCD's L2.
template <typename T>
constexpr int kSpmvWaves = sizeof(T) == 8 ? 8 : 4;
constexpr int kSpmvWavesFew = 16;
constexpr long long kSpmvFew = 256;  // groups: one per CU

// rowmap: row of each (group, lane), -1 padding.  fam: per (group, lane) the
// number of periodic slaves whose rows follow the lane's (a master), kFamSlave
// for a slave's row, 0 otherwise.  With fold set the epilogue applies bc3per:
// a master's sum takes its slaves' sums in ascending order from LDS and the
// slaves get zero, as k_fold_vec does in a launch of its own (5 to 14 us per
// product, as long as the whole product up to 16^3).
// gate (nullable): the product is skipped when *gate is set (a Krylov
// iteration enqueued before the host knew that the last one had converged).
template <typename T, typename Acc, int W>
__global__ void __launch_bounds__(W * kGroup) k_spmv(
    const T* __restrict__ vals, const int* __restrict__ scolp,
    const long long* __restrict__ grp_slot, const int* __restrict__ rowmap,
    const uint8_t* __restrict__ fam, const double* __restrict__ p, double* __restrict__ q,
    long long n, long long ngroups, int fold, const int* gate, long long* t0) {
  if (gate && *gate) return;
  if (t0 && blockIdx.x == 0 && threadIdx.x == 0) *t0 = wall_clock64();
  __shared__ Acc part[W][5][kGroup];
  const long long per = (gridDim.x + 7) / 8;
  const long long g = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (g >= ngroups) return;  // whole workgroup
  const int w = threadIdx.x / kGroup, r = threadIdx.x % kGroup;
  const long long s0 = grp_slot[g] + w, s1 = grp_slot[g + 1];
  const long long row = rowmap[g * kGroup + r];
  const int nf = fold ? fam[g * kGroup + r] : 0;
  Acc t[5] = {0, 0, 0, 0, 0};
  // software pipeline: the gathers of p for the next slot and the column
  // index of the one after are issued before the block of this slot is
  // consumed (padding lanes read column 0 and zero blocks)
  Acc pc[5] = {0, 0, 0, 0, 0};
  if (s0 < s1) {
    const long long j0 = scolp[s0 * kGroup + r];
#pragma unroll
    for (int f = 0; f < 5; ++f) pc[f] = (Acc)p[j0 + f * n];
  }
  long long jn = s0 + W < s1 ? scolp[(s0 + W) * kGroup + r] : 0;
  for (long long s = s0; s < s1; s += W) {
    Acc pn[5] = {0, 0, 0, 0, 0};
    if (s + W < s1) {
#pragma unroll
      for (int f = 0; f < 5; ++f) pn[f] = (Acc)p[jn + f * n];
      if (s + 2 * W < s1) jn = scolp[(s + 2 * W) * kGroup + r];
    }
    Acc a[25];
    load_slot(vals + s * (25 * kGroup), r, a);
#pragma unroll
    for (int i = 0; i < 5; ++i)
      t[i] += a[i] * pc[0] + a[5 + i] * pc[1] + a[10 + i] * pc[2] + a[15 + i] * pc[3] +
              a[20 + i] * pc[4];
#pragma unroll
    for (int f = 0; f < 5; ++f) pc[f] = pn[f];
  }
#pragma unroll
  for (int f = 0; f < 5; ++f) part[w][f][r] = t[f];
  __syncthreads();
  if (row < 0) return;
  auto rowsum = [&](int f, int rr) {
    Acc v = part[0][f][rr];
#pragma unroll
    for (int k = 1; k < W; ++k) v += part[k][f][rr];
    return (double)v;
  };
  for (int f = w; f < 5; f += W) {
    double v = nf == kFamSlave ? 0.0 : rowsum(f, r);
    if (nf > 0 && nf < kFamSlave)
      for (int k = 1; k <= nf; ++k) v += rowsum(f, r + k);
    q[row + f * n] = v;
  }
}

// Transpose matvec without the periodic maps: q_j = sum_i B_ij^T x_i over
// the blocks of column j, B_ij read at the slot tslot of (i, j); scol gives
// the raw columns i of row j (the graph is structurally symmetric).
template <typename T>
__global__ void __launch_bounds__(256) k_spmv_t(const T* __restrict__ vals, const int* __restrict__ scol,
                                                const uint32_t* __restrict__ tslot,
                                                const long long* __restrict__ grp_slot,
                                                const int* __restrict__ rowmap,
                                                const double* __restrict__ x, double* __restrict__ q,
                                                long long n, long long ngroups) {
  const long long at = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const long long g = at / kGroup;
  const int r = (int)(at % kGroup);
  if (g >= ngroups) return;
  const long long row = rowmap[at];
  if (row < 0) return;
  double t[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (long long s = grp_slot[g]; s < grp_slot[g + 1]; ++s) {
    const long long i = scol[s * kGroup + r];
    const uint32_t ts = tslot[s * kGroup + r];
    const T* blk = vals + (size_t)(ts >> 6) * (25 * kGroup);
    const int tr = (int)(ts & 63);
    double xi[5];
#pragma unroll
    for (int f = 0; f < 5; ++f) xi[f] = x[i + f * n];
#pragma unroll
    for (int gg = 0; gg < 5; ++gg) {
      double a = 0.0;
#pragma unroll
      for (int f = 0; f < 5; ++f) a += (double)blk[slot_pos<T>(f + 5 * gg, tr)] * xi[f];
      t[gg] += a;
    }
  }
#pragma unroll
  for (int f = 0; f < 5; ++f) q[row + f * n] = t[f];
}

// slaves take their master's value (the transpose of the periodic fold)
__global__ void k_per_copy_vec(double* v, const int* master, const int* ptr, const int* slave,
                               int nfold, long long n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nfold) return;
  const long long m = master[i];
  for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
    const long long s = slave[k];
#pragma unroll
    for (int f = 0; f < 5; ++f) v[s + f * n] = v[m + f * n];
  }
}

// r = b - q (true residual of the refinement loop)
__global__ void k_sub(double* r, const double* b, const double* q, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    r[i] = b[i] - q[i];
}

// plain copy, 16 B per lane (calibration of the memory counters)
__global__ void k_copy(double2* __restrict__ dst, const double2* __restrict__ src, long long n2) {
  // one 16-byte element per lane, no loop: the fastest plain copy measured
  // on MI355X (6.2 TB/s for 859 MB; grid-stride loops reached 4.6-5.2)
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n2) dst[i] = src[i];
}

// padded assembled blocks -> lhsK(25,nnz) (double) and back
template <typename T>
__global__ void k_aos_to_ref(const T* __restrict__ aos, double* __restrict__ ref, long long nnz) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= 25 * nnz) return;
  const long long k = i / 25;
  ref[i] = (double)aos[(size_t)aos_stride<T>() * k + (i - 25 * k)];
}
__global__ void k_ref_to_aos(const double* __restrict__ ref, double* __restrict__ aos,
                             long long nnz) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= (long long)aos_stride<double>() * nnz) return;
  const long long k = i / aos_stride<double>(), e = i - (long long)aos_stride<double>() * k;
  aos[i] = e < 25 ? ref[25 * k + e] : 0.0;
}


// bc3per: master += slaves (ascending), slaves zeroed; one lane per master
// and plane
__global__ void k_fold_vec(double* v, const int* master, const int* ptr, const int* slave,
                           int nfold, long long n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nfold) return;
  double* p = v + (size_t)blockIdx.y * n;
  const long long m = master[i];
  double s = p[m];
  for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
    s += p[slave[k]];
    p[slave[k]] = 0.0;
  }
  p[m] = s;
}

// ---------------- deterministic reductions ----------------
// A reduction writes one partial per workgroup (sums of its wavefronts, added
// in order); the partials are added in a fixed order, by k_finish for a single
// inner product (k_dot), or by the workgroup that arrives last for the sums
// inside k_gs_dots, k_gs_update, k_nodes and k_product_nodes.  The only atomic
// is the arrival count (arrive_last): results do not depend on timing.
//
// Wavefront sum on the vector ALU (row shifts, then the two row broadcasts:
// no LDS traffic), the same in every lane.
template <int kCtrl, int kRows>
__device__ inline double dpp_move(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, kCtrl, kRows, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, kRows, 0xf, false);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// v of one lane (a uniform index) in every lane
__device__ inline double from_lane(double v, int lane) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double wave_sum(double v) {
  v += dpp_move<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of each row of
  v += dpp_move<0x112, 0xf>(v);  // 16 holds the row's sum
  v += dpp_move<0x114, 0xf>(v);
  v += dpp_move<0x118, 0xf>(v);
  v += dpp_move<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v += dpp_move<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  return from_lane(v, 63);
}

__device__ inline void block_partial(double v, double* part) {
  __shared__ double ws[kRedThreads / 64];
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) ws[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kRedThreads / 64; ++w) s += ws[w];
    part[blockIdx.x] = s;
  }
}

// *out = the sum of np partials, in a fixed order by one workgroup
__global__ void __launch_bounds__(kRedThreads) k_finish(const double* part, int np, double* out) {
  double s = 0.0;
  for (int b = threadIdx.x; b < np; b += blockDim.x) s += part[b];
  block_partial(s, out);
}

// Reductions take one pass of kUnroll independent, coalesced loads per
// thread (launch_dot's grid), so every load of a thread is in flight
// at once; a grid-stride tail covers vectors larger than the grid.
constexpr int kUnroll = 8;

__global__ void __launch_bounds__(kRedThreads) k_dot(const double* a, const double* b, long long n,
                                                     double* part) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  double v[kUnroll];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) v[u] = 0.0;
  for (; i + (kUnroll - 1) * stride < n; i += kUnroll * stride) {
    double x[kUnroll], y[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      x[u] = a[i + u * stride];
      y[u] = b[i + u * stride];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] += x[u] * y[u];
  }
  for (; i < n; i += stride) v[0] += a[i] * b[i];
  double t = 0.0;
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) t += v[u];
  block_partial(t, part);
}

// ---------------- Gram-Schmidt and the Hessenberg recurrence ----------------
// One Krylov iteration after its product w = K w_i (solgmr.f:598-669), in two
// launches and without the host: k_gs_dots, k_gs_update.
//
// Basis vectors stay unnormalised, u_j = w_j / n_j; the norms n_j are scalars
// of GmDev, so no pass over memory only divides by a norm.
//
// The orthogonalisation is the modified Gram-Schmidt of the reference with its
// inner products taken in one pass: with d_k = (u_k, w) of the incoming w, MGS
// subtracts h_k u_k with
//     h_1 = d_1,  h_k = d_k - sum_{j<k} (u_k, u_j) h_j
// (each h_k is the product of u_k with w less the earlier directions), so one
// pass over the basis forms every d_k and the new row (u_i, u_j) of the
// products of the basis, a triangular substitution of at most 60 rows gives
// the h_k, and a second pass subtracts.  Two reads of the basis per iteration
// against MGS's i + 1 dependent steps of two reads and a write each; bound by
// those reads from 100^3 on (128^3: 6 TB/s), by the launches below 32^3.
// Per iteration with the norm, the scaling and the Hessenberg column, 12
// vectors: 41 us at 64^3 (FP64; one launch per MGS step 68 us), 9 us at 4^3
// (40 us and a wait for the host).
//
// Reductions: a workgroup writes its partial sums, the workgroup that arrives
// last adds them in index order (the value does not depend on which one that
// is) and does the scalar work of the step: the coefficients (k_gs_dots), or
// the norm, the Givens rotations, the convergence test, at the end of a cycle
// the back substitution, and the iteration's result to the host
// (k_gs_update).  The partials cross the XCDs' L2 caches: they are written
// and read with agent-scope accesses, and a wait for the writes' completion
// stands before the arrival count.
__device__ inline void part_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double part_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// true in every thread of the workgroup that arrives last; its partial sums
// have to be stored before.  The counter is zero again afterwards.
__device__ inline bool arrive_last(unsigned* cnt) {
  __shared__ int last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned at =
        __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = at == gridDim.x - 1;
    if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return last != 0;
}

// Workgroups of both kernels: 16 wavefronts, at most kGsBlocks of them (two
// per CU), so that the last one has at most 8 partials per lane and sum to
// add, all in flight together.  Each agent-scope read goes to memory: with
// 1024 workgroups of 4 wavefronts that read theirs one after the other the
// tail took most of k_gs_dots at 64^3 (41 us at nv = 8).
constexpr int kGsThreads = 1024;
constexpr int kGsBlocks = 512;

// sum of np <= kGsBlocks partials by one wavefront, in a fixed order
__device__ inline double wave_sum_partials(const double* part, int np) {
  const int lane = threadIdx.x & 63;
  double v[kGsBlocks / 64];
#pragma unroll
  for (int u = 0; u < kGsBlocks / 64; ++u)
    v[u] = lane + 64 * u < np ? part_load(part + lane + 64 * u) : 0.0;
  double s = 0.0;
#pragma unroll
  for (int u = 0; u < kGsBlocks / 64; ++u) s += v[u];
  return wave_sum(s);
}

struct GsArgs {
  double* w;             // the product, then the new basis vector
  const double* basis;   // w_0 .. w_{nv-1}
  long long n, kstr;     // length, stride between basis vectors (even)
  int nv, K, minIters;   // nv: the iteration number, 1..K
  int unit;              // w is the product of u_i, not of w_i
  int clocked;           // the product's time is GmDev::t0 to the dots' start; else 0
  double unorm, epsnrm;  // of the cycle
  double n0;             // norm of the start vector as stored
  double* part;          // 2 nv channels of `chan` partials
  long long chan;
  GmDev* gm;
  GmHost* host;          // the iteration's slot
  unsigned seq;          // the iteration's token for the host
};

// pairs of elements per lane and pass
constexpr int kGsU = 2;

// d_k = (w_k, w) and (w_k, w_i), raw, for the nv basis vectors.  Wavefront
// v + 4 s of a workgroup takes the vectors v, v + 4, ... on the s-th quarter
// of the workgroup's elements, so each holds at most kT pairs of sums (kT =
// ceil(nv / 4)); w and w_i are read by four wavefronts together and come from
// L1 for three of them.
template <int kT>
__global__ void __launch_bounds__(kGsThreads) k_gs_dots(GsArgs A) {
  GmDev& gm = *A.gm;
  if (A.nv > 1 && gm.done) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    gm.t1 = wall_clock64();
    if (!A.clocked) gm.t0 = gm.t1;
  }
  __shared__ double red[4][2 * kGmMax], D[2 * kGmMax], nr[kGmMax];
  __shared__ double G[kGmMax * (kGmMax - 1) / 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wv = wave & 3, quarter = wave >> 2;
  const int nv = A.nv;
  const long long np2 = (A.n + 1) / 2;  // pairs; the last may hold one element
  const phg_d2* w2 = reinterpret_cast<const phg_d2*>(A.w);
  const phg_d2* u2 = reinterpret_cast<const phg_d2*>(A.basis + (size_t)(nv - 1) * A.kstr);
  const phg_d2* b2[kT];
#pragma unroll
  for (int t = 0; t < kT; ++t) {
    const int j = wv + 4 * t;
    b2[t] = reinterpret_cast<const phg_d2*>(A.basis + (size_t)(j < nv ? j : nv - 1) * A.kstr);
  }
  double a1[kT], a2[kT];
#pragma unroll
  for (int t = 0; t < kT; ++t) a1[t] = a2[t] = 0.0;
  const long long step = gridDim.x * (256LL * kGsU);
  for (long long p = (blockIdx.x * 4LL + quarter) * (64 * kGsU) + lane; p < np2; p += step) {
    phg_d2 x[kGsU], z[kGsU];
#pragma unroll
    for (int u = 0; u < kGsU; ++u) {
      const long long i = p + 64 * u;
      const bool in = i < np2;
      x[u] = in ? w2[i] : phg_d2{0.0, 0.0};
      z[u] = in ? u2[i] : phg_d2{0.0, 0.0};
      // past an odd length the pair's second element is padding
      if (2 * i + 1 >= A.n) x[u].y = z[u].y = 0.0;
    }
#pragma unroll
    for (int t = 0; t < kT; ++t) {
#pragma unroll
      for (int u = 0; u < kGsU; ++u) {
        const long long i = p + 64 * u;
        phg_d2 b = b2[t][i < np2 ? i : p];
        if (2 * i + 1 >= A.n) b.y = 0.0;
        a1[t] += b.x * x[u].x + b.y * x[u].y;
        a2[t] += b.x * z[u].x + b.y * z[u].y;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < kT; ++t) {
    const int j = wv + 4 * t;
    if (j < nv) {
      const double s1 = wave_sum(a1[t]), s2 = wave_sum(a2[t]);
      if (lane == 0) {
        red[quarter][2 * j] = s1;
        red[quarter][2 * j + 1] = s2;
      }
    }
  }
  if ((int)threadIdx.x < nv) nr[threadIdx.x] = nv > 1 ? gm.nrm[threadIdx.x] : A.n0;
  __syncthreads();
  if ((int)threadIdx.x < 2 * nv) {
    const int ch = threadIdx.x;
    const double s = red[0][ch] + red[1][ch] + red[2][ch] + red[3][ch];
    D[ch] = s;
    if (gridDim.x > 1) part_store(A.part + (size_t)ch * A.chan + blockIdx.x, s);
  }
  if (gridDim.x > 1 && !arrive_last(&gm.cnt)) return;
  // rows 1 .. nv - 2 of the strict lower triangle, row k at k (k - 1) / 2
  for (int e = threadIdx.x; e < (nv - 1) * (nv - 2) / 2; e += kGsThreads) G[e] = gm.G[e];
  if (gridDim.x > 1)
    for (int ch = wave; ch < 2 * nv; ch += kGsThreads / 64) {
      const double s = wave_sum_partials(A.part + (size_t)ch * A.chan, gridDim.x);
      if (lane == 0) D[ch] = s;
    }
  __syncthreads();
  if (wave != 0) return;
  // one wavefront from here: lane k holds d_k
  const int i = nv - 1;
  const double ni = nr[i], nk = lane < nv ? nr[lane] : 1.0, nw = A.unit ? 1.0 : ni;
  double d = lane < nv ? D[2 * lane] / (nk * nw) : 0.0;
  if (lane < i) {
    const double g = D[2 * lane + 1] / (nk * ni);
    G[i * (i - 1) / 2 + lane] = g;
    gm.G[i * (i - 1) / 2 + lane] = g;
  }
  __builtin_amdgcn_wave_barrier();
  for (int j = 0; j < i; ++j) {
    const double hj = from_lane(d, j);
    if (lane > j && lane < nv) d -= G[lane * (lane - 1) / 2 + j] * hj;
  }
  if (lane < nv) {
    gm.h[lane] = d;
    gm.coef[lane] = -d / nk;
  }
  if (lane == 0) {
    gm.scale = 1.0 / nw;
    if (nv == 1) {
      gm.nrm[0] = A.n0;
      gm.done = 0;
      gm.e[0] = A.unorm;
      gm.acc_spmv = gm.acc_gs = 0;
    }
  }
}

// w <- scale w - sum_k h_k w_k / n_k (scale 1 / n_i) and its norm; then the
// Hessenberg column's rotations (solgmr.f:645-663), the convergence test and,
// when the cycle ends, the back substitution (solgmr.f:681-686).
__global__ void __launch_bounds__(kGsThreads) k_gs_update(GsArgs A) {
  GmDev& gm = *A.gm;
  if (A.nv > 1 && gm.done) return;
  __shared__ double cf[kGmMax], ws[kGsThreads / 64];
  const int nv = A.nv, i = nv - 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((int)threadIdx.x < nv) cf[threadIdx.x] = gm.coef[threadIdx.x];
  const double a = gm.scale;
  // the step's scalars, loaded before the wait for the other workgroups:
  // lane k holds row k of the column
  double hk = wave == 0 && lane < nv ? gm.h[lane] : 0.0;
  const double cs = wave == 0 && lane < i ? gm.cs[lane] : 0.0;
  const double sn = wave == 0 && lane < i ? gm.sn[lane] : 0.0;
  const double ei = gm.e[i];
  __syncthreads();
  const long long np2 = (A.n + 1) / 2;
  phg_d2* w2 = reinterpret_cast<phg_d2*>(A.w);
  const phg_d2* b2 = reinterpret_cast<const phg_d2*>(A.basis);
  const long long bs = A.kstr / 2;
  double acc = 0.0;
  for (long long p = blockIdx.x * (long long)kGsThreads + threadIdx.x; p < np2;
       p += gridDim.x * (long long)kGsThreads) {
    phg_d2 x = w2[p] * a;
    int j = 0;
    for (; j + 4 <= nv; j += 4) {
      phg_d2 b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = b2[(j + t) * bs + p];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        x.x += cf[j + t] * b[t].x;
        x.y += cf[j + t] * b[t].y;
      }
    }
    for (; j < nv; ++j) {
      const phg_d2 b = b2[j * bs + p];
      x.x += cf[j] * b.x;
      x.y += cf[j] * b.y;
    }
    if (2 * p + 1 < A.n) {
      w2[p] = x;
      acc += x.x * x.x + x.y * x.y;
    } else {
      A.w[2 * p] = x.x;
      acc += x.x * x.x;
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) ws[wave] = acc;
  __syncthreads();
  double sq = wave == 0 ? wave_sum(lane < kGsThreads / 64 ? ws[lane] : 0.0) : 0.0;
  if (gridDim.x > 1) {
    if (threadIdx.x == 0) part_store(A.part + blockIdx.x, sq);
    if (!arrive_last(&gm.cnt)) return;
    if (wave == 0) sq = wave_sum_partials(A.part, gridDim.x);
  }
  if (wave != 0) return;
  const double nrm = sqrt(sq);
  // rotations of the earlier columns, in order: (j, j + 1)
  double top = from_lane(hk, 0);
  for (int j = 0; j < i; ++j) {
    const double c = from_lane(cs, j), s = from_lane(sn, j), lo = from_lane(hk, j + 1);
    const double t = c * top + s * lo;
    top = -s * top + c * lo;
    if (lane == j) hk = t;
  }
  const double rho = sqrt(top * top + nrm * nrm);
  const double c = top / rho, s = nrm / rho;
  const double e1 = -s * ei, e0 = c * ei;
  if (lane == i) hk = rho;
  if (lane < nv) gm.R[(size_t)i * kGmMax + lane] = hk;
  const double echeck = fabs(e1);
  const bool conv = echeck <= A.epsnrm && nv >= A.minIters;
  const bool done = conv || nv >= A.K;
  if (lane == 0) {
    gm.nrm[nv] = nrm;
    gm.cs[i] = c;
    gm.sn[i] = s;
    gm.e[i] = e0;
    gm.e[nv] = e1;
  }
  if (done) {
    double ek = lane < i ? gm.e[lane] : (lane == i ? e0 : 0.0);
    const double nk = lane < nv ? gm.nrm[lane] : 1.0;
    double y = 0.0;
    for (int j = i; j >= 0; --j) {
      const double rj = j == i ? hk : (lane <= j ? gm.R[(size_t)j * kGmMax + lane] : 0.0);
      const double yj = from_lane(ek, j) / from_lane(rj, j);
      if (lane == j) y = yj;
      if (lane < j) ek = ek - yj * rj;
    }
    if (lane < nv) gm.y[lane] = y / nk;
  }
  if (lane == 0) {
    const long long t2 = wall_clock64();
    const long long tp = gm.acc_spmv + gm.t1 - gm.t0, tg = gm.acc_gs + t2 - gm.t1;
    gm.acc_spmv = tp;
    gm.acc_gs = tg;
    gm.iKs = nv;
    gm.done = done ? 1 : 0;
    GmHost* h = A.host;
    __hip_atomic_store(&h->done, done ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&h->echeck, echeck, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&h->acc_spmv, tp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&h->acc_gs, tg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&h->seq, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// u = src / sqrt(*sq); norm_out <- sqrt(*sq) (written by one lane)
__global__ void k_scale(double* u, const double* src, long long n, const double* sq,
                        double* norm_out) {
  const double nrm = sqrt(*sq);
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i == 0 && norm_out) *norm_out = nrm;
  for (; i < n; i += (long long)gridDim.x * blockDim.x) u[i] = src[i] / nrm;
}

// dy (+)= sum_k y_k u_k, k ascending (solgmr.f:690-692), over the cycle's
// directions: the first nz from zb (network directions), the others from the
// basis; the coefficients, each with its vector's 1/norm, as the cycle left
// them in gm.  Four directions' loads in flight per lane; bound by the bytes of
// the directions.
__global__ void __launch_bounds__(256) k_combine(double* __restrict__ dy,
                                                 const double* __restrict__ basis, long long kstr,
                                                 const double* __restrict__ zb, long long zstr,
                                                 int nz, const GmDev* __restrict__ gm, long long n,
                                                 int add) {
  __shared__ double cf[kGmMax];
  const int k = gm->iKs;
  if ((int)threadIdx.x < k) cf[threadIdx.x] = gm->y[threadIdx.x];
  __syncthreads();
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    double v = add ? dy[i] : 0.0;
    int j = 0;
    for (; j < k && j < nz; ++j) v = v + cf[j] * zb[(size_t)j * zstr + i];
#pragma unroll 4
    for (; j < k; ++j) v = v + cf[j] * basis[(size_t)j * kstr + i];
    dy[i] = v;
  }
}

// ---------------- nodal work after the assembly ----------------
// The assembly leaves res (5) and BDiag (25) per node contiguous and the wall
// elements' contributions apart.  Per node: wall contributions, the Dirichlet
// rows and columns (bc3res.f:25-153, bc3bdg.f:25-330) and the periodic fold
// (res: master += slaves ascending, slaves zero, bc3res.f:157-163; BDiag:
// master += slaves, slaves copy it, bc3bdg.f:338-352).  With kSolve also what
// SolGMRs does per node before its Krylov loop: tnanq's count on res and
// BDiag, rmes, the LU factors, L^-1 res (also into the start vector) and the
// two sums of squares (solgmr.f:459-490), so each node's 30 values are read
// once and its 40 written once.
//
// k_boundary_nodes forms the sums of the few nodes with several sources (a
// periodic family, wall faces) with one lane per value, so that their chains
// of dependent loads run side by side; in k_nodes' own lanes they held up
// nearly every wavefront of a box (27.9 us at 4^3, 557 us at 128^3 against
// 15 and 310 us for both kernels).  k_nodes is bound by its bytes (0.5
// KB per node) from 64^3 on, by launches below.
constexpr int kNodeThreads = 256;
constexpr int kNodeBlocks = 1024;

struct NodeArgs {
  const double* ares;      // 5 per node
  const double* abd;       // 25 per node
  const double* wres;      // 5 per contribution
  int nspec;
  const int* sptr;         // members of a boundary group
  const int* smem;
  const int* wptr;         // wall contributions of a member
  double* ssum;            // 32 per group: BDiag (25), res (5)
  const int2* info;        // boundary group, family (-1 without)
  const uint8_t* bcm;
  double* res;
  double* rmes;
  double* start;
  double* bdiag;
  double* raw;             // BDiag before factorisation, nullable
  long long n;
  int prec;
  double* part;            // 3 channels of kNodeBlocks partials
  GmDev* gm;
  SolveHost* host;
  unsigned seq;
};

// value e of a node after the Dirichlet rows and columns: e < 25 BDiag (row
// e % 5, column e / 5), else res
__device__ inline double masked(double v, int e, uint8_t m) {
  if (e >= 25) return (m >> (e - 25)) & 1 ? 0.0 : v;
  const int i = e % 5, j = e / 5;
  return ((m >> i) & 1) || ((m >> j) & 1) ? (i == j ? 1.0 : 0.0) : v;
}

// one lane per (group, value)
__global__ void __launch_bounds__(256) k_boundary_nodes(NodeArgs A) {
  const long long at = blockIdx.x * 256LL + threadIdx.x;
  const int g = (int)(at >> 5), e = (int)(at & 31);
  if (g >= A.nspec || e >= 30 || (e < 25 && !A.prec)) return;
  double s = 0.0;
  for (int q = A.sptr[g]; q < A.sptr[g + 1]; ++q) {
    const long long k = A.smem[q];
    double v = e < 25 ? A.abd[25 * k + e] : A.ares[5 * k + e - 25];
    if (e >= 25) {
      const int w1 = A.wptr[q + 1];
#pragma unroll 4
      for (int w = A.wptr[q]; w < w1; ++w) v += A.wres[5 * (size_t)w + e - 25];
    }
    s += masked(v, e, A.bcm[k]);
  }
  A.ssum[32 * (size_t)g + e] = s;
}

__device__ inline double is_bad(double x) { return x != x || fabs(x) > 1.0e10 ? 1.0 : 0.0; }

template <bool kSolve>
__global__ void __launch_bounds__(kNodeThreads) k_nodes(NodeArgs A) {
  const int t = threadIdx.x;
  const long long n = A.n;
  // agent scope: the last workgroup reads it, perhaps from another XCD
  if (blockIdx.x == 0 && t == 0)
    __hip_atomic_store(&A.gm->ta[3], wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  double s_res = 0.0, s_rmes = 0.0, bad = 0.0;
  for (long long k = blockIdx.x * (long long)kNodeThreads + t; k < n;
       k += gridDim.x * (long long)kNodeThreads) {
    const int2 in = A.info[k];
    const uint8_t m = A.bcm[k];
    const bool sp = in.x >= 0;
    const double* rr = sp ? A.ssum + 32 * (size_t)in.x + 25 : A.ares + 5 * k;
    const double* rb = sp ? A.ssum + 32 * (size_t)in.x : A.abd + 25 * k;
    // a family's sums belong to its master; the slaves' res is zero
    const bool slave = in.y >= 0 && A.smem[A.sptr[in.x]] != k;
    double r[5], a[5][5];
#pragma unroll
    for (int f = 0; f < 5; ++f) r[f] = rr[f];
    if (A.prec) {
#pragma unroll
      for (int j = 0; j < 5; ++j)
#pragma unroll
        for (int i = 0; i < 5; ++i) a[i][j] = rb[i + 5 * j];
    }
    if (!sp && m) {
#pragma unroll
      for (int f = 0; f < 5; ++f) r[f] = masked(r[f], 25 + f, m);
      if (A.prec) {
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < 5; ++i) a[i][j] = masked(a[i][j], i + 5 * j, m);
      }
    }
    if (slave) {
#pragma unroll
      for (int f = 0; f < 5; ++f) r[f] = 0.0;
    }
    if constexpr (kSolve) {
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        A.rmes[k + f * n] = r[f];
        bad += is_bad(r[f]);
        s_rmes += r[f] * r[f];
      }
      if (A.prec) {
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < 5; ++i) {
            bad += is_bad(a[i][j]);
            if (A.raw) A.raw[k + (i + 5 * j) * n] = a[i][j];
          }
        lu_factor(a);
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < 5; ++i) A.bdiag[k + (i + 5 * j) * n] = a[i][j];
      } else {
        // the factors of an earlier call (solgmr.f:471)
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < 5; ++i) {
            a[i][j] = A.bdiag[k + (i + 5 * j) * n];
            bad += is_bad(a[i][j]);
          }
      }
      lu_solve_lower(a, r);
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        A.res[k + f * n] = r[f];
        A.start[k + f * n] = r[f];
        s_res += r[f] * r[f];
      }
    } else {
#pragma unroll
      for (int f = 0; f < 5; ++f) A.res[k + f * n] = r[f];
      if (A.prec) {
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < 5; ++i) A.bdiag[k + (i + 5 * j) * n] = a[i][j];
      }
    }
  }
  if constexpr (kSolve) {
    __shared__ double ws[3][kNodeThreads / 64];
    auto block_sums = [&](double out[3]) {
      s_res = wave_sum(s_res);
      s_rmes = wave_sum(s_rmes);
      bad = wave_sum(bad);
      if ((t & 63) == 0) {
        ws[0][t >> 6] = s_res;
        ws[1][t >> 6] = s_rmes;
        ws[2][t >> 6] = bad;
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < 3; ++c) out[c] = ws[c][0] + ws[c][1] + ws[c][2] + ws[c][3];
    };
    double sum[3];
    block_sums(sum);
    if (t == 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) part_store(A.part + c * kNodeBlocks + blockIdx.x, sum[c]);
    }
    if (!arrive_last(&A.gm->cnt)) return;
    double v[3][kNodeBlocks / kNodeThreads];
#pragma unroll
    for (int u = 0; u < kNodeBlocks / kNodeThreads; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int b = t + kNodeThreads * u;
        v[c][u] = b < (int)gridDim.x ? part_load(A.part + c * kNodeBlocks + b) : 0.0;
      }
    s_res = s_rmes = bad = 0.0;
#pragma unroll
    for (int u = 0; u < kNodeBlocks / kNodeThreads; ++u) {
      s_res += v[0][u];
      s_rmes += v[1][u];
      bad += v[2][u];
    }
    block_sums(sum);
    if (t != 0) return;
    SolveHost* h = A.host;
    const long long now = wall_clock64();
    const long long ta3 =
        __hip_atomic_load(&A.gm->ta[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const long long ta[5] = {A.gm->ta[0], A.gm->ta[1], A.gm->ta[2], ta3, now};
    __hip_atomic_store(&h->sumsq, sum[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&h->sumsq_m, sum[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&h->bad, sum[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#pragma unroll
    for (int k = 0; k < 5; ++k)
      __hip_atomic_store(&h->ta[k], ta[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&h->seq, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ---------------- the FP64 tangent's product around its element kernel ----------------
// k_product_in: per node the direction as the elements read it, v at the
// periodic master with the constrained components zero.  kLu: v = U^-1 src of
// the master (the refinement's U^-1 dy), also stored in planes for
// k_product_nodes.
template <bool kLu>
__global__ void __launch_bounds__(256) k_product_in(const double* __restrict__ src,
                                                    const double* __restrict__ D,
                                                    const int* __restrict__ iper,
                                                    const uint8_t* __restrict__ bcm,
                                                    double* __restrict__ vp,
                                                    double* __restrict__ v, long long n) {
  const long long k = blockIdx.x * 256LL + threadIdx.x;
  if (k >= n) return;
  const long long m = iper[k];
  const uint8_t c = bcm[k];
  double r[5];
#pragma unroll
  for (int f = 0; f < 5; ++f) r[f] = src[m + f * n];
  if constexpr (kLu) {
    double d[5][5];
#pragma unroll
    for (int j = 0; j < 5; ++j)
#pragma unroll
      for (int i = 0; i <= j; ++i) d[i][j] = D[(i + 5 * j) * n + m];
#pragma unroll
    for (int i = 4; i >= 0; --i) {
      double s = r[i];
#pragma unroll
      for (int q = 4; q > i; --q) s -= r[q] * d[i][q];
      r[i] = d[i][i] * s;
    }
#pragma unroll
    for (int f = 0; f < 5; ++f) v[k + f * n] = r[f];
  }
  double2* o = reinterpret_cast<double2*>(vp + 8 * k);
#pragma unroll
  for (int f = 0; f < 5; ++f) r[f] = (c >> f) & 1 ? 0.0 : r[f];
  o[0] = make_double2(r[0], r[1]);
  o[1] = make_double2(r[2], r[3]);
  o[2] = make_double2(r[4], 0.0);
}

struct ProductArgs {
  const long long* goff;   // the node incidence layout, 64-node groups
  const int* inc;
  const double* out;       // element products at their slots there
  const double* v;         // direction, 5 planes
  const int* iper;
  const uint8_t* bcm;
  const int2* info;        // boundary group, family (-1 without)
  const int* sptr;
  const int* smem;
  int nmem;                // members, 0: no sums apart
  double* msum;            // 8 per member: the slaves' sums
  double* w;               // the product (without kResid)
  const double* rmes;
  const double* bdiag;
  double* start;
  long long n;
  double* part;            // kNodeBlocks partials
  GmDev* gm;
  SolveHost* host;
  unsigned seq;
};

// values f0 .. f0 + kF - 1 of the node's sum of element products in element
// order; a constrained value f is the unit diagonals of its element blocks,
// cnt(k) v(iper(k))_f (bc3lhs.f:55-235: one per element containing the node)
template <int kF>
__device__ __forceinline__ void node_product(const ProductArgs& A, long long k, int f0,
                                             double acc[kF]) {
  const long long o0 = A.goff[k >> 6];
  const int deg = (int)((A.goff[(k >> 6) + 1] - o0) >> 6);
  const uint8_t m = A.bcm[k];
  int cnt = 0;
#pragma unroll
  for (int f = 0; f < kF; ++f) acc[f] = 0.0;
  long long slot = o0 + (k & 63);
#pragma unroll 4
  for (int j = 0; j < deg; ++j, slot += 64) {
    const bool on = A.inc[slot] >= 0;
    cnt += on;
#pragma unroll
    for (int f = 0; f < kF; ++f) {
      const double r = A.out[slot * 5 + f0 + f];
      acc[f] += on ? r : 0.0;
    }
  }
  if (m) {
    const long long mm = A.iper[k];
#pragma unroll
    for (int f = 0; f < kF; ++f)
      if ((m >> (f0 + f)) & 1) acc[f] = (double)cnt * A.v[mm + (f0 + f) * A.n];
  }
}

// the periodic slaves' sums, one lane per value (in the masters' lanes they
// would hold up nearly every wavefront of a box, see k_boundary_nodes)
__global__ void __launch_bounds__(256) k_product_members(ProductArgs A) {
  const long long at = blockIdx.x * 256LL + threadIdx.x;
  const int q = (int)(at >> 3), f = (int)(at & 7);
  if (q >= A.nmem || f >= 5) return;
  const long long k = A.smem[q];
  const int2 in = A.info[k];
  if (in.y < 0 || A.sptr[in.x] == q) return;
  double s[1];
  node_product<1>(A, k, f, s);
  A.msum[8 * (size_t)q + f] = s[0];
}

// per node the product with the slaves folded into their master (bc3per:
// ascending, slaves zero); kResid: instead r = L^-1 (rmes - product) into
// start and the sum of its squares to the host, with seq.  Bound by the element
// products' 40 bytes per node and element from 64^3 on (0.49 ms at 128^3, 4.5
// TB/s), by launches below: with k_product_in, the element kernel and
// k_product_members it replaces the refinement's twelve launches and two waits
// (a mixed step of three iterations at 16^3: 1.41 -> 1.30 ms).
template <bool kResid>
__global__ void __launch_bounds__(kNodeThreads) k_product_nodes(ProductArgs A) {
  const int t = threadIdx.x;
  const long long n = A.n;
  double sq = 0.0;
  for (long long k = blockIdx.x * (long long)kNodeThreads + t; k < n;
       k += gridDim.x * (long long)kNodeThreads) {
    double r[5];
    node_product<5>(A, k, 0, r);
    const int2 in = A.info[k];
    if (in.y >= 0) {
      const int q0 = A.sptr[in.x], q1 = A.sptr[in.x + 1];
      if (A.smem[q0] == k) {
        for (int q = q0 + 1; q < q1; ++q) {
          double s[5];
          if (A.nmem > 0) {
#pragma unroll
            for (int f = 0; f < 5; ++f) s[f] = A.msum[8 * (size_t)q + f];
          } else {
            node_product<5>(A, A.smem[q], 0, s);
          }
#pragma unroll
          for (int f = 0; f < 5; ++f) r[f] += s[f];
        }
      } else {
#pragma unroll
        for (int f = 0; f < 5; ++f) r[f] = 0.0;
      }
    }
    if constexpr (kResid) {
      double a[5][5];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = j + 1; i < 5; ++i) a[i][j] = A.bdiag[k + (i + 5 * j) * n];
#pragma unroll
      for (int f = 0; f < 5; ++f) r[f] = A.rmes[k + f * n] - r[f];
      lu_solve_lower(a, r);
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        A.start[k + f * n] = r[f];
        sq += r[f] * r[f];
      }
    } else {
#pragma unroll
      for (int f = 0; f < 5; ++f) A.w[k + f * n] = r[f];
    }
  }
  if constexpr (kResid) {
    __shared__ double ws[kNodeThreads / 64];
    auto block_sum = [&](double v) {
      v = wave_sum(v);
      __syncthreads();
      if ((t & 63) == 0) ws[t >> 6] = v;
      __syncthreads();
      return ws[0] + ws[1] + ws[2] + ws[3];
    };
    const double s = block_sum(sq);
    if (t == 0) part_store(A.part + blockIdx.x, s);
    if (!arrive_last(&A.gm->cnt)) return;
    double v[kNodeBlocks / kNodeThreads];
#pragma unroll
    for (int u = 0; u < kNodeBlocks / kNodeThreads; ++u) {
      const int b = t + kNodeThreads * u;
      v[u] = b < (int)gridDim.x ? part_load(A.part + b) : 0.0;
    }
    sq = 0.0;
#pragma unroll
    for (int u = 0; u < kNodeBlocks / kNodeThreads; ++u) sq += v[u];
    const double all = block_sum(sq);
    if (t != 0) return;
    __hip_atomic_store(&A.host->rsq, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&A.host->rseq, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Small host arrays, between device memory and pinned host memory.  To the host
// one workgroup, which then stores the token; 16 otherwise.  Bound by the bus's
// latency: all arrays of a call in one launch (4 to 8 us for 5 KB to 128 KB).
__global__ void __launch_bounds__(1024) k_small_copy(SmallCopy S, unsigned* done, unsigned token) {
  for (int a = 0; a < S.count; ++a) {
    unsigned* d = static_cast<unsigned*>(S.seg[a].dst);
    const unsigned* s = static_cast<const unsigned*>(S.seg[a].src);
    const unsigned n = (unsigned)S.seg[a].words;
#pragma unroll 4
    for (unsigned i = blockIdx.x * 1024 + threadIdx.x; i < n; i += gridDim.x * 1024) d[i] = s[i];
  }
  if (!done) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(done, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_end_mark(SolveHost* h, unsigned seq) {
  __hip_atomic_store(&h->end, wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __hip_atomic_store(&h->end_seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------- layout conversion ----------------
template <typename T>
__global__ void k_csr_to_slots(const double* ref, T* slots, const uint32_t* c2s, long long nnz) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint32_t qs = c2s[k];
  T* dst = slots + (size_t)(qs >> 6) * (25 * kGroup);
#pragma unroll
  for (int e = 0; e < 25; ++e) dst[slot_pos<T>(e, (int)(qs & 63))] = (T)ref[k * 25 + e];
}

template <typename T>
__global__ void k_slots_to_csr(const T* slots, double* ref, const uint32_t* c2s, long long nnz) {
  long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint32_t qs = c2s[k];
  const T* src = slots + (size_t)(qs >> 6) * (25 * kGroup);
#pragma unroll
  for (int e = 0; e < 25; ++e) ref[k * 25 + e] = (double)src[slot_pos<T>(e, (int)(qs & 63))];
}

// ---------------- itrPredict / itrCorrect / itrUpdate / itrBC ----------------
// One lane per node forms the node's new (y, ac), sets the Dirichlet values
// on y (temperature, no-slip velocity, pressure; itrbc.f:60-139) and writes
// them; a periodic master writes its slaves' too (itrbc.f:141-178: they copy
// y and ac), so a slave's own lane writes nothing.
struct StateArgs {
  double* y;
  double* ac;
  const double* yold;
  const double* acold;
  const double* dy;
  const uint8_t* bcm;
  const double* BC;
  const int2* info;
  const int* fmaster;
  const int* fptr;
  const int* fslave;
  long long n;
  double f1, f2;
};

// kMode 0: itrPredict, same-velocity predictor (itrPC.f:67-73): y = yold,
//          ac = acold f1
//       1: itrCorrect (itrPC.f:128-148): y -= Dy, ac = acold f1 + (y - yold) f2
//       2: itrUpdate (itrPC.f:204-207) of (y, ac) = the old state towards
//          (yold, acold) = the new one: ac += (acold - ac) f1, y += (yold - y) f2
template <int kMode>
__global__ void k_state(StateArgs A) {
  const long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const long long n = A.n;
  if (k >= n) return;
  const int fam = A.info[k].y;
  if (fam >= 0 && A.fmaster[fam] != k) return;
  double v[5], a[5];
  const int from[5] = {1, 2, 3, 0, 4};  // Dy is in equation order
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    const long long i = k + f * n;
    if constexpr (kMode == 0) {
      v[f] = A.yold[i];
      a[f] = A.acold[i] * A.f1;
    } else if constexpr (kMode == 1) {
      v[f] = A.y[i] - A.dy[k + from[f] * n];
      a[f] = A.acold[i] * A.f1 + (v[f] - A.yold[i]) * A.f2;
    } else {
      a[f] = A.ac[i] + (A.acold[i] - A.ac[i]) * A.f1;
      v[f] = A.y[i] + (A.yold[i] - A.y[i]) * A.f2;
    }
  }
  const uint8_t m = A.bcm[k];
  if (m & 16) v[4] = A.BC[k + n];
  if (m & 2) {
    v[0] = A.BC[k + 2 * n];
    v[1] = A.BC[k + 3 * n];
    v[2] = A.BC[k + 4 * n];
  }
  if (m & 1) v[3] = A.BC[k];
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    A.y[k + f * n] = v[f];
    A.ac[k + f * n] = a[f];
  }
  if (fam < 0) return;
  for (int q = A.fptr[fam]; q < A.fptr[fam + 1]; ++q) {
    const long long s = A.fslave[q];
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      A.y[s + f * n] = v[f];
      A.ac[s + f * n] = a[f];
    }
  }
}

inline int grid_for(long long n, int threads) {
  long long b = (n + threads - 1) / threads;
  return (int)(b < 1 ? 1 : b);
}

}  // namespace

int launch_i3lu(phg_ctx* c, double* diag, double* r, int code) {
  const long long n = c->nshg;
  const int g = grid_for(n, 256);
  if (code == 0)
    k_lu_fact<<<g, 256, 0, c->stream>>>(diag, n);
  else if (code == 1)
    k_lu_forward<<<g, 256, 0, c->stream>>>(diag, r, n);
  else if (code == 2)
    k_lu_backward<<<g, 256, 0, c->stream>>>(diag, r, n);
  else if (code == 3)
    k_lu_product<<<g, 256, 0, c->stream>>>(diag, r, n);
  else {
    phg_set_error("i3LU: unsupported code %d", code);
    return PHG_EINVAL;
  }
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_spsi3pre(phg_ctx* c) {
  PHG_TRY(require_matrix(c, "Spsi3pre"));
  const int g = (int)c->ngroups, nt = kPreWaves * kGroup;
  if (c->precision == PHG_MIXED)
    k_spsi3pre<float, float><<<g, nt, 0, c->stream>>>(
        c->lhs_aos32, c->lhs32, c->slot2csr, c->scol, c->grp_slot, c->rowmap, c->bdiag, c->nshg);
  else
    k_spsi3pre<double, double><<<g, nt, 0, c->stream>>>(
        c->lhs_aos, c->lhs64, c->slot2csr, c->scol, c->grp_slot, c->rowmap, c->bdiag, c->nshg);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_spmv(phg_ctx* c, const double* p, double* q, bool fold, const int* gate,
                long long* t0) {
  PHG_TRY(require_matrix(c, "SparseAp"));
  const int g = (int)((c->ngroups + 7) / 8 * 8);  // one workgroup per group, XCD-strided
  const int in_group = fold && c->fam_in_group ? 1 : 0;
  auto run = [&](auto vals, auto waves) {
    constexpr int W = decltype(waves)::value;
    k_spmv<std::remove_pointer_t<decltype(vals)>, double, W><<<g, W * kGroup, 0, c->stream>>>(
        vals, c->scolp, c->grp_slot, c->rowmap, c->fam, p, q, c->nshg, c->ngroups, in_group, gate,
        t0);
  };
  auto pick = [&](auto vals) {
    using T = std::remove_pointer_t<decltype(vals)>;
    if (c->ngroups <= kSpmvFew)
      run(vals, std::integral_constant<int, kSpmvWavesFew>{});
    else
      run(vals, std::integral_constant<int, kSpmvWaves<T>>{});
  };
  if (c->precision == PHG_MIXED)
    pick(c->lhs32);
  else
    pick(c->lhs64);
  PHG_HIP(hipGetLastError());
  // a family of more than kGroup rows: the rows lie in several groups.  The
  // fold runs whatever the gate says: on a skipped product's old output it
  // is harmless (nothing reads that vector any more)
  return fold && !c->fam_in_group ? launch_bc3per(c, q, 5) : 0;
}

// q = K^T x for the periodic-folded operator K = F A G of the matvec:
// K^T = F A^T G (G copies masters to slaves, F folds slaves into masters).
// x is overwritten by G x.
int launch_spmv_t(phg_ctx* c, double* x, double* q) {
  if (!c->tslot) {
    phg_set_error("transpose matvec: slot map not built");
    return PHG_EINVAL;
  }
  if (c->nfold > 0) {
    k_per_copy_vec<<<(c->nfold + 255) / 256, 256, 0, c->stream>>>(x, c->fold_master, c->fold_ptr,
                                                                  c->fold_slave, c->nfold, c->nshg);
    PHG_HIP(hipGetLastError());
  }
  const int g = grid_for(c->ngroups * kGroup, 256);
  if (c->precision == PHG_MIXED)
    k_spmv_t<float><<<g, 256, 0, c->stream>>>(c->lhs32, c->scol, c->tslot, c->grp_slot, c->rowmap,
                                              x, q, c->nshg, c->ngroups);
  else
    k_spmv_t<double><<<g, 256, 0, c->stream>>>(c->lhs64, c->scol, c->tslot, c->grp_slot,
                                               c->rowmap, x, q, c->nshg, c->ngroups);
  PHG_HIP(hipGetLastError());
  return launch_bc3per(c, q, 5);
}

int launch_sub(phg_ctx* c, double* r, const double* b, const double* q, long long n) {
  int g = (int)std::min<long long>(grid_for(n, 256), 16384);
  k_sub<<<g, 256, 0, c->stream>>>(r, b, q, n);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_copy(phg_ctx* c, double* dst, const double* src, long long n) {
  if (n & 1) {  // copied as 16-byte pairs
    phg_set_error("copy: odd length %lld", n);
    return PHG_EINVAL;
  }
  const long long n2 = n / 2;
  const int g = grid_for(n2, 256);
  k_copy<<<g, 256, 0, c->stream>>>(reinterpret_cast<double2*>(dst),
                                   reinterpret_cast<const double2*>(src), n2);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_aos_to_ref(phg_ctx* c, double* ref) {
  const long long n = 25 * c->nnz;
  if (c->precision == PHG_MIXED)
    k_aos_to_ref<float><<<grid_for(n, 256), 256, 0, c->stream>>>(c->lhs_aos32, ref, c->nnz);
  else
    k_aos_to_ref<double><<<grid_for(n, 256), 256, 0, c->stream>>>(c->lhs_aos, ref, c->nnz);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_ref_to_aos(phg_ctx* c, const double* ref) {
  const long long n = (long long)aos_stride<double>() * c->nnz;
  k_ref_to_aos<<<grid_for(n, 256), 256, 0, c->stream>>>(ref, c->lhs_aos, c->nnz);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_bc3per(phg_ctx* c, double* v, int nq) {
  if (c->nfold <= 0) return 0;
  k_fold_vec<<<dim3((c->nfold + 255) / 256, nq), 256, 0, c->stream>>>(
      v, c->fold_master, c->fold_ptr, c->fold_slave, c->nfold, c->nshg);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_dot(phg_ctx* c, const double* a, const double* b, long long n, double* out) {
  // workgroups so that one unrolled pass covers n, at most red_blocks
  const int g = (int)std::min<long long>(grid_for(n, kRedThreads * kUnroll), c->red_blocks);
  k_dot<<<g, kRedThreads, 0, c->stream>>>(a, b, n, c->red_part);
  PHG_HIP(hipGetLastError());
  k_finish<<<1, kRedThreads, 0, c->stream>>>(c->red_part, g, out);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_gs(phg_ctx* c, double* w, int iK, bool unit, bool clocked, double unorm, double epsnrm,
              double n0, unsigned seq) {
  if (iK < 1 || iK >= kGmMax) {
    phg_set_error("Gram-Schmidt: iteration %d outside 1..%d", iK, kGmMax - 1);
    return PHG_EINVAL;
  }
  GsArgs A{};
  A.w = w;
  A.basis = c->krylov;
  A.n = 5 * c->nshg;
  A.kstr = c->kstr;
  A.nv = iK;
  A.K = c->prm.Kspace;
  A.minIters = c->prm.minIters;
  A.unit = unit ? 1 : 0;
  A.clocked = clocked ? 1 : 0;
  A.unorm = unorm;
  A.epsnrm = epsnrm;
  A.n0 = n0;
  A.part = c->red_part;
  A.chan = c->red_blocks;
  A.gm = c->gm;
  A.host = c->h_gm + iK;
  A.seq = seq;
  const long long np2 = (A.n + 1) / 2;
  const int gd = (int)std::min<long long>(grid_for(np2, 256 * kGsU), kGsBlocks);
  const int gu = (int)std::min<long long>(grid_for(np2, kGsThreads), kGsBlocks);
  // Widths up to 20 vectors, the longest cycle of the workloads, so that hardly
  // a wavefront loads a vector twice; one width above, whose wavefronts load 15
  // vectors whatever iK is (the last again) and spill 33 words.  Per iteration
  // with the update, 64^3, FP64, against one launch per Gram-Schmidt step: 21 to
  // 24 vectors 178 us (266), 25 to 32 206 (352), 41 to 60 304 (634).
  const int t = (iK + 3) / 4;
  if (t <= 1)
    k_gs_dots<1><<<gd, kGsThreads, 0, c->stream>>>(A);
  else if (t == 2)
    k_gs_dots<2><<<gd, kGsThreads, 0, c->stream>>>(A);
  else if (t == 3)
    k_gs_dots<3><<<gd, kGsThreads, 0, c->stream>>>(A);
  else if (t <= 5)
    k_gs_dots<5><<<gd, kGsThreads, 0, c->stream>>>(A);
  else
    k_gs_dots<15><<<gd, kGsThreads, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  k_gs_update<<<gu, kGsThreads, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_scale(phg_ctx* c, double* u, const double* src, long long n, const double* sq_ptr,
                 double* norm_out) {
  int g = (int)std::min<long long>(grid_for(n, 256), 16384);
  k_scale<<<g, 256, 0, c->stream>>>(u, src, n, sq_ptr, norm_out);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_combine(phg_ctx* c, double* dy, const double* zb, int nz, bool add) {
  const long long n = 5 * c->nshg;
  int g = (int)std::min<long long>(grid_for(n, 256), 16384);
  k_combine<<<g, 256, 0, c->stream>>>(dy, c->krylov, c->kstr, zb, n, nz, c->gm, n, add ? 1 : 0);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_nodes(phg_ctx* c, bool prec, bool solve, double* raw, double* start) {
  NodeArgs A{};
  A.ares = c->acc_res;
  A.abd = c->acc_bd;
  A.wres = c->wres;
  A.nspec = c->nspec;
  A.sptr = c->sptr;
  A.smem = c->smem;
  A.wptr = c->wptr;
  A.ssum = c->ssum;
  A.info = c->ninfo;
  A.bcm = c->bcm;
  A.res = c->res;
  A.rmes = c->rmes;
  A.start = start;
  A.bdiag = c->bdiag;
  A.raw = raw;
  A.n = c->nshg;
  A.prec = prec ? 1 : 0;
  A.part = c->red_part;
  A.gm = c->gm;
  A.host = c->h_sol;
  if (c->nspec > 0) {
    k_boundary_nodes<<<grid_for(32LL * c->nspec, 256), 256, 0, c->stream>>>(A);
    PHG_HIP(hipGetLastError());
  }
  const int g = std::min(grid_for(c->nshg, kNodeThreads), kNodeBlocks);
  if (solve) {
    A.seq = ++c->sol_seq;
    k_nodes<true><<<g, kNodeThreads, 0, c->stream>>>(A);
  } else {
    k_nodes<false><<<g, kNodeThreads, 0, c->stream>>>(A);
  }
  PHG_HIP(hipGetLastError());
  return 0;
}

namespace {

ProductArgs product_args(phg_ctx* c, const double* v) {
  ProductArgs A{};
  A.goff = c->inc_goff;
  A.inc = c->inc;
  A.out = c->resid;
  A.v = v;
  A.iper = c->iper;
  A.bcm = c->bcm;
  A.info = c->ninfo;
  A.sptr = c->sptr;
  A.smem = c->smem;
  // below half a wavefront per SIMD the masters' lanes take their slaves' chains
  // along in less time than a launch (a product at 4913 nodes 98.5 -> 92 us)
  A.nmem = c->nfold > 0 && c->nshg > 32768 ? c->nmem : 0;
  A.msum = c->msum;
  A.n = c->nshg;
  A.part = c->red_part;
  A.gm = c->gm;
  A.host = c->h_sol;
  return A;
}

int launch_members(phg_ctx* c, const ProductArgs& A) {
  if (A.nmem > 0) {
    k_product_members<<<grid_for(8LL * A.nmem, 256), 256, 0, c->stream>>>(A);
    PHG_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace

int launch_tangent_product(phg_ctx* c, const double* v, double* w) {
  const long long n = c->nshg;
  k_product_in<false><<<grid_for(n, 256), 256, 0, c->stream>>>(v, nullptr, c->iper, c->bcm,
                                                              c->vpack, nullptr, n);
  PHG_HIP(hipGetLastError());
  PHG_TRY(launch_jv(c));
  ProductArgs A = product_args(c, v);
  A.w = w;
  PHG_TRY(launch_members(c, A));
  k_product_nodes<false><<<grid_for(n, kNodeThreads), kNodeThreads, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_tangent_residual(phg_ctx* c, const double* dy, double* v, double* start) {
  const long long n = c->nshg;
  k_product_in<true><<<grid_for(n, 256), 256, 0, c->stream>>>(dy, c->bdiag, c->iper, c->bcm,
                                                             c->vpack, v, n);
  PHG_HIP(hipGetLastError());
  PHG_TRY(launch_jv(c));
  ProductArgs A = product_args(c, v);
  A.rmes = c->rmes;
  A.bdiag = c->bdiag;
  A.start = start;
  A.seq = ++c->res_seq;
  PHG_TRY(launch_members(c, A));
  const int g = std::min(grid_for(n, kNodeThreads), kNodeBlocks);
  k_product_nodes<true><<<g, kNodeThreads, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_small_copy(phg_ctx* c, const SmallCopy& S, unsigned* done) {
  k_small_copy<<<done ? 1 : 16, 1024, 0, c->stream>>>(S, done, done ? ++c->copy_seq : 0);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_end_mark(phg_ctx* c) {
  k_end_mark<<<1, 1, 0, c->stream>>>(c->h_sol, c->sol_seq);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_csr_to_slots(phg_ctx* c, const double* ref, double* slots) {
  k_csr_to_slots<double><<<grid_for(c->nnz, 256), 256, 0, c->stream>>>(ref, slots, c->csr2slot,
                                                                       c->nnz);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_slots_to_csr(phg_ctx* c, const double* slots, double* ref) {
  k_slots_to_csr<double><<<grid_for(c->nnz, 256), 256, 0, c->stream>>>(slots, ref, c->csr2slot,
                                                                       c->nnz);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_slots_to_csr32(phg_ctx* c, const float* slots, double* ref) {
  k_slots_to_csr<float><<<grid_for(c->nnz, 256), 256, 0, c->stream>>>(slots, ref, c->csr2slot,
                                                                      c->nnz);
  PHG_HIP(hipGetLastError());
  return 0;
}

static StateArgs state_args(const phg_ctx* c, double* y, double* ac, const double* yold,
                            const double* acold) {
  StateArgs A{};
  A.y = y;
  A.ac = ac;
  A.yold = yold;
  A.acold = acold;
  A.bcm = c->bcm;
  A.BC = c->BCv;
  A.info = c->ninfo;
  A.fmaster = c->fold_master;
  A.fptr = c->fold_ptr;
  A.fslave = c->fold_slave;
  A.n = c->nshg;
  return A;
}

int launch_predict(phg_ctx* c) {
  // The reference's other predictors (ipred 2-4, itrPC.f:75-119) call
  // itrBC with iBC, BC, iper and ilwork undeclared in itrPredict, so they
  // are implicitly typed uninitialised scalars passed where arrays belong:
  // the reference defines no result for them.
  if (c->prm.ipred != 1) {
    phg_set_error("phg_predict: ipred %d; only the same-velocity predictor (ipred 1, "
                  "itrPC.f:67-73) has a defined result in the reference", c->prm.ipred);
    return PHG_EINVAL;
  }
  StateArgs A = state_args(c, c->y, c->ac, c->yold, c->acold);
  A.f1 = 1.0 - c->prm.almi / c->prm.gami;
  k_state<0><<<grid_for(c->nshg, 256), 256, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_correct(phg_ctx* c) {
  StateArgs A = state_args(c, c->y, c->ac, c->yold, c->acold);
  A.dy = c->dy;
  A.f1 = 1.0 - c->prm.almi / c->prm.gami;
  A.f2 = c->prm.almi * c->prm.Dtgl / c->prm.gami / c->prm.alfi;
  k_state<1><<<grid_for(c->nshg, 256), 256, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_update(phg_ctx* c) {
  StateArgs A = state_args(c, c->yold, c->acold, c->y, c->ac);
  A.f1 = 1.0 / c->prm.almi;
  A.f2 = 1.0 / c->prm.alfi;
  k_state<2><<<grid_for(c->nshg, 256), 256, 0, c->stream>>>(A);
  PHG_HIP(hipGetLastError());
  return 0;
}

int launch_yshuffle(phg_ctx* c, const double* src, double* dst, bool new2old) {
  const long long n = c->nshg;
  k_yshuffle<<<grid_for(n, 256), 256, 0, c->stream>>>(src, dst, n, new2old ? 1 : 0);
  PHG_HIP(hipGetLastError());
  return 0;
}
