// Eigen-decomposition of the closure scatter (the first-call basis).
//   symmetric_eigen   eigenvalues and eigenvectors of 0.5 (A + A^T) for a batch of small
//                     fp32 matrices (n <= 128), eigenvalues ascending and eigenvectors as
//                     columns, the contract of torch.linalg.eigh that closure_basis calls
//                     (recap/sparse/closure.py:75-81).
//
// One workgroup per matrix.  One-sided cyclic Jacobi (Hestenes 1958; Golub & Van Loan, Matrix
// Computations, 4th ed., sec. 8.6.3) on the columns of G = B V, B the symmetrised input and V
// the accumulated rotations: a rotation of columns x, y makes them orthogonal, and when all
// are, V diagonalises B^2 and so B, with lambda_i = v_i . g_i.  The columns live in registers,
// one element per lane (two for n > 64), so a rotation is wave-local: one dot product per
// pair and two FMAs per element, the cosines kept as a scale factor per column.  The rounds
// follow the circle ordering (Brent & Luk 1985) as a ring: every wave holds 8 adjacent pair
// slots, the upper columns move one slot to the right and the lower ones to the left
// after every round, so only the two columns that leave a wave go through LDS, and one
// barrier per round is enough.  Latency bounds it (a chain of a reduction, the rotation's
// square roots and the exchange, per round) and VALU issue, about 0.83 us a round for 10-12
// sweeps of 128 rounds: 1.28 ms for 12 matrices of order 128 and 0.31 ms for 4 of order 64.
// (The two-sided form, both matrices in LDS, moved 256 KB through it per round behind two
// barriers: 3.84 and 1.05 ms, with eigenvalue errors of 1.7e-6 of the largest against
// 2.8e-7 here.)
//
// V^T B^2 V = diag leaves eigenvalues +s and -s of an indefinite B undetermined, so a result
// with a negative eigenvalue, or one that is no eigenvector, is computed again from
// B + mu I, mu the spectral norm the first pass gives; a scatter (positive semidefinite)
// never takes that branch.
#include "kernels.hpp"

namespace recap {

namespace {

constexpr int kEigenMax = 128;
// |x . y| <= tol |x| |y| counts as orthogonal: a few times the rounding of a 128-term dot
// product.  A sweep that finds every pair so ends the loop; a sweep cap bounds it whatever
// the input.
constexpr float kEigenTol = 5.0e-7f;
// Rounds between two renormalisations of the scaled columns (their scale factors stay above
// 0.7^32 and the column norms are computed afresh).
constexpr int kRenorm = 32;

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(x), CTRL, 0xf, 0xf, true));
}

constexpr int kPairs = 8;            // pair slots of a wave
constexpr int kLanes = 64 / kPairs;  // lanes that hold one slot's scalars

// Wave sums of 8 values at once: lane l gets the sum of p[l / 8] over all 64 lanes.  The
// first steps add two lanes' halves of two values into one register: 20 instructions.
__device__ __forceinline__ float group_sums(const float (&p)[kPairs]) {
  float half[4];  // p[i] in lanes 0-31, p[i + 4] in lanes 32-63
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[i]), __float_as_uint(p[i + 4]), false, false);
    half[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  float row[2];  // p[i + 2 r] in row r of 16 lanes
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(half[i]), __float_as_uint(half[i + 2]), false, false);
    row[i] = dpp_add<0x128>(__uint_as_float(r[0]) + __uint_as_float(r[1]));  // + row_ror:8
  }
  float x = (threadIdx.x & 8) ? row[1] : row[0];
  x = dpp_add<0x141>(x);    // + row_half_mirror
  x = dpp_add<0xb1>(x);     // + quad_perm 1,0,3,2
  return dpp_add<0x4e>(x);  // + quad_perm 2,3,0,1
}

__device__ __forceinline__ float from_group(float x, int k) {  // wave-uniform value of group k
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(x), k * kLanes));
}

// E elements of a column per lane (row lane + 64 e), NW waves of kPairs slots.  Four slots a
// wave (twice the waves) took 1.52 ms at order 128, sixteen 1.37 ms, eight 1.28 ms: the
// instructions that every wave repeats (reduction, rotation, exchange) against the waves
// that hide their latency.
template <int E, int NW>
__global__ __launch_bounds__(64 * NW) void symmetric_eigen_kernel(EigenArgs a) {
  constexpr int kEigenThreads = 64 * NW;
  constexpr int P = kPairs;
  constexpr int SLOTS = P * NW;         // 2 * SLOTS columns
  static_assert(2 * SLOTS == 64 * E, "every column has a place");
  constexpr int kCols = 2 * SLOTS;
  struct Column { float g[E], v[E]; };
  struct Scalars { float norm2, scale; int index, pad; };  // |x|^2, its factor, input column
  __shared__ __attribute__((aligned(16))) float V[kEigenMax * kEigenMax];
  __shared__ __attribute__((aligned(16))) float A[kEigenMax * kEigenMax];
  // During the sweeps the two matrices' storage holds the columns and scalars that move.
  auto& box = *reinterpret_cast<Column (*)[2][2][NW][64]>(A);   // [parity][upper, lower][wave]
  auto& sc = *reinterpret_cast<Scalars (*)[2][2][SLOTS]>(V);
  static_assert(sizeof(Column) * 4 * NW * 64 <= sizeof(A) && sizeof(Scalars) * 4 * SLOTS <= sizeof(V), "storage");
  __shared__ float lam[kEigenMax], size2[kEigenMax], off2[kEigenMax];
  __shared__ int rank[kEigenMax];
  __shared__ int rotated;
  const int t = threadIdx.x, n = a.n, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int slot = P * wave + lane / kLanes;   // the pair slot whose scalars this lane holds
  const bool leader = lane % kLanes == 0;
  const float* src = a.a + (int64_t)blockIdx.x * n * n;

  // The columns are those of the input times a power of two that brings its largest element
  // to [1, 2): the squared norms and their products stay in range for any input.
  float top = 0.0f;
  for (int i = t; i < n * n; i += kEigenThreads) top = fmaxf(top, fabsf(src[i]));
  for (int off = 32; off >= 1; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
  if (lane == 0) lam[wave] = top;
  __syncthreads();
  for (int i = 0; i < NW; ++i) top = fmaxf(top, lam[i]);
  __syncthreads();   // lam is written again below
  const int power = top > 0.0f && top < INFINITY ? ilogbf(top) : 0;

  Column up[P], lo[P];
  Scalars su, sl;   // of this lane's slot
  float shift = 0.0f;
  for (int attempt = 0; attempt < 2; ++attempt) {
    // Column c of B + shift I; columns and rows past n are zero (and never rotate).
    auto load = [&](int c) {
      Column x;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int r = lane + 64 * e;
        x.g[e] = (r < n && c < n)
                     ? 0.5f * (ldexpf(src[r * n + c], -power) + ldexpf(src[c * n + r], -power))
                     : 0.0f;
        x.v[e] = r == c ? 1.0f : 0.0f;
        if (r == c && c < n) x.g[e] += shift;
      }
      return x;
    };
#pragma unroll
    for (int i = 0; i < P; ++i) {
      up[i] = load(P * wave + i);
      lo[i] = load(SLOTS + P * wave + i);
    }
    su = Scalars{0.0f, 1.0f, slot, 0};
    sl = Scalars{0.0f, 1.0f, SLOTS + slot, 0};
    int parity = 0;

    // Columns multiplied by their factors, and their squared norms.
    auto renormalise = [&]() {
      float pu[P], pl[P];
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const float fu = from_group(su.scale, i), fl = from_group(sl.scale, i);
        pu[i] = pl[i] = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          up[i].g[e] *= fu; up[i].v[e] *= fu;
          lo[i].g[e] *= fl; lo[i].v[e] *= fl;
          pu[i] = fmaf(up[i].g[e], up[i].g[e], pu[i]);
          pl[i] = fmaf(lo[i].g[e], lo[i].g[e], pl[i]);
        }
      }
      su.norm2 = group_sums(pu); su.scale = 1.0f;
      sl.norm2 = group_sums(pl); sl.scale = 1.0f;
    };

    for (int sweep = 0; sweep < a.max_sweeps; ++sweep) {
      bool any = false;
      if (t == 0) rotated = 0;
      // kCols rounds: one more than the circle needs, so that they split into P at a time.
      for (int round = 0; round < kCols; round += P) {
        if (round % kRenorm == 0) renormalise();
#pragma unroll
        for (int r = 0; r < P; ++r) {
          // The registers rotate instead of the columns: slot i's upper column is in
          // up[(i - r) mod P], its lower one in lo[(i + r) mod P].
          auto u = [&](int i) -> Column& { return up[(i - r + P) % P]; };
          auto l = [&](int i) -> Column& { return lo[(i + r) % P]; };
          float dots[P];
#pragma unroll
          for (int i = 0; i < P; ++i) {
            dots[i] = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) dots[i] = fmaf(u(i).g[e], l(i).g[e], dots[i]);
          }
          const float xy = group_sums(dots) * (su.scale * sl.scale);
          const bool turn = fabsf(xy) > kEigenTol * __builtin_amdgcn_sqrtf(su.norm2 * sl.norm2);
          if (__any(turn)) {
            any = true;
            // t = tan of the smaller angle that makes the pair orthogonal; x <- c (x - t y),
            // y <- c (y + t x), the factor c going to the columns' scales.
            const float tau = (sl.norm2 - su.norm2) * 0.5f * __builtin_amdgcn_rcpf(xy);
            const float mag = __builtin_amdgcn_rcpf(fabsf(tau) + __builtin_amdgcn_sqrtf(fmaf(tau, tau, 1.0f)));
            const float tn = turn ? copysignf(mag, tau) : 0.0f;
            const float c = turn ? __builtin_amdgcn_rsqf(fmaf(tn, tn, 1.0f)) : 1.0f;
            const float fu = tn * sl.scale * __builtin_amdgcn_rcpf(su.scale);
            const float fl = tn * su.scale * __builtin_amdgcn_rcpf(sl.scale);
            su.norm2 = turn ? fmaf(-tn, xy, su.norm2) : su.norm2;
            sl.norm2 = turn ? fmaf(tn, xy, sl.norm2) : sl.norm2;
            su.scale *= c;
            sl.scale *= c;
#pragma unroll
            for (int i = 0; i < P; ++i) {
              const float wu = from_group(fu, i), wl = from_group(fl, i);
#pragma unroll
              for (int e = 0; e < E; ++e) {
                const float gx = u(i).g[e], vx = u(i).v[e];
                u(i).g[e] = fmaf(-wu, l(i).g[e], gx);
                u(i).v[e] = fmaf(-wu, l(i).v[e], vx);
                l(i).g[e] = fmaf(wl, gx, l(i).g[e]);
                l(i).v[e] = fmaf(wl, vx, l(i).v[e]);
              }
            }
          }
          // Move on by one slot: upper columns right, lower ones left, turning at the ends;
          // the upper column of slot 0 stays and slot 0's lower one becomes slot 1's upper.
          Column &leave_u = u(P - 1), &leave_l = l(0);   // also the places of those that arrive
          box[parity][0][wave][lane] = leave_u;
          box[parity][1][wave][lane] = leave_l;
          if (leader) {
            if (slot == 0) sc[parity][0][0] = su;
            else if (slot == SLOTS - 1) sc[parity][1][SLOTS - 1] = su;
            else sc[parity][0][slot + 1] = su;
            if (slot == 0) sc[parity][0][1] = sl;
            else sc[parity][1][slot - 1] = sl;
          }
          __syncthreads();
          if (wave == 0) {
            leave_u = u(0);
            u(0) = leave_l;
          } else {
            leave_u = box[parity][0][wave - 1][lane];
          }
          leave_l = wave == NW - 1 ? box[parity][0][wave][lane] : box[parity][1][wave + 1][lane];
          su = sc[parity][0][slot];
          sl = sc[parity][1][slot];
          parity ^= 1;
        }
      }
      if (any) rotated = 1;
      __syncthreads();
      const int more = rotated;
      __syncthreads();   // read by every thread before the next sweep clears it
      if (!more) break;
    }
    renormalise();

    // Rayleigh quotients, squared column norms and squared residuals |g - lambda v|^2.
    auto quotients = [&](Column (&x)[P], const Scalars& s) {
      float vg[P], vv[P], rr[P];
#pragma unroll
      for (int i = 0; i < P; ++i) {
        vg[i] = vv[i] = rr[i] = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          vg[i] = fmaf(x[i].v[e], x[i].g[e], vg[i]);
          vv[i] = fmaf(x[i].v[e], x[i].v[e], vv[i]);
        }
      }
      const float q = group_sums(vg) / group_sums(vv);
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const float qi = from_group(q, i);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float d = fmaf(-qi, x[i].v[e], x[i].g[e]);
          rr[i] = fmaf(d, d, rr[i]);
        }
      }
      const float res = group_sums(rr);
      if (leader) {
        lam[s.index] = q;
        size2[s.index] = s.norm2;
        off2[s.index] = res;
      }
    };
    quotients(up, su);   // every P rounds the registers are back in slot order
    quotients(lo, sl);
    __syncthreads();
    float top2 = 0.0f;
    for (int i = lane; i < n; i += 64) top2 = fmaxf(top2, size2[i]);
    for (int off = 32; off >= 1; off >>= 1) top2 = fmaxf(top2, __shfl_xor(top2, off, 64));
    const float norm = sqrtf(top2);   // the spectral norm of B (first attempt; of its scaled copy)
    bool redo = false;
    for (int i = lane; i < n; i += 64)
      redo |= lam[i] < -2.0e-6f * norm ||
              sqrtf(off2[i]) > fmaf(1.0e-3f, sqrtf(size2[i]), 4.0e-6f * norm);
    redo = __any(redo);
    __syncthreads();
    if (attempt == 1 || !redo) break;   // the same in every wave
    shift = 1.01f * norm;
  }

  // V row by row for the products below, column c at its input index.
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int cu = __builtin_amdgcn_readlane(su.index, i * kLanes);
    const int cl = __builtin_amdgcn_readlane(sl.index, i * kLanes);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      V[(lane + 64 * e) * kEigenMax + cu] = up[i].v[e];
      V[(lane + 64 * e) * kEigenMax + cl] = lo[i].v[e];
    }
  }
  for (int i = t; i < n; i += kEigenThreads) lam[i] = ldexpf(lam[i] - shift, power);
  __syncthreads();

  // One Newton-Schulz step towards the nearest orthogonal matrix, V <- V (3I - V^T V) / 2,
  // removes the rounding drift the sweeps of rotations leave in V's orthogonality (~1e-5
  // at n = 128, down to ~1e-6) without moving it off the eigenvectors.
  const int n4 = (n + 3) / 4;
  for (int tile = t; tile < n4 * n4; tile += kEigenThreads) {
    const int i0 = 4 * (tile / n4), j0 = 4 * (tile % n4);
    float e[4][4] = {};
    for (int r = 0; r < n; ++r) {
      const float4 vi = *reinterpret_cast<const float4*>(&V[r * kEigenMax + i0]);
      const float4 vj = *reinterpret_cast<const float4*>(&V[r * kEigenMax + j0]);
      const float xi[4] = {vi.x, vi.y, vi.z, vi.w}, xj[4] = {vj.x, vj.y, vj.z, vj.w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) e[u][w] = fmaf(xi[u], xj[w], e[u][w]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        A[(i0 + u) * kEigenMax + j0 + w] = e[u][w] - ((i0 + u == j0 + w) ? 1.0f : 0.0f);
  }
  __syncthreads();
  {
    // A row of V times E, kEigenThreads / 64 threads per two rows' 64 E columns: accumulated,
    // then written back after every thread has finished reading V.
    constexpr int kRows = 64 * E, kPer = kRows * kRows / kEigenThreads;   // elements a thread
    constexpr int kThreadsPerRow = kRows / kPer;
    static_assert(kPer % 4 == 0 && kPer * kThreadsPerRow == kRows, "whole rows");
    const int i = t / kThreadsPerRow, j0 = kPer * (t % kThreadsPerRow);
    float acc[kPer];
#pragma unroll
    for (int w = 0; w < kPer; ++w) acc[w] = 0.0f;
    if (i < n) {
      for (int r = 0; r < n; ++r) {
        const float v = V[i * kEigenMax + r];
#pragma unroll
        for (int w = 0; w < kPer; ++w) acc[w] = fmaf(v, A[r * kEigenMax + j0 + w], acc[w]);
      }
    }
    __syncthreads();
    if (i < n) {
#pragma unroll
      for (int w = 0; w < kPer; ++w)
        if (j0 + w < n) V[i * kEigenMax + j0 + w] -= 0.5f * acc[w];
    }
    __syncthreads();
  }

  // Ascending order of the n eigenvalues, ties to the lower index.
  for (int i = t; i < n; i += kEigenThreads) {
    const float li = lam[i];
    int rk = 0;
    for (int j = 0; j < n; ++j) {
      const float lj = lam[j];
      rk += (lj < li) || (lj == li && j < i);
    }
    rank[i] = rk;
    a.values[(int64_t)blockIdx.x * n + rk] = li;
  }
  __syncthreads();
  float* dst = a.vectors + (int64_t)blockIdx.x * n * n;
  for (int idx = t; idx < n * n; idx += kEigenThreads) {
    const int i = idx / n, j = idx % n;
    dst[i * n + rank[j]] = V[i * kEigenMax + j];
  }
}

}  // namespace

hipError_t run_symmetric_eigen(const EigenArgs& a, hipStream_t s) {
  if (a.n < 1 || a.n > kEigenMax || a.batch < 1) return hipErrorInvalidValue;
  if (a.n <= 64)
    hipLaunchKernelGGL((symmetric_eigen_kernel<1, 4>), dim3(a.batch), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((symmetric_eigen_kernel<2, 8>), dim3(a.batch), dim3(512), 0, s, a);
  return hipGetLastError();
}

}  // namespace recap
