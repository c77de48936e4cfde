// Eigen-decomposition of the closure scatter (the first-call basis).
//   symmetric_eigen   eigenvalues and eigenvectors of 0.5 (A + A^T) for a batch of small
//                     fp32 matrices (n <= 128), eigenvalues ascending and eigenvectors as
//                     columns, the contract of torch.linalg.eigh that closure_basis calls
//                     (recap/sparse/closure.py:75-81).
//
// One workgroup per matrix; the matrix and the accumulated rotations live in registers at the
// head dimensions 64 and 128, in LDS (2 x 64 KB) at other orders.  Two-sided cyclic Jacobi
// (Golub & Van Loan, Matrix Computations, 4th ed., alg. 8.5.2 with the symmetric 2x2 Schur rotation of alg. 8.5.1) in the parallel
// round-robin ordering of Brent & Luk (1985): a sweep is m - 1 rounds (m = n rounded up
// to even) of m/2 disjoint index pairs, rotated at once.  In LDS a round is two barriers: the m/2
// threads that own a pair compute its rotation and publish it with the pair, then every
// thread applies J_k^T B J_l to whole 2x2 blocks (k, l) of the matrix, so the row and
// column passes need no barrier between them, and V <- V J to the rotation matrix.
//
// Off-diagonal entries are only ever formed from off-diagonal entries, so the rounding
// noise they carry shrinks with them and the relative test of Demmel & Veselic (1992),
// |a_pq| <= tol sqrt(|a_pp a_qq|), is reached; a sweep that rotates nothing ends the loop,
// and a fixed sweep cap bounds it whatever the input.
#include "kernels.hpp"

namespace recap {

namespace {

constexpr int kEigenMax = 128;
constexpr int kEigenThreads = 1024;    // 4 waves per SIMD hide the LDS latency of a round
constexpr float kEigenTol = 1.0e-7f;   // ~ 2 fp32 ulps of 1

// Pair k of round r in the circle ordering of m (even) indices: every unordered pair once
// per sweep of m - 1 rounds.
__device__ __forceinline__ void round_pair(int m, int r, int k, int& p, int& q) {
  if (k == 0) { p = m - 1; q = r; return; }
  const int c = m - 1;
  p = r + k; if (p >= c) p -= c;
  q = r - k; if (q < 0) q += c;
}

// From the converged V and the diagonal (lam) to the sorted outputs, by THREADS threads; A is
// scratch and rank an LDS array of kEigenMax.
template <int THREADS>
__device__ __forceinline__ void finish(const EigenArgs& a, float* A, float* V, float* lam, int* rank) {
  const int t = threadIdx.x, n = a.n;
  // One Newton-Schulz step towards the nearest orthogonal matrix, V <- V (3I - V^T V) / 2,
  // removes the rounding drift the sweeps of rotations leave in V's orthogonality (~1e-5
  // at n = 128, down to ~1e-6) without moving it off the eigenvectors.
  const int n4 = (n + 3) / 4;
  for (int tile = t; tile < n4 * n4; tile += THREADS) {
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
    // THREADS / 128 threads per row: a piece of row i of V (E) accumulated, then written back
    // after every thread has finished reading V.
    constexpr int kPer = kEigenMax * kEigenMax / THREADS;
    const int i = t / (kEigenMax / kPer), j0 = kPer * (t % (kEigenMax / kPer));
    float acc[kPer];
#pragma unroll
    for (int w = 0; w < kPer; ++w) acc[w] = 0.0f;
    if (i < n && j0 < n) {
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
  }

  // Ascending order of the n real eigenvalues, ties to the lower index (the padded index
  // n, when n is odd, is an isolated zero row and is dropped).
  for (int i = t; i < n; i += THREADS) {
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
  for (int idx = t; idx < n * n; idx += THREADS) {
    const int i = idx / n, j = idx % n;
    dst[i * n + rank[j]] = V[i * kEigenMax + j];
  }
}


__global__ __launch_bounds__(kEigenThreads) void symmetric_eigen_kernel(EigenArgs a) {
  __shared__ __attribute__((aligned(16))) float A[kEigenMax * kEigenMax];
  __shared__ __attribute__((aligned(16))) float V[kEigenMax * kEigenMax];
  __shared__ float rot_c[kEigenMax / 2], rot_s[kEigenMax / 2];
  __shared__ int pair_p[kEigenMax / 2], pair_q[kEigenMax / 2];
  __shared__ float lam[kEigenMax];
  __shared__ int rank[kEigenMax];
  __shared__ int rotated;
  const int t = threadIdx.x, n = a.n, m = a.m, half = m / 2;
  // Fixed work map of a round: pair column l = t % 64 for every block (k, l) and rotation
  // column of this thread, pair rows k = t / 64 + 16 j (blocks) and V rows i = t / 64 + 16 j.
  const int l = t & 63, k0 = t >> 6;
  const float* src = a.a + (int64_t)blockIdx.x * n * n;

  // The whole 128 x 128 storage is defined (zero outside n x n, V = I) so the tiled
  // products below may read past n.
  for (int idx = t; idx < kEigenMax * kEigenMax; idx += kEigenThreads) {
    const int i = idx >> 7, j = idx & (kEigenMax - 1);
    float x = 0.0f;
    if (i < n && j < n) x = 0.5f * (src[i * n + j] + src[j * n + i]);
    A[idx] = x;
    V[idx] = (i == j) ? 1.0f : 0.0f;
  }
  if (t == 0) rotated = 0;
  __syncthreads();

  for (int sweep = 0; sweep < a.max_sweeps; ++sweep) {
    for (int r = 0; r < m - 1; ++r) {
      if (t < half) {
        int p, q;
        round_pair(m, r, t, p, q);
        const float app = A[p * kEigenMax + p], aqq = A[q * kEigenMax + q];
        const float apq = A[p * kEigenMax + q];
        float c = 1.0f, s = 0.0f;
        if (fabsf(apq) > kEigenTol * sqrtf(fabsf(app * aqq)) && apq != 0.0f) {
          // t = tan(theta) of the smaller rotation that zeroes a_pq (alg. 8.5.1).
          const float tau = (aqq - app) / (2.0f * apq);
          const float tn = copysignf(1.0f, tau) / (fabsf(tau) + sqrtf(1.0f + tau * tau));
          c = 1.0f / sqrtf(1.0f + tn * tn);
          s = tn * c;
          rotated = 1;
        }
        rot_c[t] = c; rot_s[t] = s;
        pair_p[t] = p; pair_q[t] = q;
      }
      __syncthreads();
      if (l < half) {
        const int pl = pair_p[l], ql = pair_q[l];
        const float cl = rot_c[l], sl = rot_s[l];
        // B <- J^T B J over 2x2 blocks: rows (p_k, q_k), columns (p_l, q_l).
#pragma unroll
        for (int j = 0; j < kEigenMax / 2 / (kEigenThreads / 64); ++j) {
          const int k = k0 + (kEigenThreads / 64) * j;
          if (k >= half) break;
          const int pk = pair_p[k], qk = pair_q[k];
          const float ck = rot_c[k], sk = rot_s[k];
          if (k == l) {
            // Diagonal block: the closed form, with the zeroed entry set exactly.
            const float apq = A[pk * kEigenMax + qk];
            const float tn = (ck != 0.0f) ? sk / ck : 0.0f;
            A[pk * kEigenMax + pk] -= tn * apq;
            A[qk * kEigenMax + qk] += tn * apq;
            if (sk != 0.0f) { A[pk * kEigenMax + qk] = 0.0f; A[qk * kEigenMax + pk] = 0.0f; }
            continue;
          }
          const float b_pp = A[pk * kEigenMax + pl], b_pq = A[pk * kEigenMax + ql];
          const float b_qp = A[qk * kEigenMax + pl], b_qq = A[qk * kEigenMax + ql];
          // rows: r_p = c_k b_p - s_k b_q, r_q = s_k b_p + c_k b_q
          const float r_pp = ck * b_pp - sk * b_qp, r_pq = ck * b_pq - sk * b_qq;
          const float r_qp = sk * b_pp + ck * b_qp, r_qq = sk * b_pq + ck * b_qq;
          // columns: x_p = c_l r_p - s_l r_q, x_q = s_l r_p + c_l r_q
          A[pk * kEigenMax + pl] = cl * r_pp - sl * r_pq;
          A[pk * kEigenMax + ql] = sl * r_pp + cl * r_pq;
          A[qk * kEigenMax + pl] = cl * r_qp - sl * r_qq;
          A[qk * kEigenMax + ql] = sl * r_qp + cl * r_qq;
        }
        // V <- V J: columns (p_l, q_l) of rows i.
#pragma unroll
        for (int j = 0; j < kEigenMax / (kEigenThreads / 64); ++j) {
          const int i = k0 + (kEigenThreads / 64) * j;
          if (i >= m) break;
          const float vp = V[i * kEigenMax + pl], vq = V[i * kEigenMax + ql];
          V[i * kEigenMax + pl] = cl * vp - sl * vq;
          V[i * kEigenMax + ql] = sl * vp + cl * vq;
        }
      }
      __syncthreads();
    }
    const int any = rotated;   // read by every thread after the round's last barrier
    __syncthreads();
    if (t == 0) rotated = 0;
    __syncthreads();
    if (!any) break;
  }

  for (int i = t; i < n; i += kEigenThreads) lam[i] = A[i * kEigenMax + i];
  __syncthreads();
  finish<kEigenThreads>(a, A, V, lam, rank);
}

// The rotation that zeroes a_pq (alg. 8.5.1): t = tan(theta) of the smaller angle; c = 1 and
// s = 0 for an entry that is small already.  Branch-free, so that the test's chain of operations
// and the rotation's run side by side (a two-layer schedule with two 4 x 64 decompositions: 2040 ->
// 1973 us; at 128 no difference); a rotation that is not taken may divide by zero, and its result
// is dropped.
__device__ __forceinline__ bool jacobi_rotation(float app, float aqq, float apq, float& c, float& s) {
  const bool turn = fabsf(apq) > kEigenTol * sqrtf(fabsf(app * aqq)) && apq != 0.0f;
  const float tau = (aqq - app) / (2.0f * apq);
  const float tn = copysignf(1.0f, tau) / (fabsf(tau) + sqrtf(1.0f + tau * tau));
  const float ct = 1.0f / sqrtf(1.0f + tn * tn);
  c = turn ? ct : 1.0f;
  s = turn ? tn * ct : 0.0f;
  return turn;
}

// The same sweeps for n = N = 64 or 128 (the head dimensions) with A and V in registers, every
// element by the operations of the kernel above, which took these orders before (values and
// vectors compared bit for bit then, on 16 batches: scatters, indefinite, diagonal, rank 3, zero).
// Slot k of a round is its pair k; a lane holds one slot's rows (two elements, row p and row q of
// a column) and a wave eight slots' columns, so a 2 x 2 block (k, l) is in one lane.  From a
// round to the next the circle ordering moves every column and every row by one
// slot (q's right, p's left, p of slot 0 staying, q of the last slot turning into its p, p of
// slot 1 into q of slot 0): rows move by lane shifts, columns by the register renaming of an
// eightfold unrolled loop, and only the two columns that leave a wave go through LDS, with one
// barrier a round.  VALU issue bounds it, about 400 instructions a wave and round (the blocks'
// and V's rotations 190, the row moves 85, the rotation itself with its IEEE divisions and
// roots 75), two waves a SIMD at N = 128, 1.65 us a round.  The kernel above moves both matrices
// through LDS, 256 KB a round, behind two barriers: 3.84 ms for 12 matrices of order 128 and
// 1.05 ms for 4 of order 64; here 1.91 and 0.53 ms.
template <int N>
__global__ __launch_bounds__(4 * N) void symmetric_eigen_ring_kernel(EigenArgs a) {
  constexpr int SLOTS = N / 2, P = 8, NW = SLOTS / P, E = N / 64, THREADS = 64 * NW;
  static_assert(THREADS == 4 * N && (N - 1) % P == P - 1, "whole waves; a sweep ends at the 8th round");
  struct Column { float gp, gq, v[E]; };  // rows p and q of this lane's slot; rows lane + 64 e of V
  __shared__ __attribute__((aligned(16))) float A[kEigenMax * kEigenMax];
  __shared__ __attribute__((aligned(16))) float V[kEigenMax * kEigenMax];
  __shared__ float lam[kEigenMax];
  __shared__ int rank[kEigenMax];
  // During the sweeps the matrices' storage holds, for alternate rounds, the columns that move
  // and the entries a_pq of the next round's pairs.
  auto& box = *reinterpret_cast<Column (*)[2][2][NW][64]>(A);   // [parity][q, p][wave][lane]
  auto& entry = *reinterpret_cast<float (*)[2][64]>(V);         // [parity][slot]
  static_assert(sizeof(Column) * 4 * NW * 64 <= sizeof(A), "storage");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int mine = lane - P * wave;   // the column of this wave whose slot is this lane's
  const bool first = lane == 0, last = lane == SLOTS - 1;
  const float* src = a.a + (int64_t)blockIdx.x * N * N;

  // Round 0: p of slot 0 is N - 1 and its q is 0, slot k >= 1 holds p = k and q = N - 1 - k.
  auto p_index = [](int k) { return k == 0 ? N - 1 : k; };
  auto q_index = [](int k) { return k == 0 ? 0 : N - 1 - k; };
  const int slot = lane & (SLOTS - 1);
  auto load = [&](int j) {
    Column x;
    const int rp = p_index(slot), rq = q_index(slot);
    x.gp = 0.5f * (src[rp * N + j] + src[j * N + rp]);
    x.gq = 0.5f * (src[rq * N + j] + src[j * N + rq]);
#pragma unroll
    for (int e = 0; e < E; ++e) x.v[e] = lane + 64 * e == j ? 1.0f : 0.0f;
    return x;
  };
  Column pc[P], qc[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    pc[i] = load(p_index(P * wave + i));
    qc[i] = load(q_index(P * wave + i));
  }

  // The diagonal is only ever read by the rotation of its own pair, so every wave keeps all of
  // it, slot k's a_pp and a_qq in lane k, and the columns' own diagonal elements are not kept
  // up (they stay bounded).
  float app = src[p_index(slot) * (N + 1)], aqq = src[q_index(slot) * (N + 1)];
  app = 0.5f * (app + app);
  aqq = 0.5f * (aqq + aqq);
  int parity = 0;
#pragma unroll
  for (int i = 0; i < P; ++i)
    if (mine == i && lane < SLOTS) entry[0][lane] = qc[i].gp;
  __syncthreads();

  for (int sweep = 0; sweep < a.max_sweeps; ++sweep) {
    bool any = false;
    for (int round = 0;; round += P) {
#pragma unroll
      for (int r = 0; r < P; ++r) {
        if (r == P - 1 && round + r == N - 1) break;   // N - 1 rounds a sweep
        // Slot i's p column is in pc[(i + r) mod P], its q column in qc[(i - r) mod P].
        auto p = [&](int i) -> Column& { return pc[(i + r) % P]; };
        auto q = [&](int i) -> Column& { return qc[(i - r + P) % P]; };
        // Every wave computes every slot's rotation, slot k in lane k.
        const float apq = entry[parity][slot];
        parity ^= 1;
        float ck, sk;
        // (At N = 64 the upper lanes hold no slot; what they compute is not used.)
        const bool turn = jacobi_rotation(app, aqq, apq, ck, sk) && lane < SLOTS;
        if (__any(turn)) {   // the same in every wave; without a rotation nothing changes
          any = true;
          // Diagonal blocks: the closed form, with the zeroed entries set exactly.
          const float tn = sk / ck;
          app = fmaf(-tn, apq, app);
          aqq = fmaf(tn, apq, aqq);
          const int zeroed = sk != 0.0f ? mine : -1;
#pragma unroll
          for (int i = 0; i < P; ++i) {
            const float cl = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(ck), P * wave + i));
            const float sl = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(sk), P * wave + i));
            Column &cp = p(i), &cq = q(i);
            // rows: r_p = c_k b_p - s_k b_q, r_q = s_k b_p + c_k b_q
            const float r_pp = fmaf(ck, cp.gp, -(sk * cp.gq)), r_pq = fmaf(ck, cq.gp, -(sk * cq.gq));
            const float r_qp = fmaf(sk, cp.gp, ck * cp.gq), r_qq = fmaf(sk, cq.gp, ck * cq.gq);
            // columns: x_p = c_l r_p - s_l r_q, x_q = s_l r_p + c_l r_q
            cp.gp = fmaf(cl, r_pp, -(sl * r_pq));
            cq.gq = fmaf(sl, r_qp, cl * r_qq);
            const float x_pq = fmaf(sl, r_pp, cl * r_pq), x_qp = fmaf(cl, r_qp, -(sl * r_qq));
            cq.gp = zeroed == i ? 0.0f : x_pq;
            cp.gq = zeroed == i ? 0.0f : x_qp;
#pragma unroll
            for (int e = 0; e < E; ++e) {
              const float vp = cp.v[e], vq = cq.v[e];
              cp.v[e] = fmaf(cl, vp, -(sl * vq));
              cq.v[e] = fmaf(sl, vp, cl * vq);
            }
          }
        }
        // Rows move by one slot, in every column and in the diagonal.
        auto move_rows = [&](float& xp, float& xq) {
          constexpr int kLeft = 0x130, kRight = 0x138;   // wave_shl:1, wave_shr:1
          const int gp = (int)__float_as_uint(xp), gq = (int)__float_as_uint(xq);
          int up = __builtin_amdgcn_update_dpp(gq, gp, kLeft, 0xf, 0xf, false);  // lane + 1's p
          if constexpr (SLOTS < 64) up = last ? gq : up;   // (of 64, the last keeps the old value)
          const int uq = __builtin_amdgcn_update_dpp(up, gq, kRight, 0xf, 0xf, false);
          xp = first ? xp : __uint_as_float((unsigned)up);
          xq = __uint_as_float((unsigned)uq);
        };
#pragma unroll
        for (int i = 0; i < P; ++i) {
          move_rows(pc[i].gp, pc[i].gq);
          move_rows(qc[i].gp, qc[i].gq);
        }
        move_rows(app, aqq);
        // The next round's a_pq: the q column of slot k >= 1 is this round's of slot k - 1, that
        // of slot 0 this round's p column of slot 1.
        float next = p(1).gp;
#pragma unroll
        for (int i = 0; i < P; ++i) next = mine == i + 1 ? q(i).gp : next;
        if (lane < SLOTS && ((mine >= 1 && mine <= P) || (wave == 0 && first))) entry[parity][lane] = next;
        // Columns move by one slot: out of this wave through LDS, the others by renaming.
        Column &leave_q = q(P - 1), &leave_p = p(0);
        box[parity][0][wave][lane] = leave_q;
        box[parity][1][wave][lane] = leave_p;
        __syncthreads();   // (a wave is at most one round ahead of another: two parities do)
        if (wave == 0) {
          leave_q = p(1);
          p(1) = leave_p;
        } else {
          leave_q = box[parity][0][wave - 1][lane];
        }
        leave_p = wave == NW - 1 ? box[parity][0][wave][lane] : box[parity][1][wave + 1][lane];
      }
      if (round + P - 1 == N - 1) break;
    }
    // Seven rounds into the unrolled loop: the columns back to the registers of round 0.
    Column np[P], nq[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      np[i] = pc[(i + P - 1) % P];
      nq[i] = qc[(i + 1) % P];
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      pc[i] = np[i];
      qc[i] = nq[i];
    }
    if (!any) break;   // the same in every wave
  }
  __syncthreads();   // the last columns and entries are read before V is written

#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int k = P * wave + i, jp = p_index(k), jq = q_index(k);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      V[(lane + 64 * e) * kEigenMax + jp] = pc[i].v[e];
      V[(lane + 64 * e) * kEigenMax + jq] = qc[i].v[e];
    }
  }
  if (t < SLOTS) {
    lam[p_index(slot)] = app;
    lam[q_index(slot)] = aqq;
  }
  __syncthreads();
  finish<THREADS>(a, A, V, lam, rank);
}

}  // namespace

hipError_t run_symmetric_eigen(const EigenArgs& a, hipStream_t s) {
  if (a.n < 1 || a.n > kEigenMax || a.m != a.n + (a.n & 1) || a.batch < 1)
    return hipErrorInvalidValue;
  if (a.n == 128) {
    hipLaunchKernelGGL(symmetric_eigen_ring_kernel<128>, dim3(a.batch), dim3(512), 0, s, a);
    return hipGetLastError();
  }
  if (a.n == 64) {
    hipLaunchKernelGGL(symmetric_eigen_ring_kernel<64>, dim3(a.batch), dim3(256), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(symmetric_eigen_kernel, dim3(a.batch), dim3(kEigenThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace recap
