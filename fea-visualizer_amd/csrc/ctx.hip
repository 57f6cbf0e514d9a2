// ctx.hip -- mesh context: idx_map, CSR pattern and deterministic P1
// assembly of the stiffness K, mass M and advection A matrices on the GPU.
//
// Reference behaviour restated (tvumcc/fea-visualizer):
//   idx_map                 src/FEM/FEMContext.cpp:224-240
//   K (surface gradients)   src/FEM/FEMContext.cpp:70-113
//   M (|J|/24 [2 1 1;..])   src/FEM/FEMContext.cpp:119-150
//   A (area/3 v.grad phi_j) src/FEM/FEMContext.cpp:156-202
//   max row nonzeros        src/FEM/FEMContext.cpp:207-219
// The pattern is the set of (idx(i), idx(j)) over triangles sharing i and j
// that pass the boundary filter, sorted per row, explicit zeros kept -- the
// pattern Eigen's setFromTriplets builds, which every system matrix of the
// reference shares.  Values are summed per entry in (element, i, j) order, the
// order setFromTriplets sums duplicate triplets in, without atomics: one
// thread owns one row and walks the row vertex's incident triangles in
// ascending element order.
#include "femhip_ctx.h"
#include "femhip_geom.h"

#include <algorithm>
#include <cstring>

namespace femhip {

namespace {

__global__ void k_keep(const uint8_t* onb, int nv, int bc, int* keep) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nv) keep[i] = (bc == FEM_NEUMANN || !onb[i]) ? 1 : 0;
}

__global__ void k_idx_map(const uint8_t* onb, int nv, int bc, const int* offs, int* idx, int* row2v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  bool keep = (bc == FEM_NEUMANN || !onb[i]);
  int r = keep ? offs[i] : -1;
  idx[i] = r;
  if (keep) row2v[r] = i;
}

// Incidence counts: each triangle counted once per distinct vertex.
__global__ void k_inc_count(const uint32_t* tri, int ntri, int* cnt) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntri) return;
  uint32_t a = tri[3 * (size_t)t], b = tri[3 * (size_t)t + 1], c = tri[3 * (size_t)t + 2];
  atomicAdd(&cnt[a], 1);
  if (b != a) atomicAdd(&cnt[b], 1);
  if (c != a && c != b) atomicAdd(&cnt[c], 1);
}

__global__ void k_inc_fill(const uint32_t* tri, int ntri, const int* inc_ptr, int* cursor, int* inc) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntri) return;
  uint32_t v3[3] = {tri[3 * (size_t)t], tri[3 * (size_t)t + 1], tri[3 * (size_t)t + 2]};
  for (int a = 0; a < 3; a++) {
    bool dup = false;
    for (int q = 0; q < a; q++) dup |= (v3[q] == v3[a]);
    if (dup) continue;
    int pos = inc_ptr[v3[a]] + atomicAdd(&cursor[v3[a]], 1);
    inc[pos] = t;
  }
}

// Atomic fill order is arbitrary; sorting each vertex's list restores the
// ascending element order the summation relies on.
__global__ void k_inc_sort(const int* inc_ptr, int nv, int* inc) {
  int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  int lo = inc_ptr[v], hi = inc_ptr[v + 1];
  for (int i = lo + 1; i < hi; i++) {
    int key = inc[i];
    int j = i - 1;
    while (j >= lo && inc[j] > key) {
      inc[j + 1] = inc[j];
      j--;
    }
    inc[j + 1] = key;
  }
}

// Distinct columns of row r (vertex i) in ascending order: the unknowns of the
// incident triangles' vertices (those that pass the boundary filter, which for
// a vertex that has a row are the ones with an unknown).  mode 0 counts, mode 1
// writes col_idx and the diagonal position.
//
// Bound by latency: a thread's chain is incidence -> triangle -> unknown, then
// the merge.  kChunk triangles are loaded at once and merged into a sorted list
// of the thread's own in LDS (rows hold ~7 entries); a row past kListCap
// entries searches its next larger column over the triangles again and again.
// The search alone, for every row, took 131 us a launch at 261K rows, the list
// 23.
constexpr int kChunk = 3;
constexpr int kListCap = 16;
__global__ void __launch_bounds__(kBlock) k_row_cols(const uint32_t* __restrict__ tri, const int* __restrict__ idx,
                                                     const int* __restrict__ row2v, const int* __restrict__ inc_ptr,
                                                     const int* __restrict__ inc, int n, int mode,
                                                     int* __restrict__ cnt, const int* __restrict__ rp,
                                                     int* __restrict__ ci, int* __restrict__ diag) {
  __shared__ int list[kListCap][kBlock];
  const int r = blockIdx.x * kBlock + threadIdx.x, tid = threadIdx.x;
  if (r >= n) return;
  const int i = row2v[r];
  const int lo = inc_ptr[i], hi = inc_ptr[i + 1];
  int c = 0;
  bool fits = true;
  for (int e0 = lo; e0 < hi && fits; e0 += kChunk) {
    int col[kChunk][3];
#pragma unroll
    for (int u = 0; u < kChunk; u++) {
      const size_t t = 3 * (size_t)inc[min(e0 + u, hi - 1)];
#pragma unroll
      for (int b = 0; b < 3; b++) col[u][b] = idx[tri[t + b]];
    }
#pragma unroll
    for (int u = 0; u < kChunk; u++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const int w = col[u][b];
        if (w < 0) continue;
        int q = c;  // list[0..q) < w
        while (q > 0 && list[q - 1][tid] > w) q--;
        if (q > 0 && list[q - 1][tid] == w) continue;
        if (c == kListCap) {
          fits = false;
          continue;
        }
        for (int m = c; m > q; m--) list[m][tid] = list[m - 1][tid];
        list[q][tid] = w;
        c++;
      }
  }
  const int out = mode == 1 ? rp[r] : 0;
  int dpos = -1;
  if (fits) {
    if (mode == 1)
      for (int q = 0; q < c; q++) {
        const int w = list[q][tid];
        ci[out + q] = w;
        if (w == r) dpos = out + q;
      }
  } else {
    c = 0;
    for (int last = -1;; c++) {
      int best = INT32_MAX;
      for (int e = lo; e < hi; e++)
        for (int b = 0; b < 3; b++) {
          const int w = idx[tri[3 * (size_t)inc[e] + b]];
          if (w > last && w < best) best = w;
        }
      if (best == INT32_MAX) break;
      if (mode == 1) {
        ci[out + c] = best;
        if (best == r) dpos = out + c;
      }
      last = best;
    }
  }
  if (mode == 0) cnt[r] = c;
  else diag[r] = dpos;
}

// Position of col in the ascending cols[0..m); col is there.
__device__ inline int find_slot(const int* cols, int m, int col) {
  int lo = 0;
  while (m > 1) {
    const int half = m >> 1;
    if (cols[lo + half] <= col) lo += half;
    m -= half;
  }
  return lo;
}

// K, M, A of the mesh and M's row sums.  A thread owns a row and walks the row
// vertex's triangles in ascending element order.
//
// Bound by latency and by the FP64 divides of the geometry (each triangle is
// formed by its three rows).  The workgroup's rows are one stretch of the CSR
// arrays, so their columns and sums stay in LDS and the stretch is written
// once, in whole lines; kChunk triangles' vertices are in flight at once.
// Accumulating in global memory instead chained a search of the row's columns
// and three read-modify-writes per triangle corner: 409 us at 261K rows, 68
// now.  Blocks whose rows average more than kAsmRow entries (~7 on a surface)
// still accumulate there.
constexpr int kAsmBlock = 64, kAsmRow = 8, kAsmCap = kAsmBlock * kAsmRow;
__global__ void __launch_bounds__(kAsmBlock) k_assemble(
    const float* __restrict__ xyz, const uint32_t* __restrict__ tri, const uint8_t* __restrict__ onb,
    const int* __restrict__ idx, const int* __restrict__ row2v, const int* __restrict__ inc_ptr,
    const int* __restrict__ inc, const int* __restrict__ rp, const int* __restrict__ ci, int n, int bc, double vx,
    double vy, double vz, const double* __restrict__ vel_e, int normalize, const double* __restrict__ kappa_e,
    double* __restrict__ K, double* __restrict__ M, double* __restrict__ A, double* __restrict__ lumped) {
  __shared__ int s_ci[kAsmCap];
  __shared__ double s_K[kAsmCap], s_M[kAsmCap], s_A[kAsmCap];
  const int row0 = blockIdx.x * kAsmBlock, tid = threadIdx.x;
  const int base = rp[row0], end = rp[min(n, row0 + kAsmBlock)];
  const bool staged = end - base <= kAsmCap;
  if (staged)
    for (int s = tid; s < end - base; s += kAsmBlock) {
      s_ci[s] = ci[base + s];
      s_K[s] = 0.0;
      s_M[s] = 0.0;
      s_A[s] = 0.0;
    }
  __syncthreads();
  const int r = row0 + tid;
  // cols, k, m, a: the row's m_row columns and sums, in LDS or in memory
  auto row = [&](const int* cols, int m_row, double* k, double* m, double* a) __attribute__((always_inline)) {
    const int i = row2v[r];
    const bool bi = onb[i] != 0;
    const int hi = inc_ptr[i + 1];
    for (int e0 = inc_ptr[i]; e0 < hi; e0 += kChunk) {
      int t[kChunk];
      uint32_t v[kChunk][3];
      float p[kChunk][3][3];
      int col[kChunk][3];
      bool bw[kChunk][3];
#pragma unroll
      for (int u = 0; u < kChunk; u++) t[u] = inc[min(e0 + u, hi - 1)];
#pragma unroll
      for (int u = 0; u < kChunk; u++)
#pragma unroll
        for (int b = 0; b < 3; b++) v[u][b] = tri[3 * (size_t)t[u] + b];
#pragma unroll
      for (int u = 0; u < kChunk; u++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
          for (int q = 0; q < 3; q++) p[u][b][q] = xyz[3 * (size_t)v[u][b] + q];
          col[u][b] = idx[v[u][b]];
          bw[u][b] = onb[v[u][b]] != 0;
        }
#pragma unroll
      for (int u = 0; u < kChunk; u++) {
        if (e0 + u >= hi) break;
        Geo G;
        elem_geom_at(p[u], G);
        const double kap = kappa_e ? kappa_e[t[u]] : 1.0;
        const double mo = G.jdet / 24.0;
        double vel[3] = {vx, vy, vz};
        if (vel_e)
          for (int q = 0; q < 3; q++) vel[q] = vel_e[3 * (size_t)t[u] + q];
        // FEMContext.cpp:179-180: tangential projection, then normalised
        const double nn = G.nrm[0] * G.nrm[0] + G.nrm[1] * G.nrm[1] + G.nrm[2] * G.nrm[2];
        const double vd = (vel[0] * G.nrm[0] + vel[1] * G.nrm[1] + vel[2] * G.nrm[2]) / nn;
        double tvel[3];
        for (int q = 0; q < 3; q++) tvel[q] = vel[q] - vd * G.nrm[q];
        if (normalize) {
          const double z = tvel[0] * tvel[0] + tvel[1] * tvel[1] + tvel[2] * tvel[2];
          if (z > 0.0) {
            const double sz = sqrt(z);
            for (int q = 0; q < 3; q++) tvel[q] = tvel[q] / sz;
          }
        }
        const double jd6 = G.jdet / 6.0;
        // the row vertex is one corner (a degenerate triangle may repeat it)
        unsigned corners = 0;
#pragma unroll
        for (int c = 0; c < 3; c++) corners |= v[u][c] == (uint32_t)i ? 1u << c : 0u;
        while (corners) {
          const int c = __ffs(corners) - 1;
          corners &= corners - 1;
          double gc[3];
#pragma unroll
          for (int q = 0; q < 3; q++) gc[q] = c == 0 ? G.g[0][q] : c == 1 ? G.g[1][q] : G.g[2][q];
#pragma unroll
          for (int b = 0; b < 3; b++) {
            const bool keep_km = (bc == FEM_NEUMANN) || (!bi && !bw[u][b]);  // FEMContext.cpp:99,136
            const bool keep_a = !bi && !bw[u][b];                            // FEMContext.cpp:188
            if (!keep_km && !keep_a) continue;
            const int s = find_slot(cols, m_row, col[u][b]);
            if (keep_km) {
              const double kab = G.area * (gc[0] * G.g[b][0] + gc[1] * G.g[b][1] + gc[2] * G.g[b][2]);  // elem_kab
              k[s] += kap * kab;
              m[s] += (c == b) ? 2.0 * mo : mo;
            }
            if (keep_a) a[s] += jd6 * (tvel[0] * G.g[b][0] + tvel[1] * G.g[b][1] + tvel[2] * G.g[b][2]);
          }
        }
      }
    }
    double acc = 0.0;
    for (int s = 0; s < m_row; s++) acc += m[s];
    lumped[r] = acc;
  };
  if (r < n) {
    const int lo = rp[r], m_row = rp[r + 1] - lo;
    if (staged) {
      row(s_ci + (lo - base), m_row, s_K + (lo - base), s_M + (lo - base), s_A + (lo - base));
    } else {
      for (int s = lo; s < lo + m_row; s++) {
        K[s] = 0.0;
        M[s] = 0.0;
        A[s] = 0.0;
      }
      row(ci + lo, m_row, K + lo, M + lo, A + lo);
    }
  }
  __syncthreads();
  if (staged)
    for (int s = tid; s < end - base; s += kAsmBlock) {
      K[base + s] = s_K[s];
      M[base + s] = s_M[s];
      A[base + s] = s_A[s];
    }
}

// Position of (c, r) for every CSR entry (r, c); the pattern is structurally
// symmetric, so A^T reuses row_ptr / col_idx with permuted values.
__global__ void k_tperm(const int* rp, const int* ci, int n, int* tperm) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  for (int s = rp[r]; s < rp[r + 1]; s++) {
    int c = ci[s];
    int lo = rp[c], hi = rp[c + 1];
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (ci[mid] < r) lo = mid + 1;
      else hi = mid;
    }
    tperm[s] = lo;
  }
}

}  // namespace

void ctx_free(fem_ctx* c) {
  if (!c) return;
  void* ptrs[] = {c->d_slabs[0], c->d_slabs[1], c->d_kappa_e, c->d_vel_e};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

int ctx_assemble(fem_ctx* c, const fem_assembly_params* prm) {
  int rc = 0;
  fem_assembly_params p;
  if (prm) {
    p = *prm;
  } else {
    std::memset(&p, 0, sizeof(p));
    p.velocity[0] = 1.0;  // AdvectionDiffusionParameters default (1,0,0)
    p.normalize_velocity = 1;
  }
  // Element coefficients, in host or device memory, go to buffers that the
  // context keeps: freeing them waited for the device and unmapped 17 MB,
  // 3.1 ms of an assembly with 520K triangles.
  const double *kappa = nullptr, *vel = nullptr;
  auto take = [&](const double* src, size_t count, double** buf, const double** out) -> int {
    if (!src) return 0;
    if (!*buf) *buf = dalloc<double>(count, &rc);
    if (!*buf) return rc;
    FEM_HIP(hipMemcpyAsync(*buf, src, sizeof(double) * count, hipMemcpyDefault, c->stream));
    *out = *buf;
    return 0;
  };
  if (int r = take(p.kappa_e, (size_t)c->ntri, &c->d_kappa_e, &kappa)) return r;
  if (int r = take(p.velocity_e, 3 * (size_t)c->ntri, &c->d_vel_e, &vel)) return r;
  c->normalize = p.normalize_velocity;
  for (int q = 0; q < 3; q++) c->velocity[q] = p.velocity[q];
  if (c->n > 0) {
    hipLaunchKernelGGL(k_assemble, dim3(div_up(c->n, kAsmBlock)), dim3(kAsmBlock), 0, c->stream, c->d_xyz, c->d_tri,
                       c->d_onb, c->d_idx, c->d_row2v, c->d_inc_ptr, c->d_inc, c->d_rp, c->d_ci, c->n, c->bc,
                       p.velocity[0], p.velocity[1], p.velocity[2], vel, p.normalize_velocity,
                       kappa, c->d_K, c->d_M, c->d_A, c->d_lumped);
    FEM_HIP(hipGetLastError());
  }
  FEM_HIP(hipStreamSynchronize(c->stream));
  c->version++;
  return 0;
}

int ctx_create(const fem_mesh* mesh, int bc, fem_ctx** out) {
  int rc = 0;
  fem_ctx* c = new fem_ctx();
  c->nv = mesh->num_vertices;
  c->ntri = mesh->num_triangles;
  c->bc = bc;
  const int nv = c->nv, nt = c->ntri;
  uint32_t top = 0;  // a plain maximum: the loop vectorises
  for (long long q = 0; q < 3LL * nt; q++) top = std::max(top, mesh->triangles[q]);
  if (nt > 0 && top >= (uint32_t)nv) {
    ctx_free(c);
    set_error("fem_ctx_create: triangle index out of range");
    return FEM_ERR_INVALID;
  }
#define CK(x)                  \
  do {                         \
    int rc_ = (x);             \
    if (rc_) {                 \
      ctx_free(c);             \
      return rc_;              \
    }                          \
  } while (0)
#define CKH(x)                                  \
  do {                                          \
    hipError_t e_ = (x);                        \
    if (e_ != hipSuccess) {                     \
      ctx_free(c);                              \
      return hip_fail(e_, #x);                  \
    }                                           \
  } while (0)
  CKH(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  // One slab for the mesh and the rows, whose number the host counts from the
  // boundary flags, and one for the entries: an allocation each instead of 19
  // (and as many frees, each a wait for the device), and no wait for a count
  // but the entries'.
  int n = 0;
  for (int i = 0; i < nv; i++) n += (bc == FEM_NEUMANN || !mesh->on_boundary[i]) ? 1 : 0;
  c->n = n;
  size_t need = 0;
  auto place = [&](size_t bytes) {
    const size_t at = need;
    need += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t o_xyz = place(sizeof(float) * 3 * (size_t)nv), o_tri = place(sizeof(uint32_t) * 3 * (size_t)nt);
  const size_t o_onb = place((size_t)nv), o_idx = place(sizeof(int) * ((size_t)nv + 1));
  const size_t o_ptr = place(sizeof(int) * ((size_t)nv + 1)), o_inc = place(sizeof(int) * 3 * (size_t)nt);
  const size_t o_keep = place(sizeof(int) * ((size_t)nv + 1)), o_scan = place(sizeof(int) * scan_scratch(nv + 1));
  const size_t o_row = place(sizeof(int) * ((size_t)n + 1)), o_rp = place(sizeof(int) * ((size_t)n + 1));
  const size_t o_diag = place(sizeof(int) * ((size_t)n + 1)), o_lump = place(sizeof(double) * ((size_t)n + 1));
  char* slab = c->d_slabs[0] = dalloc<char>(need, &rc);
  if (rc) { ctx_free(c); return rc; }
  c->d_xyz = (float*)(slab + o_xyz);
  c->d_tri = (uint32_t*)(slab + o_tri);
  c->d_onb = (uint8_t*)(slab + o_onb);
  c->d_idx = (int*)(slab + o_idx);
  c->d_inc_ptr = (int*)(slab + o_ptr);
  c->d_inc = (int*)(slab + o_inc);
  c->d_row2v = (int*)(slab + o_row);
  c->d_rp = (int*)(slab + o_rp);
  c->d_diag = (int*)(slab + o_diag);
  c->d_lumped = (double*)(slab + o_lump);
  int* keep = (int*)(slab + o_keep);  // keep flags and their scan, then the incidence cursors
  int* scan = (int*)(slab + o_scan);
  hipStream_t st = c->stream;
  CKH(hipMemcpyAsync(c->d_xyz, mesh->xyz, sizeof(float) * 3 * nv, hipMemcpyHostToDevice, st));
  CKH(hipMemcpyAsync(c->d_tri, mesh->triangles, sizeof(uint32_t) * 3 * nt, hipMemcpyHostToDevice, st));
  CKH(hipMemcpyAsync(c->d_onb, mesh->on_boundary, (size_t)nv, hipMemcpyHostToDevice, st));
  // idx_map: exclusive scan of the keep flags (FEMContext.cpp:224-240)
  if (nv > 0) {
    hipLaunchKernelGGL(k_keep, dim3(div_up(nv, kBlock)), dim3(kBlock), 0, st, c->d_onb, nv, bc, keep);
    CK(exclusive_scan_i32(keep, keep, nv, scan, st));
    hipLaunchKernelGGL(k_idx_map, dim3(div_up(nv, kBlock)), dim3(kBlock), 0, st, c->d_onb, nv, bc, keep,
                       c->d_idx, c->d_row2v);
  }
  // vertex -> incident triangles, ascending
  CKH(hipMemsetAsync(c->d_inc_ptr, 0, sizeof(int) * (nv + 1), st));
  if (nt > 0)
    hipLaunchKernelGGL(k_inc_count, dim3(div_up(nt, kBlock)), dim3(kBlock), 0, st, c->d_tri, nt, c->d_inc_ptr);
  CK(exclusive_scan_i32(c->d_inc_ptr, c->d_inc_ptr, nv + 1, scan, st));
  CKH(hipMemsetAsync(keep, 0, sizeof(int) * (nv + 1), st));
  if (nt > 0) {
    hipLaunchKernelGGL(k_inc_fill, dim3(div_up(nt, kBlock)), dim3(kBlock), 0, st, c->d_tri, nt, c->d_inc_ptr,
                       keep, c->d_inc);
  }
  if (nv > 0)
    hipLaunchKernelGGL(k_inc_sort, dim3(div_up(nv, kBlock)), dim3(kBlock), 0, st, c->d_inc_ptr, nv, c->d_inc);
  // CSR pattern: count, scan, fill
  if (n > 0) {
    hipLaunchKernelGGL(k_row_cols, dim3(div_up(n, kBlock)), dim3(kBlock), 0, st, c->d_tri, c->d_idx,
                       c->d_row2v, c->d_inc_ptr, c->d_inc, n, 0, c->d_rp, nullptr, nullptr, nullptr);
    CKH(hipMemsetAsync(c->d_rp + n, 0, sizeof(int), st));
    CKH(hipGetLastError());
    CK(exclusive_scan_i32(c->d_rp, c->d_rp, n + 1, scan, st));
  } else {
    CKH(hipMemsetAsync(c->d_rp, 0, sizeof(int), st));
  }
  // the host copy of row_ptr: the number of entries and the longest row
  // (FEMContext.cpp:207-219)
  c->h_rp.resize((size_t)n + 1);
  CKH(hipMemcpyAsync(c->h_rp.data(), c->d_rp, sizeof(int) * (n + 1), hipMemcpyDeviceToHost, st));
  CKH(hipStreamSynchronize(st));
  const int nnz = c->h_rp[n];
  c->nnz = nnz;
  c->max_row = 0;
  for (int r = 0; r < n; r++) c->max_row = std::max(c->max_row, c->h_rp[r + 1] - c->h_rp[r]);
  need = 0;
  const size_t o_ci = place(sizeof(int) * ((size_t)nnz + 1)), o_tp = place(sizeof(int) * ((size_t)nnz + 1));
  const size_t o_K = place(sizeof(double) * ((size_t)nnz + 1)), o_M = place(sizeof(double) * ((size_t)nnz + 1));
  const size_t o_A = place(sizeof(double) * ((size_t)nnz + 1));
  slab = c->d_slabs[1] = dalloc<char>(need, &rc);
  if (rc) { ctx_free(c); return rc; }
  c->d_ci = (int*)(slab + o_ci);
  c->d_tperm = (int*)(slab + o_tp);
  c->d_K = (double*)(slab + o_K);
  c->d_M = (double*)(slab + o_M);
  c->d_A = (double*)(slab + o_A);
  if (n > 0) {
    hipLaunchKernelGGL(k_row_cols, dim3(div_up(n, kBlock)), dim3(kBlock), 0, st, c->d_tri, c->d_idx,
                       c->d_row2v, c->d_inc_ptr, c->d_inc, n, 1, nullptr, c->d_rp, c->d_ci, c->d_diag);
    hipLaunchKernelGGL(k_tperm, dim3(div_up(n, kBlock)), dim3(kBlock), 0, st, c->d_rp, c->d_ci, n, c->d_tperm);
    CKH(hipGetLastError());
  }
  CK(ctx_assemble(c, nullptr));
#undef CK
#undef CKH
  *out = c;
  return 0;
}

}  // namespace femhip

namespace femhip {
namespace {

// smooth_normals.glsl:22-57 without atomics: each vertex sums, over its
// incident triangles in ascending order, the unnormalised normal of the
// triangle whose vertices are moved along their normals by
// min(1, extrusion * max(0, value)).  FP32 as the shader.
__global__ void k_smooth_normals(int nv, const float* xyz, const uint32_t* tri, const int* inc_ptr, const int* inc,
                                 const float* nrm, const float* val, float extrusion, float* out) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f;
  for (int e = inc_ptr[v]; e < inc_ptr[v + 1]; e++) {
    const uint32_t* t = tri + 3 * (size_t)inc[e];
    float p[3][3];
    for (int a = 0; a < 3; a++) {
      const size_t w = t[a];
      const float h = fminf(1.0f, extrusion * fmaxf(0.0f, val[w]));
      for (int q = 0; q < 3; q++) p[a][q] = xyz[3 * w + q] + h * nrm[3 * w + q];
    }
    const float e1[3] = {p[1][0] - p[0][0], p[1][1] - p[0][1], p[1][2] - p[0][2]};
    const float e2[3] = {p[2][0] - p[0][0], p[2][1] - p[0][1], p[2][2] - p[0][2]};
    s0 += e1[1] * e2[2] - e1[2] * e2[1];
    s1 += e1[2] * e2[0] - e1[0] * e2[2];
    s2 += e1[0] * e2[1] - e1[1] * e2[0];
  }
  out[3 * (size_t)v] = s0;
  out[3 * (size_t)v + 1] = s1;
  out[3 * (size_t)v + 2] = s2;
}

}  // namespace

// normals/out: device [nv][3]; values: device [nv].
int ctx_smooth_normals_device(fem_ctx* c, const float* d_nrm, const float* d_val, float extrusion, float* d_out,
                              hipStream_t st) {
  if (c->nv == 0) return 0;
  hipLaunchKernelGGL(k_smooth_normals, dim3(div_up(c->nv, kBlock)), dim3(kBlock), 0, st, c->nv, c->d_xyz, c->d_tri,
                     c->d_inc_ptr, c->d_inc, d_nrm, d_val, extrusion, d_out);
  FEM_HIP(hipGetLastError());
  return 0;
}

int ctx_smooth_normals(fem_ctx* c, const float* nrm, const float* val, float extrusion, float* out) {
  const size_t nv = (size_t)c->nv;
  if (nv == 0) return 0;
  int rc = 0;
  float* d = dalloc<float>(7 * nv, &rc);  // normals, values, output
  if (!d) return rc;
  float *dn = d, *dv = d + 3 * nv, *dout = d + 4 * nv;
  hipError_t e = hipMemcpyAsync(dn, nrm, sizeof(float) * 3 * nv, hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(dv, val, sizeof(float) * nv, hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) {
    rc = ctx_smooth_normals_device(c, dn, dv, extrusion, dout, c->stream);
    if (!rc) e = hipMemcpyAsync(out, dout, sizeof(float) * 3 * nv, hipMemcpyDeviceToHost, c->stream);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  (void)hipFree(d);
  if (e != hipSuccess) return hip_fail(e, "smooth_normals");
  return rc;
}

}  // namespace femhip
